// mg_strip.h -- red-black SOR (sors.f90:93-260) on register strips: FP32, the
// mixed form's correction equation in the fixed schedule of poisson.hip, and
// FP64, the reference's sweeps and residuals.
//
// A lane holds two neighbouring columns (i even, i + 1) of R rows (first row
// even), so every row of a colour pass updates the same one of the two nodes
// in all lanes and nothing diverges.  A node's horizontal neighbours are the
// lane's other node and one DPP move from the next lane, its vertical ones
// the lane's own rows; only a strip's first and last row need values of
// another strip, exchanged through LDS once per colour pass.  The products
// aw u and an u that the reference's expression takes of every neighbour are
// made once, when a node changes, and serve its four neighbours.  Against a
// region held in LDS (six LDS reads and the index arithmetic per node and
// pass) a node costs eleven FP32 operations, ten where aw = an, and a pass
// two LDS reads and two writes per strip.
//
// Every expression keeps the operations and the order of sor_update, getres,
// full_weight and prolong_node in poisson.hip, so a sweep gives the same bits
// whichever form runs it.
#pragma once

#include "lepic_internal.h"

namespace lepic_mg {

// value of the next lane to the west (east) of the wave; zero at its ends
__device__ __forceinline__ float from_west(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x138, 0xf, 0xf, true));   // wave_shr:1
}
__device__ __forceinline__ float from_east(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x130, 0xf, 0xf, true));   // wave_shl:1
}

__device__ __forceinline__ double from_west(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x138, 0xf, 0xf, true);
  return __hiloint2double(__builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x138, 0xf, 0xf, true), lo);
}
__device__ __forceinline__ double from_east(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x130, 0xf, 0xf, true);
  return __hiloint2double(__builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x130, 0xf, 0xf, true), lo);
}

// om1 = 1 - omega, rac = 1 / ac rounded, racl (FP64) what the rounding left
template <typename T> struct StripCoef;
template <> struct StripCoef<float> {
  float aw, an, ac, om, om1, rac;
};
template <> struct StripCoef<double> {
  double aw, an, ac, om, om1, rac, racl;
};

// The coefficients as values the compiler keeps in scalar registers: it would
// load them from the kernel's arguments again for every node of a pass.
template <typename T>
__device__ __forceinline__ StripCoef<T> strip_hold(StripCoef<T> k) {
  asm volatile("" : "+s"(k.aw), "+s"(k.an), "+s"(k.ac), "+s"(k.om), "+s"(k.om1), "+s"(k.rac));
  if constexpr (sizeof(T) == 8) asm volatile("" : "+s"(k.racl));
  return k;
}

// v where the mask's bits are set, u elsewhere: one bitfield insert, where a
// select on a condition becomes a branch around the node's whole update
__device__ __forceinline__ float strip_select(uint32_t m, float v, float u) {
  return __uint_as_float((m & __float_as_uint(v)) | (~m & __float_as_uint(u)));
}
__device__ __forceinline__ double strip_select(uint32_t m, double v, double u) {
  const uint32_t hi = (m & (uint32_t)__double2hiint(v)) | (~m & (uint32_t)__double2hiint(u));
  const uint32_t lo = (m & (uint32_t)__double2loint(v)) | (~m & (uint32_t)__double2loint(u));
  return __hiloint2double((int)hi, (int)lo);
}
__device__ __forceinline__ float strip_clear(uint32_t m, float v) { return __uint_as_float(m & __float_as_uint(v)); }
__device__ __forceinline__ double strip_clear(uint32_t m, double v) {
  return __hiloint2double((int)(m & (uint32_t)__double2hiint(v)), (int)(m & (uint32_t)__double2loint(v)));
}
__device__ __forceinline__ uint32_t strip_mask(bool b) { return b ? 0xFFFFFFFFu : 0u; }

// u: state, p = aw u, q = an u (ISO: aw = an and only p is used), b:
// right-hand side, m: all bits set where bcnd <= 0 (walls keep u, which is
// zero there).
template <typename T, int R, bool ISO>
struct Strip {
  T u[R][2], p[R][2], q[R][2], b[R][2];
  uint32_t m[R][2];
  __device__ __forceinline__ T north(int r, int P) const { return ISO ? p[r][P] : q[r][P]; }   // an u
  __device__ __forceinline__ void products(const StripCoef<T>& k, int r, int P) {
    p[r][P] = k.aw * u[r][P];
    if (!ISO) q[r][P] = k.an * u[r][P];
  }
};

// a pair of neighbouring nodes, aligned like one
template <typename T> struct __attribute__((packed, aligned(sizeof(T)))) P2 { T x, y; };
using F2 = P2<float>;
using D2 = P2<double>;
struct __attribute__((packed, aligned(1))) B2 { int8_t x, y; };

// sor_update of node (r, P) given an u of its northern and southern neighbours
template <int R, bool ISO, int P>
__device__ __forceinline__ void strip_update(Strip<float, R, ISO>& s, const StripCoef<float>& k, int r, float qn, float qs) {
  const float pw = P ? s.p[r][0] : from_west(s.p[r][1]), pe = P ? from_east(s.p[r][0]) : s.p[r][1];
  const float x = s.b[r][P] - pw - qn - qs - pe;
  const float v = k.om1 * s.u[r][P] + k.om * x * k.rac;
  s.u[r][P] = strip_select(s.m[r][P], v, s.u[r][P]);
  s.products(k, r, P);
}

// getres of node (r, P), zero on walls (the restriction counts bcnd <= 0 nodes only)
template <typename T, int R, bool ISO, int P>
__device__ __forceinline__ T strip_resid(const Strip<T, R, ISO>& s, const StripCoef<T>& k, int r, T qn, T qs) {
  const T pw = P ? s.p[r][0] : from_west(s.p[r][1]), pe = P ? from_east(s.p[r][0]) : s.p[r][1];
  const T v = s.b[r][P] - (pw + pe + qn + qs + k.ac * s.u[r][P]);
  return strip_clear(s.m[r][P], v);
}

// Edge rows in LDS (an u), for each colour (0 red, 1 black) the first and the
// last row of every strip: ed[(2 colour + last) * E + (strip + 1) * Lx + lane].
// o is the lane's own entry; the guard strips before the first and after the
// last are zero.
template <typename T>
struct Edges {
  T* ed;
  int E, Lx, o;
  bool write;                  // the lane belongs to a strip
};

// One colour pass: red (i + j odd) is the second node of even rows and the
// first of odd ones.
template <int R, bool ISO, bool RED>
__device__ __forceinline__ void strip_pass(Strip<float, R, ISO>& s, const StripCoef<float>& k, const Edges<float>& e) {
  constexpr int E0 = RED ? 1 : 0, O0 = 1 - E0;            // position in even and odd rows
  constexpr int other = RED ? 1 : 0, own = 1 - other;     // colours of the neighbours and of the pass
  const float above = e.ed[(2 * other) * e.E + e.o + e.Lx], below = e.ed[(2 * other + 1) * e.E + e.o - e.Lx];
#pragma unroll
  for (int r = 1; r + 1 < R; ++r) {
    if (r & 1) strip_update<R, ISO, O0>(s, k, r, s.north(r + 1, O0), s.north(r - 1, O0));
    else strip_update<R, ISO, E0>(s, k, r, s.north(r + 1, E0), s.north(r - 1, E0));
  }
  strip_update<R, ISO, E0>(s, k, 0, s.north(1, E0), below);
  strip_update<R, ISO, O0>(s, k, R - 1, above, s.north(R - 2, O0));
  if (e.write) {
    e.ed[(2 * own) * e.E + e.o] = s.north(0, E0);
    e.ed[(2 * own + 1) * e.E + e.o] = s.north(R - 1, O0);
  }
}

// Orders the strips' LDS traffic: a block barrier, or inside one wave, whose
// LDS operations complete in order, a fence for the compiler.
template <bool WAVE>
__device__ __forceinline__ void strip_sync() {
  if (WAVE) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  } else {
    __syncthreads();
  }
}

// nsw red-black sweeps; the black edges of the starting state are in LDS.  A
// pass writes only its own colour's edges and reads the other's, so one
// synchronisation per pass suffices.
template <int R, bool ISO, bool WAVE>
__device__ __forceinline__ void strip_sweeps(Strip<float, R, ISO>& s, const StripCoef<float>& k, int nsw, const Edges<float>& e) {
  for (int it = 0; it < nsw; ++it) {
    strip_pass<R, ISO, true>(s, k, e);
    strip_sync<WAVE>();
    strip_pass<R, ISO, false>(s, k, e);
    strip_sync<WAVE>();
  }
}

// the black edges of a starting state that is not zero
template <typename T, int R, bool ISO>
__device__ __forceinline__ void strip_publish_black(const Strip<T, R, ISO>& s, const Edges<T>& e) {
  if (e.write) {
    e.ed[2 * e.E + e.o] = s.north(0, 0);
    e.ed[3 * e.E + e.o] = s.north(R - 1, 1);
  }
}

// Full weighting (mg.f90:386-414) of the residuals at the coarse nodes of the
// strip, the second node of every odd row.  out[t]: coarse node of row 2t + 1.
// All edges are in LDS; contains two synchronisations.
template <typename T, int R, bool ISO, bool WAVE>
__device__ __forceinline__ void strip_restrict(const Strip<T, R, ISO>& s, const StripCoef<T>& k, const Edges<T>& e,
                                               T out[R / 2]) {
  T g[R + 1][2];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    T n0, n1, s0, s1;          // an u of the two nodes' northern and southern neighbours
    if (r + 1 < R) { n0 = s.north(r + 1 < R ? r + 1 : r, 0); n1 = s.north(r + 1 < R ? r + 1 : r, 1); }
    else { n0 = e.ed[2 * e.E + e.o + e.Lx]; n1 = e.ed[e.o + e.Lx]; }          // even row: black, red
    if (r > 0) { s0 = s.north(r > 0 ? r - 1 : r, 0); s1 = s.north(r > 0 ? r - 1 : r, 1); }
    else { s0 = e.ed[e.E + e.o - e.Lx]; s1 = e.ed[3 * e.E + e.o - e.Lx]; }     // odd row: red, black
    g[r][0] = strip_resid<T, R, ISO, 0>(s, k, r, n0, s0);
    g[r][1] = strip_resid<T, R, ISO, 1>(s, k, r, n1, s1);
  }
  strip_sync<WAVE>();          // every edge has been read
  if (e.write) {
    e.ed[e.o] = g[0][0];
    e.ed[2 * e.E + e.o] = g[0][1];
  }
  strip_sync<WAVE>();
  g[R][0] = e.ed[e.o + e.Lx];
  g[R][1] = e.ed[2 * e.E + e.o + e.Lx];
  T ge[R + 1];                 // the first node of the next lane
#pragma unroll
  for (int r = 0; r <= R; ++r) ge[r] = from_east(g[r][0]);
#pragma unroll
  for (int t = 0; t < R / 2; ++t) {
    const int c = 2 * t + 1;
    const T v = ((T)4 * g[c][1] + (T)2 * (ge[c] + g[c - 1][1] + g[c][0] + g[c + 1][1]) + ge[c + 1] + ge[c - 1] +
                 g[c - 1][0] + g[c + 1][0]) / (T)16;
    out[t] = strip_clear(s.m[c][1], v);
  }
}

// The bilinear correction (mg.f90:585-611) of the strip's nodes added to u on
// bcnd <= 0 nodes.  c[t]: coarse values (ci - 1, ci) of coarse row j0/2 + t,
// ci = i0/2 + 1, for the strip's first row j0 and first column i0.
template <typename T, int R, bool ISO>
__device__ __forceinline__ void strip_prolong(Strip<T, R, ISO>& s, const P2<T> c[R / 2 + 1]) {
#pragma unroll
  for (int t = 0; t < R / 2; ++t) {
    const P2<T> a = c[t], b = c[t + 1];
    const T v[2][2] = {{(b.y + a.y + a.x + b.x) / (T)4, (b.y + a.y) / (T)2}, {(b.y + b.x) / (T)2, b.y}};
#pragma unroll
    for (int d = 0; d < 2; ++d)
#pragma unroll
      for (int P = 0; P < 2; ++P)
        s.u[2 * t + d][P] = strip_select(s.m[2 * t + d][P], s.u[2 * t + d][P] + v[d][P], s.u[2 * t + d][P]);
  }
}

// ---- FP64: the reference's sweeps with the residual of every sweep ----

// x / ac, correctly rounded as the reference's division: the quotient from the
// reciprocal in two parts is within one unit in the last place, so the
// remainder is exact and one correction rounds it right (Markstein's theorem,
// IBM J. Res. Dev. 34, 1990); four operations where the general division
// takes a dozen.
__device__ __forceinline__ double strip_div(double x, const StripCoef<double>& k) {
  const double q = __builtin_fma(x, k.rac, x * k.racl);
  return __builtin_fma(__builtin_fma(-k.ac, q, x), k.rac, q);
}

// sors.f90:108-110 of node (r, P).  The residual (sors.f90:348-349 order) is
// taken where its neighbours are at hand: a black node's of this sweep right
// after its update, a red node's of the sweep before right before it.
// Returns |residual|, zero on walls.
template <int R, bool ISO, int P, bool RED, bool RES, bool UPD>
__device__ __forceinline__ double strip_node64(Strip<double, R, ISO>& s, const StripCoef<double>& k, int r, double qn,
                                               double qs) {
  const double pw = P ? s.p[r][0] : from_west(s.p[r][1]), pe = P ? from_east(s.p[r][0]) : s.p[r][1];
  const double u = s.u[r][P], b = s.b[r][P];
  double res = 0.0;
  if (RES && RED) res = b - (pw + qn + qs + pe + k.ac * u);
  if (UPD) {
    const double v = k.om1 * u + strip_div(k.om * (b - pw - qn - qs - pe), k);
    s.u[r][P] = strip_select(s.m[r][P], v, u);
    s.products(k, r, P);
  }
  if (RES && !RED) res = b - (pw + qn + qs + pe + k.ac * s.u[r][P]);
  return RES ? fabs(strip_clear(s.m[r][P], res)) : 0.0;
}

// One colour pass; UPD false: the residual of the red nodes alone.
template <int R, bool ISO, bool RED, bool RES, bool UPD>
__device__ __forceinline__ double strip_pass64(Strip<double, R, ISO>& s, const StripCoef<double>& k,
                                               const Edges<double>& e) {
  constexpr int E0 = RED ? 1 : 0, O0 = 1 - E0;            // position in even and odd rows
  constexpr int other = RED ? 1 : 0, own = 1 - other;     // colours of the neighbours and of the pass
  const double above = e.ed[(2 * other) * e.E + e.o + e.Lx], below = e.ed[(2 * other + 1) * e.E + e.o - e.Lx];
  double rr = 0.0;
#pragma unroll
  for (int r = 1; r + 1 < R; ++r) {
    if (r & 1) rr += strip_node64<R, ISO, O0, RED, RES, UPD>(s, k, r, s.north(r + 1, O0), s.north(r - 1, O0));
    else rr += strip_node64<R, ISO, E0, RED, RES, UPD>(s, k, r, s.north(r + 1, E0), s.north(r - 1, E0));
  }
  rr += strip_node64<R, ISO, E0, RED, RES, UPD>(s, k, 0, s.north(1, E0), below);
  rr += strip_node64<R, ISO, O0, RED, RES, UPD>(s, k, R - 1, above, s.north(R - 2, O0));
  if (UPD && e.write) {
    e.ed[(2 * own) * e.E + e.o] = s.north(0, E0);
    e.ed[(2 * own + 1) * e.E + e.o] = s.north(R - 1, O0);
  }
  return rr;
}

// A region's u, b and bc on the lane's strip: columns i0, i0 + 1, rows j0 .. +
// R - 1; all loads are issued before the first is used, from clamped
// positions.  uin null: zero.  The outer walls come from uw, the level's
// array 0: the other state buffers hold the nodes between them.
template <int R, bool ISO>
__device__ __forceinline__ void strip_region_load(Strip<double, R, ISO>& s, const double* uin, const double* uw,
                                                  const double* b, const int8_t* bc, int n1, int n2, int i0, int j0) {
  const int W = n1 + 3;
  const bool oki = i0 >= 0 && i0 <= n1 + 1, okb = i0 >= 2 && i0 <= n1;
  D2 lu[R], lb[R];
  B2 lc[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int j = j0 + r;
    const bool ok = oki && j >= 1 && j <= n2 + 1;
    const int64_t q = ok ? (int64_t)j * W + i0 : (int64_t)2 * W + 2;
    const int64_t qb = okb && j >= 2 && j <= n2 ? (int64_t)(j - 1) * (n1 + 1) + (i0 - 1) : (int64_t)(n1 + 2);
    lu[r] = D2{0.0, 0.0};
    if (uin) {
      const double* base = i0 == 0 || i0 == n1 + 1 || j == 1 || j == n2 + 1 ? uw : uin;
      lu[r] = *(const D2*)(base + q);
    }
    lb[r] = *(const D2*)(b + qb);
    lc[r] = *(const B2*)(bc + q);
    if (!ok) lc[r] = B2{1, 1};
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const bool ok = oki && j0 + r >= 1 && j0 + r <= n2 + 1;
    s.m[r][0] = strip_mask(lc[r].x <= 0);
    s.m[r][1] = strip_mask(lc[r].y <= 0);
    s.u[r][0] = ok ? lu[r].x : 0.0;
    s.u[r][1] = ok ? lu[r].y : 0.0;
    s.b[r][0] = lb[r].x;
    s.b[r][1] = lb[r].y;
  }
}

// ---------------------------------------------------------------------------
// one visit of a multi-block level
// ---------------------------------------------------------------------------
struct TileArgs {
  const float* u_in;           // state before the visit; null: zero (down visits)
  float* u_out;                // state after it; null when phi takes it
  const float* b;
  const int8_t* bc;
  int n1, n2;
  StripCoef<float> k;
  int nsw, halo;               // sweeps; halo nodes around a tile (even)
  const float* e2h;            // up visit: the coarse correction to prolong
  float* r2h;                  // last launch of a down visit: the coarse right-hand side
  double* phi;                 // finest up visit: phi += the correction
};

// A block's region is 128 columns x NW R rows: a tile and a halo of 2 nodes
// per sweep (validity shrinks by one node per colour pass; 2 more where the
// restriction reads the residual one node past the tile).  Tiles start at
// (2, 2): the outer walls are never updated.
template <int R, int NW, bool ISO>
__global__ __launch_bounds__(64 * NW) void k_tile32(TileArgs A) {
  constexpr int E = (NW + 2) * 64;
  __shared__ float ed[4 * E];
  for (int q = threadIdx.x; q < 4 * E; q += 64 * NW) ed[q] = 0.0f;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int n1 = A.n1, n2 = A.n2, W = n1 + 3;
  const int TX = 128 - 2 * A.halo, TY = NW * R - 2 * A.halo;
  const int i0 = 2 + (int)blockIdx.x * TX - A.halo + 2 * lane;
  const int j0 = 2 + (int)blockIdx.y * TY - A.halo + w * R;
  const bool oki = i0 >= 2 && i0 <= n1;
  const StripCoef<float> k = strip_hold(A.k);
  // what leaves the block: the tile's nodes
  const bool colo = oki && 2 * lane >= A.halo && 2 * lane < 128 - A.halo;
  const int lr0 = w * R;
  bool own[R];
#pragma unroll
  for (int r = 0; r < R; ++r)
    own[r] = colo && lr0 + r >= A.halo && lr0 + r < NW * R - A.halo && j0 + r <= n2;
  D2 ph[R];
  if (A.phi) {                 // loaded with the state, not after the sweeps
#pragma unroll
    for (int r = 0; r < R; ++r)
      ph[r] = *(const D2*)(A.phi + (own[r] ? (int64_t)(j0 + r) * W + i0 : (int64_t)2 * W + 2));
  }
  Strip<float, R, ISO> s;
  {
    F2 lu[R], lb[R];
    B2 lc[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int j = j0 + r;
      const bool ok = oki && j >= 2 && j <= n2;
      const int64_t q = ok ? (int64_t)j * W + i0 : (int64_t)2 * W + 2;
      const int64_t qb = ok ? (int64_t)(j - 1) * (n1 + 1) + (i0 - 1) : (int64_t)(n1 + 2);
      lu[r] = A.u_in ? *(const F2*)(A.u_in + q) : F2{0.0f, 0.0f};
      lb[r] = *(const F2*)(A.b + qb);
      lc[r] = *(const B2*)(A.bc + q);
      if (!ok) lc[r] = B2{1, 1};
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      s.m[r][0] = strip_mask(lc[r].x <= 0);
      s.m[r][1] = strip_mask(lc[r].y <= 0);
      s.u[r][0] = strip_select(s.m[r][0], lu[r].x, 0.0f);
      s.u[r][1] = strip_select(s.m[r][1], lu[r].y, 0.0f);
      s.b[r][0] = lb[r].x;
      s.b[r][1] = lb[r].y;
    }
  }
  if (A.e2h) {
    const int m1 = n1 / 2, m2 = n2 / 2, Wc = m1 + 3;
    const int ci = min(max(i0 / 2 + 1, 2), m1 + 1);
    F2 c[R / 2 + 1];
#pragma unroll
    for (int t = 0; t <= R / 2; ++t) {
      const int cj = min(max((j0 >> 1) + t, 1), m2 + 1);
      c[t] = *(const F2*)(A.e2h + (int64_t)cj * Wc + ci - 1);
    }
    strip_prolong<float, R, ISO>(s, c);
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    s.products(k, r, 0);
    s.products(k, r, 1);
  }
  Edges<float> e{ed, E, 64, (w + 1) * 64 + lane, true};
  __syncthreads();
  if (A.u_in) {
    strip_publish_black<float, R, ISO>(s, e);
    __syncthreads();
  }
  strip_sweeps<R, ISO, false>(s, k, A.nsw, e);
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if (!own[r]) continue;
    const int64_t q = (int64_t)(j0 + r) * W + i0;
    if (A.phi) {
      if (s.m[r][0]) A.phi[q] = ph[r].x + (double)s.u[r][0];
      if (s.m[r][1]) A.phi[q + 1] = ph[r].y + (double)s.u[r][1];
    } else {
      *(F2*)(A.u_out + q) = F2{s.u[r][0], s.u[r][1]};
    }
  }
  if (A.r2h) {                 // block-uniform
    float out[R / 2];
    strip_restrict<float, R, ISO, false>(s, k, e, out);
    const int m1 = n1 / 2;
#pragma unroll
    for (int t = 0; t < R / 2; ++t) {
      const int r = 2 * t + 1, j = j0 + r;
      if (!own[r] || i0 + 1 > n1) continue;
      A.r2h[(int64_t)((j + 1) / 2 - 1) * (m1 + 1) + i0 / 2] = out[t];
    }
  }
}

// ---------------------------------------------------------------------------
// a level of the single-workgroup kernel, arrays in LDS
// ---------------------------------------------------------------------------
template <typename T>
struct StripLevel {
  int n1, n2;
  int Lx, SW, nst;             // lanes per strip row ((n1 + 1) / 2), strips per wave, strips
  int inv;                     // 65536 / Lx + 1: lane / Lx = lane inv >> 16 for lane < 64, Lx <= 64
  StripCoef<T> k;
};

// the lane's strip of a level: wave w holds strips w SW .. w SW + SW - 1,
// each Lx lanes.  The last column pair of a strip holds a wall (value zero),
// so the DPP move from the neighbouring strip's lane brings a zero.
struct StripPos {
  int strip, lx, i0;
  bool act;
};

template <typename T>
__device__ __forceinline__ StripPos strip_pos(const StripLevel<T>& L, int w) {
  const int lane = threadIdx.x & 63;
  StripPos p;
  const int q = (lane * L.inv) >> 16;
  p.lx = lane - q * L.Lx;
  p.strip = w * L.SW + q;
  p.act = q < L.SW && p.strip < L.nst;
  p.i0 = 2 + 2 * p.lx;
  return p;
}

// All loads are issued before the first is used, from clamped positions.
template <typename T, int R, bool ISO>
__device__ __forceinline__ void strip_load(Strip<T, R, ISO>& s, const StripLevel<T>& L, const StripPos& p, const T* u,
                                           const T* b, const int8_t* bc) {
  const int W = L.n1 + 3;
  int8_t c[R][2];
  T lu[R][2];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int j = min(2 + p.strip * R + r, L.n2), i = min(p.i0, L.n1);
    const int q = p.act ? j * W + i : 2 * W + 2;
    const int qb = p.act ? (j - 1) * (L.n1 + 1) + i - 1 : L.n1 + 2;
    c[r][0] = bc[q];
    c[r][1] = bc[q + 1];
    s.b[r][0] = b[qb];
    s.b[r][1] = b[qb + 1];
    if (u) {
      lu[r][0] = u[q];
      lu[r][1] = u[q + 1];
    }
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const bool ok = p.act && 2 + p.strip * R + r <= L.n2 && p.i0 <= L.n1;
#pragma unroll
    for (int P = 0; P < 2; ++P) {
      s.m[r][P] = strip_mask(ok && c[r][P] <= 0);
      s.u[r][P] = u ? strip_clear(s.m[r][P], lu[r][P]) : (T)0;
    }
  }
}

// The lane's edges: zero guards below the first and above the last strip, and
// the starting state's black edges (north: their an u).
template <typename T, int R, bool ISO>
__device__ __forceinline__ void strip_edges(const Strip<T, R, ISO>& s, const StripLevel<T>& L, const StripPos& p,
                                            const Edges<T>& e) {
  if (!p.act) return;
  if (p.strip == 0) e.ed[e.E + p.lx] = e.ed[3 * e.E + p.lx] = (T)0;
  if (p.strip == L.nst - 1) e.ed[e.o + e.Lx] = e.ed[2 * e.E + e.o + e.Lx] = (T)0;
  strip_publish_black<T, R, ISO>(s, e);
}

// where the lane reads and writes its edges
template <typename T>
__device__ __forceinline__ Edges<T> strip_edge_pos(const StripLevel<T>& L, const StripPos& p, T* ed) {
  return Edges<T>{ed, (L.nst + 2) * L.Lx, L.Lx, p.act ? (p.strip + 1) * L.Lx + p.lx : L.Lx, p.act};
}

// the coarse correction u2 around the strip, prolonged onto it
template <typename T, int R, bool ISO>
__device__ __forceinline__ void strip_prolong_from(Strip<T, R, ISO>& s, const StripLevel<T>& L, const StripPos& p,
                                                   const T* u2) {
  const int m1 = L.n1 / 2, m2 = L.n2 / 2;
  P2<T> c[R / 2 + 1];
#pragma unroll
  for (int t = 0; t <= R / 2; ++t) {
    const int cj = min((p.act ? p.strip : 0) * (R / 2) + 1 + t, m2 + 1);
    const int q = cj * (m1 + 3) + min(p.i0 / 2, m1);
    c[t] = P2<T>{u2[q], u2[q + 1]};
  }
  strip_prolong<T, R, ISO>(s, c);
}

// Down visit: nsw sweeps from zero, the state to u, the restricted residual
// to the coarse right-hand side b2.
template <int R, bool ISO, bool WAVE>
__device__ __forceinline__ void strip_down(const StripLevel<float>& L, const StripCoef<float>& kl, int nsw, float* ed, float* u,
                                           const float* b, const int8_t* bc, float* b2) {
  const StripCoef<float> k = strip_hold(kl);
  const StripPos p = strip_pos(L, WAVE ? 0 : (int)(threadIdx.x >> 6));
  const Edges<float> e = strip_edge_pos(L, p, ed);
  Strip<float, R, ISO> s;
  strip_load<float, R, ISO>(s, L, p, nullptr, b, bc);
#pragma unroll
  for (int r = 0; r < R; ++r) s.p[r][0] = s.p[r][1] = s.q[r][0] = s.q[r][1] = 0.0f;
  strip_edges<float, R, ISO>(s, L, p, e);
  strip_sync<WAVE>();
  strip_sweeps<R, ISO, WAVE>(s, k, nsw, e);
  const int W = L.n1 + 3, m1 = L.n1 / 2, j0 = 2 + p.strip * R;
  if (p.act && p.i0 <= L.n1) {
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (j0 + r <= L.n2) {
        u[(j0 + r) * W + p.i0] = s.u[r][0];
        u[(j0 + r) * W + p.i0 + 1] = s.u[r][1];
      }
  }
  float out[R / 2];
  strip_restrict<float, R, ISO, WAVE>(s, k, e, out);
  if (p.act && p.i0 + 1 <= L.n1) {
#pragma unroll
    for (int t = 0; t < R / 2; ++t)
      if (j0 + 2 * t + 1 <= L.n2) b2[(j0 / 2 + t) * (m1 + 1) + p.i0 / 2] = out[t];
  }
  strip_sync<WAVE>();
}

// Up visit: the coarse correction u2 prolonged onto u, nsw sweeps, the state
// to u, to the global array gu, or added to phi.
template <int R, bool ISO, bool WAVE>
__device__ __forceinline__ void strip_up(const StripLevel<float>& L, const StripCoef<float>& kl, int nsw, float* ed, float* u,
                                         const float* b, const int8_t* bc, const float* u2, float* gu, double* phi) {
  const StripCoef<float> k = strip_hold(kl);
  const StripPos p = strip_pos(L, WAVE ? 0 : (int)(threadIdx.x >> 6));
  const Edges<float> e = strip_edge_pos(L, p, ed);
  Strip<float, R, ISO> s;
  strip_load<float, R, ISO>(s, L, p, u, b, bc);
  const int W = L.n1 + 3, j0 = 2 + p.strip * R;
  strip_prolong_from<float, R, ISO>(s, L, p, u2);
#pragma unroll
  for (int r = 0; r < R; ++r) {
    s.products(k, r, 0);
    s.products(k, r, 1);
  }
  strip_edges<float, R, ISO>(s, L, p, e);
  strip_sync<WAVE>();
  strip_sweeps<R, ISO, WAVE>(s, k, nsw, e);
  if (p.act && p.i0 <= L.n1) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (j0 + r > L.n2) continue;
      const int q = (j0 + r) * W + p.i0;
      if (phi) {
        if (s.m[r][0]) phi[q] = phi[q] + (double)s.u[r][0];
        if (s.m[r][1]) phi[q + 1] = phi[q + 1] + (double)s.u[r][1];
      } else if (gu) {
        gu[q] = s.u[r][0];
        gu[q + 1] = s.u[r][1];
      } else {
        u[q] = s.u[r][0];
        u[q + 1] = s.u[r][1];
      }
    }
  }
  strip_sync<WAVE>();
}

// ---- FP64 visits ----

// sum over the participants, the same value in every participant; ws holds
// two banks of 16 wave sums used alternately (par), so a bank is rewritten
// only after the barriers of a whole sweep
template <bool WAVE>
__device__ __forceinline__ double strip_sum(double v, double* ws, int par) {
  v = lepic::wave_sum(v);
  if (WAVE) return v;
  const int w = threadIdx.x >> 6, nw = blockDim.x >> 6;
  double* bank = ws + 16 * par;
  if ((threadIdx.x & 63) == 0) bank[w] = v;
  __syncthreads();
  double t = 0.0;
  for (int q = 0; q < nw; ++q) t += bank[q];
  return t;
}

// What a visit needs of the exit test (sors.f90:371-377), and its outcome.
struct VisitTest {
  int dig, nr;
  double eps;
  double* ws;                  // strip_sum's banks
  int ks;
  double res;
};

// Sweeps until the exit test ends the visit; the black edges of the starting
// state are in LDS.  The red nodes' residual after sweep k comes with the red
// pass of sweep k + 1, whose result is dropped when the test ends the visit;
// all edges are then in LDS again.  Ends with a synchronisation.
template <int R, bool ISO, bool WAVE>
__device__ __forceinline__ void strip_sweeps64(Strip<double, R, ISO>& s, const StripCoef<double>& k, VisitTest& v,
                                               const Edges<double>& e) {
  double red[R], prev = 0.0;
  strip_pass64<R, ISO, true, false, true>(s, k, e);
  for (v.ks = 1;; ++v.ks) {
    strip_sync<WAVE>();
    const double rb = strip_pass64<R, ISO, false, true, true>(s, k, e);
    strip_sync<WAVE>();
#pragma unroll
    for (int r = 0; r < R; ++r) red[r] = s.u[r][1 - (r & 1)];
    const double rr = strip_pass64<R, ISO, true, true, true>(s, k, e);
    v.res = strip_sum<WAVE>(rr + rb, v.ws, v.ks & 1);
    const bool stop = v.dig == 0 ? v.res <= v.eps : prev > 0.0 && v.res / prev <= 0.6;
    if (stop || v.ks >= v.nr) break;
    prev = v.res;
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    s.u[r][1 - (r & 1)] = red[r];
    s.products(k, r, 1 - (r & 1));
  }
  if (e.write) {
    e.ed[e.o] = s.north(0, 1);
    e.ed[e.E + e.o] = s.north(R - 1, 0);
  }
  strip_sync<WAVE>();
}

// strip_down under the exit test
template <int R, bool ISO, bool WAVE>
__device__ __forceinline__ void strip_down64(const StripLevel<double>& L, VisitTest& v, double* ed, double* u,
                                             const double* b, const int8_t* bc, double* b2) {
  const StripCoef<double> k = strip_hold(L.k);
  const StripPos p = strip_pos(L, WAVE ? 0 : (int)(threadIdx.x >> 6));
  const Edges<double> e = strip_edge_pos(L, p, ed);
  Strip<double, R, ISO> s;
  strip_load<double, R, ISO>(s, L, p, nullptr, b, bc);
#pragma unroll
  for (int r = 0; r < R; ++r) s.p[r][0] = s.p[r][1] = s.q[r][0] = s.q[r][1] = 0.0;
  strip_edges<double, R, ISO>(s, L, p, e);
  strip_sync<WAVE>();
  strip_sweeps64<R, ISO, WAVE>(s, k, v, e);
  const int W = L.n1 + 3, m1 = L.n1 / 2, j0 = 2 + p.strip * R;
  if (p.act && p.i0 <= L.n1) {
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (j0 + r <= L.n2) {
        u[(j0 + r) * W + p.i0] = s.u[r][0];
        u[(j0 + r) * W + p.i0 + 1] = s.u[r][1];
      }
  }
  double out[R / 2];
  strip_restrict<double, R, ISO, WAVE>(s, k, e, out);
  if (p.act && p.i0 + 1 <= L.n1) {
#pragma unroll
    for (int t = 0; t < R / 2; ++t)
      if (j0 + 2 * t + 1 <= L.n2) b2[(j0 / 2 + t) * (m1 + 1) + p.i0 / 2] = out[t];
  }
  strip_sync<WAVE>();
}

// strip_up under the exit test; the state goes to u, or to gu where not null
template <int R, bool ISO, bool WAVE>
__device__ __forceinline__ void strip_up64(const StripLevel<double>& L, VisitTest& v, double* ed, double* u,
                                           const double* b, const int8_t* bc, const double* u2, double* gu) {
  const StripCoef<double> k = strip_hold(L.k);
  const StripPos p = strip_pos(L, WAVE ? 0 : (int)(threadIdx.x >> 6));
  const Edges<double> e = strip_edge_pos(L, p, ed);
  Strip<double, R, ISO> s;
  strip_load<double, R, ISO>(s, L, p, u, b, bc);
  strip_prolong_from<double, R, ISO>(s, L, p, u2);
#pragma unroll
  for (int r = 0; r < R; ++r) {
    s.products(k, r, 0);
    s.products(k, r, 1);
  }
  strip_edges<double, R, ISO>(s, L, p, e);
  strip_sync<WAVE>();
  strip_sweeps64<R, ISO, WAVE>(s, k, v, e);
  const int W = L.n1 + 3, j0 = 2 + p.strip * R;
  if (p.act && p.i0 <= L.n1) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (j0 + r > L.n2) continue;
      const int q = (j0 + r) * W + p.i0;
      if (gu) {
        gu[q] = s.u[r][0];
        gu[q + 1] = s.u[r][1];
      } else {
        u[q] = s.u[r][0];
        u[q + 1] = s.u[r][1];
      }
    }
  }
  strip_sync<WAVE>();
}

}  // namespace lepic_mg
