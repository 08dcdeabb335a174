// poisson.hip -- iterative_solver (iterative_solver.f90:1-69), the MG
// V-cycle (mg.f90:1-232) and red-black SOR with adaptive sweep control
// (sors.f90:1-435).
//
// A kernel launch costs about 3 us on MI355X whatever it does, and a grid-wide
// software barrier costs more, so the solver is organised to launch few
// kernels and to need no grid synchronisation:
//  * FP64 fine ("multi-block") levels run k_visit64: each block holds a tile
//    and a halo of 2S+1 nodes on register strips (mg_strip.h) and performs S
//    red-black sweeps on it, recomputing the halo redundantly instead of
//    exchanging it.  After every sweep it writes the tile to that sweep's
//    state buffer (kRot = 9 rotating buffers per level, for a continuation's
//    up to 8 sweeps) and its share of the L1 residual.  The exit test of
//    sors.f90:371-377 for those sweeps is taken at the start of the next
//    launch (or by the kernel that consumes the level), by every block from
//    the same partial sums in the same order, so all blocks agree and no
//    atomics or host round trips are needed.  A visit
//    takes two launches, of which the second mostly finds it finished.  An up
//    visit prolongs the coarse correction while it loads; the restriction
//    needs the visit's outcome and is a kernel of its own (k_restrict64).
//    Between the V-cycles the finest state stays in its buffer; the solve's
//    end moves it to phi.
//  * Coarse levels (at most mg_tail_nodes nodes) run in one workgroup that
//    performs the whole lower part of the V-cycle (down sweeps, restrictions,
//    the coarsest solve, prolongations and up sweeps), with the levels that
//    fit in its LDS (up to 158 KB) held there: k_tail_strips, or k_tail where a
//    level is too wide for strips or is the finest one in FP64.
//  * Mixed mode runs each visit of a multi-block level in one launch of
//    k_tile32 (mg_strip.h): the sweeps of a fixed count on register strips,
//    with the prolongation on load, the restriction after the last sweep, and
//    on the finest level the correction added to phi.  The sweep counts and
//    so every buffer are known at launch, nothing is read back but the
//    V-cycle's FP64 residual.
// FP64 mode computes the reference's expressions in their order (no
// contraction), so a sweep is bit-identical to sors.f90; only the order of
// the L1 residual sum differs.  Mixed mode runs the same V-cycle in FP32 on
// the correction equation inside an FP64 iterative-refinement loop whose
// FP64 residual keeps the reference's convergence definition.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <type_traits>
#include <vector>

#include "lepic_internal.h"
#include "mg_strip.h"

using namespace lepic;
using namespace lepic_mg;

namespace {

constexpr int kVisitLog = 2 * kMaxLevels;     // ig = 1 .. 2ng-1
constexpr size_t kTailLds = 160 * 1024 - 2048;  // dynamic LDS of k_tail (static arrays take < 2 KB)
constexpr int kTailThreads = 1024;
constexpr int kS = kSweepsPerLaunch;          // most sweeps of one launch (kRot - 1 state buffers ahead)
constexpr int kDefaultTailNodes = 5000;
constexpr int kResidBlocks = 2048;            // most blocks of the FP64 finest-level residual
// byte offset of the residual partials behind the scalars and the visit log
constexpr size_t kPartialsOff = (64 * 8 + kVisitLog * sizeof(int) + 7) / 8 * 8;
constexpr size_t kScalarBytes = kPartialsOff + kResidBlocks * 8;
constexpr int kNr = 10;                       // sweep limit of sors.f90:63-64
// Mixed form: the FP32 correction V-cycle is a preconditioner inside FP64
// refinement to the unchanged tolerance, so its schedule is chosen, not
// taken from the reference's exit test (sors.f90:371-377).  The finest level
// (when multi-block) runs a fixed 4 down / 3 up red-black sweeps at omega
// 1.15: the reference's omega 1.4 (iterative_solver.f90:27) damps the
// highest frequencies less, and its exit test stops these visits after 2
// sweeps on plasma solves and runs them to 10 near electrodes.  The other
// multi-block levels and the tail levels above the coarsest run the 10 down
// / 2 up sweeps the test gives them on plasma solves, without the per-sweep
// residuals and sums the test needs; the coarsest level keeps the test.
// Measured: 1024^2 argon box 4 -> 3 V-cycles per solve.
constexpr int kFineDn = 4, kFineUp = 3;
constexpr float kFineOmega = 1.15f;
constexpr int kFixDn = kNr, kFixUp = 2;
constexpr int kWaveNodes = 320;               // tail levels with at most this many interior nodes run in one wave

// mixed form: a visit's sweeps run in one launch of k_tile32 unless its tiles,
// small behind a deep halo (84 x 20 nodes for 10 sweeps and the restriction),
// then need more than two blocks per CU; two launches of 5 sweeps cost one
// more load and launch (about 5 us) but sweep 1.8 instead of 4.9 times the
// tiles' nodes
constexpr int kTileMaxBlocks = 512, kTileSplit = 5;

// ---- SOR update of one node (sors.f90:108-110 / 238-240) ----
// FP64 divides like the reference; the FP32 smoother of the mixed form
// multiplies by the reciprocal (the FP64 refinement sets the final accuracy)
template <typename T>
__device__ __forceinline__ T sor_update(T u, T b, T uW, T uN, T uS, T uE, T aw, T an, T ac, T omega) {
  if constexpr (sizeof(T) == 4)
    return (1.0f - omega) * u + omega * (b - aw * uW - an * uN - an * uS - aw * uE) * (1.0f / ac);
  else
    return ((T)1.0 - omega) * u + omega * (b - aw * uW - an * uN - an * uS - aw * uE) / ac;
}

// ---- residual of one node, sors.f90:348-349 order ----
template <typename T>
__device__ __forceinline__ double sor_resid(T u, T b, T uW, T uN, T uS, T uE, T aw, T an, T ac) {
  return (double)(b - (aw * uW + an * uN + an * uS + aw * uE + ac * u));
}

// ---- getres, mg.f90:512-547 order (aw, ae, an, as, ac) ----
template <typename T, typename PU, typename PB>
__device__ __forceinline__ T getres(PU u, PB b, int ir, int jr, int n1, T aw, T an, T ac) {
  const int64_t W = n1 + 3;
  const int64_t c = (int64_t)jr * W + ir;
  T uij = u[c], un = u[c + W], us = u[c - W], ue = u[c + 1], uw = u[c - 1];
  T urhs = b[(int64_t)(jr - 1) * (n1 + 1) + (ir - 1)];
  return urhs - (aw * uw + aw * ue + an * un + an * us + ac * uij);
}

// mg.f90:386-414: the weighted sum of the centre residual g9 and the eight
// around it (g1 north-east, then clockwise), each counted when its flag holds
template <typename T>
__device__ __forceinline__ T full_weight(T g9, T g1, T g2, T g3, T g4, T g5, T g6, T g7, T g8, bool f1, bool f2,
                                         bool f3, bool f4, bool f5, bool f6, bool f7, bool f8) {
  const T r9 = g9;
  const T r1 = f1 ? g1 : (T)0, r2 = f2 ? g2 : (T)0, r3 = f3 ? g3 : (T)0, r4 = f4 ? g4 : (T)0;
  const T r5 = f5 ? g5 : (T)0, r6 = f6 ? g6 : (T)0, r7 = f7 ? g7 : (T)0, r8 = f8 ? g8 : (T)0;
  return ((T)4.0 * r9 + (T)2.0 * (r2 + r4 + r6 + r8) + r1 + r3 + r5 + r7) / (T)16.0;
}

// full-weighted residual of coarse node (i,j), mg.f90:386-414.  The nine
// fine residuals are evaluated unconditionally (at a position clamped into
// the interior when the reference skips one), so all loads issue at once;
// the reference's conditions select which of them count.
template <typename T, typename PU, typename PB, typename PC>
__device__ __forceinline__ T restrict_node(PU u, PB b, PC bc, int i, int j, int n1, int n2, T aw, T an, T ac) {
  const int ir = 2 * i - 1, jr = 2 * j - 1;
  const int64_t W = n1 + 3;
  auto B = [&](int a, int c) { return bc[(int64_t)c * W + a]; };
  auto G = [&](int a, int c) {
    a = a < 1 ? 1 : (a > n1 + 1 ? n1 + 1 : a);
    c = c < 1 ? 1 : (c > n2 + 1 ? n2 + 1 : c);
    return getres(u, b, a, c, n1, aw, an, ac);
  };
  const bool xe = ir != n1 + 1, xw = ir != 1, yn = jr != n2 + 1, ys = jr != 1;
  const bool f1 = xe && yn && B(ir + 1, jr + 1) <= 0;
  const bool f2 = xe && B(ir + 1, jr) <= 0;
  const bool f3 = B(ir + 1, jr - 1) <= 0 && xe && ys;
  const bool f4 = B(ir, jr - 1) <= 0 && ys;
  const bool f5 = B(ir - 1, jr - 1) <= 0 && xw && ys;
  const bool f6 = B(ir - 1, jr) <= 0 && xw;
  const bool f7 = B(ir - 1, jr + 1) <= 0 && xw && yn;
  const bool f8 = B(ir, jr + 1) <= 0 && yn;
  const T g9 = G(ir, jr), g1 = G(ir + 1, jr + 1), g2 = G(ir + 1, jr), g3 = G(ir + 1, jr - 1);
  const T g4 = G(ir, jr - 1), g5 = G(ir - 1, jr - 1), g6 = G(ir - 1, jr), g7 = G(ir - 1, jr + 1);
  const T g8 = G(ir, jr + 1);
  return full_weight<T>(g9, g1, g2, g3, g4, g5, g6, g7, g8, f1, f2, f3, f4, f5, f6, f7, f8);
}

// bilinear add of coarse node (i,j)'s correction to its four fine nodes,
// mg.f90:585-611
template <typename T, typename PU, typename PC, typename PE>
__device__ __forceinline__ void prolong_node(PU u, PC bc, int n1, PE e2h, int m1, int i, int j) {
  const int64_t Wc = m1 + 3, W = n1 + 3;
  T r1 = e2h[(int64_t)j * Wc + i], r2 = e2h[(int64_t)(j - 1) * Wc + i];
  T r3 = e2h[(int64_t)(j - 1) * Wc + i - 1], r4 = e2h[(int64_t)j * Wc + i - 1];
  const int ir = 2 * i - 1, jr = 2 * j - 1;
  const int64_t c = (int64_t)jr * W + ir;
  if (bc[c] <= 0) u[c] = u[c] + r1;
  if (bc[c - W] <= 0) u[c - W] = u[c - W] + (r1 + r2) / (T)2.0;
  if (bc[c - W - 1] <= 0) u[c - W - 1] = u[c - W - 1] + (r1 + r2 + r3 + r4) / (T)4.0;
  if (bc[c - 1] <= 0) u[c - 1] = u[c - 1] + (r1 + r4) / (T)2.0;
}

// ---------------------------------------------------------------------------
// visit control of multi-block levels (FP64)
// ---------------------------------------------------------------------------
// What the exit test of a launch reads: the partial sums of the launch's
// sweeps by nb1 blocks, of the sweep before them by nb0.
struct StopTest {
  const double* partials;
  int stride, nb0, nb1;
  int dig, nr;
  double eps;
};

// sors.f90:371-377 for sweeps kf .. kt (of one launch): the first sweep after
// which the reference stops (0 if none), from the blocks' partial sums of the
// L1 residual in a fixed order (lane strides, then a tree); the sweep before
// the visit's first counts as zero.  Called by every thread of a block, which
// all get the same answer; a wave sums one sweep at a time.  s_res: kS + 1
// doubles.
__device__ int first_stop(const StopTest& T, int kf, int kt, double* s_res, double* r_out) {
  const int lane = threadIdx.x & 63, nw = blockDim.x >> 6;
  for (int m = threadIdx.x >> 6; m <= kt - kf + 1; m += nw) {
    const int k = kf - 1 + m;
    double s = 0.0;
    if (k >= 1) {
      const double* p = T.partials + (size_t)(k % kRing) * T.stride;
      const int nb = m == 0 ? T.nb0 : T.nb1;
      for (int q = lane; q < nb; q += 64) s += p[q];
      s = wave_sum(s);
    }
    if (lane == 0) s_res[m] = s;
  }
  __syncthreads();
  double prev = s_res[0];
  for (int k = kf; k <= kt; ++k) {
    const double rk = s_res[k - kf + 1];
    bool stop = (T.dig == 0) ? (rk <= T.eps) : (prev > 0.0 && rk / prev <= 0.6);
    if (k >= T.nr) stop = true;
    if (stop) {
      *r_out = rk;
      return k;
    }
    prev = rk;
  }
  return 0;
}

struct VisitRef {
  LevelCtrl* ctrl;
  StopTest t;              // of the visit's last launch
  int epoch, ig;
  int nexec;               // sweeps launched in the visit
  int klast0;              // sweeps before the visit's last launch
  int* visit;
  double* vres;
};

struct Resolved {
  int ks;                  // sweeps of the visit (0: not finished)
  int buf;                 // rotating buffer holding the state after them
  double res;
};

// Outcome of a visit after all its launches; every block of the consuming
// kernel evaluates it (all threads) and one records it.
__device__ Resolved resolve_visit(const VisitRef& V, bool writer, double* s_res) {
  LevelCtrl* c = V.ctrl;
  const int c0 = c->cur[(V.epoch - 1) & 1];
  Resolved out{0, 0, 0.0};
  if (c->done_epoch == V.epoch) {
    out.ks = c->ksor;
    out.res = c->res;
  } else {
    out.ks = first_stop(V.t, V.klast0 + 1, V.nexec, s_res, &out.res);
  }
  if (out.ks) out.buf = (c0 + out.ks) % kRot;
  if (writer && out.ks && threadIdx.x == 0) {
    c->cur[V.epoch & 1] = out.buf;
    V.visit[V.ig] = out.ks;
    V.vres[V.ig] = out.res;
  }
  return out;
}

// ---------------------------------------------------------------------------
// multi-block levels (FP64)
// ---------------------------------------------------------------------------
constexpr int kVR = 4;                        // rows of a strip
constexpr int kVisitMaxWaves = 16;

struct VisitArgs {
  double* rot[kRot];
  const double* b;
  const int8_t* bc;
  int n1, n2;
  StripCoef<double> k;
  LevelCtrl* ctrl;
  double* partials;
  StopTest t;              // of the visit's previous launch
  int epoch;
  int k0, kexec, kchk;     // sweeps k0+1 .. k0+kexec; the previous launch's kchk .. k0 (kchk 0: no test)
  int halo_x, halo_y;      // region around a tile; halo_y a multiple of kVR
  int zero;                // the visit starts from zero
  const double* crot[kRot];   // up visit's first launch: the coarse correction (null: none), from the buffer
  int coarse_mb;              // that the coarse level's visit ends in, or from buffer 0
  VisitRef vc;
};

// Sweeps of a visit on one tile (see the file comment).  Bound by VALU issue:
// an update costs 19 FP64 operations where aw = an (four of them the
// division), its residual 8 more, against six LDS reads, the index arithmetic
// and a division of a dozen operations per node and pass on a region in LDS,
// the residual in a third pass.  1025 x 513 nodes, 5 sweeps: 34-39 us so
// before, 16 now; 257 x 129: 14, now 9; a launch that finds the visit finished
// takes 4.5 us either way.  The region of 128
// columns x kVR rows per wave is the tile and a halo of 2 kexec + 1 nodes at
// least (validity shrinks by one node per colour pass, and the residual reads
// one more).  Tiles start at (2, 2).  A wave takes part only in the sweeps
// whose outcome still reaches the tile, and only waves of tile rows (halo_y is
// a multiple of a strip's rows) evaluate residuals and write states.
template <bool ISO>
__global__ __launch_bounds__(64 * kVisitMaxWaves) void k_visit64(VisitArgs A) {
  __shared__ double ed[4 * (kVisitMaxWaves + 2) * 64];
  __shared__ double ws[kS][kVisitMaxWaves];
  __shared__ double s_res[2][kS + 1];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
  const int E = (nw + 2) * 64;
  const int n1 = A.n1, n2 = A.n2;
  const int TX = 128 - 2 * A.halo_x, TY = nw * kVR - 2 * A.halo_y;
  const int i0 = 2 + (int)blockIdx.x * TX - A.halo_x + 2 * lane;
  const int j0 = 2 + (int)blockIdx.y * TY - A.halo_y + w * kVR;
  const int bid = blockIdx.y * gridDim.x + blockIdx.x;
  LevelCtrl* c = A.ctrl;
  const int c0 = c->cur[(A.epoch - 1) & 1];
  Strip<double, kVR, ISO> s;
  strip_region_load<kVR, ISO>(s, A.zero ? nullptr : A.rot[(c0 + A.k0) % kRot], A.rot[0], A.b, A.bc, n1, n2, i0, j0);
  if (A.kchk > 0) {
    // Another block may record the stop while this one looks, so every wave
    // takes part in the test; a stop recorded by an earlier launch counts
    // whatever the test says of sweeps that were not run.
    const int done = __hip_atomic_load(&c->done_epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    double r = 0.0;
    const int ks = first_stop(A.t, A.kchk, A.k0, s_res[0], &r);
    if (done == A.epoch) return;
    if (ks) {
      if (bid == 0 && threadIdx.x == 0) {
        c->ksor = ks;
        c->res = r;
        __hip_atomic_store(&c->done_epoch, A.epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      return;
    }
  }
  if (A.crot[0]) {
    int cb = 0;
    if (A.coarse_mb) cb = resolve_visit(A.vc, bid == 0, s_res[1]).buf;
    const double* e2h = A.crot[cb];
    const int m1 = n1 / 2, m2 = n2 / 2, Wc = m1 + 3;
    const int ci = min(max(i0 / 2 + 1, 2), m1 + 1);
    D2 e[kVR / 2 + 1];
#pragma unroll
    for (int t = 0; t <= kVR / 2; ++t) {
      const int cj = min(max((j0 >> 1) + t, 1), m2 + 1);
      e[t] = *(const D2*)(e2h + (int64_t)cj * Wc + ci - 1);
    }
    strip_prolong<double, kVR, ISO>(s, e);
  }
  const StripCoef<double> k = strip_hold(A.k);
#pragma unroll
  for (int r = 0; r < kVR; ++r) {
    s.products(k, r, 0);
    s.products(k, r, 1);
  }
  Edges<double> e{ed, E, 64, (w + 1) * 64 + lane, true};
  if (w == 0) ed[E + lane] = ed[3 * E + lane] = 0.0;
  if (w == nw - 1) ed[e.o + 64] = ed[2 * E + e.o + 64] = 0.0;
  strip_publish_black<double, kVR, ISO>(s, e);
  __syncthreads();
  const int P = 2 * A.kexec, dist = min(kVR * w + kVR - 1, kVR * (nw - w) - 1);
  const int last = (dist + 2 + P - A.halo_y) / 2;            // the wave's last sweep
  const bool own = kVR * w >= A.halo_y && kVR * (w + 1) <= kVR * nw - A.halo_y;
  const bool colo = 2 * lane >= A.halo_x && 2 * lane < 128 - A.halo_x && i0 <= n1;
  const int W = n1 + 3;
  auto log = [&](int it, double rr) {                        // the wave's share of sweep it's residual
    const double t = wave_sum(colo ? rr : 0.0);
    if (lane == 0) ws[it - 1][w] = t;
  };
  double rb = 0.0;
  for (int it = 1; it <= A.kexec; ++it) {
    if (it <= last) {
      if (own && it > 1) log(it - 1, rb + strip_pass64<kVR, ISO, true, true, true>(s, k, e));
      else strip_pass64<kVR, ISO, true, false, true>(s, k, e);
    }
    __syncthreads();
    if (it <= last) {
      if (own) {
        rb = strip_pass64<kVR, ISO, false, true, true>(s, k, e);
        double* uout = A.rot[(c0 + A.k0 + it) % kRot];
        if (colo) {
#pragma unroll
          for (int r = 0; r < kVR; ++r)
            if (j0 + r <= n2) *(D2*)(uout + (int64_t)(j0 + r) * W + i0) = D2{s.u[r][0], s.u[r][1]};
        }
      } else {
        strip_pass64<kVR, ISO, false, false, true>(s, k, e);
      }
    }
    __syncthreads();
  }
  if (own) log(A.kexec, rb + strip_pass64<kVR, ISO, true, true, false>(s, k, e));
  __syncthreads();
  const int w0 = A.halo_y / kVR, nown = nw - 2 * w0;
  for (int it = 1 + w; it <= A.kexec; it += nw) {
    const double t = wave_sum(lane < nown ? ws[it - 1][w0 + lane] : 0.0);
    if (lane == 0) A.partials[(size_t)((A.k0 + it) % kRing) * A.t.stride + bid] = t;
  }
}

// restriction, mg.f90:335-444, from a multi-block level: resolves the fine
// level's down visit and writes the coarse right-hand side
struct RestrictArgs {
  VisitRef vf;
  const double* frot[kRot];
  const double* fb;
  const int8_t* fbc;
  int n1, n2;
  StripCoef<double> k;
  double* r2h;
};

// A block's region is 128 x 32 nodes with 2 around the tile; bound by latency
// (the visit's outcome, then the loads): 1025 x 513 nodes 20 us with every
// residual's neighbours read from memory, 7.8 so.
constexpr int kRestrictWaves = 8;
template <bool ISO>
__global__ __launch_bounds__(64 * kRestrictWaves) void k_restrict64(RestrictArgs A) {
  constexpr int NW = kRestrictWaves, E = (NW + 2) * 64;
  __shared__ double ed[4 * E];
  __shared__ double s_res[kS + 1];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int n1 = A.n1, n2 = A.n2, m1 = n1 / 2;
  const int bid = blockIdx.y * gridDim.x + blockIdx.x;
  const int i0 = (int)blockIdx.x * 124 + 2 * lane, j0 = (int)blockIdx.y * (NW * kVR - 4) + w * kVR;
  const int buf = resolve_visit(A.vf, bid == 0, s_res).buf;
  Strip<double, kVR, ISO> s;
  strip_region_load<kVR, ISO>(s, A.frot[buf], A.frot[0], A.fb, A.fbc, n1, n2, i0, j0);
  const StripCoef<double> k = strip_hold(A.k);
#pragma unroll
  for (int r = 0; r < kVR; ++r) {
    s.products(k, r, 0);
    s.products(k, r, 1);
  }
  Edges<double> e{ed, E, 64, (w + 1) * 64 + lane, true};
  if (w == 0) ed[E + lane] = ed[3 * E + lane] = 0.0;
  if (w == NW - 1) ed[e.o + 64] = ed[2 * E + e.o + 64] = 0.0;
  strip_publish_black<double, kVR, ISO>(s, e);
  ed[e.o] = s.north(0, 1);                         // red edges
  ed[E + e.o] = s.north(kVR - 1, 0);
  __syncthreads();
  double out[kVR / 2];
  strip_restrict<double, kVR, ISO, false>(s, k, e, out);
  if (lane == 0 || lane == 63 || i0 + 1 > n1) return;
#pragma unroll
  for (int t = 0; t < kVR / 2; ++t) {
    const int r = 2 * t + 1, lr = w * kVR + r, j = j0 + r;
    if (lr < 2 || lr >= NW * kVR - 2 || j > n2) continue;
    A.r2h[(int64_t)((j + 1) / 2 - 1) * (m1 + 1) + i0 / 2] = out[t];
  }
}

// The host waits for one kernel per V-cycle, which writes what the host needs
// straight into its memory and then the sequence number the host polls.
// Against a copy, an event and the runtime's completion handling this takes
// about 9 us off a V-cycle (128^2, four of them: 290 to 254 us a solve).
struct ReportArgs {
  SolveReport* out;
  uint64_t seq;
  const int* visit;
  const double* vres;
};

// wave 0; lane `ig` reports ks and res instead of what the log holds (-1: none)
__device__ void write_report(const ReportArgs& A, int ig, int ks, double res, double resid) {
  const int lane = threadIdx.x;
  if (lane < kVisitLog) {
    A.out->visit[lane] = lane == ig ? ks : A.visit[lane];
    A.out->vres[lane] = lane == ig ? res : A.vres[lane];
  }
  if (lane == 0) {
    A.out->status = ks;
    A.out->resid = resid;
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "");   // system scope
  if (lane == 0) __hip_atomic_store(&A.out->seq, A.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// end of a V-cycle on a multi-block finest level (FP64): records the up visit
__global__ __launch_bounds__(64 * (kS + 1)) void k_finish64(VisitRef V, ReportArgs A) {
  __shared__ double s_res[kS + 1];
  const Resolved r = resolve_visit(V, true, s_res);
  if (threadIdx.x < 64) write_report(A, r.ks ? V.ig : -1, r.ks, r.res, 0.0);
}

// end of the others: the finest residual's partial sums in a fixed order
constexpr int kReportThreads = 256;
__global__ __launch_bounds__(kReportThreads) void k_report(const double* __restrict__ partials, int nb, ReportArgs A) {
  __shared__ double ws[kReportThreads / 64];
  double r = 0.0;
  for (int q = threadIdx.x; q < nb; q += kReportThreads) r += partials[q];
  r = wave_sum(r);
  if ((threadIdx.x & 63) == 0) ws[threadIdx.x >> 6] = r;
  __syncthreads();
  if (threadIdx.x < 64) write_report(A, -1, 0, 0.0, ((ws[0] + ws[1]) + ws[2]) + ws[3]);
}

// end of a solve: the finest level's state from buffer `u_in` to phi (buffer 0)
__global__ __launch_bounds__(256) void k_settle64(double* __restrict__ phi, const double* __restrict__ u_in,
                                                  const int8_t* __restrict__ bc, int64_t n, LevelCtrl* c) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q == 0) c->cur[0] = c->cur[1] = 0;
  if (q < n && bc[q] == -1) phi[q] = u_in[q];
}

// Mixed mode with the finest level in k_tail: phi += e (bcnd <= 0 nodes) at
// the end of a V-cycle (otherwise the last up visit adds its own state).
__global__ __launch_bounds__(256) void k_add_corr(double* __restrict__ phi, const float* __restrict__ e,
                                                  const int8_t* __restrict__ bc, int64_t n) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q < n && bc[q] <= 0) phi[q] = phi[q] + (double)e[q];
}

// FP64 L1 residual of phi on the finest level (the reference's definition,
// sors.f90:348-349 order); in mixed mode it also becomes the FP32 right-hand
// side of the next correction equation (zero on walls).  A thread takes two columns of kResidRows rows,
// all loads before the first use: 1025^2 nodes (22 MB) 6.2 us, 10.4 with a row
// per block and a node per thread at a time.  k_report sums the blocks'
// partial sums: letting the block that ends last do it takes as long at 129^2
// (each block then makes its writes visible to the others) and 16 us longer at
// 1025^2.
constexpr int kResidRows = 4, kResidThreads = 256;
__global__ __launch_bounds__(kResidThreads) void k_resid64(const double* __restrict__ u, const double* __restrict__ b,
                                                           const int8_t* __restrict__ bc, int n1, int n2, double aw,
                                                           double an, double ac, float* __restrict__ bf,
                                                           double* __restrict__ partials) {
  constexpr int R = kResidRows, NT = kResidThreads;
  __shared__ double ws[NT / 64];
  const int W = n1 + 3, np = n1 / 2;                       // column pairs (2, 3), (4, 5) ...
  const int64_t n = (int64_t)np * ((n2 - 1 + R - 1) / R);
  double sum = 0.0;
  for (int64_t q = (int64_t)blockIdx.x * NT + threadIdx.x; q < n; q += (int64_t)gridDim.x * NT) {
    const int i0 = 2 + 2 * (int)(q % np), j0 = 2 + R * (int)(q / np);
    D2 um[R + 2], bb[R];
    double uw[R], ue[R];
    B2 m[R];
#pragma unroll
    for (int r = 0; r < R + 2; ++r) um[r] = *(const D2*)(u + (int64_t)min(j0 + r - 1, n2 + 1) * W + i0);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int64_t c = (int64_t)min(j0 + r, n2 + 1) * W + i0;
      uw[r] = u[c - 1];
      ue[r] = u[c + 2];
      m[r] = *(const B2*)(bc + c);
      bb[r] = *(const D2*)(b + (int64_t)(min(j0 + r, n2 + 1) - 1) * (n1 + 1) + i0 - 1);
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (j0 + r > n2) break;
      double r0 = 0.0, r1 = 0.0;
      if (m[r].x == -1) r0 = bb[r].x - (aw * uw[r] + an * um[r + 2].x + an * um[r].x + aw * um[r + 1].y + ac * um[r + 1].x);
      if (m[r].y == -1) r1 = bb[r].y - (aw * um[r + 1].x + an * um[r + 2].y + an * um[r].y + aw * ue[r] + ac * um[r + 1].y);
      if (bf) *(F2*)(bf + (int64_t)(j0 + r - 1) * (n1 + 1) + i0 - 1) = F2{(float)r0, (float)r1};
      sum += fabs(r0) + fabs(r1);
    }
  }
  sum = wave_sum(sum);
  if ((threadIdx.x & 63) == 0) ws[threadIdx.x >> 6] = sum;
  __syncthreads();
  if (threadIdx.x == 0) partials[blockIdx.x] = ((ws[0] + ws[1]) + ws[2]) + ws[3];
}

__global__ void k_cold_start(double* __restrict__ u, const int8_t* __restrict__ bc, int64_t n) {
  int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q < n && bc[q] == -1) u[q] = 0.0;
}

__global__ void k_copy_interior(double* __restrict__ u, const double* __restrict__ g,
                                const int8_t* __restrict__ bc, int64_t n) {
  int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q < n && bc[q] == -1) u[q] = g[q];
}

// ---------------------------------------------------------------------------
// single-workgroup kernel for the coarse levels Ls..ng
// ---------------------------------------------------------------------------
template <typename T>
struct TLevel {
  int n1, n2;
  T aw, an, ac;
  T* gu;                   // global arrays
  T* gb;
  const int8_t* gbc;
  int lds;                 // 1: held in LDS at the offsets below
  uint32_t ou, ob, obc;
};

template <typename T>
struct TailArgs {
  int Ls, ng, k;
  int fix_dn, fix_up;      // levels above the coarsest: fixed down / up sweep counts (0: the exit test)
  T omega;
  double eps;
  const int8_t* bc_img;    // bc arrays of the LDS-resident levels, in their LDS layout at offset 0
  int bc_bytes;
  int* visit;
  double* vres;
  TLevel<T> lv[kMaxLevels + 1];
};

// Sum over the block in a fixed order (wave trees, then a tree over the wave
// sums that every wave evaluates the same way); the caller guarantees a
// barrier since the previous call's reads of ws.
__device__ inline double block_sum_1024(double v, double* ws) {
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) ws[threadIdx.x >> 6] = v;
  __syncthreads();
  const int lane = threadIdx.x & 63, nw = blockDim.x >> 6;
  return wave_sum(lane < nw ? ws[lane] : 0.0);
}

// explicit address spaces, so LDS-resident levels use ds_ instructions and
// global ones global_ instructions instead of flat accesses
template <typename T> using lds_p = __attribute__((address_space(3))) T*;
template <typename T> using glb_p = __attribute__((address_space(1))) T*;

// red-black SOR at one tail level; lanes walk columns, waves walk rows
template <typename T, typename PU, typename PB, typename PC>
__device__ void t_smooth(PU u, PB b, PC bc, int n1, int n2, T aw, T an, T ac, T omega, double eps, int dig,
                         int nr, double* ws, int* ksor_out, double* res_out) {
  const int W = n1 + 3;
  const int hw = (n1 + 2) / 2;   // slots of one colour per row
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, nw = blockDim.x >> 6;
  double res_s = 0.0, res = 0.0;
  int ksor = 0;
  constexpr int NB = sizeof(T) == 8 ? 1 : 2;  // rows per wave whose loads are issued together
  for (int k = 1; k <= nr; ++k) {
    for (int color = 1; color >= 0; --color) {  // red (i+j odd) then black
      for (int j0 = 1 + wv; j0 <= n2 + 1; j0 += NB * nw) {
        for (int mm = lane; mm < hw; mm += 64) {
          int x[NB], xb[NB];
          bool act[NB];
          T c[NB], w[NB], e[NB], n[NB], so[NB], bb[NB];
#pragma unroll
          for (int q = 0; q < NB; ++q) {
            const int j = j0 + q * nw;
            const int i = 1 + 2 * mm + ((color ^ ((j + 1) & 1)) & 1);
            act[q] = j <= n2 + 1 && i <= n1 + 1;
            x[q] = act[q] ? j * W + i : W + 1;
            xb[q] = act[q] ? (j - 1) * (n1 + 1) + (i - 1) : 0;
            const int8_t mq = bc[x[q]];
            act[q] = act[q] & (mq <= 0);
            c[q] = u[x[q]]; w[q] = u[x[q] - 1]; e[q] = u[x[q] + 1];
            n[q] = u[x[q] + W]; so[q] = u[x[q] - W]; bb[q] = b[xb[q]];
          }
#pragma unroll
          for (int q = 0; q < NB; ++q)
            if (act[q]) u[x[q]] = sor_update(c[q], bb[q], w[q], n[q], so[q], e[q], aw, an, ac, omega);
        }
      }
      __syncthreads();
    }
    double r = 0.0;
    for (int j0 = 1 + wv; j0 <= n2 + 1; j0 += NB * nw)
      for (int i = 1 + lane; i <= n1 + 1; i += 64) {
        int x[NB], xb[NB];
        bool act[NB];
        T c[NB], w[NB], e[NB], n[NB], so[NB], bb[NB];
#pragma unroll
        for (int q = 0; q < NB; ++q) {
          const int j = j0 + q * nw;
          act[q] = j <= n2 + 1;
          x[q] = act[q] ? j * W + i : W + 1;
          xb[q] = act[q] ? (j - 1) * (n1 + 1) + (i - 1) : 0;
          const int8_t mq = bc[x[q]];
          act[q] = act[q] & (mq == -1);
          c[q] = u[x[q]]; w[q] = u[x[q] - 1]; e[q] = u[x[q] + 1];
          n[q] = u[x[q] + W]; so[q] = u[x[q] - W]; bb[q] = b[xb[q]];
        }
#pragma unroll
        for (int q = 0; q < NB; ++q)
          if (act[q]) r += fabs(sor_resid(c[q], bb[q], w[q], n[q], so[q], e[q], aw, an, ac));
      }
    res = block_sum_1024(r, ws);
    ksor += 1;
    bool stop;
    if (dig == 0) stop = res <= eps;
    else stop = res_s > 0.0 && (res / res_s) <= 0.6;
    if (stop) break;
    res_s = res;
  }
  *ksor_out = ksor;
  *res_out = res;
}

// Interior node of participant m in a colour's pass (t_smooth_fused).
__device__ __forceinline__ int colour_node(int m, bool red, int n1p) {
  const int q = 2 * m + (red ? 1 : 0);
  return (n1p & 1) ? q : q ^ ((q / n1p) & 1);
}

// Red-black sweeps of one tail level with the residual folded into the
// sweeps.  Where n1+1 is odd, interior node q = (j-1)(n1+1) + (i-1) is red
// (i+j odd) exactly when q is odd, so a participant handles red nodes 2m+1 and
// black nodes 2m for m = tid + P*r, r < R, with the indices computed once.
// Where n1+1 is even (a coarsest level of an odd number of cells along x) the
// nodes of a pair 2m, 2m+1 lie in one row and have the two colours, the other
// way round in every second row (colour_node).
// The residual after sweep k is the black nodes' residual, taken right after
// their update (their red neighbours are final), plus the red nodes'
// residual, taken in the red pass of sweep k+1 from the same loads as that
// pass's update; the update is stored only if the exit test (sors.f90:371-377)
// lets sweep k+1 run.  Expressions and exit tests are those of t_smooth.
// WAVE: wave 0 alone (P = 64, no block barriers); else the whole block.
template <typename T, int R, bool WAVE, typename PU, typename PB, typename PC>
__device__ __forceinline__ void t_smooth_fused(PU u, PB b, PC bc, int n1, int n2, T aw, T an, T ac, T omega, double eps,
                               int dig, int nr, double* ws, int* ksor_out, double* res_out, int nfix) {
  const int W = n1 + 3, n1p = n1 + 1;
  const int nint = n1p * (n2 + 1);
  const int P = WAVE ? 64 : (int)blockDim.x;
  const int tid = WAVE ? (int)(threadIdx.x & 63) : (int)threadIdx.x;
  int xr[R], qr[R], xk[R], qk[R];
  bool ur[R], rr[R], uk[R], rk[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int m = tid + P * r;
    int q = colour_node(m, true, n1p);
    bool ok = q < nint;
    q = ok ? q : 0;
    int x = (q / n1p + 1) * W + q % n1p + 1;
    int8_t mq = bc[x];
    xr[r] = x; qr[r] = q; ur[r] = ok && mq <= 0; rr[r] = ok && mq == -1;
    q = colour_node(m, false, n1p);
    ok = q < nint;
    q = ok ? q : 0;
    x = (q / n1p + 1) * W + q % n1p + 1;
    mq = bc[x];
    xk[r] = x; qk[r] = q; uk[r] = ok && mq <= 0; rk[r] = ok && mq == -1;
  }
  // in block mode the last item of a level is often held by a few waves
  // only: waves that hold none skip it (a wave-uniform branch after the
  // other items' loads, so those still issue together)
  bool wr[R], wk[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    wr[r] = WAVE || r + 1 < R || __ballot(2 * (tid + P * r) + 1 < nint) != 0;
    wk[r] = WAVE || r + 1 < R || __ballot(2 * (tid + P * r) < nint) != 0;
  }
  T cand[R];
  auto red_pass = [&](bool want_res) {
    double rs = 0.0;
    T c[R], w[R], e[R], nn[R], so[R], bb[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (!wr[r]) continue;
      c[r] = u[xr[r]]; w[r] = u[xr[r] - 1]; e[r] = u[xr[r] + 1];
      nn[r] = u[xr[r] + W]; so[r] = u[xr[r] - W]; bb[r] = b[qr[r]];
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (!wr[r]) continue;
      if (want_res && rr[r]) rs += fabs(sor_resid(c[r], bb[r], w[r], nn[r], so[r], e[r], aw, an, ac));
      cand[r] = sor_update(c[r], bb[r], w[r], nn[r], so[r], e[r], aw, an, ac, omega);
    }
    return rs;
  };
  auto store_red = [&]() {
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (ur[r]) u[xr[r]] = cand[r];
  };
  auto black_pass = [&]() {
    double rs = 0.0;
    T c[R], w[R], e[R], nn[R], so[R], bb[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (!wk[r]) continue;
      c[r] = u[xk[r]]; w[r] = u[xk[r] - 1]; e[r] = u[xk[r] + 1];
      nn[r] = u[xk[r] + W]; so[r] = u[xk[r] - W]; bb[r] = b[qk[r]];
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (!wk[r]) continue;
      T v = c[r];
      if (uk[r]) {
        v = sor_update(c[r], bb[r], w[r], nn[r], so[r], e[r], aw, an, ac, omega);
        u[xk[r]] = v;
      }
      if (rk[r]) rs += fabs(sor_resid(v, bb[r], w[r], nn[r], so[r], e[r], aw, an, ac));
    }
    return rs;
  };
  if (nfix > 0) {  // a fixed count without residuals or exit test (mixed form)
    for (int k = 1; k <= nfix; ++k) {
      red_pass(false);
      store_red();
      strip_sync<WAVE>();
      black_pass();
      strip_sync<WAVE>();
    }
    *ksor_out = nfix;
    *res_out = 0.0;
    return;
  }
  // sweep 1
  red_pass(false);
  store_red();
  strip_sync<WAVE>();
  double rb = black_pass();
  strip_sync<WAVE>();
  int k = 1;
  double res_s = 0.0, res = 0.0;
  for (;;) {
    const double rs = red_pass(true);
    res = strip_sum<WAVE>(rs + rb, ws, k & 1);
    bool stop;
    if (dig == 0) stop = res <= eps;
    else stop = res_s > 0.0 && (res / res_s) <= 0.6;
    if (stop || k >= nr) break;
    res_s = res;
    store_red();
    strip_sync<WAVE>();
    rb = black_pass();
    strip_sync<WAVE>();
    ++k;
  }
  // the last red pass only read; the next phase may overwrite nothing it read
  strip_sync<WAVE>();
  *ksor_out = k;
  *res_out = res;
}

// items per participant and colour of a level, 0 if above kFusedMaxR
constexpr int kFusedMaxR = 3;
static_assert((kWaveNodes + 1) / 2 <= 64 * kFusedMaxR, "wave-mode levels must fit the fused smoother");
__device__ __forceinline__ int fused_items(int n1, int n2, int P) {
  const int half = ((n1 + 1) * (n2 + 1) + 1) / 2;
  const int R = (half + P - 1) / P;
  return R <= kFusedMaxR ? R : 0;
}

// LDS-resident levels run the fused smoother with one or three items per
// participant (two-item levels take the three-item form with one masked);
// levels in global memory, or larger than three items, run t_smooth.  Few
// instantiations keep the kernel's code small: it is fetched anew by the CU
// that runs each launch.
template <typename T, bool WAVE, typename PU, typename PB, typename PC>
__device__ __forceinline__ bool t_smooth_fused_any(PU u, PB b, PC bc, int n1, int n2, T aw, T an, T ac, T omega,
                                                   double eps, int dig, int nr, double* ws, int* ks, double* res,
                                                   int nfix) {
  const int R = fused_items(n1, n2, WAVE ? 64 : (int)blockDim.x);
  if (R == 1) {
    t_smooth_fused<T, 1, WAVE>(u, b, bc, n1, n2, aw, an, ac, omega, eps, dig, nr, ws, ks, res, nfix);
    return true;
  }
  if (R == 2 || R == 3) {
    t_smooth_fused<T, 3, WAVE>(u, b, bc, n1, n2, aw, an, ac, omega, eps, dig, nr, ws, ks, res, nfix);
    return true;
  }
  return false;
}

// nfix > 0: exactly nfix sweeps, no residuals (LDS-resident levels of the
// mixed form); 0: the reference's exit test
template <typename T, bool WAVE = false>
__device__ __forceinline__ void smooth_level(const TLevel<T>& L, T* u, T* b, const int8_t* bc, T omega, double eps,
                                             int dig, int nr, double* ws, int* ks, double* res, int nfix = 0) {
  if (L.lds && t_smooth_fused_any<T, WAVE>((lds_p<T>)u, (lds_p<const T>)b, (lds_p<const int8_t>)bc, L.n1, L.n2,
                                           L.aw, L.an, L.ac, omega, eps, dig, nr, ws, ks, res, nfix))
    return;
  if constexpr (!WAVE) {
    if (L.lds)
      t_smooth<T>((lds_p<T>)u, (lds_p<const T>)b, (lds_p<const int8_t>)bc, L.n1, L.n2, L.aw, L.an, L.ac, omega,
                  eps, dig, nr, ws, ks, res);
    else
      t_smooth<T>((glb_p<T>)u, (glb_p<const T>)b, (glb_p<const int8_t>)bc, L.n1, L.n2, L.aw, L.an, L.ac, omega,
                  eps, dig, nr, ws, ks, res);
  }
}

// restriction of level l onto l+1 and prolongation of l+1 onto l by the
// participants (tid, P); LDS-resident pairs of levels use LDS-typed pointers
template <typename T, typename PU, typename PB, typename PC, typename PUC, typename PBC, typename PCC>
__device__ __forceinline__ void tail_restrict_p(const TLevel<T>& F, const TLevel<T>& C, PU uf, PB bf, PC bcf,
                                                PUC e2h, PBC r2h, PCC bcc, int tid, int P) {
  for (int q = tid; q < (C.n1 + 3) * (C.n2 + 3); q += P) e2h[q] = (T)0;
  for (int q = tid; q < (C.n1 + 1) * (C.n2 + 1); q += P) {
    const int i = q % (C.n1 + 1) + 1, j = q / (C.n1 + 1) + 1;
    T out = (T)0;
    if (bcc[j * (C.n1 + 3) + i] <= 0) out = restrict_node<T>(uf, bf, bcf, i, j, F.n1, F.n2, F.aw, F.an, F.ac);
    r2h[q] = out;
  }
}

template <typename T>
__device__ __forceinline__ void tail_restrict(const TLevel<T>& F, const TLevel<T>& C, T* uf, T* bf,
                                              const int8_t* bcf, T* e2h, T* r2h, const int8_t* bcc, int tid,
                                              int P) {
  if (F.lds && C.lds)
    tail_restrict_p<T>(F, C, (lds_p<const T>)uf, (lds_p<const T>)bf, (lds_p<const int8_t>)bcf, (lds_p<T>)e2h,
                       (lds_p<T>)r2h, (lds_p<const int8_t>)bcc, tid, P);
  else
    tail_restrict_p<T>(F, C, (const T*)uf, (const T*)bf, bcf, e2h, r2h, bcc, tid, P);
}

template <typename T, typename PU, typename PC, typename PE>
__device__ __forceinline__ void tail_prolong_p(const TLevel<T>& F, const TLevel<T>& C, PU uf, PC bcf, PE uc,
                                               int tid, int P) {
  for (int q = tid; q < (C.n1 + 1) * (C.n2 + 1); q += P)
    prolong_node<T>(uf, bcf, F.n1, uc, C.n1, q % (C.n1 + 1) + 1, q / (C.n1 + 1) + 1);
}

template <typename T>
__device__ __forceinline__ void tail_prolong(const TLevel<T>& F, const TLevel<T>& C, T* uf, const int8_t* bcf,
                                             const T* uc, int tid, int P) {
  if (F.lds && C.lds)
    tail_prolong_p<T>(F, C, (lds_p<T>)uf, (lds_p<const int8_t>)bcf, (lds_p<const T>)uc, tid, P);
  else
    tail_prolong_p<T>(F, C, uf, bcf, uc, tid, P);
}

// Block copies of `bytes` bytes between 16-byte aligned global and LDS
// buffers: every thread issues its 16-byte loads (up to four) before it
// stores, so a copy costs one memory latency instead of one per loop trip.
typedef int v4i __attribute__((ext_vector_type(4)));

template <typename VD, typename VS, typename BD, typename BS>
__device__ __forceinline__ void copy_block(VD d4, VS s4, BD d1, BS s1, int bytes) {
  const int nv = bytes >> 4;
  for (int q0 = threadIdx.x; q0 < nv; q0 += 4 * (int)blockDim.x) {
    v4i v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int q = q0 + k * (int)blockDim.x;
      if (q < nv) v[k] = s4[q];
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int q = q0 + k * (int)blockDim.x;
      if (q < nv) d4[q] = v[k];
    }
  }
  for (int q = (nv << 4) + (int)threadIdx.x; q < bytes; q += blockDim.x) d1[q] = s1[q];
}

__device__ __forceinline__ void copy_g2l(char* lds_dst, const void* src, int bytes) {
  copy_block((lds_p<v4i>)lds_dst, (glb_p<const v4i>)src, (lds_p<char>)lds_dst, (glb_p<const char>)src, bytes);
}

__device__ __forceinline__ void copy_l2g(void* dst, const char* lds_src, int bytes) {
  copy_block((glb_p<v4i>)dst, (lds_p<const v4i>)lds_src, (glb_p<char>)dst, (lds_p<const char>)lds_src, bytes);
}

// three global-to-LDS copies whose loads are all issued before any store
// (segments of up to 4 x 16 x blockDim bytes take one memory latency)
__device__ __forceinline__ void copy3_g2l(char* d0, const void* s0, int n0, char* d1, const void* s1, int n1,
                                          char* d2, const void* s2, int n2) {
  lds_p<v4i> d[3] = {(lds_p<v4i>)d0, (lds_p<v4i>)d1, (lds_p<v4i>)d2};
  glb_p<const v4i> sv[3] = {(glb_p<const v4i>)s0, (glb_p<const v4i>)s1, (glb_p<const v4i>)s2};
  const int nb[3] = {n0, n1, n2};
  const int P = blockDim.x, t = threadIdx.x;
  v4i v[3][4];
#pragma unroll
  for (int g = 0; g < 3; ++g)
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int q = t + k * P;
      if (q < (nb[g] >> 4)) v[g][k] = sv[g][q];
    }
#pragma unroll
  for (int g = 0; g < 3; ++g)
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int q = t + k * P;
      if (q < (nb[g] >> 4)) d[g][q] = v[g][k];
    }
  // what is left: vectors beyond 4 per thread, then the last bytes
  char* dc[3] = {d0, d1, d2};
  const void* sc[3] = {s0, s1, s2};
#pragma unroll
  for (int g = 0; g < 3; ++g) {
    for (int q = t + 4 * P; q < (nb[g] >> 4); q += P) d[g][q] = sv[g][q];
    for (int q = (nb[g] & ~15) + t; q < nb[g]; q += P)
      ((lds_p<char>)dc[g])[q] = ((glb_p<const char>)sc[g])[q];
  }
}

template <typename T>
__global__ __launch_bounds__(kTailThreads) void k_tail(TailArgs<T> A) {
  extern __shared__ __align__(16) char smem[];
  __shared__ double ws[32];
  __shared__ T* sU[kMaxLevels + 1];
  __shared__ T* sB[kMaxLevels + 1];
  __shared__ const int8_t* sBC[kMaxLevels + 1];
  const int Ls = A.Ls, ng = A.ng;
  if (threadIdx.x == 0) {
    for (int l = Ls; l <= ng; ++l) {
      const TLevel<T>& L = A.lv[l];
      sU[l] = L.lds ? (T*)(smem + L.ou) : L.gu;
      sB[l] = L.lds ? (T*)(smem + L.ob) : L.gb;
      sBC[l] = L.lds ? (const int8_t*)(smem + L.obc) : L.gbc;
    }
  }
  __syncthreads();
  {
    // one memory latency for all of it: the bc image of the resident levels
    // and, when resident, u and b of the first level
    const TLevel<T>& L = A.lv[Ls];
    const int ub = L.lds ? (L.n1 + 3) * (L.n2 + 3) * (int)sizeof(T) : 0;
    const int bb = L.lds ? (L.n1 + 1) * (L.n2 + 1) * (int)sizeof(T) : 0;
    copy3_g2l(smem, A.bc_img, A.bc_bytes, smem + L.ou, L.gu, ub, smem + L.ob, L.gb, bb);
  }
  __syncthreads();
  int ks;
  double res = 0.0;
  // levels from Lw down are run by wave 0 alone (no block barriers)
  int Lw = ng + 1;
  for (int l = ng; l >= Ls && A.lv[l].lds && (A.lv[l].n1 + 1) * (A.lv[l].n2 + 1) <= kWaveNodes; --l) Lw = l;
  const int tid = threadIdx.x, P = blockDim.x;
  for (int l = Ls; l < ng && l < Lw; ++l) {  // down leg: ig = l
    const TLevel<T>& F = A.lv[l];
    smooth_level<T>(F, sU[l], sB[l], sBC[l], A.omega, A.eps, l - ng, kNr, ws, &ks, &res, A.fix_dn);
    if (tid == 0) { A.visit[l] = ks; A.vres[l] = res; }
    tail_restrict<T>(F, A.lv[l + 1], sU[l], sB[l], sBC[l], sU[l + 1], sB[l + 1], sBC[l + 1], tid, P);
    __syncthreads();
  }
  if (Lw <= ng) {
    if (tid < 64) {
      for (int l = Lw; l < ng; ++l) {
        const TLevel<T>& F = A.lv[l];
        smooth_level<T, true>(F, sU[l], sB[l], sBC[l], A.omega, A.eps, l - ng, kNr, ws, &ks, &res, A.fix_dn);
        if (tid == 0) { A.visit[l] = ks; A.vres[l] = res; }
        tail_restrict<T>(F, A.lv[l + 1], sU[l], sB[l], sBC[l], sU[l + 1], sB[l + 1], sBC[l + 1], tid, 64);
        strip_sync<true>();
      }
      smooth_level<T, true>(A.lv[ng], sU[ng], sB[ng], sBC[ng], A.omega, A.eps, 0, A.k == 1 ? 1000000 : kNr, ws,
                            &ks, &res);
      if (tid == 0) { A.visit[ng] = ks; A.vres[ng] = res; }
      for (int l = ng - 1; l >= Lw; --l) {
        const TLevel<T>& F = A.lv[l];
        tail_prolong<T>(F, A.lv[l + 1], sU[l], sBC[l], (const T*)sU[l + 1], tid, 64);
        strip_sync<true>();
        smooth_level<T, true>(F, sU[l], sB[l], sBC[l], A.omega, A.eps, ng - l, kNr, ws, &ks, &res, A.fix_up);
        if (tid == 0) { A.visit[2 * ng - l] = ks; A.vres[2 * ng - l] = res; }
      }
    }
    __syncthreads();
  } else {  // coarsest: ig = ng; the first V-cycle iterates to eps (sors.f90:63-64)
    smooth_level<T>(A.lv[ng], sU[ng], sB[ng], sBC[ng], A.omega, A.eps, 0, A.k == 1 ? 1000000 : kNr, ws, &ks,
                    &res);
    if (tid == 0) { A.visit[ng] = ks; A.vres[ng] = res; }
  }
  for (int l = std::min(Lw, ng) - 1; l >= Ls; --l) {  // up leg: ig = 2ng - l
    const TLevel<T>& F = A.lv[l];
    tail_prolong<T>(F, A.lv[l + 1], sU[l], sBC[l], (const T*)sU[l + 1], tid, P);
    __syncthreads();
    smooth_level<T>(F, sU[l], sB[l], sBC[l], A.omega, A.eps, ng - l, kNr, ws, &ks, &res, A.fix_up);
    if (tid == 0) { A.visit[2 * ng - l] = ks; A.vres[2 * ng - l] = res; }
  }
  const TLevel<T>& L = A.lv[Ls];
  if (L.lds) copy_l2g(L.gu, smem + L.ou, (L.n1 + 3) * (L.n2 + 3) * (int)sizeof(T));
}

// The same work on register strips (mg_strip.h): every level above the
// coarsest runs its sweeps from registers, its arrays in LDS between the
// visits.  Levels whose strips fit one wave run in wave 0 without block
// barriers.  The coarsest level keeps the exit test of sors.f90:371-377 on the
// arrays in LDS, in FP64 every level does (strip_sweeps64).  Bound by the
// latency of the passes one after the other.  FP32 at 65^2 nodes and below: 28
// us a launch against 60 for k_tail, of 65e3 cycles: load 4e3, down visits 13e3
// (65^2), 9e3 (33^2), 6.2-6.9e3 each below, up visits 2.5-5.2e3; a pass costs
// about 225 cycles in one wave, most of them the LDS exchange.  FP64 at 65 x 33
// nodes and below: 44 us against 87 for k_tail.
template <typename T>
struct TailStripLevel {
  StripLevel<T> s;
  int two;                     // strips of 2 rows (else 4); always in wave 0
  uint32_t ou, ob, obc;        // LDS offsets of the correction, right-hand side and bc arrays
};

template <typename T>
struct TailStripArgs {
  int Ls, ng, k;
  int Lw;                      // levels Ls .. Lw-1 by the whole block, Lw .. ng-1 by wave 0
  int cw;                      // the coarsest level by wave 0
  int fix_dn, fix_up;          // FP32: the sweeps of a visit
  double eps;
  const int8_t* bc_img;
  int bc_bytes;
  uint32_t u_begin, u_end, oed;
  const T* gb;                 // level Ls: right-hand side, and where its correction goes
  T* gu;
  double* phi;                 // FP32, not null when Ls is the finest level
  T omega, caw, can, cac;      // coarsest level
  int* visit;
  double* vres;
  TailStripLevel<T> lv[kMaxLevels + 1];
};

template <typename T, bool ISO>
__global__ __launch_bounds__(kTailThreads) void k_tail_strips(TailStripArgs<T> A) {
  extern __shared__ __align__(16) char smem[];
  __shared__ double ws[32];
  const int Ls = A.Ls, ng = A.ng, tid = threadIdx.x;
  auto U = [&](int l) { return (T*)(smem + A.lv[l].ou); };
  auto B = [&](int l) { return (T*)(smem + A.lv[l].ob); };
  auto M = [&](int l) { return (const int8_t*)(smem + A.lv[l].obc); };
  T* ed = (T*)(smem + A.oed);
  {
    const StripLevel<T>& L = A.lv[Ls].s;
    copy3_g2l(smem, A.bc_img, A.bc_bytes, smem + A.lv[Ls].ob, A.gb, (L.n1 + 1) * (L.n2 + 1) * (int)sizeof(T), smem,
              A.bc_img, 0);
  }
  for (uint32_t q = A.u_begin + 16u * tid; q < A.u_end; q += 16u * blockDim.x)
    *(float4*)(smem + q) = make_float4(0.f, 0.f, 0.f, 0.f);
  __syncthreads();
  int ks = 0;
  double res = 0.0;
  TLevel<T> C;
  C.n1 = A.lv[ng].s.n1; C.n2 = A.lv[ng].s.n2;
  C.aw = A.caw; C.an = A.can; C.ac = A.cac;
  C.gu = nullptr; C.gb = nullptr; C.gbc = nullptr;
  C.lds = 1;
  C.ou = C.ob = C.obc = 0;
  const int nr = A.k == 1 ? 1000000 : kNr;
  auto down = [&](int l, auto rows, auto wave) {
    constexpr int R = decltype(rows)::value;
    constexpr bool W = decltype(wave)::value;
    const StripLevel<T>& L = A.lv[l].s;
    if constexpr (sizeof(T) == 4) {
      strip_down<R, ISO, W>(L, L.k, A.fix_dn, ed, U(l), B(l), M(l), B(l + 1));
      if (tid == 0) A.visit[l] = A.fix_dn;
    } else {
      VisitTest v{l - ng, kNr, A.eps, ws, 0, 0.0};
      strip_down64<R, ISO, W>(L, v, ed, U(l), B(l), M(l), B(l + 1));
      if (tid == 0) { A.visit[l] = v.ks; A.vres[l] = v.res; }
    }
  };
  auto up = [&](int l, auto rows, auto wave) {
    constexpr int R = decltype(rows)::value;
    constexpr bool W = decltype(wave)::value;
    const StripLevel<T>& L = A.lv[l].s;
    T* gu = l == Ls ? A.gu : nullptr;
    if constexpr (sizeof(T) == 4) {
      strip_up<R, ISO, W>(L, L.k, A.fix_up, ed, U(l), B(l), M(l), U(l + 1), gu, l == Ls ? A.phi : nullptr);
      if (tid == 0) A.visit[2 * ng - l] = A.fix_up;
    } else {
      VisitTest v{ng - l, kNr, A.eps, ws, 0, 0.0};
      strip_up64<R, ISO, W>(L, v, ed, U(l), B(l), M(l), U(l + 1), gu);
      if (tid == 0) { A.visit[2 * ng - l] = v.ks; A.vres[2 * ng - l] = v.res; }
    }
  };
  using Two = std::integral_constant<int, 2>;
  using Four = std::integral_constant<int, 4>;
  for (int l = Ls; l < A.Lw; ++l) {
    if (A.lv[l].two) down(l, Two{}, std::false_type{});
    else down(l, Four{}, std::false_type{});
  }
  if (A.cw) {
    if (tid < 64) {
      for (int l = A.Lw; l < ng; ++l) down(l, Two{}, std::true_type{});
      smooth_level<T, true>(C, U(ng), B(ng), M(ng), A.omega, A.eps, 0, nr, ws, &ks, &res);
      if (tid == 0) { A.visit[ng] = ks; A.vres[ng] = res; }
      for (int l = ng - 1; l >= A.Lw; --l) up(l, Two{}, std::true_type{});
    }
  } else {                     // Lw == ng
    smooth_level<T>(C, U(ng), B(ng), M(ng), A.omega, A.eps, 0, nr, ws, &ks, &res);
    if (tid == 0) { A.visit[ng] = ks; A.vres[ng] = res; }
  }
  __syncthreads();
  for (int l = A.Lw - 1; l >= Ls; --l) {
    if (A.lv[l].two) up(l, Two{}, std::false_type{});
    else up(l, Four{}, std::false_type{});
  }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
template <typename T>
T* rot_of(Level& L, int r) { return (T*)L.rot[r]; }

template <typename T>
T* u_of(Level& L, bool f32) { return f32 ? (T*)L.uf : (T*)L.u; }

template <typename T>
T* b_of(Level& L, bool f32) { return f32 ? (T*)L.bf : (T*)L.b; }

int* d_visit_of(lepic_ctx* ctx) { return (int*)(ctx->d_scalar + 64); }
double* d_vres_of(lepic_ctx* ctx) { return ctx->d_scalar + 32; }

// A launch of kexec sweeps: the halo, the waves of a block and the grid.
struct VisitShape {
  int hx, hy, nw;
  dim3 g;
  int nb() const { return (int)(g.x * g.y); }
};

// The fewest waves of 8, 12, 16 whose launch has at most one block per CU
// (a block of 8 waves passes its rows in half the time of one of 16, but halos
// cost it more of them: 8-row tiles in 32 rows against 40 in 64 for 5 sweeps);
// larger grids take 16.
constexpr int kVisitBlocks = 256;

VisitShape visit_shape(const Level& L, int kexec) {
  VisitShape S;
  S.hx = 2 * kexec + 2;
  S.hy = (2 * kexec + 1 + kVR - 1) / kVR * kVR;
  const int tx = 128 - 2 * S.hx;
  for (S.nw = 8;; S.nw += 4) {
    const int ty = S.nw * kVR - 2 * S.hy;
    if (ty < 8) continue;
    S.g = dim3((unsigned)((L.n1 - 1 + tx - 1) / tx), (unsigned)((L.n2 - 1 + ty - 1) / ty));
    if (S.nw == kVisitMaxWaves || S.nb() <= kVisitBlocks) return S;
  }
}

// How a multi-block level's FP64 visit runs: the reference's exit test
// (sors.f90:371-377) decides; one launch of `first` sweeps (one more than the
// same visit took in the previous V-cycle: most visits then finish in one
// launch of a small halo) and one of the others up to kNr, which first tests
// the first one's sweeps and returns at once when the visit has stopped there.
constexpr int kFirstMax = 5;
static_assert(kNr - 2 <= kS && kFirstMax <= kS && kNr - kFirstMax <= kS, "a visit takes two launches");

VisitRef visit_ref(lepic_ctx* ctx, int l, int epoch, int dig, int nr, int ig, double eps, int nexec, int klast0,
                   int before) {
  Level& L = ctx->lv[l];
  VisitRef v;
  v.ctrl = ctx->d_ctrl + l;
  v.t = StopTest{L.partials, L.part_stride, before ? visit_shape(L, before).nb() : 0,
                 visit_shape(L, nexec - klast0).nb(), dig, nr, eps};
  v.epoch = epoch; v.ig = ig;
  v.nexec = nexec;
  v.klast0 = klast0;
  v.visit = d_visit_of(ctx);
  v.vres = d_vres_of(ctx);
  return v;
}

// the down or up visit of a V-cycle
VisitRef cycle_visit_ref(lepic_ctx* ctx, int l, int epoch, bool up, double eps) {
  const int f = up ? ctx->lv[l].first_up : ctx->lv[l].first_dn, ng = ctx->ng;
  return visit_ref(ctx, l, epoch, up ? ng - l : l - ng, kNr, up ? 2 * ng - l : l, eps, kNr, f, f);
}

StripCoef<double> strip_coef64(const Level& L) {
  StripCoef<double> k;
  k.aw = L.aw; k.an = L.an; k.ac = L.ac;
  k.om = 1.4;                                     // iterative_solver.f90:27
  k.om1 = 1.0 - k.om;
  k.rac = 1.0 / k.ac;
  k.racl = std::fma(-k.rac, k.ac, 1.0) / k.ac;
  return k;
}

VisitArgs visit_args(lepic_ctx* ctx, int l, int epoch, int dig, int nr, double eps) {
  Level& L = ctx->lv[l];
  VisitArgs A{};
  for (int r = 0; r < kRot; ++r) A.rot[r] = rot_of<double>(L, r);
  A.b = L.b;
  A.bc = L.bc;
  A.n1 = L.n1; A.n2 = L.n2;
  A.k = strip_coef64(L);
  A.ctrl = ctx->d_ctrl + l;
  A.partials = L.partials;
  A.t = StopTest{L.partials, L.part_stride, 0, 0, dig, nr, eps};
  A.epoch = epoch;
  return A;
}

// one launch: sweeps k0+1 .. k0+kexec; the one before it ran sweeps kchk .. k0
int launch_sweeps(lepic_ctx* ctx, int l, VisitArgs& A, int k0, int kexec, int kchk) {
  const Level& L = ctx->lv[l];
  const VisitShape S = visit_shape(L, kexec);
  A.k0 = k0; A.kexec = kexec; A.kchk = kchk;
  A.halo_x = S.hx; A.halo_y = S.hy;
  if (L.aw == L.an) hipLaunchKernelGGL(k_visit64<true>, S.g, dim3(64 * S.nw), 0, ctx->stream, A);
  else hipLaunchKernelGGL(k_visit64<false>, S.g, dim3(64 * S.nw), 0, ctx->stream, A);
  LEPIC_HIP(hipGetLastError());
  A.t.nb0 = A.t.nb1;                              // for the launch after it
  A.t.nb1 = S.nb();
  A.zero = 0;
  A.crot[0] = nullptr;
  return 0;
}

// the down or up visit of a V-cycle; the up visit starts with the prolonged
// correction of the level below
int launch_visit(lepic_ctx* ctx, int l, int epoch, bool up, double eps) {
  Level& L = ctx->lv[l];
  const int ng = ctx->ng, first = up ? L.first_up : L.first_dn;
  VisitArgs A = visit_args(ctx, l, epoch, up ? ng - l : l - ng, kNr, eps);
  A.zero = !up && l > 1;
  if (up) {
    Level& C = ctx->lv[l + 1];
    for (int r = 0; r < kRot; ++r) A.crot[r] = C.mb ? rot_of<double>(C, r) : C.u;
    A.coarse_mb = C.mb;
    if (C.mb) A.vc = cycle_visit_ref(ctx, l + 1, epoch, true, eps);
  }
  if (int rc = launch_sweeps(ctx, l, A, 0, first, 0)) return rc;
  return launch_sweeps(ctx, l, A, first, kNr - first, 1);
}

// ---- mixed form: visits of fixed sweep counts in k_tile32 ----
StripCoef<float> strip_coef(const Level& L, float omega) {
  StripCoef<float> k;
  k.aw = (float)L.aw; k.an = (float)L.an; k.ac = (float)L.ac;
  k.om = omega; k.om1 = 1.0f - omega; k.rac = 1.0f / k.ac;
  return k;
}

bool strip_iso(const Level& L) { return (float)L.aw == (float)L.an; }

// One launch of nsw sweeps.  Bound by VALU issue (eleven instructions of about
// 4.7 cycles per node and pass) behind the launch's load latency of about
// 3 us.  Regions of 128 columns by 4 rows for each of 16 waves, four waves per
// SIMD to cover the LDS exchange (8 waves x 8 rows: 9.9, 11.9, 11.7, 11.3 us
// for the four down visits of 1025^2 .. 129^2 against 9.2, 12.3, 10.6, 10.0);
// fewer waves, whose passes take less long, where the launch then still has at
// most one block per CU (129^2: 4 sweeps 7.0 us with 16 waves, 5.1 with 8; 3 sweeps
// 7.3, 5.4).  The sweeps on a region in LDS that this replaces took 23.5 us for
// the 1025^2 down visit (4 sweeps) and 29.6, 20.4, 21.2 us for the 10 sweeps of
// the others in two launches each.
template <int NW>
void launch_tile_of(lepic_ctx* ctx, const Level& L, const TileArgs& A, dim3 g) {
  if (strip_iso(L)) hipLaunchKernelGGL((k_tile32<4, NW, true>), g, dim3(64 * NW), 0, ctx->stream, A);
  else hipLaunchKernelGGL((k_tile32<4, NW, false>), g, dim3(64 * NW), 0, ctx->stream, A);
}

int launch_tile32(lepic_ctx* ctx, const Level& L, TileArgs A) {
  A.halo = 2 * A.nsw + (A.r2h ? 2 : 0);
  const int tx = 128 - 2 * A.halo;
  for (int nw = 8;; nw += 4) {
    const int ty = 4 * nw - 2 * A.halo;
    if (ty < 8) continue;
    const dim3 g((unsigned)((L.n1 - 1 + tx - 1) / tx), (unsigned)((L.n2 - 1 + ty - 1) / ty));
    if (nw < 16 && (int64_t)g.x * g.y > kVisitBlocks) continue;
    if (nw == 8) launch_tile_of<8>(ctx, L, A, g);
    else if (nw == 12) launch_tile_of<12>(ctx, L, A, g);
    else launch_tile_of<16>(ctx, L, A, g);
    LEPIC_HIP(hipGetLastError());
    return 0;
  }
}

TileArgs tile_args(lepic_ctx* ctx, int l) {
  Level& L = ctx->lv[l];
  TileArgs A{};
  A.b = L.bf; A.bc = L.bc; A.n1 = L.n1; A.n2 = L.n2;
  A.k = strip_coef(L, l == 1 ? kFineOmega : 1.4f);
  return A;
}

// down visit of level l: from zero into rot[0], the restricted residual to
// level l + 1's right-hand side
int tile_down(lepic_ctx* ctx, int l) {
  Level& L = ctx->lv[l];
  const int nsw = l == 1 ? kFineDn : kFixDn;
  TileArgs A = tile_args(ctx, l);
  A.u_out = rot_of<float>(L, 0);
  const int h = 2 * nsw + 2;
  const int64_t nb = (int64_t)((L.n1 - 1 + 127 - 2 * h) / (128 - 2 * h)) * ((L.n2 - 1 + 63 - 2 * h) / (64 - 2 * h));
  A.nsw = nsw;
  if (nsw > kTileSplit && nb > kTileMaxBlocks) {
    A.nsw = kTileSplit;
    A.u_out = rot_of<float>(L, 1);
    if (int rc = launch_tile32(ctx, L, A)) return rc;
    A.u_in = rot_of<float>(L, 1);
    A.u_out = rot_of<float>(L, 0);
    A.nsw = nsw - kTileSplit;
  }
  A.r2h = ctx->lv[l + 1].bf;
  return launch_tile32(ctx, L, A);
}

// up visit: rot[0] and the prolonged correction of level l + 1 into rot[1], on
// the finest level added to phi
int tile_up(lepic_ctx* ctx, int l) {
  Level& L = ctx->lv[l];
  Level& C = ctx->lv[l + 1];
  TileArgs A = tile_args(ctx, l);
  A.u_in = rot_of<float>(L, 0);
  if (l == 1) A.phi = ctx->phi;
  else A.u_out = rot_of<float>(L, 1);
  A.e2h = C.mb ? rot_of<float>(C, 1) : C.uf;
  A.nsw = l == 1 ? kFineUp : kFixUp;
  return launch_tile32(ctx, L, A);
}

int launch_restrict(lepic_ctx* ctx, int l, int epoch, double eps) {
  Level& F = ctx->lv[l];
  Level& C = ctx->lv[l + 1];
  RestrictArgs A;
  A.vf = cycle_visit_ref(ctx, l, epoch, false, eps);
  for (int r = 0; r < kRot; ++r) A.frot[r] = rot_of<double>(F, r);
  A.fb = F.b;
  A.fbc = F.bc;
  A.n1 = F.n1; A.n2 = F.n2;
  A.k = strip_coef64(F);
  A.r2h = C.b;
  constexpr int tx = 124, ty = kRestrictWaves * kVR - 4;
  const dim3 g((unsigned)((F.n1 - 1 + tx - 1) / tx), (unsigned)((F.n2 - 1 + ty - 1) / ty));
  if (F.aw == F.an) hipLaunchKernelGGL(k_restrict64<true>, g, dim3(64 * kRestrictWaves), 0, ctx->stream, A);
  else hipLaunchKernelGGL(k_restrict64<false>, g, dim3(64 * kRestrictWaves), 0, ctx->stream, A);
  LEPIC_HIP(hipGetLastError());
  return 0;
}

// The bc arrays of levels ng .. Lr, coarsest first, each from a 16-byte
// boundary: rebuilt when the boundary or the layout changes.
int tail_bc_image(lepic_ctx* ctx, int Lr, bool f32) {
  const int key = Lr * 2 + (f32 ? 1 : 0);
  if (ctx->tail_bc_key == key) return 0;
  auto bytes_of = [&](int l) { return (size_t)(ctx->lv[l].n1 + 3) * (ctx->lv[l].n2 + 3); };
  size_t total = 0;
  for (int l = ctx->ng; l >= Lr; --l) total = (total + bytes_of(l) + 15) & ~size_t(15);
  if (total > ctx->tail_bc_cap) {
    if (ctx->d_tail_bc) LEPIC_HIP(hipFree(ctx->d_tail_bc));
    LEPIC_HIP(hipMalloc(&ctx->d_tail_bc, total));
    ctx->tail_bc_cap = total;
  }
  size_t off = 0;
  for (int l = ctx->ng; l >= Lr; --l) {
    LEPIC_HIP(hipMemcpyAsync(ctx->d_tail_bc + off, ctx->lv[l].bc, bytes_of(l), hipMemcpyDeviceToDevice, ctx->stream));
    off = (off + bytes_of(l) + 15) & ~size_t(15);
  }
  ctx->tail_bc_key = key;
  return 0;
}

// k_tail_strips' layout, or false where a level above the coarsest does not fit
// its strips (wider than 128 columns or more than 16 waves) or the LDS, or
// holds wall values (FP64, the finest level).
template <typename T>
bool tail_strips_plan(lepic_ctx* ctx, TailStripArgs<T>& A, size_t& lds, int& threads) {
  if (ctx->Lc == ctx->ng) return false;   // the coarsest level alone
  if (sizeof(T) == 8 && ctx->Lc == 1) return false;
  const int ng = ctx->ng, Ls = ctx->Lc;
  auto al = [](size_t x) { return (x + 15) & ~size_t(15); };
  A.Ls = Ls; A.ng = ng; A.Lw = ng;
  int waves = 4;
  size_t ed = 0;
  for (int l = Ls; l < ng; ++l) {
    const Level& L = ctx->lv[l];
    TailStripLevel<T>& V = A.lv[l];
    StripLevel<T>& S = V.s;
    S.n1 = L.n1; S.n2 = L.n2;
    S.Lx = (L.n1 + 1) / 2;
    if (S.Lx > 64) return false;
    S.SW = 64 / S.Lx;
    S.inv = 65536 / S.Lx + 1;
    // strips of two rows where they fit four waves, one per SIMD; strips of
    // four rows where a level has work for every SIMD anyway (65^2: 13e3
    // cycles a down visit in 8 waves of 4 rows, 18e3 in 4 waves of 8)
    V.two = ((L.n2 - 1 + 1) / 2 + S.SW - 1) / S.SW <= 4;
    const int R = V.two ? 2 : 4;
    S.nst = (L.n2 - 1 + R - 1) / R;
    const int w = (S.nst + S.SW - 1) / S.SW;
    if (w > 16) return false;
    if (w == 1 && V.two) A.Lw = std::min(A.Lw, l);
    else if (A.Lw < l) return false;
    waves = std::max(waves, w);
    if constexpr (sizeof(T) == 4) S.k = strip_coef(L, 1.4f);
    else S.k = strip_coef64(L);
    ed = std::max(ed, (size_t)4 * (S.nst + 2) * S.Lx * sizeof(T));
  }
  const Level& C = ctx->lv[ng];
  A.lv[ng].s.n1 = C.n1; A.lv[ng].s.n2 = C.n2;
  A.cw = (C.n1 + 1) * (C.n2 + 1) <= kWaveNodes ? 1 : 0;
  if (!A.cw && A.Lw < ng) return false;
  size_t off = 0;
  for (int l = ng; l >= Ls; --l) {
    A.lv[l].obc = (uint32_t)off;
    off = al(off + (size_t)(ctx->lv[l].n1 + 3) * (ctx->lv[l].n2 + 3));
  }
  A.bc_bytes = (int)off;
  A.u_begin = (uint32_t)off;
  for (int l = ng; l >= Ls; --l) {
    A.lv[l].ou = (uint32_t)off;
    off = al(off + (size_t)(ctx->lv[l].n1 + 3) * (ctx->lv[l].n2 + 3) * sizeof(T));
  }
  A.u_end = (uint32_t)off;
  for (int l = ng; l >= Ls; --l) {
    A.lv[l].ob = (uint32_t)off;
    off = al(off + (size_t)(ctx->lv[l].n1 + 1) * (ctx->lv[l].n2 + 1) * sizeof(T));
  }
  A.oed = (uint32_t)off;
  lds = off + ed;
  threads = 64 * waves;
  return lds <= kTailLds;
}

template <typename T>
int launch_tail(lepic_ctx* ctx, bool f32, int k, double eps);

// levels Ls .. ng of a V-cycle on strips where the plan allows, else in the
// generic kernel, which starts from the state in global memory: zero on
// coarser levels
template <typename T>
int launch_lower(lepic_ctx* ctx, int k, double eps) {
  constexpr bool f32 = sizeof(T) == 4;
  TailStripArgs<T> A{};
  size_t lds = 0;
  int threads = 0;
  Level& L = ctx->lv[ctx->Lc];
  if (!tail_strips_plan(ctx, A, lds, threads)) {
    const int64_t n = (int64_t)(L.n1 + 3) * (L.n2 + 3);
    if (f32 || ctx->Lc > 1)
      if (int rc = zero_async(ctx, u_of<T>(L, f32), n * sizeof(T))) return rc;
    if (int rc = launch_tail<T>(ctx, f32, k, eps)) return rc;
    if (f32 && ctx->Lc == 1) {
      hipLaunchKernelGGL(k_add_corr, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, ctx->stream, ctx->phi,
                         (const float*)L.uf, (const int8_t*)ctx->bc, n);
      LEPIC_HIP(hipGetLastError());
    }
    return 0;
  }
  if (int rc = tail_bc_image(ctx, ctx->Lc, f32)) return rc;
  A.k = k; A.eps = eps;
  A.fix_dn = kFixDn; A.fix_up = kFixUp;
  A.bc_img = ctx->d_tail_bc;
  A.gb = b_of<T>(L, f32);
  A.gu = u_of<T>(L, f32);
  A.phi = ctx->Lc == 1 ? ctx->phi : nullptr;
  const Level& C = ctx->lv[ctx->ng];
  A.omega = (T)1.4; A.caw = (T)C.aw; A.can = (T)C.an; A.cac = (T)C.ac;
  A.visit = d_visit_of(ctx);
  A.vres = d_vres_of(ctx);
  static bool attr_set = false;   // per instantiation
  if (!attr_set) {
    LEPIC_HIP(hipFuncSetAttribute((const void*)k_tail_strips<T, true>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kTailLds));
    LEPIC_HIP(hipFuncSetAttribute((const void*)k_tail_strips<T, false>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kTailLds));
    attr_set = true;
  }
  if ((T)L.aw == (T)L.an)
    hipLaunchKernelGGL((k_tail_strips<T, true>), dim3(1), dim3(threads), lds, ctx->stream, A);
  else hipLaunchKernelGGL((k_tail_strips<T, false>), dim3(1), dim3(threads), lds, ctx->stream, A);
  LEPIC_HIP(hipGetLastError());
  return 0;
}

template <typename T>
int launch_tail(lepic_ctx* ctx, bool f32, int k, double eps) {
  TailArgs<T> A{};
  A.Ls = ctx->Lc; A.ng = ctx->ng; A.k = k; A.omega = (T)1.4; A.eps = eps;
  // mixed form: the tail levels above the coarsest run the counts the exit
  // test gives them on plasma solves, without the per-sweep sums the test
  // needs
  A.fix_dn = f32 ? kFixDn : 0;
  A.fix_up = f32 ? kFixUp : 0;
  A.visit = d_visit_of(ctx);
  A.vres = d_vres_of(ctx);
  auto al = [](size_t x) { return (x + 15) & ~size_t(15); };
  // residency, coarsest first, until the LDS budget is spent; the LDS holds
  // the bc arrays of the resident levels first, then their u and b
  int Lr = ctx->ng + 1;   // finest resident level
  size_t need_all = 0;
  for (int l = ctx->ng; l >= ctx->Lc; --l) {
    const Level& L = ctx->lv[l];
    const size_t need = al((size_t)(L.n1 + 3) * (L.n2 + 3) * sizeof(T)) +
                        al((size_t)(L.n1 + 1) * (L.n2 + 1) * sizeof(T)) + al((size_t)(L.n1 + 3) * (L.n2 + 3));
    if (need_all + need > kTailLds) break;
    need_all += need;
    Lr = l;
  }
  size_t off = 0;
  for (int l = ctx->ng; l >= Lr; --l) {
    const Level& L = ctx->lv[l];
    A.lv[l].obc = (uint32_t)off;
    off = al(off + (size_t)(L.n1 + 3) * (L.n2 + 3));
  }
  const size_t bc_bytes = off;
  for (int l = ctx->ng; l >= ctx->Lc; --l) {
    Level& L = ctx->lv[l];
    TLevel<T>& C = A.lv[l];
    C.n1 = L.n1; C.n2 = L.n2; C.aw = (T)L.aw; C.an = (T)L.an; C.ac = (T)L.ac;
    C.gu = u_of<T>(L, f32); C.gb = b_of<T>(L, f32); C.gbc = L.bc;
    C.lds = l >= Lr ? 1 : 0;
    if (C.lds) {
      C.ou = (uint32_t)off; off = al(off + (size_t)(L.n1 + 3) * (L.n2 + 3) * sizeof(T));
      C.ob = (uint32_t)off; off = al(off + (size_t)(L.n1 + 1) * (L.n2 + 1) * sizeof(T));
    }
  }
  if (int rc = tail_bc_image(ctx, Lr, f32)) return rc;
  A.bc_img = ctx->d_tail_bc;
  A.bc_bytes = (int)bc_bytes;
  static bool attr_set = false;   // per instantiation; the attribute is per kernel
  if (!attr_set) {
    LEPIC_HIP(hipFuncSetAttribute((const void*)k_tail<T>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                  (int)kTailLds));
    attr_set = true;
  }
  hipLaunchKernelGGL(k_tail<T>, dim3(1), dim3(kTailThreads), off, ctx->stream, A);
  LEPIC_HIP(hipGetLastError());
  return 0;
}

// slot 0: what the host waits for next; slot 1: the starting residual, which it
// reads when it has something to wait for
ReportArgs report_args(lepic_ctx* ctx, int slot = 0) {
  return ReportArgs{ctx->d_report + slot, ++ctx->report_seq[slot], d_visit_of(ctx), d_vres_of(ctx)};
}

int launch_finish64(lepic_ctx* ctx, const VisitRef& v) {
  hipLaunchKernelGGL(k_finish64, dim3(1), dim3(64 * (kS + 1)), 0, ctx->stream, v, report_args(ctx));
  LEPIC_HIP(hipGetLastError());
  return 0;
}

int launch_report(lepic_ctx* ctx, int nb, int slot = 0) {
  hipLaunchKernelGGL(k_report, dim3(1), dim3(kReportThreads), 0, ctx->stream, (const double*)ctx->d_partials, nb,
                     report_args(ctx, slot));
  LEPIC_HIP(hipGetLastError());
  return 0;
}

// One FP64 V-cycle (mg.f90:85-225): levels 1..Ls-1 multi-block, Ls..ng in one
// workgroup; then the end-of-cycle kernel.
int vcycle64(lepic_ctx* ctx, int k, double eps) {
  const int Ls = ctx->Lc;
  const int e_dn = ctx->mg_epoch + 1, e_up = ctx->mg_epoch + 2;
  ctx->mg_epoch += 2;
  for (int l = 1; l < Ls; ++l) {  // down leg
    if (int rc = launch_visit(ctx, l, e_dn, false, eps)) return rc;
    if (int rc = launch_restrict(ctx, l, e_dn, eps)) return rc;
  }
  if (int rc = launch_lower<double>(ctx, k, eps)) return rc;
  for (int l = Ls - 1; l >= 1; --l)  // up leg
    if (int rc = launch_visit(ctx, l, e_up, true, eps)) return rc;
  return ctx->lv[1].mb ? launch_finish64(ctx, cycle_visit_ref(ctx, 1, e_up, true, eps)) : launch_report(ctx, 0);
}

// One V-cycle of the mixed form on the FP32 correction equation; adds the
// correction to phi.
int vcycle32(lepic_ctx* ctx, int k, double eps, bool begun) {
  for (int l = begun ? 2 : 1; l < ctx->Lc; ++l)
    if (int rc = tile_down(ctx, l)) return rc;
  if (int rc = launch_lower<float>(ctx, k, eps)) return rc;
  for (int l = ctx->Lc - 1; l >= 1; --l)
    if (int rc = tile_up(ctx, l)) return rc;
  return 0;
}

double alpha_of(lepic_ctx* ctx) {
  // iterative_solver.f90:22-23
  return std::fabs((double)((ctx->g.n1 + 1) * (ctx->g.n2 + 1)) * ctx->lv[1].ac) * 1.0;
}

// FP64 residual of phi, reported; fills the FP32 right-hand side when fill_f32
int launch_resid64(lepic_ctx* ctx, bool fill_f32, const double* u = nullptr, int slot = 0) {
  Level& L = ctx->lv[1];
  const int64_t n = (int64_t)(L.n1 / 2) * ((L.n2 - 1 + kResidRows - 1) / kResidRows);
  const int nb = (int)std::min<int64_t>(std::max<int64_t>((n + kResidThreads - 1) / kResidThreads, 1), kResidBlocks);
  hipLaunchKernelGGL(k_resid64, dim3(nb), dim3(kResidThreads), 0, ctx->stream, u ? u : (const double*)ctx->phi,
                     (const double*)ctx->rhs, (const int8_t*)ctx->bc, L.n1, L.n2, L.aw, L.an, L.ac,
                     fill_f32 ? L.bf : nullptr, ctx->d_partials);
  LEPIC_HIP(hipGetLastError());
  return launch_report(ctx, nb, slot);
}

// Waits for the slot's report launched last.  The stream is asked now and
// then, so that an error on it ends the wait.
int read_report(lepic_ctx* ctx, int* visit, double* vres, int slot = 0) {
  const SolveReport* h = ctx->h_report + slot;
  auto arrived = [&]() { return __atomic_load_n(&h->seq, __ATOMIC_ACQUIRE) == ctx->report_seq[slot]; };
  for (uint32_t spin = 1; !arrived(); ++spin) {
    if (spin % 65536 != 0) continue;
    const hipError_t q = hipStreamQuery(ctx->stream);
    if (q == hipErrorNotReady) continue;
    LEPIC_HIP(q);
    if (!arrived()) return ctx->fail(LEPIC_ERR_STATE, "a V-cycle ended without its report");
  }
  std::memcpy(vres, h->vres, sizeof(h->vres));
  std::memcpy(visit, h->visit, sizeof(h->visit));
  return 0;
}

}  // namespace

namespace lepic {

int poisson_setup(lepic_ctx* ctx) {
  const int ng = ctx->ng;
  const double eps0 = ctx->g.eps0;
  const bool mixed = ctx->g.precision == LEPIC_MIXED;
  for (int l = 1; l <= ng; ++l) {
    Level& L = ctx->lv[l];
    L.n1 = ctx->g.n1 >> (l - 1);
    L.n2 = ctx->g.n2 >> (l - 1);
    const double f = (double)(1 << (l - 1));  // h2=2.d0*h, h4=4.d0*h ... (mg.f90:59-80)
    L.h1 = f * ctx->g.h1;
    L.h2 = f * ctx->g.h2;
    L.aw = eps0 / (L.h1 * L.h1);  // mg.h:11-15
    L.an = eps0 / (L.h2 * L.h2);
    L.ac = -(L.an + L.an + L.aw + L.aw);
    const size_t nn = (size_t)(L.n1 + 3) * (L.n2 + 3), nr = (size_t)(L.n1 + 1) * (L.n2 + 1);
    if (l == 1) {
      L.u = ctx->phi;
      L.b = ctx->rhs;
      L.bc = ctx->bc;
    } else {
      LEPIC_HIP(hipMalloc(&L.u, nn * 8));
      LEPIC_HIP(hipMemsetAsync(L.u, 0, nn * 8, ctx->stream));
      LEPIC_HIP(hipMalloc(&L.b, nr * 8));
      LEPIC_HIP(hipMemsetAsync(L.b, 0, nr * 8, ctx->stream));
      LEPIC_HIP(hipMalloc(&L.bc, nn));
      LEPIC_HIP(hipMemsetAsync(L.bc, 1, nn, ctx->stream));
    }
    if (mixed) {
      LEPIC_HIP(hipMalloc(&L.uf, nn * 4));
      LEPIC_HIP(hipMemsetAsync(L.uf, 0, nn * 4, ctx->stream));
      LEPIC_HIP(hipMalloc(&L.bf, nr * 4));
      LEPIC_HIP(hipMemsetAsync(L.bf, 0, nr * 4, ctx->stream));
    }
  }
  // levels with more nodes than the tail threshold run multi-block; the
  // coarsest level always runs in the single workgroup (unless ng = 1)
  const int64_t tail_nodes = ctx->g.mg_tail_nodes > 0 ? ctx->g.mg_tail_nodes : kDefaultTailNodes;
  ctx->Lc = ng;
  for (int l = 1; l <= ng; ++l) {
    const Level& L = ctx->lv[l];
    if ((int64_t)(L.n1 + 1) * (L.n2 + 1) <= tail_nodes) { ctx->Lc = l; break; }
  }
  if (ng == 1 && (int64_t)(ctx->lv[1].n1 + 1) * (ctx->lv[1].n2 + 1) > tail_nodes) ctx->Lc = 2;
  for (int l = 1; l < ctx->Lc && l <= ng; ++l) {
    Level& L = ctx->lv[l];
    L.mb = true;
    const size_t nn = (size_t)(L.n1 + 3) * (L.n2 + 3);
    if (mixed) {
      // the states after the down and the up visit; walls stay zero
      L.rot[0] = L.uf;
      LEPIC_HIP(hipMalloc(&L.rot[1], nn * 4));
      LEPIC_HIP(hipMemsetAsync(L.rot[1], 0, nn * 4, ctx->stream));
      continue;
    }
    L.first_dn = L.first_up = kFirstMax;
    L.rot[0] = L.u;
    for (int r = 1; r < kRot; ++r) {
      LEPIC_HIP(hipMalloc(&L.rot[r], nn * 8));
      LEPIC_HIP(hipMemsetAsync(L.rot[r], 0, nn * 8, ctx->stream));
    }
    L.part_stride = 0;
    for (int k = 1; k <= kS; ++k) L.part_stride = std::max(L.part_stride, visit_shape(L, k).nb());
    const size_t np = (size_t)kRing * L.part_stride;
    LEPIC_HIP(hipMalloc(&L.partials, np * 8));
    LEPIC_HIP(hipMemsetAsync(L.partials, 0, np * 8, ctx->stream));
  }
  LEPIC_HIP(hipMalloc(&ctx->d_ctrl, (kMaxLevels + 1) * sizeof(LevelCtrl)));
  LEPIC_HIP(hipMemsetAsync(ctx->d_ctrl, 0, (kMaxLevels + 1) * sizeof(LevelCtrl), ctx->stream));
  ctx->mg_epoch = 0;
  // one allocation: 64 doubles of scalars (the visit residuals from 32), the
  // visit log, then the FP64 residual's block partials
  LEPIC_HIP(hipMalloc(&ctx->d_scalar, kScalarBytes));
  LEPIC_HIP(hipMemsetAsync(ctx->d_scalar, 0, kScalarBytes, ctx->stream));
  ctx->d_partials = (double*)((char*)ctx->d_scalar + kPartialsOff);
  if (!ctx->h_report) {
    LEPIC_HIP(hipHostMalloc((void**)&ctx->h_report, 2 * sizeof(SolveReport), hipHostMallocMapped | hipHostMallocCoherent));
    std::memset((void*)ctx->h_report, 0, 2 * sizeof(SolveReport));
    LEPIC_HIP(hipHostGetDevicePointer((void**)&ctx->d_report, ctx->h_report, 0));
  }
  return 0;
}

void poisson_teardown(lepic_ctx* ctx) {
  for (int l = 1; l <= kMaxLevels; ++l) {
    Level& L = ctx->lv[l];
    for (int r = 1; r < kRot; ++r)
      if (L.rot[r]) (void)hipFree(L.rot[r]);
    if (L.partials) (void)hipFree(L.partials);
  }
  if (ctx->d_tail_bc) (void)hipFree(ctx->d_tail_bc);
  ctx->d_tail_bc = nullptr;
  ctx->tail_bc_cap = 0;
  ctx->tail_bc_key = -1;
}

int poisson_solve(lepic_ctx* ctx, double eps, int ncycl, int start, lepic_solve_info* info,
                  int32_t* log, int32_t log_cap) {
  const int ng = ctx->ng;
  const bool mixed = ctx->g.precision == LEPIC_MIXED;
  const int64_t n = ctx->nodes;
  const dim3 g1((unsigned)((n + 255) / 256));
  if (ng == 1 && mixed) return ctx->fail(LEPIC_ERR_UNSUPPORTED, "ng=1 runs in FP64 only");
  const double alpha = alpha_of(ctx);
  int visit[kVisitLog];
  double vres[kVisitLog];
  double res = 0.0, res_s = 0.0, ktot = 0.0;
  info->nlog = 0;
  info->start_used = start;
  info->res0_alt = -1.0;
  if (start == LEPIC_START_NET) {
    // the network's guess replaces the previous phi only if it lowers the
    // initial residual; otherwise the solve starts from the previous phi
    info->start_used = LEPIC_START_PREV;
    const int g = net_probe_due(ctx) ? net_guess(ctx, ctx->phi_given) : 1;
    if (g < 0) return g;
    if (g == 0) {
      double r_prev = 0.0, r_net = 0.0;
      if (int rc = launch_resid64(ctx, false)) return rc;
      if (int rc = read_report(ctx, visit, vres)) return rc;
      r_prev = ctx->h_report->resid;
      if (int rc = launch_resid64(ctx, false, ctx->phi_given)) return rc;
      if (int rc = read_report(ctx, visit, vres)) return rc;
      r_net = ctx->h_report->resid;
      net_probe_result(ctx, r_net > 0.0 ? r_prev / r_net : HUGE_VAL);
      if (r_net < r_prev) {
        hipLaunchKernelGGL(k_copy_interior, g1, dim3(256), 0, ctx->stream, ctx->phi,
                           (const double*)ctx->phi_given, (const int8_t*)ctx->bc, n);
        info->start_used = LEPIC_START_NET;
        info->res0_alt = r_prev / alpha;
      } else {
        info->res0_alt = r_net / alpha;
      }
    }
  } else if (start == LEPIC_START_COLD) {
    hipLaunchKernelGGL(k_cold_start, g1, dim3(256), 0, ctx->stream, ctx->phi, (const int8_t*)ctx->bc, n);
  } else if (start == LEPIC_START_GIVEN) {
    hipLaunchKernelGGL(k_copy_interior, g1, dim3(256), 0, ctx->stream, ctx->phi,
                       (const double*)ctx->phi_given, (const int8_t*)ctx->bc, n);
  }
  LEPIC_HIP(hipGetLastError());
  // residual of the starting guess; in mixed mode it also fills the FP32
  // right-hand side of the first correction equation
  // (the first V-cycle runs whatever it is, so nothing waits for it here)
  if (int rc = launch_resid64(ctx, mixed, nullptr, 1)) return rc;
  int k = 1;
  info->status = 0;
  // FP64 with a multi-block finest level: the buffer that holds its state
  // (the visits' sweeps add up), and the state's way back to phi
  int state = 0;
  auto settle = [&]() -> int {
    if (state == 0) return 0;
    hipLaunchKernelGGL(k_settle64, g1, dim3(256), 0, ctx->stream, ctx->phi, (const double*)ctx->lv[1].rot[state],
                       (const int8_t*)ctx->bc, n, ctx->d_ctrl + 1);
    LEPIC_HIP(hipGetLastError());
    return 0;
  };
  // mixed form: the next V-cycle's first visit is launched, the residual before
  // the V-cycle and the least that it is expected to leave of it
  bool begun = false;
  double r_last = 0.0, gain = 0.002;
  auto read_start = [&]() -> int {
    int v0[kVisitLog];
    double r0[kVisitLog];
    if (int rc = read_report(ctx, v0, r0, 1)) return rc;
    info->res0 = r_last = ctx->h_report[1].resid / alpha;
    return 0;
  };
  for (;;) {
    if (ng == 1 && ctx->lv[1].mb) {
      // red-black SOR alone on a multi-block grid (mg.f90:197-198 with
      // ng=1): the first call iterates to eps (up to 10^6 sweeps), later
      // calls do 10; launches go in batches with a host check in between
      const int nr = (k == 1) ? 1000000 : kNr;
      const int e = ++ctx->mg_epoch;
      int k0 = 0, ks = 0;
      VisitArgs A = visit_args(ctx, 1, e, 0, nr, alpha * eps);
      while (k0 < nr) {
        const int k_end = std::min(nr, k0 + 16 * kFirstMax);
        for (int kchk = 0; k0 < k_end; k0 += kFirstMax) {   // nr is a multiple of kFirstMax
          if (int rc = launch_sweeps(ctx, 1, A, k0, kFirstMax, kchk)) return rc;
          kchk = k0 + 1;
        }
        if (int rc = launch_finish64(ctx, visit_ref(ctx, 1, e, 0, nr, 1, alpha * eps, k0, k0 - kFirstMax,
                                                    kFirstMax))) return rc;
        if (int rc = read_report(ctx, visit, vres)) return rc;
        ks = ctx->h_report->status;
        if (ks) break;
      }
      if (!ks) return ctx->fail(LEPIC_ERR_STATE, "SOR visit did not finish");
    } else if (!mixed) {
      if (int rc = vcycle64(ctx, k, alpha * eps)) return rc;
      if (int rc = read_report(ctx, visit, vres)) return rc;
    } else {
      // FP32 correction V-cycle on the FP64 residual, then phi += e; the new
      // FP64 residual is both the convergence test and the next right-hand side
      if (int rc = vcycle32(ctx, k, alpha * eps, begun)) return rc;
      if (int rc = launch_resid64(ctx, true)) return rc;
      if (k == 1)
        if (int rc = read_start()) return rc;
      // The next V-cycle's first visit writes nothing that a solve that ends
      // here would keep, so it is launched before the report is read where
      // another V-cycle is as good as certain (a reduction of more than three
      // times the last V-cycle's would be needed to stop, or of 500 in the
      // first): it covers the host's wait and the launch's way to the device.
      // Per solve of two to four V-cycles on 128x128 256 -> 250 us, on
      // 1024x1024 630 -> 621 us.
      begun = k < ncycl && ctx->Lc > 1 && r_last * gain > eps;
      if (begun)
        if (int rc = tile_down(ctx, 1)) return rc;
      if (int rc = read_report(ctx, visit, vres)) return rc;
      vres[2 * ng - 1] = ctx->h_report->resid;
      const double r = ctx->h_report->resid / alpha;
      gain = 0.3 * r / r_last;
      r_last = r;
    }
    if (k == 1 && !mixed)
      if (int rc = read_start()) return rc;
    const int nvis = 2 * ng - 1;
    if (ctx->lv[1].mb && !mixed) state = (state + visit[1] + (ng > 1 ? visit[nvis] : 0)) % kRot;
    if (ng > 1)
      for (int l = 1; l < ctx->Lc; ++l) {
        Level& L = ctx->lv[l];
        if (!L.mb) continue;
        if (!mixed) {
          // one sweep more than last time: a spare sweep costs less than a
          // continuation launch when the count grows by one
          L.first_dn = std::min(std::max(visit[l] + 1, 2), kFirstMax);
          L.first_up = std::min(std::max(visit[2 * ng - l] + 1, 2), kFirstMax);
        } else {   // the mixed form's fixed counts
          visit[l] = l == 1 ? kFineDn : kFixDn;
          visit[2 * ng - l] = l == 1 ? kFineUp : kFixUp;
        }
      }
    for (int ig = 1; ig <= nvis; ++ig) {
      int l = ig < ng ? ig : (ig > ng ? 2 * ng - ig : ng);
      ktot += (double)visit[ig] / std::pow(2.0, 2 * (l - 1));
      if (log && info->nlog < log_cap) log[info->nlog] = visit[ig];
      info->nlog++;
    }
    res = vres[nvis] / alpha;
    if (k == 1) res_s = res;
    else if (std::fabs(res / res_s) > 10.0) {
      info->vcycles = k;
      info->res = res;
      if (int rc = settle()) return rc;
      return ctx->fail(LEPIC_ERR_DIVERGED, "PDE solver is diverging (iterative_solver.f90:42-49)");
    }
    if (res <= eps || k == ncycl) break;
    ++k;
  }
  if (int rc = settle()) return rc;
  info->vcycles = k;
  info->status = (res <= eps) ? 0 : 1;
  info->res = res;
  info->ktot = ktot;
  return net_after_solve(ctx);
}

}  // namespace lepic
