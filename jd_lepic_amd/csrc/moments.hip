// moments.hip -- averaged particle moments on the GPU: part_moments
// (utils.f90:1-136), calc_avg (utils.f90:138-265) and the phi/E averages
// of the main loop (main.f90:903-944).
//
// part_moments: one block per 1024-slot particle segment (the particle
// layout of the mover), thread t owning four consecutive slots; each
// particle adds k1*kq*w*(|v|^2, vx, vy, vz) to the four nodes around its
// half-step-back position on the grid coarsened by size_na.  Runs of
// particles in one coarse cell are summed in registers over a thread's
// slots, then over adjacent lanes (segmented DPP sums), go to an LDS window
// of coarse nodes around the segment's first particle and from there to the
// FP64 moment grid, one atomic per node and quantity of a segment.  A
// particle's cell and weights are the reference's bit for bit; the order of
// the sums differs from its serial loop, and k1 kq multiplies a run's sum
// instead of every term.  calc_avg and the phi/E averages are elementwise over
// nodes.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "lepic_internal.h"

using namespace lepic;

namespace {

struct MomArgs {
  const int32_t* seg;            // particles per segment
  // FP64 form
  const double *x, *y, *vx, *vy, *vz;
  // mixed form
  const int32_t* cell;
  const float *fx, *fy, *fvx, *fvy, *fvz;
  const int8_t* bc;              // fine bcnd: kq = 2 where bc != -1
  int n1, size_na, na1, na2;
  double h1, h2, xmax, ymax, half_dt, k1;
  ExactDiv d1, d2;               // the coarse cell's sides, size_na h
  double* pm;                    // (na2+1)(na1+1) x 4: |v|^2, vx, vy, vz
};

// LDS window of coarse nodes, kMomX0 columns left and kMomY0 rows below the
// segment's first particle: a sorted segment spans up to 1024 / (particles
// per cell) columns of one row and drifts a few cells between sorts; runs in
// cells outside go to the moment grid directly.  16 KB of LDS would let nine
// blocks on a CU; the registers (94) let five.
constexpr int kMomCols = 64, kMomRows = 8, kMomX0 = 8, kMomY0 = 3;
constexpr int kMomWin = kMomCols * kMomRows;

// a run's sums (corner, quantity) into the window or the moment grid, scaled
// by k1 and each corner's kq: at the fine node next to the coarse node's, as
// utils.f90:103-135 indexes it.  A factor 2 is exact, so it is applied to the
// sum instead of every particle.
__device__ __forceinline__ void mom_flush(const MomArgs& a, double (*win)[4], int wx0, int wy0, int ix, int iy,
                                          const double acc[16]) {
  const int ixf = a.size_na * ix - (a.size_na - 1), iyf = a.size_na * iy - (a.size_na - 1);
  const bool in = ix >= wx0 && ix + 1 < wx0 + kMomCols && iy >= wy0 && iy + 1 < wy0 + kMomRows;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const int dx = (c == 1 || c == 2) ? 1 : 0, dy = c >= 2 ? 1 : 0;
    const double k = (a.bc[(int64_t)(iyf + dy) * (a.n1 + 3) + ixf + dx] != -1 ? 2.0 : 1.0) * a.k1;
    if (in) {
      double* w = win[(iy + dy - wy0) * kMomCols + ix + dx - wx0];
#pragma unroll
      for (int q = 0; q < 4; ++q)
        __builtin_amdgcn_ds_atomic_fadd_f64((__attribute__((address_space(3))) double*)(w + q), k * acc[4 * c + q]);
    } else if (ix + dx <= a.na1 + 1 && iy + dy <= a.na2 + 1) {
      double* m = a.pm + 4 * ((int64_t)(iy + dy - 1) * (a.na1 + 1) + (ix + dx - 1));
#pragma unroll
      for (int q = 0; q < 4; ++q) atomic_add_f64(m + q, k * acc[4 * c + q]);
    }
  }
}

// one stage of the segmented sum: the values CTRL lanes back join the lanes
// whose run reaches them (one change of the active lanes for all sixteen)
template <int CTRL, int ROWS>
__device__ __forceinline__ void mom_stage(double acc[16], bool take) {
  double o[16];
#pragma unroll
  for (int c = 0; c < 16; ++c) o[c] = dpp_move<CTRL, ROWS>(acc[c]);
  if (take) {
#pragma unroll
    for (int c = 0; c < 16; ++c) acc[c] += o[c];
  }
}

// Bound by FP64 issue: about 90 operations a particle and 290 a wave of 256
// particles for the lane sums, against 24 B (mixed) or 40 B (FP64) read.
// 26.2e6 particles at 100 per cell, mixed, size_na 2: 0.213 ms, 2.95 TB/s of
// the 24 B a particle; 7.11 ms with 16 atomics on the moment grid per thread.
// The divisions by the cell's sides round as the reference's (a product with
// the rounded reciprocal, 0.205 ms, puts a particle on a coarse column in the
// cell below it now and then, and its place is 1.3 times less exact).
template <bool MIXED>
__global__ __launch_bounds__(kBlock) void k_part_moments(MomArgs a) {
  __shared__ double win[kMomWin][4];
  __shared__ int s_w[2];
  const int t = threadIdx.x, lane = t & 63;
  const int cnt = a.seg[blockIdx.x];
  if (cnt <= 0) return;          // block-uniform
  const int64_t i0 = (int64_t)blockIdx.x * kChunk + (int64_t)kItems * t;
  const int nv = min(max(cnt - kItems * t, 0), kItems);
  double X[kItems], Y[kItems], V[kItems][3];
  // the arrays are padded to whole segments: vector loads past the count stay inside
  if (MIXED) {
    const int4 c4 = *(const int4*)(a.cell + i0);
    const float4 fx4 = *(const float4*)(a.fx + i0), fy4 = *(const float4*)(a.fy + i0);
    const float4 u4 = *(const float4*)(a.fvx + i0), v4 = *(const float4*)(a.fvy + i0), w4 = *(const float4*)(a.fvz + i0);
    const int c[4] = {c4.x, c4.y, c4.z, c4.w};
    const float fx[4] = {fx4.x, fx4.y, fx4.z, fx4.w}, fy[4] = {fy4.x, fy4.y, fy4.z, fy4.w};
    const float u[4] = {u4.x, u4.y, u4.z, u4.w}, v[4] = {v4.x, v4.y, v4.z, v4.w}, w[4] = {w4.x, w4.y, w4.z, w4.w};
#pragma unroll
    for (int k = 0; k < kItems; ++k) {
      X[k] = ((double)((c[k] & 0xFFFF) - 1) + (double)fx[k]) * a.h1;
      Y[k] = ((double)((c[k] >> 16) - 1) + (double)fy[k]) * a.h2;
      V[k][0] = u[k]; V[k][1] = v[k]; V[k][2] = w[k];
    }
  } else {
#pragma unroll
    for (int k = 0; k < kItems; k += 2) {
      const double2 x2 = *(const double2*)(a.x + i0 + k), y2 = *(const double2*)(a.y + i0 + k);
      const double2 u2 = *(const double2*)(a.vx + i0 + k), v2 = *(const double2*)(a.vy + i0 + k);
      const double2 w2 = *(const double2*)(a.vz + i0 + k);
      X[k] = x2.x; X[k + 1] = x2.y; Y[k] = y2.x; Y[k + 1] = y2.y;
      V[k][0] = u2.x; V[k + 1][0] = u2.y; V[k][1] = v2.x; V[k + 1][1] = v2.y; V[k][2] = w2.x; V[k + 1][2] = w2.y;
    }
  }
  for (int e = t; e < 4 * kMomWin; e += kBlock) (&win[0][0])[e] = 0.0;
  if (t == 0) {
    s_w[0] = max((int)(X[0] * a.d1.r) + 1 - kMomX0, 1);
    s_w[1] = max((int)(Y[0] * a.d2.r) + 1 - kMomY0, 1);
  }
  __syncthreads();
  const int wx0 = s_w[0], wy0 = s_w[1];
  // running sum of consecutive particles in one coarse cell
  int cur = -1;
  double acc[16];                // [corner][|v|^2, vx, vy, vz]
#pragma unroll
  for (int c = 0; c < 16; ++c) acc[c] = 0.0;
  const int S = a.na1 + 3;
#pragma unroll
  for (int k = 0; k < kItems; ++k) {
    const double vx = V[k][0], vy = V[k][1], vz = V[k][2];
    const double xp = X[k] - vx * a.half_dt, yp = Y[k] - vy * a.half_dt;
    if (k >= nv || !(xp <= a.xmax && xp >= 0.0 && yp <= a.ymax && yp >= 0.0)) continue;
    const int ix = (int)div_finite(xp, a.d1) + 1, iy = (int)div_finite(yp, a.d2) + 1;
    const double px = div_finite(ix * a.d1.h - xp, a.d1), py = div_finite(iy * a.d2.h - yp, a.d2);
    const int key = iy * S + ix;
    if (key != cur) {
      if (cur >= 0) mom_flush(a, win, wx0, wy0, cur % S, cur / S, acc);
      cur = key;
#pragma unroll
      for (int c = 0; c < 16; ++c) acc[c] = 0.0;
    }
    const double e = vx * vx + vy * vy + vz * vz;
    const double ki[4] = {px * py, (1.0 - px) * py, (1.0 - px) * (1.0 - py), px * (1.0 - py)};
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      acc[4 * c] = fma(ki[c], e, acc[4 * c]);
      acc[4 * c + 1] = fma(ki[c], vx, acc[4 * c + 1]);
      acc[4 * c + 2] = fma(ki[c], vy, acc[4 * c + 2]);
      acc[4 * c + 3] = fma(ki[c], vz, acc[4 * c + 3]);
    }
  }
  // the run that ends the thread, over runs of equal cell in adjacent lanes
  const uint64_t act = __ballot(cur >= 0);
  if (act != 0) {                // wave-uniform
    const int kk = cur >= 0 ? cur : -2 - lane;
    const int kp = __shfl_up(kk, 1, 64);
    const uint64_t heads = __ballot(lane == 0 || kp != kk);
    if (__popcll(heads & act) != __popcll(act)) {
      const int s = 63 - __builtin_clzll(heads & ((2ull << lane) - 1ull));
      mom_stage<0x111, 0xf>(acc, lane - 1 >= s && (lane & 15) >= 1);
      mom_stage<0x112, 0xf>(acc, lane - 2 >= s && (lane & 15) >= 2);
      mom_stage<0x114, 0xf>(acc, lane - 4 >= s && (lane & 15) >= 4);
      mom_stage<0x118, 0xf>(acc, lane - 8 >= s && (lane & 15) >= 8);
      mom_stage<0x142, 0xa>(acc, (lane & 16) && (lane & ~15) - 1 >= s);
      mom_stage<0x143, 0xc>(acc, lane >= 32 && s <= 31);
    }
    const bool tail = lane == 63 || ((heads >> (lane + 1)) & 1ull);
    if (tail && cur >= 0) mom_flush(a, win, wx0, wy0, cur % S, cur / S, acc);
  }
  __syncthreads();
  for (int e = t; e < 4 * kMomWin; e += kBlock) {
    const double v = (&win[0][0])[e];
    const int nd = e >> 2, ix = wx0 + nd % kMomCols, iy = wy0 + nd / kMomCols;
    if (v != 0.0 && ix <= a.na1 + 1 && iy <= a.na2 + 1)
      atomic_add_f64(a.pm + 4 * ((int64_t)(iy - 1) * (a.na1 + 1) + (ix - 1)) + (e & 3), v);
  }
}

struct AvgArgs {
  const double* np;              // fine density of the species
  const double* sink;            // ss2D(2) of the species
  const double* src;             // ss2D(1) of the species
  const double* pm;
  const int8_t* bc;
  int n1, size_na, na1, na2;
  double mass_over_qe, k;        // mass/qe, Nm/Vc
  double* out;                   // data_pavg of the species: (na2+1)(na1+1) x 7
};

__global__ void k_calc_avg(AvgArgs a) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= (int64_t)(a.na1 + 1) * (a.na2 + 1)) return;
  const int ix = (int)(q % (a.na1 + 1)) + 1, iy = (int)(q / (a.na1 + 1)) + 1;
  const int64_t f = (int64_t)(a.size_na * iy - (a.size_na - 1)) * (a.n1 + 3) + (a.size_na * ix - (a.size_na - 1));
  const double* m = a.pm + 4 * q;
  double* o = a.out + 7 * q;
  const double n = a.np[f], jx = m[1], jy = m[2], jz = m[3];
  o[0] = o[0] + n;
  o[2] = o[2] + jx;
  o[3] = o[3] + jy;
  o[4] = o[4] + jz;
  double Tp = 0.0;
  if (n > 0) Tp = a.mass_over_qe * (1.0 / 3.0) * (m[0] / n - (jx * jx + jy * jy + jz * jz) / (n * n));
  if (Tp > 0) o[1] = o[1] + Tp;
  o[5] = o[5] + a.src[f] * a.k;
  o[6] = o[6] + a.sink[f] * a.k;
}

__global__ void k_phi_avg(const double* __restrict__ phi, const double* __restrict__ E, int64_t nodes,
                          double* __restrict__ out) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= nodes) return;
  out[3 * q] += phi[q];
  out[3 * q + 1] += E[2 * q];
  out[3 * q + 2] += E[2 * q + 1];
}

unsigned nblk(int64_t n) { return (unsigned)((n + 255) / 256); }


// ---- charge and energy totals ----------------------------------------------
constexpr int kTotBlocks = 1024;   // per-block partials, summed on the host in block order

// Block sum in a fixed order: waves by xor-shuffles, then the four wave sums
// in wave order.
__device__ __forceinline__ double block_sum256(double v, double* s_w) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  if ((threadIdx.x & 63) == 0) s_w[threadIdx.x >> 6] = v;
  __syncthreads();
  return s_w[0] + s_w[1] + s_w[2] + s_w[3];
}

// sum |v|^2 over the particles of one species (either layout); blocks stride
// over the segments, threads over a segment's slots
__global__ __launch_bounds__(256) void k_species_v2(const int32_t* __restrict__ seg, int64_t nseg,
                                                    const double* __restrict__ vx, const double* __restrict__ vy,
                                                    const double* __restrict__ vz, const float* __restrict__ fvx,
                                                    const float* __restrict__ fvy, const float* __restrict__ fvz,
                                                    double* __restrict__ partial) {
  __shared__ double s_w[4];
  double s = 0.0;
  for (int64_t g = blockIdx.x; g < nseg; g += gridDim.x) {
    const int cnt = seg[g];
    for (int j = threadIdx.x; j < cnt; j += 256) {
      const int64_t i = g * kChunk + j;
      double a, b, c;
      if (vx) { a = vx[i]; b = vy[i]; c = vz[i]; }
      else { a = fvx[i]; b = fvy[i]; c = fvz[i]; }
      s += a * a + b * b + c * c;
    }
  }
  const double t = block_sum256(s, s_w);
  if (threadIdx.x == 0) partial[blockIdx.x] = t;
}

// sum |E|^2 over the interior nodes (bcnd == -1)
__global__ __launch_bounds__(256) void k_field_e2(const double* __restrict__ E, const int8_t* __restrict__ bc,
                                                  int64_t nodes, double* __restrict__ partial) {
  __shared__ double s_w[4];
  double s = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < nodes; i += (int64_t)gridDim.x * 256)
    if (bc[i] == -1) s += E[2 * i] * E[2 * i] + E[2 * i + 1] * E[2 * i + 1];
  const double t = block_sum256(s, s_w);
  if (threadIdx.x == 0) partial[blockIdx.x] = t;
}

// launch one of the sums above with nb blocks and add the partials in order
template <typename Launch>
int sum_partials(lepic_ctx* ctx, int nb, Launch launch, double* out) {
  static_assert(kTotBlocks <= kPinnedDoubles, "partials fit the pinned scratch");
  if (!ctx->d_diag) LEPIC_HIP(hipMalloc(&ctx->d_diag, kTotBlocks * 8));
  launch(ctx->d_diag);
  LEPIC_HIP(hipGetLastError());
  LEPIC_HIP(hipMemcpyAsync(ctx->h_pinned, ctx->d_diag, (size_t)nb * 8, hipMemcpyDeviceToHost, ctx->stream));
  LEPIC_HIP(hipStreamSynchronize(ctx->stream));
  double t = 0.0;
  for (int b = 0; b < nb; ++b) t += ctx->h_pinned[b];
  *out = t;
  return 0;
}
}  // namespace

extern "C" {

int lepic_moments_reset(lepic_ctx* ctx) {
  if (!ctx) return LEPIC_ERR_ARG;
  Moments& M = ctx->mom;
  if (M.data) LEPIC_HIP(hipFree(M.data));
  if (M.phi) LEPIC_HIP(hipFree(M.phi));
  if (M.pm) LEPIC_HIP(hipFree(M.pm));
  M = Moments{};
  return 0;
}

int lepic_moments_accumulate(lepic_ctx* ctx, int32_t size_na) {
  if (!ctx || size_na < 1) return LEPIC_ERR_ARG;
  if (!ctx->boundary_set) return ctx->fail(LEPIC_ERR_STATE, "lepic_set_boundary not called");
  if (ctx->g.n1 % size_na || ctx->g.n2 % size_na)
    return ctx->fail(LEPIC_ERR_ARG, "size_na must divide n1 and n2 (read_input.f90:109-111)");
  Moments& M = ctx->mom;
  if (M.size_na && M.size_na != size_na)
    return ctx->fail(LEPIC_ERR_STATE, "size_na changed since the last reset");
  const int na1 = ctx->g.n1 / size_na, na2 = ctx->g.n2 / size_na;
  const int64_t nc = (int64_t)(na1 + 1) * (na2 + 1);
  if (!M.size_na) {
    M.size_na = size_na;
    LEPIC_HIP(hipMalloc(&M.data, (size_t)nc * 7 * ctx->nsp * 8));
    LEPIC_HIP(hipMalloc(&M.phi, (size_t)ctx->nodes * 3 * 8));
    LEPIC_HIP(hipMalloc(&M.pm, (size_t)nc * 4 * 8));
    if (int rc = zero_async(ctx, M.data, (size_t)nc * 7 * ctx->nsp * 8)) return rc;
    if (int rc = zero_async(ctx, M.phi, (size_t)ctx->nodes * 3 * 8)) return rc;
  }
  const bool mixed = ctx->g.precision == LEPIC_MIXED;
  for (int p = 0; p < ctx->nsp; ++p) {
    Species& s = ctx->sp[p];
    if (int rc = zero_async(ctx, M.pm, (size_t)nc * 4 * 8)) return rc;
    MomArgs a{};
    const int b = s.cur;
    a.seg = s.seg[b];
    if (mixed) {
      a.cell = s.cell[b];
      a.fx = s.f[b][0]; a.fy = s.f[b][1]; a.fvx = s.f[b][3]; a.fvy = s.f[b][4]; a.fvz = s.f[b][5];
    } else {
      a.x = s.d[b][0]; a.y = s.d[b][1]; a.vx = s.d[b][3]; a.vy = s.d[b][4]; a.vz = s.d[b][5];
    }
    a.bc = ctx->bc;
    a.n1 = ctx->g.n1; a.size_na = size_na; a.na1 = na1; a.na2 = na2;
    a.h1 = ctx->g.h1; a.h2 = ctx->g.h2;
    const double ha1 = size_na * ctx->g.h1, ha2 = size_na * ctx->g.h2;
    a.d1 = exact_div(ha1); a.d2 = exact_div(ha2);
    a.xmax = ctx->g.n1 * ctx->g.h1; a.ymax = ctx->g.n2 * ctx->g.h2;
    a.half_dt = ctx->g.dt / 2.0;
    a.k1 = s.Nm / (ha1 * ha2 * ctx->g.zmax);
    a.pm = M.pm;
    const int64_t nb = nseg_of(s);
    if (nb > 0) {
      if (mixed) hipLaunchKernelGGL(k_part_moments<true>, dim3((unsigned)nb), dim3(kBlock), 0, ctx->stream, a);
      else hipLaunchKernelGGL(k_part_moments<false>, dim3((unsigned)nb), dim3(kBlock), 0, ctx->stream, a);
      LEPIC_HIP(hipGetLastError());
    }
    AvgArgs g{};
    g.np = s.np; g.sink = s.sink; g.src = s.src; g.pm = M.pm; g.bc = ctx->bc;
    g.n1 = ctx->g.n1; g.size_na = size_na; g.na1 = na1; g.na2 = na2;
    g.mass_over_qe = s.mass / ctx->g.qe;
    g.k = s.Nm / (ctx->g.h1 * ctx->g.h2 * ctx->g.zmax);
    g.out = M.data + (size_t)p * nc * 7;
    hipLaunchKernelGGL(k_calc_avg, dim3(nblk(nc)), dim3(256), 0, ctx->stream, g);
    LEPIC_HIP(hipGetLastError());
    // ss2D = 0 after the average (main.f90:931, plt_src = 0)
    if (int rc = zero_async(ctx, s.sink, ctx->nodes * 8)) return rc;
    if (int rc = zero_async(ctx, s.src, ctx->nodes * 8)) return rc;
  }
  hipLaunchKernelGGL(k_phi_avg, dim3(nblk(ctx->nodes)), dim3(256), 0, ctx->stream, (const double*)ctx->phi,
                     (const double*)ctx->E, ctx->nodes, M.phi);
  LEPIC_HIP(hipGetLastError());
  M.count += 1;
  return 0;
}

int lepic_moments_get(lepic_ctx* ctx, double* data_pavg, double* phi_avg, int32_t* count) {
  if (!ctx) return LEPIC_ERR_ARG;
  Moments& M = ctx->mom;
  if (count) *count = M.count;
  if (!M.size_na) return (data_pavg || phi_avg) ? ctx->fail(LEPIC_ERR_STATE, "no moments accumulated") : 0;
  const int64_t nc = (int64_t)(ctx->g.n1 / M.size_na + 1) * (ctx->g.n2 / M.size_na + 1);
  if (data_pavg) {
    LEPIC_HIP(hipMemcpyAsync(data_pavg, M.data, (size_t)nc * 7 * ctx->nsp * 8, hipMemcpyDeviceToHost, ctx->stream));
  }
  if (phi_avg) {
    LEPIC_HIP(hipMemcpyAsync(phi_avg, M.phi, (size_t)ctx->nodes * 3 * 8, hipMemcpyDeviceToHost, ctx->stream));
  }
  LEPIC_HIP(hipStreamSynchronize(ctx->stream));
  return 0;
}

int lepic_species_totals(lepic_ctx* ctx, int32_t ptype, double* out) {
  if (!ctx || !out || ptype < 1 || ptype > ctx->nsp) return LEPIC_ERR_ARG;
  int64_t n = 0;
  if (int rc = lepic_get_count(ctx, ptype, &n)) return rc;
  Species& s = ctx->sp[ptype - 1];
  const int64_t nseg = nseg_of(s);
  double v2 = 0.0;
  if (nseg > 0) {
    const int nb = (int)std::min<int64_t>(nseg, kTotBlocks);
    const int b = s.cur;
    const bool mixed = ctx->g.precision == LEPIC_MIXED;
    if (int rc = sum_partials(ctx, nb, [&](double* part) {
          hipLaunchKernelGGL(k_species_v2, dim3(nb), dim3(256), 0, ctx->stream, (const int32_t*)s.seg[b], nseg,
                             mixed ? nullptr : (const double*)s.d[b][3], mixed ? nullptr : (const double*)s.d[b][4],
                             mixed ? nullptr : (const double*)s.d[b][5], mixed ? (const float*)s.f[b][3] : nullptr,
                             mixed ? (const float*)s.f[b][4] : nullptr, mixed ? (const float*)s.f[b][5] : nullptr,
                             part);
        }, &v2))
      return rc;
  }
  out[0] = (double)n;
  out[1] = 0.5 * s.Nm * s.mass * v2;
  out[2] = s.Nm * s.charge * (double)n;
  return 0;
}

int lepic_field_energy(lepic_ctx* ctx, double* W) {
  if (!ctx || !W) return LEPIC_ERR_ARG;
  if (!ctx->boundary_set) return ctx->fail(LEPIC_ERR_STATE, "lepic_set_boundary not called");
  const int nb = (int)std::min<int64_t>((ctx->nodes + 255) / 256, kTotBlocks);
  double e2 = 0.0;
  if (int rc = sum_partials(ctx, nb, [&](double* part) {
        hipLaunchKernelGGL(k_field_e2, dim3(nb), dim3(256), 0, ctx->stream, (const double*)ctx->E,
                           (const int8_t*)ctx->bc, ctx->nodes, part);
      }, &e2))
    return rc;
  *W = 0.5 * ctx->g.eps0 * e2 * ctx->g.h1 * ctx->g.h2 * ctx->g.zmax;
  return 0;
}

}  // extern "C"

