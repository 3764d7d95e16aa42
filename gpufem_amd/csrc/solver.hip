// ELL SpMV and the Jacobi-preconditioned CG in FP64.
//
// Rows are visited in 256-row tiles in grid-stride order, with workgroup
// ids remapped so that each XCD (workgroups are dispatched round-robin over
// the 8 XCDs) owns a contiguous part of every window of tiles: the
// x-gathers of neighbouring rows then hit the same L2.
//
// SpMV variants (chosen per matrix by the tuner in solve.cpp):
//   kThreadU1/U4/U8  one thread per row, slots streamed 1/4/8 at a time
//                    (more loads in flight per thread); same summation
//                    order as the reference's Axy, so all three are bitwise
//                    identical.
//   kTile2/kTile4    2 or 4 waves share a 64-row tile, each taking every
//                    2nd/4th slot; partial sums combined through LDS.
//   kNode2/kNode3    thread per row over the d x d node blocks of a 2D / 3D
//                    FEM matrix: one node column per d slots and the d
//                    entries of x read together (fewer loads, 4/d instead of
//                    4 column bytes per entry); bitwise equal to kThreadU1.
//   kBsell2/kBsell3  thread per node row of the block-sliced copy, four
//                    slices per workgroup in grid-stride sweeps.
//   kBsell2G/3G      the same with one workgroup per four-slice group (one
//                    sweep; the dispatcher balances unequal slices).
//
// Inside an iteration the slice-group variants run the split kernels while the
// matrix stays in the last-level cache (iter_variant).
//
// CG schedules: three launches per iteration (k_spmv_pq, k_update,
// k_direction), or two (k_split_product, k_split_update; k_split_check after a
// chunk of them), with all scalars in a device PcgState, so the host can
// enqueue or graph-replay chunks of iterations; or one cooperative
// persistent kernel (k_pcg_persistent, k_split_persistent) with a grid barrier
// after each of those steps.  A small system takes hundreds of iterations in one
// launch of one workgroup under any schedule (k_single).  Every block reduces the per-block partials in the same fixed
// order, so all blocks take the same convergence decision and results are
// bitwise reproducible for a given matrix and variant.  The SpMV kernel may
// run on a grid of its own (the slice-group variants): k_update reduces its
// spmv_grid p.q partials, and the persistent kernel plays the same logical
// SpMV workgroups in turn.  No workgroup waits on another inside a kernel
// but the persistent one: on gfx950 an agent-scope release writes back the
// XCD's L2, far too costly once per workgroup per SpMV.
#include <algorithm>

#include "device_common.hpp"
#include "gf_internal.hpp"
#include "launch.hpp"

namespace gf {

struct PcgState {
  double rho[2];  // r.z, double-buffered by iteration parity
  double rr;      // r.r after the last update
  double bnorm2;  // b.b
  double rtol2;   // rtol^2
  // two-launch iteration: iterations done, by parity (a launch of parity P
  // reads itv[P] and writes itv[P ^ 1], rho[P] likewise: no workgroup of it
  // can see the value it leaves); it: the count at the last check
  int32_t itv[2];
  int32_t it;
  int32_t done;
  int32_t status;
  int32_t maxit;
};

struct GridBarrier {
  unsigned long long count;  // arrivals since the launch began (monotonic)
  int abort;
  int pad;
};

namespace {

using namespace dev;

// ---------------------------------------------------------------------------
// standalone SpMV (multi-RHS by repeated sweeps)
// ---------------------------------------------------------------------------
template <int V>
__global__ __launch_bounds__(kNT) void k_spmv(int64_t n, const double* __restrict__ val,
                                              const int32_t* __restrict__ col,
                                              const int32_t* __restrict__ rownnz,
                                              const double* __restrict__ x,
                                              double* __restrict__ y, BsellView bs) {
  for_rows_spmv<V, double>(logical_block(), gridDim.x, n, val, col, rownnz, x,
                           [&](int64_t i, double v) { y[i] = v; }, bs);
}

// block-sliced copy: node columns (padding blocks point at the row's own
// node, whose x entries exist) and values (padding blocks are zero)
__global__ void k_bsell_cols(BsellView bs, int d, int64_t n, const int32_t* __restrict__ col,
                             const int32_t* __restrict__ rownnz, int32_t* __restrict__ bcol) {
  for (int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; t < bs.nslices * 64;
       t += int64_t(gridDim.x) * blockDim.x) {
    const int64_t sl = t >> 6;
    const int lane = int(t & 63);
    const int32_t R = bs.perm[t];
    const int64_t b0 = bs.sptr[sl], w = bs.sptr[sl + 1] - b0;
    const int32_t cnt = R >= 0 ? rownnz[int64_t(d) * R] / d : 0;
    for (int64_t j = 0; j < w; ++j)
      bcol[(b0 + j) * 64 + lane] =
          j < cnt ? col[int64_t(d) * R + j * d * n] / d : (R >= 0 ? R : 0);
  }
}

__global__ void k_bsell_offsets(BsellView bs, const int32_t* __restrict__ bcol,
                                int16_t* __restrict__ coff, int* overflow) {
  for (int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; t < bs.nslices * 64;
       t += int64_t(gridDim.x) * blockDim.x) {
    const int64_t sl = t >> 6;
    const int lane = int(t & 63);
    const int32_t R = bs.perm[t];
    const int32_t base = R >= 0 ? R : 0;
    const int64_t b0 = bs.sptr[sl], w = bs.sptr[sl + 1] - b0;
    bool bad = false;
    for (int64_t j = 0; j < w; ++j) {
      const int32_t d = bcol[(b0 + j) * 64 + lane] - base;
      bad |= d < -32768 || d > 32767;
      coff[(b0 + j) * 64 + lane] = int16_t(d);
    }
    if (bad) atomicOr(overflow, 1);
  }
}

__global__ void k_bsell_vals(BsellView bs, int d, int64_t n, const double* __restrict__ val,
                             const int32_t* __restrict__ rownnz, double* __restrict__ bval) {
  for (int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; t < bs.nslices * 64;
       t += int64_t(gridDim.x) * blockDim.x) {
    const int64_t sl = t >> 6;
    const int lane = int(t & 63);
    const int32_t R = bs.perm[t];
    const int64_t b0 = bs.sptr[sl], w = bs.sptr[sl + 1] - b0;
    const int32_t cnt = R >= 0 ? rownnz[int64_t(d) * R] / d : 0;
    for (int64_t j = 0; j < w; ++j)
      for (int r = 0; r < d; ++r)
        for (int e = 0; e < d; ++e)
          bval[bsell_vidx(d * d, b0 + j, r * d + e, lane)] =
              j < cnt ? val[int64_t(d) * R + r + (j * d + e) * n] : 0.0;
  }
}

// The inverse: the ELL values of the live slots from the block-sliced copy
// (padding slots of the ELL rows keep their zeros).
__global__ void k_bsell_to_ell(BsellView bs, int d, int64_t n, const double* __restrict__ bval,
                               const int32_t* __restrict__ rownnz, double* __restrict__ val) {
  for (int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; t < bs.nslices * 64;
       t += int64_t(gridDim.x) * blockDim.x) {
    const int64_t sl = t >> 6;
    const int lane = int(t & 63);
    const int32_t R = bs.perm[t];
    if (R < 0) continue;
    const int64_t b0 = bs.sptr[sl];
    const int32_t cnt = rownnz[int64_t(d) * R] / d;
    for (int64_t j = 0; j < cnt; ++j)
      for (int e = 0; e < d; ++e)
        for (int r = 0; r < d; ++r)
          val[int64_t(d) * R + r + (j * d + e) * n] = bval[bsell_vidx(d * d, b0 + j, r * d + e, lane)];
  }
}

__global__ void k_build_coln(int64_t n, int32_t nbw, int d, const int32_t* col, int32_t* coln) {
  const int64_t total = n * nbw;
  for (int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; t < total;
       t += int64_t(gridDim.x) * blockDim.x) {
    const int64_t j = t / n, i = t - j * n;
    coln[t] = col[i + j * d * n] / d;
  }
}

// plain streaming copy, 16 bytes per thread per step (the bandwidth probe)
typedef double v2d __attribute__((ext_vector_type(2)));
__global__ __launch_bounds__(kNT) void k_stream_copy(const v2d* __restrict__ src,
                                                     v2d* __restrict__ dst, int64_t n16) {
  for (int64_t i = int64_t(blockIdx.x) * kNT + threadIdx.x; i < n16; i += int64_t(gridDim.x) * kNT)
    dst[i] = __builtin_nontemporal_load(src + i);
}

__global__ void k_jacobi_inv(int64_t n, const double* val, const int32_t* diag, double* dinv) {
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += int64_t(gridDim.x) * blockDim.x) {
    const int32_t s = diag[i];
    const double d = s >= 0 ? val[i + int64_t(s) * n] : 0.0;
    dinv[i] = 1.0 / d;
  }
}

// ---------------------------------------------------------------------------
// PCG phases (shared by the multi-launch and the persistent schedules)
// ---------------------------------------------------------------------------
// q = K p over the rows of logical SpMV workgroup lb of nlb; returns this
// thread's part of p.q
template <int V>
__device__ inline double phase_spmv_pq(const PcgBuffers& B, int lb, int nlb) {
  double pq = 0.0;
  for_rows_spmv<V, double>(lb, nlb, B.n, B.val, B.col, B.rownnz, B.p, [&](int64_t i, double qi) {
    B.q[i] = qi;
    pq += B.p[i] * qi;
  }, B.bs);
  return pq;
}

__device__ inline void phase_update(const PcgBuffers& B, double alpha, double* rz_out,
                                    double* rr_out) {
  double rz = 0, rr = 0;
  for_my_rows(B.n, [&](int64_t i) {
    B.x[i] += alpha * B.p[i];
    const double ri = B.r[i] - alpha * B.q[i];
    const double zi = B.dinv ? B.dinv[i] * ri : ri;
    B.r[i] = ri;
    B.z[i] = zi;
    rz += ri * zi;
    rr += ri * ri;
  });
  *rz_out = rz;
  *rr_out = rr;
}

__device__ inline void phase_direction(const PcgBuffers& B, double beta) {
  for_my_rows(B.n, [&](int64_t i) { B.p[i] = B.z[i] + beta * B.p[i]; });
}

// ---------------------------------------------------------------------------
// The two-launch iteration (split variants).  The direction is never stored on
// its own: the product forms p_k = z_k + beta_k p_{k-1} in its gathers and the
// update forms it again for its own rows, which then hold (z_{k+1}, p_k) in
// place; beta comes from the same sums, in the same order and with the same
// rounding as in a direction pass of its own.  An iteration, with the split
// product, against the three launches before: Brick8 64x32x32 37.0 / 43.6 us,
// Q8 512x256 53.6 / 66.0, Q8 201x67 13.2 / 18.9, Q4 64x32 9.8 / 13.5, Brick20
// 24^3 61 / 64.  A matrix that streams from memory keeps the three launches:
// there the second gather costs 23 us a product (Brick8 96^3), more than the
// direction pass it saves.
// ---------------------------------------------------------------------------
// The product's slices from `first` on in steps of nlb, `waves` waves; wave 0's
// lanes return their part of p.q
template <int D>
__device__ inline double phase_split(const PcgBuffers& B, SplitSlice first, int nlb, int waves,
                                     double beta) {
  double pq = 0.0;
  const LazyDirection<D> p{B.z, B.p, B.n / D, beta};
  double* __restrict__ q = B.q;
  for_rows_split<D>(first, nlb, waves, B.bs, B.val, B.col, p, [&](int32_t R, const double* acc) {
#pragma unroll
    for (int r = 0; r < D; ++r) {
      q[int64_t(D) * R + r] = acc[r];
      pq += p.at(R, r) * acc[r];
    }
  });
  return pq;
}

// kRows rows of a thread at a time: the loads of the first ones are issued
// before the scalars of the iteration are known (their latency and the
// reduction's overlap).  Row i = D node + e of the solver's vectors is entry
// e * nodes + node of z and p.
constexpr int kRows = 4;
struct SplitRows {
  double x[kRows], z[kRows], p[kRows], r[kRows], q[kRows], d[kRows];
};
template <int D>
__device__ inline void split_load(const PcgBuffers& B, int64_t base, int64_t stride, SplitRows* v) {
#pragma unroll
  for (int u = 0; u < kRows; ++u) {
    const int64_t i = base + u * stride;
    if (i < B.n) {
      const int64_t k = lazy_index<D>(i, B.n);
      v->z[u] = B.z[k];
      v->p[u] = B.p[k];
      v->x[u] = B.x[i];
      v->r[u] = B.r[i];
      v->q[u] = B.q[i];
      v->d[u] = B.dinv ? B.dinv[i] : 1.0;
    }
  }
}
// x += alpha p; r -= alpha q; z = M^-1 r over the rows of logical workgroup lb
// (the first ones already in v); the sums r.z and r.r of it to part2[slot]
template <int D>
__device__ inline void phase_split_update(const PcgBuffers& B, int lb, int slot, double alpha,
                                          double beta, SplitRows& v, double* sh) {
  double rz = 0.0, rr = 0.0;
  const int64_t stride = int64_t(B.nblocks) * kNT;
  for (int64_t base = int64_t(lb) * kNT + threadIdx.x;;) {
#pragma unroll
    for (int u = 0; u < kRows; ++u) {
      const int64_t i = base + u * stride;
      if (i < B.n) {
        const int64_t k = lazy_index<D>(i, B.n);
        const double pi = v.z[u] + beta * v.p[u];
        const double ri = v.r[u] - alpha * v.q[u];
        const double zi = B.dinv ? v.d[u] * ri : ri;
        B.x[i] = v.x[u] + alpha * pi;
        B.r[i] = ri;
        B.z[k] = zi;
        B.p[k] = pi;
        rz += ri * zi;
        rr += ri * ri;
      }
    }
    base += kRows * stride;
    if (base >= B.n) break;
    split_load<D>(B, base, stride, &v);
  }
  block_sum2(&rz, &rr, sh);
  if (threadIdx.x == 0) {
    B.part2[slot] = rz;
    B.part2[B.nblocks + slot] = rr;
  }
}

// Whether iteration `it` runs, from the residual sum every workgroup forms in
// the same order; `lead` sets the state when it does not.
__device__ inline bool split_goes_on(const PcgBuffers& B, int it, double rr, bool lead) {
  PcgState* st = B.st;
  if (!(rr <= st->rtol2 * st->bnorm2) && it < st->maxit) return true;
  if (lead) {
    st->rr = rr;
    st->it = it;
    st->done = 1;
  }
  return false;
}
// The iteration that breaks down reports its own residual: nothing has written
// the partials of r.r since (every workgroup finds the same p.q and leaves).
__device__ inline void split_breakdown(const PcgBuffers& B, int it, double* sh) {
  if (blockIdx.x != 0) return;
  const double rr = reduce_partials(B.part2 + B.nblocks, B.nblocks, sh);
  if (threadIdx.x != 0) return;
  B.st->rr = rr;
  B.st->it = it;
  B.st->status = GF_ERR_BREAKDOWN;
  B.st->done = 1;
}
// First launch: the stopping test, beta and q = K p.  `done` changes inside a
// launch only when none of its workgroups writes a vector, so one that starts
// late and reads it set leaves nothing undone.
// Every load that waits for nothing is issued before the first wait (the flag
// included: a finished state costs the loads of one launch).
template <int D>
__global__ __launch_bounds__(64 * split_parts(D), D == 2 ? 6 : 4) void k_split_product(
    PcgBuffers B, int parity) {
  PcgState* st = B.st;
  __shared__ double sh[2 * (kNT / 64)];
  const bool lead = blockIdx.x == 0 && threadIdx.x == 0;
  const SplitSlice first = split_slice(logical_block(), B.bs);
  const int it = st->itv[parity], done = st->done;
  const double rz_old = st->rho[parity ^ 1];
  double rz, rr;
  reduce_partials2(B.part2, B.part2 + B.nblocks, B.nblocks, &rz, &rr, sh);
  if (done || !split_goes_on(B, it, rr, lead)) return;
  if (lead) st->rho[parity] = rz;
  const double beta = split_beta(it, rz, rz_old);
  store_wave_sum(phase_split<D>(B, first, gridDim.x, split_parts(D), beta), B.part1 + blockIdx.x);
}

// Second launch: alpha and the vector updates.
template <int D>
__global__ __launch_bounds__(kNT) void k_split_update(PcgBuffers B, int parity) {
  PcgState* st = B.st;
  __shared__ double sh[2 * (kNT / 64)];
  SplitRows v;
  const int lb = logical_block();
  split_load<D>(B, int64_t(lb) * kNT + threadIdx.x, int64_t(B.nblocks) * kNT, &v);
  const bool lead = blockIdx.x == 0 && threadIdx.x == 0;
  const int it = st->itv[parity], done = st->done;
  const double rho = st->rho[parity], beta = split_beta(it, rho, st->rho[parity ^ 1]);
  const double pq = reduce_partials(B.part1, B.spmv_grid, sh);
  if (done) return;
  if (!(pq > 0.0)) return split_breakdown(B, it, sh);
  phase_split_update<D>(B, lb, blockIdx.x, rho / pq, beta, v, sh);
  if (lead) st->itv[parity ^ 1] = it + 1;
}

// The state the host reads: the last residual checked as the next iteration
// (of this parity) would check it.
__global__ __launch_bounds__(kNT) void k_split_check(PcgBuffers B, int parity) {
  if (B.st->done) return;
  __shared__ double sh[kNT / 64];
  const double rr = reduce_partials(B.part2 + B.nblocks, B.nblocks, sh);
  if (threadIdx.x == 0) {
    PcgState* st = B.st;
    st->rr = rr;
    st->it = st->itv[parity];
    (void)split_goes_on(B, st->it, rr, true);
  }
}

// ---------------------------------------------------------------------------
// Small systems in one workgroup (single_fits): `count` iterations a launch, p,
// q and x in LDS, r and 1 / diagonal in registers, four workgroup barriers an
// iteration and no other synchronisation (two launches of anything take 7 us).
// Eight waves take equal runs of the matrix's block slots.  What bounds it is
// one CU's path to the L2 (64 bytes a clock): each wave keeps the first kHeld
// slots of its run in registers for the whole launch and streams the others,
// U in flight at any time and across iterations.  Q4 64x32, 7.2 us an iteration
// (9.8 in two launches): 2.3 of reductions, barriers and vector steps, 4 of
// streaming 0.48 MB, the rest of adding; 9.9 with no loads in flight across
// steps.  A slice that several waves share is summed in wave order, and p.q is
// taken from whole rows: summed over the waves' partial rows, which cancel, it
// cost a slender plate 7 of 81 iterations.
// ---------------------------------------------------------------------------
constexpr int kSingleWaves = 8;

// v plus the value `ctrl` lanes back (row_shr, row_bcast), in the lanes that
// have one
template <int CTRL, int ROWS>
__device__ inline double dpp_add(double v) {
  const int64_t b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, int(b), CTRL, ROWS, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, int(b >> 32), CTRL, ROWS, 0xf, false);
  return v + __longlong_as_double((int64_t(hi) << 32) | uint32_t(lo));
}
// a wave's sum, in lane 63: register moves (a shuffle is a trip through the LDS)
__device__ inline double wave_sum63(double v) {
  v = dpp_add<0x111, 0xf>(v);
  v = dpp_add<0x112, 0xf>(v);
  v = dpp_add<0x114, 0xf>(v);
  v = dpp_add<0x118, 0xf>(v);
  v = dpp_add<0x142, 0xa>(v);
  return dpp_add<0x143, 0xc>(v);
}
template <int D>
constexpr int kHeld = D == 2 ? 12 : 5;

template <int D>
__global__ __launch_bounds__(64 * kSingleWaves) __attribute__((amdgpu_waves_per_eu(2, 2))) void
k_single(PcgBuffers B, int count) {
  constexpr int W = kSingleWaves, DD = D * D, H = kHeld<D>, U = D == 2 ? 4 : 2;
  constexpr int SL = kSingleSlices<D>;  // of the matrix, at most
  constexpr int SW = SL / W;            // of a wave's vector rows
  static_assert(SL % W == 0, "equal shares");
  __shared__ double p_[SL * 64 * D];    // by row
  __shared__ double q_[SL][D][64];      // by position
  __shared__ double x_[SL][D][64];
  __shared__ double edge[W][D][64];     // of the slice a wave takes over from the one before
  __shared__ int64_t s_ptr[SL + 1];
  __shared__ int s_edge[W];             // its slice, or -1
  __shared__ double red[3][W];
  PcgState* st = B.st;
  if (st->done) return;
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
  const int ns = int(B.bs.nslices);
  for (int s = threadIdx.x; s <= ns; s += 64 * W) s_ptr[s] = B.bs.sptr[s];
  // this wave's vector rows: lane of slices w, w + W, ...
  int32_t R[SW];
  double r[SW][D], d[SW][D];
#pragma unroll
  for (int k = 0; k < SW; ++k) {
    const int s = w + k * W;
    R[k] = s < ns ? B.bs.perm[s * 64 + lane] : -1;
    if (s >= ns) continue;
#pragma unroll
    for (int e = 0; e < D; ++e) {
      const int64_t i = int64_t(D) * (R[k] >= 0 ? R[k] : 0) + e;
      r[k][e] = R[k] >= 0 ? B.r[i] : 0.0;
      d[k][e] = B.dinv && R[k] >= 0 ? B.dinv[i] : 1.0;
      x_[s][e][lane] = R[k] >= 0 ? B.x[i] : 0.0;
      q_[s][e][lane] = 0.0;  // slices without blocks
      if (R[k] >= 0) p_[i] = B.p[i];
    }
  }
  __syncthreads();
  // this wave's run of block slots, and the slice it begins in
  const int64_t T = s_ptr[ns], b0 = T * w / W, b1 = T * (w + 1) / W;
  int first = 0;
  while (first < ns && s_ptr[first + 1] <= b0) ++first;
  if (lane == 0) s_edge[w] = first < ns && b1 > b0 && s_ptr[first] < b0 ? first : -1;
  double hv[H][DD];
  int32_t hc[H];
#pragma unroll
  for (int k = 0; k < H; ++k) {
    if (b0 + k < b1) {
      load_block<D, double, false>(B.val, b0 + k, lane, hv[k]);
      hc[k] = B.col[(b0 + k) * 64 + lane];
    }
  }
  // the streamed ones: U in flight
  const int64_t bs0 = b0 + H;
  double sv[U][DD];
  int32_t sc[U];
  auto fetch = [&](int u, int64_t b) {
    b = b < b1 ? b : b1 - 1;
    load_block<D, double, false>(B.val, b, lane, sv[u]);
    sc[u] = B.col[b * 64 + lane];
  };
  if (bs0 < b1) {
#pragma unroll
    for (int u = 0; u < U; ++u) fetch(u, bs0 + u);
  }
  __syncthreads();  // s_edge
  uint32_t edges[SW];  // waves whose edge belongs to this wave's slices
#pragma unroll
  for (int k = 0; k < SW; ++k) {
    edges[k] = 0;
#pragma unroll
    for (int j = 1; j < W; ++j)
      if (s_edge[j] == w + k * W) edges[k] |= 1u << j;
    edges[k] = __builtin_amdgcn_readfirstlane(edges[k]);
  }
  double rho = st->rho[0], rr = st->rr;
  int it = st->it, status = GF_OK, done = 0;
  const int maxit = st->maxit;
  const double tol2 = st->rtol2 * st->bnorm2;
  // sum of a value over the workgroup, the same in every thread
  auto leave = [&](int j, double v) {
    v = wave_sum63(v);
    if (lane == 63) red[j][w] = v;
  };
  auto total = [&](int j) {
    double t = 0.0;
#pragma unroll
    for (int k = 0; k < W; ++k) t += red[j][k];
    return t;
  };
  for (int left = count; left > 0; --left) {
    __syncthreads();  // p
    double acc[D];
#pragma unroll
    for (int e = 0; e < D; ++e) acc[e] = 0.0;
    int s = first;
    int64_t end = first < ns ? s_ptr[first + 1] : 0;
    // a slice is summed, or this wave's part of it
    auto flush = [&]() {
      double* out = s_ptr[s] >= b0 ? &q_[s][0][lane] : &edge[w][0][lane];
#pragma unroll
      for (int e = 0; e < D; ++e) {
        out[e * 64] = acc[e];
        acc[e] = 0.0;
      }
    };
    auto next = [&](int64_t b) {
      if (b < end) return;
      flush();
      do end = s_ptr[++s + 1];
      while (end <= b);
    };
    auto add = [&](const double* v, int32_t c) {
#pragma unroll
      for (int f = 0; f < D; ++f) {
        const double xv = p_[D * c + f];
#pragma unroll
        for (int e = 0; e < D; ++e) acc[e] += v[e * D + f] * xv;
      }
    };
#pragma unroll
    for (int k = 0; k < H; ++k) {
      if (b0 + k < b1) {
        next(b0 + k);
        add(hv[k], hc[k]);
      }
    }
    for (int64_t b = bs0; b < b1; b += U) {
      // the buffer of a slot takes the one U further on as soon as it is used
      // up, at the end of the run the first ones of the next iteration
      const int64_t ahead = b + U < b1 ? b + U : bs0;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (b + u < b1) {
          next(b + u);
          add(sv[u], sc[u]);
        }
        fetch(u, ahead + u);
      }
    }
    if (b1 > b0) flush();
    __syncthreads();
    // p.q from the whole sums of a row, which the residual takes too
    double pq = 0.0;
#pragma unroll
    for (int k = 0; k < SW; ++k) {
      const int sk = w + k * W;
      if (R[k] < 0) continue;
#pragma unroll
      for (int e = 0; e < D; ++e) {
        double q = q_[sk][e][lane];
        if (edges[k]) {
          for (uint32_t m = edges[k]; m; m &= m - 1) q += edge[__builtin_ctz(m)][e][lane];
          q_[sk][e][lane] = q;
        }
        pq += p_[D * R[k] + e] * q;
      }
    }
    leave(0, pq);
    __syncthreads();
    pq = total(0);
    if (!(pq > 0.0)) {
      status = GF_ERR_BREAKDOWN;
      done = 1;
      break;
    }
    const double alpha = rho / pq;
    double rz = 0.0;
    rr = 0.0;
#pragma unroll
    for (int k = 0; k < SW; ++k) {
      const int sk = w + k * W;
      if (R[k] < 0) continue;
#pragma unroll
      for (int e = 0; e < D; ++e) {
        x_[sk][e][lane] += alpha * p_[D * R[k] + e];
        r[k][e] -= alpha * q_[sk][e][lane];
        rz += r[k][e] * (d[k][e] * r[k][e]);
        rr += r[k][e] * r[k][e];
      }
    }
    leave(1, rz);
    leave(2, rr);
    __syncthreads();
    rz = total(1);
    rr = total(2);
    ++it;
    if (rr <= tol2 || it >= maxit) {
      done = 1;
      break;
    }
    const double beta = rz / rho;
    rho = rz;
#pragma unroll
    for (int k = 0; k < SW; ++k) {
      if (R[k] < 0) continue;
#pragma unroll
      for (int e = 0; e < D; ++e)
        p_[D * R[k] + e] = d[k][e] * r[k][e] + beta * p_[D * R[k] + e];
    }
  }
#pragma unroll
  for (int k = 0; k < SW; ++k) {
    if (R[k] < 0) continue;
#pragma unroll
    for (int e = 0; e < D; ++e) {
      const int64_t i = int64_t(D) * R[k] + e;
      B.x[i] = x_[w + k * W][e][lane];
      B.r[i] = r[k][e];
      B.p[i] = p_[i];
    }
  }
  if (threadIdx.x == 0) {
    st->rho[0] = rho;
    st->rr = rr;
    st->it = it;
    st->status = status;
    st->done = done;
  }
}

// r = b - q (use_x0) or x = 0, r = b; z = M^-1 r; p = z; partials r.z, r.r, b.b
// (SOA > 1: z in the two-launch iteration's order, its p_old = 0)
template <int SOA>
__global__ __launch_bounds__(kNT) void k_pcg_init(PcgBuffers B, int use_x0) {
  __shared__ double sh[kNT / 64];
  double rz = 0, rr = 0, bb = 0;
  for_my_rows(B.n, [&](int64_t i) {
    const double bi = B.b[i];
    double ri;
    if (use_x0) {
      ri = bi - B.q[i];
    } else {
      B.x[i] = 0.0;
      ri = bi;
    }
    const double zi = B.dinv ? B.dinv[i] * ri : ri;
    B.r[i] = ri;
    if constexpr (SOA > 1) {
      const int64_t k = lazy_index<SOA>(i, B.n);
      B.z[k] = zi;
      B.p[k] = 0.0;
    } else {
      B.z[i] = zi;
      B.p[i] = zi;
    }
    rz += ri * zi;
    rr += ri * ri;
    bb += bi * bi;
  });
  rz = block_sum(rz, sh);
  rr = block_sum(rr, sh);
  bb = block_sum(bb, sh);
  if (threadIdx.x == 0) {
    B.part2[blockIdx.x] = rz;
    B.part2[gridDim.x + blockIdx.x] = rr;
    B.part2[2 * gridDim.x + blockIdx.x] = bb;
  }
}

__global__ __launch_bounds__(kNT) void k_pcg_init_finish(PcgBuffers B, int nb, double rtol2,
                                                         int maxit) {
  __shared__ double sh[kNT / 64];
  const double rz = reduce_partials(B.part2, nb, sh);
  const double rr = reduce_partials(B.part2 + nb, nb, sh);
  const double bb = reduce_partials(B.part2 + 2 * nb, nb, sh);
  if (threadIdx.x == 0) {
    PcgState* st = B.st;
    st->rho[0] = rz;
    st->rho[1] = 0.0;
    st->rr = rr;
    st->bnorm2 = bb;
    st->rtol2 = rtol2;
    st->itv[0] = st->itv[1] = st->it = 0;
    st->status = GF_OK;
    st->maxit = maxit;
    st->done = (rr <= rtol2 * bb) || maxit <= 0;
  }
}

template <int V>
__global__ __launch_bounds__(kNT) void k_spmv_pq(PcgBuffers B) {
  if (B.st->done) return;
  __shared__ double sh[kNT / 64];
  const double pq = block_sum(phase_spmv_pq<V>(B, logical_block(), gridDim.x), sh);
  if (threadIdx.x == 0) B.part1[blockIdx.x] = pq;
}

__global__ __launch_bounds__(kNT) void k_update(PcgBuffers B, int parity) {
  PcgState* st = B.st;
  if (st->done) return;
  __shared__ double sh[kNT / 64];
  const double pq = reduce_partials(B.part1, B.spmv_grid, sh);
  if (!(pq > 0.0)) {
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      st->status = GF_ERR_BREAKDOWN;
      st->done = 1;
    }
    return;
  }
  double rz, rr;
  phase_update(B, st->rho[parity] / pq, &rz, &rr);
  rz = block_sum(rz, sh);
  rr = block_sum(rr, sh);
  if (threadIdx.x == 0) {
    B.part2[blockIdx.x] = rz;
    B.part2[gridDim.x + blockIdx.x] = rr;
  }
}

__global__ __launch_bounds__(kNT) void k_direction(PcgBuffers B, int parity) {
  PcgState* st = B.st;
  if (st->done) return;
  __shared__ double sh[kNT / 64];
  const int nb = gridDim.x;
  const double rz = reduce_partials(B.part2, nb, sh);
  const double rr = reduce_partials(B.part2 + nb, nb, sh);
  phase_direction(B, rz / st->rho[parity]);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    st->rho[parity ^ 1] = rz;
    st->rr = rr;
    const int it = st->it + 1;
    st->it = it;
    if (rr <= st->rtol2 * st->bnorm2 || it >= st->maxit) st->done = 1;
  }
}

// ---------------------------------------------------------------------------
// bounded grid barrier for the cooperative kernel
// ---------------------------------------------------------------------------
constexpr long kSpinLimit = 1L << 22;  // several seconds of polling: a barrier never takes that long

// Sense-free barrier on a monotonic arrival counter: arrival number a (0-based)
// belongs to barrier a / nb and waits until the counter reaches the end of
// that barrier's range.  The poll is a relaxed load (no cache maintenance per
// poll: an acquire load would invalidate the XCD's L2 on every spin, under the
// feet of the waves still gathering through it); one acquire fence follows.
__device__ inline bool grid_barrier(GridBarrier* bar, int* s_flag) {
  // the workgroup barrier makes every wave's stores complete; one agent-scope
  // release (L2 write-back) then publishes them for the other XCDs
  __syncthreads();
  if (threadIdx.x == 0) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    const unsigned long long nb = gridDim.x;
    const unsigned long long arrived =
        __hip_atomic_fetch_add(&bar->count, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const unsigned long long target = (arrived / nb + 1) * nb;
    long spins = 0;
    while (__hip_atomic_load(&bar->count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < target) {
      __builtin_amdgcn_s_sleep(1);
      if (__hip_atomic_load(&bar->abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) break;
      if (++spins > kSpinLimit) {
        __hip_atomic_store(&bar->abort, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        break;
      }
    }
    *s_flag = __hip_atomic_load(&bar->abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  }
  __syncthreads();
  return *s_flag == 0;
}

// All iterations in one launch.  The grid never exceeds the co-resident
// block count (cooperative launch), every block runs the same number of
// barriers, and the convergence test uses values every block computed
// identically, so all blocks leave the loop together.
template <int V>
__global__ __launch_bounds__(kNT) void k_pcg_persistent(PcgBuffers B, GridBarrier* bar) {
  __shared__ double sh[kNT / 64];
  __shared__ int s_flag;
  PcgState* st = B.st;
  if (st->done) return;  // read before any block can change it (it only changes at exit)
  if (threadIdx.x == 0) s_flag = 0;
  __syncthreads();
  int it = st->it;
  double rho = st->rho[it & 1];
  const double rtol2 = st->rtol2, bnorm2 = st->bnorm2;
  const int maxit = st->maxit;
  const bool lead = blockIdx.x == 0 && threadIdx.x == 0;
  const int nlb = B.spmv_grid;
  for (;;) {
    // the SpMV kernel's logical workgroups j (same rows, same partial slots)
    for (int j = blockIdx.x; j < nlb; j += gridDim.x) {
      const double pq_part = block_sum(phase_spmv_pq<V>(B, xcd_block(j, nlb), nlb), sh);
      if (threadIdx.x == 0) B.part1[j] = pq_part;
    }
    if (!grid_barrier(bar, &s_flag)) break;
    const double pq = reduce_partials(B.part1, nlb, sh);
    if (!(pq > 0.0)) {
      if (lead) {
        st->status = GF_ERR_BREAKDOWN;
        st->done = 1;
      }
      break;
    }
    double rz, rr;
    phase_update(B, rho / pq, &rz, &rr);
    rz = block_sum(rz, sh);
    rr = block_sum(rr, sh);
    if (threadIdx.x == 0) {
      B.part2[blockIdx.x] = rz;
      B.part2[gridDim.x + blockIdx.x] = rr;
    }
    if (!grid_barrier(bar, &s_flag)) break;
    rz = reduce_partials(B.part2, gridDim.x, sh);
    rr = reduce_partials(B.part2 + gridDim.x, gridDim.x, sh);
    phase_direction(B, rz / rho);
    rho = rz;
    ++it;
    const bool finished = rr <= rtol2 * bnorm2 || it >= maxit;
    if (lead) {
      st->rho[it & 1] = rz;
      st->rr = rr;
      st->it = it;
      if (finished) st->done = 1;
    }
    if (finished) break;
    if (!grid_barrier(bar, &s_flag)) break;
  }
  if (lead && s_flag) {
    st->status = GF_ERR_HIP;
    st->done = 1;
  }
}

// The two-launch iteration the same way, two grid barriers each.
template <int D>
__global__ __launch_bounds__(kNT) void k_split_persistent(PcgBuffers B, GridBarrier* bar) {
  __shared__ double sh[2 * (kNT / 64)];
  __shared__ int s_flag;
  PcgState* st = B.st;
  if (st->done) return;  // read before any block can change it (it only changes at exit)
  if (threadIdx.x == 0) s_flag = 0;
  __syncthreads();
  const int nlb = B.spmv_grid;
  const bool lead = blockIdx.x == 0 && threadIdx.x == 0;
  double rho = 0.0;
  for (int it = 0;; ++it) {
    double rz, rr;
    reduce_partials2(B.part2, B.part2 + B.nblocks, B.nblocks, &rz, &rr, sh);
    if (!split_goes_on(B, it, rr, lead)) break;
    const double beta = split_beta(it, rz, rho);
    rho = rz;
    // the product's logical workgroups j (same slices, same partial slots)
    for (int j = blockIdx.x; j < nlb; j += gridDim.x) {
      store_wave_sum(
          phase_split<D>(B, split_slice(xcd_block(j, nlb), B.bs), nlb, kNT / 64, beta),
          B.part1 + j);
      __syncthreads();  // the next slices' partial rows
    }
    if (!grid_barrier(bar, &s_flag)) break;
    const double pq = reduce_partials(B.part1, nlb, sh);
    if (!(pq > 0.0)) {
      split_breakdown(B, it, sh);
      break;
    }
    // the update's logical workgroups likewise
    for (int j = blockIdx.x; j < B.nblocks; j += gridDim.x) {
      const int lb = xcd_block(j, B.nblocks);
      SplitRows v;
      split_load<D>(B, int64_t(lb) * kNT + threadIdx.x, int64_t(B.nblocks) * kNT, &v);
      phase_split_update<D>(B, lb, j, rho / pq, beta, v, sh);
    }
    if (!grid_barrier(bar, &s_flag)) break;
  }
  if (lead && s_flag) {
    st->status = GF_ERR_HIP;
    st->done = 1;
  }
}

// nbar grid barriers and nothing else: the synchronisation cost of the
// persistent schedule (two or three per iteration) on its own grid
__global__ __launch_bounds__(kNT) void k_barrier_probe(GridBarrier* bar, int nbar) {
  __shared__ int s_flag;
  for (int k = 0; k < nbar; ++k)
    if (!grid_barrier(bar, &s_flag)) break;
}

__global__ void k_barrier_reset(GridBarrier* bar) {
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    bar->count = 0;
    bar->abort = 0;
  }
}

// ---------------------------------------------------------------------------
// residual and helpers
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kNT) void k_resid_partial(PcgBuffers B) {
  __shared__ double sh[kNT / 64];
  double s = 0.0, bb = 0.0;
  for_my_rows(B.n, [&](int64_t i) {
    const double bi = B.b[i];
    const double d = bi - B.q[i];
    s += d * d;
    bb += bi * bi;
  });
  s = block_sum(s, sh);
  bb = block_sum(bb, sh);
  if (threadIdx.x == 0) {
    B.part1[blockIdx.x] = s;
    B.part2[blockIdx.x] = bb;
  }
}

// ||b - K x|| / ||b|| (or ||b - K x|| when b = 0) from the partials above
__global__ __launch_bounds__(kNT) void k_resid_finish(PcgBuffers B, int nb, double* out) {
  __shared__ double sh[kNT / 64];
  const double s = reduce_partials(B.part1, nb, sh);
  const double bb = reduce_partials(B.part2, nb, sh);
  if (threadIdx.x == 0) out[0] = bb > 0.0 ? sqrt(s / bb) : sqrt(s);
}

// The energy functional 1/2 x.Kx - b.x (q holds K x): CG's error measure up
// to a constant, 1/2 ||x - x*||_K^2 - 1/2 ||x*||_K^2, so x beats the zero
// start when it is negative.
__global__ __launch_bounds__(kNT) void k_energy_partial(PcgBuffers B) {
  __shared__ double sh[kNT / 64];
  double xq = 0.0, xb = 0.0;
  for_my_rows(B.n, [&](int64_t i) {
    const double xi = B.x[i];
    xq += xi * B.q[i];
    xb += xi * B.b[i];
  });
  xq = block_sum(xq, sh);
  xb = block_sum(xb, sh);
  if (threadIdx.x == 0) {
    B.part1[blockIdx.x] = xq;
    B.part2[blockIdx.x] = xb;
  }
}

__global__ __launch_bounds__(kNT) void k_energy_finish(PcgBuffers B, int nb, double* out) {
  __shared__ double sh[kNT / 64];
  const double xq = reduce_partials(B.part1, nb, sh);
  const double xb = reduce_partials(B.part2, nb, sh);
  if (threadIdx.x == 0) out[0] = 0.5 * xq - xb;
}

// a right-hand side no eigenvector of a stiffness matrix is like: 0.5 to 1.5, scattered
__global__ void k_probe_rhs(int64_t n, double* b) {
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += int64_t(gridDim.x) * blockDim.x)
    b[i] = 0.5 + double((uint32_t(i) * 2654435761u) >> 8) * 0x1p-24;
}

// a state in which products run whatever the partials hold
__global__ void k_state_live(PcgState* st) {
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    st->done = 0;
    st->status = GF_OK;
    st->itv[0] = 0;
    st->maxit = INT32_MAX;
    st->it = 0;
    st->rho[0] = 1.0;
    st->bnorm2 = 1.0;
    st->rtol2 = -INFINITY;
  }
}

inline int grid_for(int64_t work, int threads, int cap) {
  int64_t b = (work + threads - 1) / threads;
  if (b < 1) b = 1;
  if (b > cap) b = cap;
  return int(b);
}

}  // namespace

size_t pcg_state_bytes() { return sizeof(PcgState); }
size_t grid_barrier_bytes() { return sizeof(GridBarrier); }

int spmv_blocks(int64_t n) {
  // enough rows per block to amortize the partition, at most kMaxPcgBlocks;
  // a multiple of 8 so the XCD remap applies
  int64_t nb = (n + 1023) / 1024;
  if (nb > kMaxPcgBlocks) nb = kMaxPcgBlocks;
  if (nb >= 8) nb &= ~int64_t(7);
  if (nb < 1) nb = 1;
  return int(nb);
}

hipError_t launch_build_coln(hipStream_t s, int64_t n, int32_t width, int d, const int32_t* col,
                             int32_t* coln) {
  if (d < 2 || width % d) return hipErrorInvalidValue;
  const int64_t total = n * (width / d);
  int64_t nb = (total + kNT - 1) / kNT;
  if (nb > 8192) nb = 8192;
  if (nb < 1) nb = 1;
  hipLaunchKernelGGL(k_build_coln, dim3(unsigned(nb)), dim3(kNT), 0, s, n, width / d, d, col, coln);
  return hipGetLastError();
}

hipError_t launch_stream_copy(hipStream_t s, const void* src, void* dst, int64_t bytes) {
  if ((bytes & 15) || (reinterpret_cast<uintptr_t>(src) & 15) || (reinterpret_cast<uintptr_t>(dst) & 15))
    return hipErrorInvalidValue;
  const int64_t n16 = bytes / 16;
  hipLaunchKernelGGL(k_stream_copy, dim3(grid_for(n16, kNT, 8192)), dim3(kNT), 0, s,
                     static_cast<const v2d*>(src), static_cast<v2d*>(dst), n16);
  return hipGetLastError();
}

hipError_t launch_bsell_cols(hipStream_t s, const BsellView& bs, int d, int64_t n,
                             const int32_t* col, const int32_t* rownnz, int32_t* bcol) {
  hipLaunchKernelGGL(k_bsell_cols, dim3(grid_for(bs.nslices * 64, kNT, 8192)), dim3(kNT), 0, s, bs,
                     d, n, col, rownnz, bcol);
  return hipGetLastError();
}

hipError_t launch_bsell_offsets(hipStream_t s, const BsellView& bs, const int32_t* bcol,
                                int16_t* coff, int* overflow) {
  hipLaunchKernelGGL(k_bsell_offsets, dim3(grid_for(bs.nslices * 64, kNT, 8192)), dim3(kNT), 0, s,
                     bs, bcol, coff, overflow);
  return hipGetLastError();
}

hipError_t launch_bsell_vals(hipStream_t s, const BsellView& bs, int d, int64_t n,
                             const double* val, const int32_t* rownnz, double* bval) {
  hipLaunchKernelGGL(k_bsell_vals, dim3(grid_for(bs.nslices * 64, kNT, 8192)), dim3(kNT), 0, s, bs,
                     d, n, val, rownnz, bval);
  return hipGetLastError();
}

hipError_t launch_bsell_to_ell(hipStream_t s, const BsellView& bs, int d, int64_t n,
                               const double* bval, const int32_t* rownnz, double* val) {
  hipLaunchKernelGGL(k_bsell_to_ell, dim3(grid_for(bs.nslices * 64, kNT, 8192)), dim3(kNT), 0, s,
                     bs, d, n, bval, rownnz, val);
  return hipGetLastError();
}

int iter_variant(int variant, int64_t bslots, int64_t n) {
  if (!is_bsell_group_variant(variant)) return variant;
  const int d = variant == kBsell2G ? 2 : 3;
  if (bslots * 64 * d * d * int64_t(sizeof(double)) > kCacheBytes ||
      iteration_bytes(bslots, d, n) > kCacheTraffic)
    return variant;
  return d == 2 ? kSplit2 : kSplit3;
}

int spmv_grid(int variant, const BsellView& bs, int nblocks) {
  if (is_split_variant(variant)) {
    // sweeps of equal size over at most kSplitBlocks workgroups
    const int64_t sweeps = std::max<int64_t>(1, (bs.nslices + kSplitBlocks - 1) / kSplitBlocks);
    int64_t nb = (bs.nslices + sweeps - 1) / sweeps;
    if (nb >= 8) nb = (nb + 7) & ~int64_t(7);  // the XCD remap needs a multiple of 8
    return int(std::max<int64_t>(1, nb));
  }
  if (!is_bsell_group_variant(variant)) return nblocks;
  int64_t nb = (bs.nslices + kNT / 64 - 1) / (kNT / 64);
  nb = (nb + 7) & ~int64_t(7);  // the XCD remap needs a multiple of 8
  if (nb > kMaxSpmvBlocks) nb = kMaxSpmvBlocks;
  if (nb < 8) nb = 8;
  return int(nb);
}

hipError_t launch_spmv(hipStream_t s, int variant, int64_t n, const double* val,
                       const int32_t* col, const int32_t* rownnz, const double* x, double* y,
                       int nrhs, const BsellView* bs) {
  const BsellView view = bs ? *bs : BsellView{nullptr, nullptr, 0, nullptr};
  if (is_bsell_variant(variant) && !view.perm) return hipErrorInvalidValue;
  const dim3 g(spmv_grid(variant, view, spmv_blocks(n)));
  for (int k = 0; k < nrhs; ++k) {
    const double* xk = x + int64_t(k) * n;
    double* yk = y + int64_t(k) * n;
    GF_DISPATCH_VARIANT(variant, k_spmv, g, s, n, val, col, rownnz, xk, yk, view);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t launch_jacobi_inv(hipStream_t s, int64_t n, const double* val,
                             const int32_t* diag, double* dinv) {
  hipLaunchKernelGGL(k_jacobi_inv, dim3(grid_for(n, 256, 8192)), dim3(256), 0, s, n, val,
                     diag, dinv);
  return hipGetLastError();
}

hipError_t launch_pcg_setup(hipStream_t s, const PcgBuffers& B, int use_x0, double rtol,
                            int maxit) {
  hipError_t e;
  if (use_x0) {
    e = launch_spmv(s, B.variant, B.n, B.val, B.col, B.rownnz, B.x, B.q, 1, &B.bs);
    if (e != hipSuccess) return e;
  }
  if (!B.single && B.iter_variant == kSplit2)
    hipLaunchKernelGGL(k_pcg_init<2>, dim3(B.nblocks), dim3(kNT), 0, s, B, use_x0);
  else if (!B.single && B.iter_variant == kSplit3)
    hipLaunchKernelGGL(k_pcg_init<3>, dim3(B.nblocks), dim3(kNT), 0, s, B, use_x0);
  else
    hipLaunchKernelGGL(k_pcg_init<1>, dim3(B.nblocks), dim3(kNT), 0, s, B, use_x0);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  hipLaunchKernelGGL(k_pcg_init_finish, dim3(1), dim3(kNT), 0, s, B, B.nblocks, rtol * rtol,
                     maxit);
  return hipGetLastError();
}

namespace {
// the product of an iteration
hipError_t launch_product(hipStream_t s, const PcgBuffers& B, int parity) {
  const dim3 g(B.spmv_grid);
  if (B.iter_variant == kSplit2) {
    hipLaunchKernelGGL(k_split_product<2>, g, dim3(64 * split_parts(2)), 0, s, B, parity);
  } else if (B.iter_variant == kSplit3) {
    hipLaunchKernelGGL(k_split_product<3>, g, dim3(64 * split_parts(3)), 0, s, B, parity);
  } else {
    GF_DISPATCH_VARIANT(B.iter_variant, k_spmv_pq, g, s, B);
  }
  return hipGetLastError();
}
// and its vector updates
hipError_t launch_updates(hipStream_t s, const PcgBuffers& B, int parity) {
  const dim3 g(B.nblocks), blk(kNT);
  if (B.iter_variant == kSplit2) {
    hipLaunchKernelGGL(k_split_update<2>, g, blk, 0, s, B, parity);
    return hipGetLastError();
  }
  if (B.iter_variant == kSplit3) {
    hipLaunchKernelGGL(k_split_update<3>, g, blk, 0, s, B, parity);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(k_update, g, blk, 0, s, B, parity);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_direction, g, blk, 0, s, B, parity);
  return hipGetLastError();
}
}  // namespace

bool single_fits(int iter_variant, int64_t n, int64_t bslots, int64_t nslices) {
  if (!is_split_variant(iter_variant)) return false;
  const int d = iter_variant == kSplit2 ? 2 : 3;
  return nslices <= (d == 2 ? kSingleSlices<2> : kSingleSlices<3>) &&
         n <= nslices * 64 * d && bslots * 64 * d * d * int64_t(sizeof(double)) <= single_bytes(d);
}

namespace {
hipError_t launch_single(hipStream_t s, const PcgBuffers& B, int count) {
  const dim3 blk(64 * kSingleWaves);
  if (B.iter_variant == kSplit2)
    hipLaunchKernelGGL(k_single<2>, dim3(1), blk, 0, s, B, count);
  else
    hipLaunchKernelGGL(k_single<3>, dim3(1), blk, 0, s, B, count);
  return hipGetLastError();
}
}  // namespace

hipError_t launch_pcg_iteration(hipStream_t s, const PcgBuffers& B, int parity) {
  const hipError_t e = launch_product(s, B, parity);
  return e != hipSuccess ? e : launch_updates(s, B, parity);
}

hipError_t launch_pcg_run(hipStream_t s, const PcgBuffers& B, int count) {
  if (B.single) return launch_single(s, B, count);
  hipError_t e = hipSuccess;
  for (int it = 0; it < count && e == hipSuccess; ++it) e = launch_pcg_iteration(s, B, it & 1);
  return e;
}

hipError_t launch_pcg_chunk(hipStream_t s, const PcgBuffers& B) {
  if (B.single) return launch_pcg_run(s, B, kSingleChunk);
  const hipError_t e = launch_pcg_run(s, B, kPcgChunk);
  return e != hipSuccess ? e : launch_pcg_check(s, B, 0);
}

hipError_t launch_pcg_check(hipStream_t s, const PcgBuffers& B, int parity) {
  if (!is_split_variant(B.iter_variant)) return hipSuccess;  // the direction pass checks
  hipLaunchKernelGGL(k_split_check, dim3(1), dim3(kNT), 0, s, B, parity);
  return hipGetLastError();
}

hipError_t launch_pcg_iteration_timed(hipStream_t s, const PcgBuffers& B, int parity,
                                      hipEvent_t spmv_start, hipEvent_t spmv_stop) {
  hipError_t e = hipEventRecord(spmv_start, s);
  if (e == hipSuccess) e = launch_product(s, B, parity);
  if (e == hipSuccess) e = hipEventRecord(spmv_stop, s);
  return e != hipSuccess ? e : launch_updates(s, B, parity);
}

int persistent_blocks(int variant, int num_cu) {
  int per_cu = 0;
  hipError_t e = hipErrorInvalidValue;
  switch (variant) {
    case kThreadU1: e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_pcg_persistent<kThreadU1>, kNT, 0); break;
    case kThreadU4: e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_pcg_persistent<kThreadU4>, kNT, 0); break;
    case kThreadU8: e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_pcg_persistent<kThreadU8>, kNT, 0); break;
    case kTile2: e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_pcg_persistent<kTile2>, kNT, 0); break;
    case kTile4: e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_pcg_persistent<kTile4>, kNT, 0); break;
    case kNode2: e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_pcg_persistent<kNode2>, kNT, 0); break;
    case kNode3: e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_pcg_persistent<kNode3>, kNT, 0); break;
    case kBsell2: e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_pcg_persistent<kBsell2>, kNT, 0); break;
    case kBsell3: e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_pcg_persistent<kBsell3>, kNT, 0); break;
    case kBsell2G: e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_pcg_persistent<kBsell2G>, kNT, 0); break;
    case kBsell3G: e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_pcg_persistent<kBsell3G>, kNT, 0); break;
    case kSplit2: e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_split_persistent<2>, kNT, 0); break;
    case kSplit3: e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_split_persistent<3>, kNT, 0); break;
    default: break;
  }
  if (e != hipSuccess || per_cu < 1) return 0;
  int64_t nb = int64_t(per_cu) * num_cu;
  if (nb > kMaxPcgBlocks) nb = kMaxPcgBlocks;
  nb &= ~int64_t(7);
  return int(nb);
}

hipError_t launch_pcg_persistent(hipStream_t s, const PcgBuffers& B, void* barrier, int num_cu) {
  if (B.single) return launch_single(s, B, INT32_MAX);
  GridBarrier* bar = static_cast<GridBarrier*>(barrier);
  hipLaunchKernelGGL(k_barrier_reset, dim3(1), dim3(64), 0, s, bar);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  PcgBuffers Bc = B;
  void* args[] = {&Bc, &bar};
  // the split kernels play the logical workgroups of both steps in turn; the
  // others' vector steps take exactly the grid of the kernel schedule.  Every
  // workgroup makes the barrier longer (1024 of them: 43 us), so a workgroup for
  // 1024 rows, from a quarter to all of the CUs; us an iteration against as many
  // as are co-resident, Q8 201x67 30 / 72, 512x256 119 / 154, Brick8 64x32x32
  // 58 / 121.
  int nb = B.nblocks;
  if (is_split_variant(B.iter_variant)) {
    nb = std::min(std::max(num_cu / 4, B.nblocks), num_cu);
    nb = std::min(nb, std::min(std::max(B.nblocks, B.spmv_grid),
                               persistent_blocks(B.iter_variant, num_cu)));
    if (nb < 1) return hipErrorInvalidConfiguration;
  }
  const dim3 g(nb), blk(kNT);
  switch (B.iter_variant) {
    case kSplit2: return hipLaunchCooperativeKernel(reinterpret_cast<const void*>(k_split_persistent<2>), g, blk, args, 0, s);
    case kSplit3: return hipLaunchCooperativeKernel(reinterpret_cast<const void*>(k_split_persistent<3>), g, blk, args, 0, s);
    case kThreadU1: return hipLaunchCooperativeKernel(reinterpret_cast<const void*>(k_pcg_persistent<kThreadU1>), g, blk, args, 0, s);
    case kThreadU4: return hipLaunchCooperativeKernel(reinterpret_cast<const void*>(k_pcg_persistent<kThreadU4>), g, blk, args, 0, s);
    case kThreadU8: return hipLaunchCooperativeKernel(reinterpret_cast<const void*>(k_pcg_persistent<kThreadU8>), g, blk, args, 0, s);
    case kTile2: return hipLaunchCooperativeKernel(reinterpret_cast<const void*>(k_pcg_persistent<kTile2>), g, blk, args, 0, s);
    case kTile4: return hipLaunchCooperativeKernel(reinterpret_cast<const void*>(k_pcg_persistent<kTile4>), g, blk, args, 0, s);
    case kNode2: return hipLaunchCooperativeKernel(reinterpret_cast<const void*>(k_pcg_persistent<kNode2>), g, blk, args, 0, s);
    case kNode3: return hipLaunchCooperativeKernel(reinterpret_cast<const void*>(k_pcg_persistent<kNode3>), g, blk, args, 0, s);
    case kBsell2: return hipLaunchCooperativeKernel(reinterpret_cast<const void*>(k_pcg_persistent<kBsell2>), g, blk, args, 0, s);
    case kBsell3: return hipLaunchCooperativeKernel(reinterpret_cast<const void*>(k_pcg_persistent<kBsell3>), g, blk, args, 0, s);
    case kBsell2G: return hipLaunchCooperativeKernel(reinterpret_cast<const void*>(k_pcg_persistent<kBsell2G>), g, blk, args, 0, s);
    case kBsell3G: return hipLaunchCooperativeKernel(reinterpret_cast<const void*>(k_pcg_persistent<kBsell3G>), g, blk, args, 0, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_barrier_probe(hipStream_t s, void* barrier, int nblocks, int nbar) {
  GridBarrier* bar = static_cast<GridBarrier*>(barrier);
  hipLaunchKernelGGL(k_barrier_reset, dim3(1), dim3(64), 0, s, bar);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  void* args[] = {&bar, &nbar};
  return hipLaunchCooperativeKernel(reinterpret_cast<const void*>(k_barrier_probe), dim3(nblocks),
                                    dim3(kNT), args, 0, s);
}

int barrier_aborted(hipStream_t s, const void* barrier, int* aborted) {
  GridBarrier h;
  hipError_t e = hipMemcpyAsync(&h, barrier, sizeof(h), hipMemcpyDeviceToHost, s);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  *aborted = e == hipSuccess ? h.abort : 1;
  return int(e);
}

hipError_t read_pcg_state(hipStream_t s, const PcgBuffers& B, PcgHostState* h) {
  PcgState st;
  hipError_t e = hipMemcpyAsync(&st, B.st, sizeof(st), hipMemcpyDeviceToHost, s);
  if (e != hipSuccess) return e;
  e = hipStreamSynchronize(s);
  if (e != hipSuccess) return e;
  h->it = st.it;
  h->done = st.done;
  h->status = st.status;
  h->rr = st.rr;
  h->bnorm2 = st.bnorm2;
  return hipSuccess;
}

hipError_t launch_spmv_pq_repeat(hipStream_t s, const PcgBuffers& B, int nrep) {
  hipLaunchKernelGGL(k_state_live, dim3(1), dim3(64), 0, s, B.st);
  hipError_t e = hipGetLastError();
  for (int i = 0; i < nrep && e == hipSuccess; ++i) e = launch_product(s, B, 0);
  return e;
}

hipError_t launch_probe_setup(hipStream_t s, const PcgBuffers& B, double* b) {
  hipLaunchKernelGGL(k_probe_rhs, dim3(grid_for(B.n, kNT, 8192)), dim3(kNT), 0, s, B.n, b);
  const hipError_t e = hipGetLastError();
  return e != hipSuccess ? e : launch_pcg_setup(s, B, 0, 0.0, INT32_MAX);
}

hipError_t launch_energy(hipStream_t s, const PcgBuffers& B, double* out_dev) {
  hipError_t e = launch_spmv(s, B.variant, B.n, B.val, B.col, B.rownnz, B.x, B.q, 1, &B.bs);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_energy_partial, dim3(B.nblocks), dim3(kNT), 0, s, B);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  hipLaunchKernelGGL(k_energy_finish, dim3(1), dim3(kNT), 0, s, B, B.nblocks, out_dev);
  return hipGetLastError();
}

hipError_t launch_true_residual(hipStream_t s, const PcgBuffers& B, double* out_dev) {
  hipError_t e = launch_spmv(s, B.variant, B.n, B.val, B.col, B.rownnz, B.x, B.q, 1, &B.bs);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_resid_partial, dim3(B.nblocks), dim3(kNT), 0, s, B);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  hipLaunchKernelGGL(k_resid_finish, dim3(1), dim3(kNT), 0, s, B, B.nblocks, out_dev);
  return hipGetLastError();
}

}  // namespace gf
