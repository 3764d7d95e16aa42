// Layer kernels of the learned warm start (BF16 storage, FP32 accumulate).
//
// The convolutions are implicit GEMMs on the gfx950 matrix cores with
// v_mfma_f32_16x16x32_bf16: one instruction multiplies a 16x32 A tile by a
// 32x16 B tile.  Lane l holds eight consecutive k of A's row l%16 and of B's
// column l%16 (k = 8(l/16) + e, the same for both operands) and receives
// D[4(l/16)+e][l%16], e = 0..3.  With A = weights (output channel x input
// channel) and B = gathered activations (input channel x voxel), each lane ends
// up owning four consecutive output channels of one voxel, so the epilogue
// stores 8 contiguous bytes per lane, and the B operand is one 16-byte load of
// eight consecutive channels per lane.
#include <cfloat>

#include "nn.hpp"

namespace gf {
namespace nn {

namespace {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef __bf16 h8 __attribute__((ext_vector_type(8)));
typedef uint32_t u4 __attribute__((ext_vector_type(4)));
// tensors are 8-byte aligned (the callers' too): 16-byte loads that need no more
typedef uint32_t u4a8 __attribute__((ext_vector_type(4), aligned(8)));

constexpr int kNT = 256;

__device__ inline float bf2f(uint16_t h) { return __uint_as_float(uint32_t(h) << 16); }

// round to nearest even; NaN stays NaN
__device__ inline uint16_t f2bf(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return 0x7fc0;
  u += 0x7fffu + ((u >> 16) & 1u);
  return uint16_t(u >> 16);
}

__device__ inline f4 mfma32(u4 a, u4 b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(h8, a),
                                                 __builtin_bit_cast(h8, b), c, 0, 0, 0);
}

// source coordinate along one axis for output coordinate v and tap offset t
__device__ inline int src_coord(int v, int t, int s, int transposed, int n) {
  int c;
  if (!transposed) {
    c = s * v + t;
  } else {
    const int d = v - t;
    if (d < 0 || (d % s) != 0) return -1;
    c = d / s;
  }
  return (c >= 0 && c < n) ? c : -1;
}

// A voxel's 27 sources: one base element plus an offset per tap that is the same
// for every voxel, and a bit per tap whose source lies inside the grid.
// Transposed with stride 2 only taps of matching parity have a source,
// (v - t) / 2 = v / 2 (rounded down) + (t < 0).
struct TapGeom {
  int64_t sx, sy, sz;  // elements per step along each axis of the source
  int stride, transposed;
  __device__ inline int axis(int t) const {
    return !transposed ? t : (stride == 1 ? -t : (t < 0 ? 1 : 0));
  }
  __device__ inline int64_t off(int tap) const {
    return axis(tap / 9 - 1) * sz + axis((tap / 3) % 3 - 1) * sy + axis(tap % 3 - 1) * sx;
  }
};
__device__ inline TapGeom tap_geom(const Vol& vin, int ld, int stride, int transposed) {
  TapGeom g;
  g.sx = ld;
  g.sy = int64_t(vin.nx) * ld;
  g.sz = int64_t(vin.ny) * vin.nx * ld;
  g.stride = stride;
  g.transposed = transposed;
  return g;
}
// valid bit k (tap offset k - 1) along one axis
__device__ inline uint32_t axis_bits(int v, int s, int transposed, int n) {
  uint32_t m = 0;
#pragma unroll
  for (int k = 0; k < 3; ++k)
    if (src_coord(v, k - 1, s, transposed, n) >= 0) m |= 1u << k;
  return m;
}
__device__ inline int axis_base(int v, int s, int transposed) {
  return !transposed ? s * v : (s == 1 ? v : v >> 1);
}
// element base and tap mask of voxel v (flat over the batch) of the output
__device__ inline uint32_t voxel_taps(int64_t v, int64_t total, const Vol& vo, const Vol& vi,
                                      int ld, int stride, int transposed, int64_t* base) {
  int x, y, z;
  int64_t b;
  if (total <= int64_t(0xffffffffu)) {  // 32-bit divisions: a tenth of the instructions
    const uint32_t nout = uint32_t(vo.nodes()), v32 = uint32_t(v);
    b = v32 / nout;
    uint32_t r = v32 - uint32_t(b) * nout;
    x = int(r % uint32_t(vo.nx));
    r /= uint32_t(vo.nx);
    y = int(r % uint32_t(vo.ny));
    z = int(r / uint32_t(vo.ny));
  } else {
    const int64_t nout = vo.nodes();
    b = v / nout;
    int64_t r = v - b * nout;
    x = int(r % vo.nx);
    r /= vo.nx;
    y = int(r % vo.ny);
    z = int(r / vo.ny);
  }
  const uint32_t mx = axis_bits(x, stride, transposed, vi.nx);
  const uint32_t my = axis_bits(y, stride, transposed, vi.ny);
  const uint32_t mz = axis_bits(z, stride, transposed, vi.nz);
  uint32_t row = 0, all = 0;
#pragma unroll
  for (int k = 0; k < 3; ++k) row |= (my >> k & 1u) ? mx << (3 * k) : 0u;
#pragma unroll
  for (int k = 0; k < 3; ++k) all |= (mz >> k & 1u) ? row << (9 * k) : 0u;
  *base = (b * vi.nodes() + (int64_t(axis_base(z, stride, transposed)) * vi.ny +
                             axis_base(y, stride, transposed)) * vi.nx +
           axis_base(x, stride, transposed)) * ld;
  return all;
}

// ---- convolution ----------------------------------------------------------------
// A wave owns VB blocks of 16 voxels and CT tiles of 16 output channels; a
// workgroup is four such waves on consecutive voxels.  The reduction runs over
// slabs of 16 input channels of one tap, two slabs per matrix instruction (the
// lower lanes the first, the upper lanes the second; an odd last slab has zero
// weights).  A 32-bit mask and one offset per tap replace the index arithmetic
// of each load, the loads are 16 bytes, and VB = 4 uses each weight fragment
// four times.  KS = 4: the four waves share the voxels, each takes a quarter of
// the slab pairs, and the partial tiles are added in LDS in wave order, for the
// coarse levels whose few voxels leave the chip idle.  The network's forward and
// data gradients on 65x33x33, batch 8: 2.7 -> 1.0 ms.
template <int VB, int CT, int KS>
__global__ __launch_bounds__(kNT) void k_conv(ConvArgs a) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t total = int64_t(a.batch) * a.vout.nodes();
  const int ncb = a.cin >> 4, nct = a.cout >> 4;
  const int ct0 = blockIdx.y * CT;
  const int kq = (lane >> 4) << 2;
  const TapGeom geom = tap_geom(a.vin, a.in_ld, a.stride, a.transposed);
  // lane l forms the indices of voxel l % (16 VB) of the wave; its block's lanes
  // get them by shuffle
  const int64_t first = (KS == 1 ? int64_t(blockIdx.x) * 4 + wave : int64_t(blockIdx.x)) * (16 * VB);
  int64_t base0 = 0;
  uint32_t mask0 = 0;
  if (const int64_t v = first + lane % (16 * VB); v < total)
    mask0 = voxel_taps(v, total, a.vout, a.vin, a.in_ld, a.stride, a.transposed, &base0);
  const uint16_t* src[VB];
  uint32_t mask[VB];
#pragma unroll
  for (int j = 0; j < VB; ++j) {
    const int from = j * 16 + (lane & 15);
    mask[j] = __shfl(mask0, from);
    src[j] = a.in + __shfl(base0, from) + a.in_off + ((lane >> 4) & 1) * 8;
  }
  f4 acc[VB][CT];
#pragma unroll
  for (int j = 0; j < VB; ++j)
#pragma unroll
    for (int c = 0; c < CT; ++c) acc[j][c] = f4{0.f, 0.f, 0.f, 0.f};
  const u4 zero = {0u, 0u, 0u, 0u};
  const bool upper = lane >= 32;
  const int npair = (27 * ncb + 1) / 2;
  const int p0 = KS == 1 ? 0 : npair * wave / KS, p1 = KS == 1 ? npair : npair * (wave + 1) / KS;
  const uint16_t* wp = a.wf + ((int64_t(p0) * nct + ct0) * 64 + lane) * 8;
  int tap = 2 * p0 / ncb, cb = 2 * p0 - tap * ncb;  // the pair's first slab
  auto fetch = [&](u4* bfr, u4* af) {
    const int cb1 = cb + 1 < ncb ? cb + 1 : 0, tap1 = cb + 1 < ncb ? tap : tap + 1;
    const int64_t off0 = geom.off(tap) + cb * 16;
    const int64_t off1 = tap1 < 27 ? geom.off(tap1) + cb1 * 16 : 0;
    const int64_t off = upper ? off1 : off0;
    const int bit = upper ? tap1 : tap;  // bit 27 is never set
    cb = cb1 + 1 < ncb ? cb1 + 1 : 0;
    tap = cb1 + 1 < ncb ? tap1 : tap1 + 1;
#pragma unroll
    for (int j = 0; j < VB; ++j)
      bfr[j] = (mask[j] >> bit & 1u) ? u4(*reinterpret_cast<const u4a8*>(src[j] + off)) : zero;
#pragma unroll
    for (int c = 0; c < CT; ++c) af[c] = *reinterpret_cast<const u4*>(wp + c * 512);
    wp += int64_t(nct) * 512;
  };
  // the next pair's operands are in flight while this one is multiplied
  u4 bfr[VB], af[CT], bnx[VB], anx[CT];
  fetch(bfr, af);
  for (int i = p0; i < p1; ++i) {
    if (i + 1 < p1) fetch(bnx, anx);
#pragma unroll
    for (int c = 0; c < CT; ++c)
#pragma unroll
      for (int j = 0; j < VB; ++j) acc[j][c] = mfma32(af[c], bfr[j], acc[j][c]);
#pragma unroll
    for (int j = 0; j < VB; ++j) bfr[j] = bnx[j];
#pragma unroll
    for (int c = 0; c < CT; ++c) af[c] = anx[c];
  }
  if constexpr (KS > 1) {  // tile q = j CT + c ends in wave q % KS
    __shared__ f4 sh[KS][VB * CT][64];
#pragma unroll
    for (int j = 0; j < VB; ++j)
#pragma unroll
      for (int c = 0; c < CT; ++c) sh[wave][j * CT + c][lane] = acc[j][c];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < VB; ++j)
#pragma unroll
      for (int c = 0; c < CT; ++c)
        if ((j * CT + c) % KS == wave) {
          f4 t = sh[0][j * CT + c][lane];
#pragma unroll
          for (int k = 1; k < KS; ++k) t += sh[k][j * CT + c][lane];
          acc[j][c] = t;
        }
  }
#pragma unroll
  for (int j = 0; j < VB; ++j) {
    const int64_t vox = first + j * 16 + (lane & 15);
    if (vox >= total) continue;
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      if (KS > 1 && (j * CT + c) % KS != wave) continue;
      const int co = (ct0 + c) * 16 + kq;
      float r[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float t = acc[j][c][e] + (a.bias ? a.bias[co + e] : 0.f);
        if (a.act) t = t > 0.f ? t : a.slope * t;
        r[e] = t;
      }
      if (a.out32) {
        float4* o = reinterpret_cast<float4*>(a.out32 + vox * a.out_ld + a.out_off + co);
        float4 w = make_float4(r[0], r[1], r[2], r[3]);
        if (a.accumulate) {
          const float4 old = *o;
          w.x += old.x;
          w.y += old.y;
          w.z += old.z;
          w.w += old.w;
        }
        *o = w;
      } else {
        uint2* o = reinterpret_cast<uint2*>(a.out + vox * a.out_ld + a.out_off + co);
        if (a.accumulate) {
          const uint2 old = *o;
          r[0] += bf2f(uint16_t(old.x & 0xffffu));
          r[1] += bf2f(uint16_t(old.x >> 16));
          r[2] += bf2f(uint16_t(old.y & 0xffffu));
          r[3] += bf2f(uint16_t(old.y >> 16));
        }
        uint2 w;
        w.x = uint32_t(f2bf(r[0])) | (uint32_t(f2bf(r[1])) << 16);
        w.y = uint32_t(f2bf(r[2])) | (uint32_t(f2bf(r[3])) << 16);
        *o = w;
      }
    }
  }
}

// ---- weight gradient ---------------------------------------------------------------
// Workgroup (chunk of voxels, block of 16 input channels, NCO tiles of 16 output
// channels), all 27 taps: tiles of 64 voxels of the 27 gathered inputs and of dz
// are staged transposed in LDS ([channel][voxel], padded rows), so that each
// MFMA operand (eight consecutive voxels of one channel) is one 16-byte LDS
// read; the waves share the taps (seven each; the last wave's seventh is the
// bias, a row of ones against dz) and the voxels are the reduction axis.  The
// next tile's loads are in flight while this one is multiplied.  Taking the
// taps together stages dz once instead of 27 times and forms a voxel's indices
// once per tile instead of once per tap and quad of channels, which bounded the
// kernel (the weight gradients of the network on 65x33x33, batch 8: 3.2 -> 0.8
// ms, the bias gradients' launches gone with them).
constexpr int kWgTile = 64;
constexpr int kWgRow = kWgTile + 8;  // LDS row stride (elements): 16-byte aligned rows
constexpr int kWgTaps = 7;           // taps per wave

template <int NCO>
__global__ __launch_bounds__(kNT) void k_wgrad(WgradArgs a) {
  __shared__ __align__(16) uint16_t sx[27 * 16 * kWgRow];
  __shared__ __align__(16) uint16_t sd[NCO * 16 * kWgRow];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
  const int64_t total = int64_t(a.batch) * a.vout.nodes();
  const int64_t v0 = int64_t(blockIdx.x) * a.chunk;
  const int64_t v1 = v0 + a.chunk < total ? v0 + a.chunk : total;
  const int ci0 = blockIdx.y * 16, co0 = blockIdx.z * NCO * 16;
  const TapGeom geom = tap_geom(a.vin, a.x_ld, a.stride, 0);
  const bool bias = a.bpart && blockIdx.y == 0;
  f4 acc[kWgTaps][NCO];
#pragma unroll
  for (int j = 0; j < kWgTaps; ++j)
#pragma unroll
    for (int c = 0; c < NCO; ++c) acc[j][c] = f4{0.f, 0.f, 0.f, 0.f};
  // this thread stages channel quad `wave` of voxel `lane`: 27 sources and the
  // quads wave, wave + 4, ... of dz
  uint2 xv[27], dv[NCO];
  auto fetch = [&](int64_t base) {
    const int64_t v = base + lane;
    int64_t at = 0;
    const uint32_t mask = v < v1 ? voxel_taps(v, total, a.vout, a.vin, a.x_ld, a.stride, 0, &at) : 0u;
    const uint16_t* x = a.x + at + a.x_off + ci0 + wave * 4;
#pragma unroll
    for (int t = 0; t < 27; ++t)
      xv[t] = (mask >> t & 1u) ? *reinterpret_cast<const uint2*>(x + geom.off(t))
                               : make_uint2(0u, 0u);
    const uint16_t* d = a.dz + v * a.dz_ld + a.dz_off + co0 + wave * 4;
#pragma unroll
    for (int c = 0; c < NCO; ++c)
      dv[c] = v < v1 ? *reinterpret_cast<const uint2*>(d + c * 16) : make_uint2(0u, 0u);
  };
  // lanes 2k and 2k + 1 swap halves, so that each writes two channels of both
  // voxels, a dword each (half the LDS writes)
  const bool odd = lane & 1;
  auto put = [&](uint16_t* row, uint2 v) {
    const uint32_t got = uint32_t(__builtin_amdgcn_mov_dpp(int(odd ? v.x : v.y), 0xB1 /* 1,0,3,2 */,
                                                           0xf, 0xf, true));
    const uint32_t lo = odd ? got : v.x, hi = odd ? v.y : got;  // the even and the odd voxel's
    uint32_t* col = reinterpret_cast<uint32_t*>(row + (wave * 4 + (odd ? 2 : 0)) * kWgRow +
                                                (lane & ~1));
    col[0] = (lo & 0xffffu) | (hi << 16);
    col[kWgRow / 2] = (lo >> 16) | (hi & 0xffff0000u);
  };
  if (v0 < v1) fetch(v0);
  for (int64_t base = v0; base < v1; base += kWgTile) {
    __syncthreads();
#pragma unroll
    for (int t = 0; t < 27; ++t) put(sx + t * 16 * kWgRow, xv[t]);
#pragma unroll
    for (int c = 0; c < NCO; ++c) put(sd + c * 16 * kWgRow, dv[c]);
    __syncthreads();
    if (base + kWgTile < v1) fetch(base + kWgTile);
    const int k0 = (lane >> 4) * 8;
#pragma unroll
    for (int kb = 0; kb < kWgTile / 32; ++kb) {
      u4 B[NCO];
#pragma unroll
      for (int c = 0; c < NCO; ++c)
        B[c] = *reinterpret_cast<const u4*>(sd + (c * 16 + (lane & 15)) * kWgRow + kb * 32 + k0);
#pragma unroll
      for (int j = 0; j < kWgTaps; ++j) {
        const int tap = wave * kWgTaps + j;
        u4 A = {0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u};  // ones
        if (tap < 27)
          A = *reinterpret_cast<const u4*>(sx + (tap * 16 + (lane & 15)) * kWgRow + kb * 32 + k0);
        if (tap < 27 || bias) {
#pragma unroll
          for (int c = 0; c < NCO; ++c) acc[j][c] = mfma32(A, B[c], acc[j][c]);
        }
      }
    }
  }
#pragma unroll
  for (int j = 0; j < kWgTaps; ++j) {
    const int tap = wave * kWgTaps + j;
    float* P = a.part + (int64_t(blockIdx.x) * 27 + tap) * a.cin * a.cout;
#pragma unroll
    for (int c = 0; c < NCO; ++c) {
      const int co = co0 + c * 16 + (lane & 15);
      if (tap < 27) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          P[int64_t(ci0 + ((lane >> 4) << 2) + e) * a.cout + co] = acc[j][c][e];
      } else if (bias && lane < 16) {
        a.bpart[int64_t(blockIdx.x) * a.cout + co] = acc[j][c][0];
      }
    }
  }
}

// out[i] = sum_c part[c * len + i] in a fixed order: kRedGroups interleaved runs
// of parts, then the runs
constexpr int kRedGroups = 8;
__global__ __launch_bounds__(kNT) void k_reduce_parts(const float* part, int np, int64_t len,
                                                      float* out) {
  constexpr int W = kNT / kRedGroups;
  __shared__ float sh[kRedGroups][W];
  const int g = threadIdx.x / W, l = threadIdx.x % W;
  for (int64_t i0 = int64_t(blockIdx.x) * W; i0 < len; i0 += int64_t(gridDim.x) * W) {
    float s = 0.f;
    if (i0 + l < len) {
#pragma unroll 4
      for (int c = g; c < np; c += kRedGroups) s += part[c * len + i0 + l];
    }
    __syncthreads();
    sh[g][l] = s;
    __syncthreads();
    if (g == 0 && i0 + l < len) {
      float t = 0.f;
#pragma unroll
      for (int k = 0; k < kRedGroups; ++k) t += sh[k][l];
      out[i0 + l] = t;
    }
  }
}

// ---- weights -> MFMA A fragments -------------------------------------------------
// (pair of 16-channel slabs, output tile, lane, e): see k_conv
__global__ void k_arrange(const float* w, uint16_t* wf, int cin, int cout, int transposed) {
  const int Cc = transposed ? cout : cin, Co = transposed ? cin : cout;
  const int ncb = Cc >> 4, nct = Co >> 4, slabs = 27 * ncb;
  const int64_t total = int64_t((slabs + 1) / 2) * nct * 512;
  for (int64_t idx = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; idx < total;
       idx += int64_t(gridDim.x) * blockDim.x) {
    const int e = int(idx & 7), lane = int((idx >> 3) & 63);
    const int64_t rest = idx >> 9;
    const int ot = int(rest % nct), slab = 2 * int(rest / nct) + (lane >> 5);
    const int tap = slab / ncb, cb = slab - tap * ncb;
    const int c = cb * 16 + ((lane >> 4) & 1) * 8 + e, o = ot * 16 + (lane & 15);
    float v = 0.f;
    if (slab < slabs)
      v = transposed ? w[(int64_t(tap) * cin + o) * cout + c]
                     : w[(int64_t(tap) * cin + c) * cout + o];
    wf[idx] = f2bf(v);
  }
}

// ---- element-wise and small reductions -----------------------------------------
__global__ void k_act_bwd(uint16_t* dy, int dy_ld, int dy_off, const uint16_t* y, int y_ld,
                          int y_off, int64_t voxels, int cq, float slope) {
  const int64_t total = voxels * cq;
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < total;
       i += int64_t(gridDim.x) * blockDim.x) {
    const int64_t v = i / cq;
    const int q = int(i - v * cq);
    uint2* pd = reinterpret_cast<uint2*>(dy + v * dy_ld + dy_off + q * 4);
    const uint2 yy = *reinterpret_cast<const uint2*>(y + v * y_ld + y_off + q * 4);
    uint2 d = *pd;
    const uint16_t ys[4] = {uint16_t(yy.x & 0xffffu), uint16_t(yy.x >> 16), uint16_t(yy.y & 0xffffu),
                            uint16_t(yy.y >> 16)};
    uint16_t ds[4] = {uint16_t(d.x & 0xffffu), uint16_t(d.x >> 16), uint16_t(d.y & 0xffffu),
                      uint16_t(d.y >> 16)};
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (!(bf2f(ys[e]) > 0.f)) ds[e] = f2bf(slope * bf2f(ds[e]));
    d.x = uint32_t(ds[0]) | (uint32_t(ds[1]) << 16);
    d.y = uint32_t(ds[2]) | (uint32_t(ds[3]) << 16);
    *pd = d;
  }
}

__device__ inline void axis_up(int f, int nc, int* i0, int* i1) {
  // fine f -> coarse neighbours (weight 1 if f even, 1/2 each if odd)
  if ((f & 1) == 0) {
    *i0 = f >> 1;
    *i1 = -1;
  } else {
    *i0 = (f - 1) >> 1;
    *i1 = (f + 1) >> 1;
    if (*i1 >= nc) *i1 = -1;
  }
}

__global__ void k_prolong(const uint16_t* in, int in_ld, int in_off, Vol vc, uint16_t* out,
                          int out_ld, int out_off, Vol vf, int batch, int cq) {
  const int64_t nf = vf.nodes(), total = int64_t(batch) * nf * cq;
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < total;
       i += int64_t(gridDim.x) * blockDim.x) {
    const int64_t v = i / cq;
    const int q = int(i - v * cq);
    const int64_t b = v / nf;
    int64_t r = v - b * nf;
    const int x = int(r % vf.nx);
    r /= vf.nx;
    const int y = int(r % vf.ny), z = int(r / vf.ny);
    int cz[2], cy[2], cx[2];
    axis_up(z, vc.nz, &cz[0], &cz[1]);
    axis_up(y, vc.ny, &cy[0], &cy[1]);
    axis_up(x, vc.nx, &cx[0], &cx[1]);
    const float wz = cz[1] >= 0 ? 0.5f : 1.f, wy = cy[1] >= 0 ? 0.5f : 1.f,
                wx = cx[1] >= 0 ? 0.5f : 1.f;
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    for (int a = 0; a < 2; ++a) {
      if (cz[a] < 0) continue;
      for (int bb = 0; bb < 2; ++bb) {
        if (cy[bb] < 0) continue;
        for (int c = 0; c < 2; ++c) {
          if (cx[c] < 0) continue;
          const float w = wz * wy * wx;
          const uint2 u = *reinterpret_cast<const uint2*>(
              in + (b * vc.nodes() + (int64_t(cz[a]) * vc.ny + cy[bb]) * vc.nx + cx[c]) * in_ld +
              in_off + q * 4);
          acc[0] += w * bf2f(uint16_t(u.x & 0xffffu));
          acc[1] += w * bf2f(uint16_t(u.x >> 16));
          acc[2] += w * bf2f(uint16_t(u.y & 0xffffu));
          acc[3] += w * bf2f(uint16_t(u.y >> 16));
        }
      }
    }
    uint2 o;
    o.x = uint32_t(f2bf(acc[0])) | (uint32_t(f2bf(acc[1])) << 16);
    o.y = uint32_t(f2bf(acc[2])) | (uint32_t(f2bf(acc[3])) << 16);
    *reinterpret_cast<uint2*>(out + v * out_ld + out_off + q * 4) = o;
  }
}

__global__ void k_prolong_bwd(const uint16_t* df, int f_ld, int f_off, Vol vf, uint16_t* dc,
                              int c_ld, int c_off, Vol vc, int batch, int cq) {
  const int64_t nc = vc.nodes(), total = int64_t(batch) * nc * cq;
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < total;
       i += int64_t(gridDim.x) * blockDim.x) {
    const int64_t v = i / cq;
    const int q = int(i - v * cq);
    const int64_t b = v / nc;
    int64_t r = v - b * nc;
    const int X = int(r % vc.nx);
    r /= vc.nx;
    const int Y = int(r % vc.ny), Z = int(r / vc.ny);
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    for (int dz = -1; dz <= 1; ++dz) {
      const int fz = 2 * Z + dz;
      if (fz < 0 || fz >= vf.nz) continue;
      const float wz = dz == 0 ? 1.f : 0.5f;
      for (int dy = -1; dy <= 1; ++dy) {
        const int fy = 2 * Y + dy;
        if (fy < 0 || fy >= vf.ny) continue;
        const float wy = dy == 0 ? 1.f : 0.5f;
        for (int dx = -1; dx <= 1; ++dx) {
          const int fx = 2 * X + dx;
          if (fx < 0 || fx >= vf.nx) continue;
          const float w = wz * wy * (dx == 0 ? 1.f : 0.5f);
          const uint2 u = *reinterpret_cast<const uint2*>(
              df + (b * vf.nodes() + (int64_t(fz) * vf.ny + fy) * vf.nx + fx) * f_ld + f_off + q * 4);
          acc[0] += w * bf2f(uint16_t(u.x & 0xffffu));
          acc[1] += w * bf2f(uint16_t(u.x >> 16));
          acc[2] += w * bf2f(uint16_t(u.y & 0xffffu));
          acc[3] += w * bf2f(uint16_t(u.y >> 16));
        }
      }
    }
    uint2 o;
    o.x = uint32_t(f2bf(acc[0])) | (uint32_t(f2bf(acc[1])) << 16);
    o.y = uint32_t(f2bf(acc[2])) | (uint32_t(f2bf(acc[3])) << 16);
    *reinterpret_cast<uint2*>(dc + v * c_ld + c_off + q * 4) = o;
  }
}

__global__ __launch_bounds__(kNT) void k_mse(const float* pred, const float* target,
                                             int64_t voxels, int c, uint16_t* dpred,
                                             float* part) {
  __shared__ float sh[kNT];
  const float scale = 2.f / float(voxels * c);
  float s = 0.f;
  for (int64_t v = int64_t(blockIdx.x) * kNT + threadIdx.x; v < voxels;
       v += int64_t(gridDim.x) * kNT) {
    uint16_t g[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) g[e] = 0;
    for (int e = 0; e < c; ++e) {
      const float d = pred[v * 16 + e] - target[v * 4 + e];
      s += d * d;
      g[e] = f2bf(scale * d);
    }
    uint4* o = reinterpret_cast<uint4*>(dpred + v * 16);
    o[0] = make_uint4(g[0] | (uint32_t(g[1]) << 16), g[2] | (uint32_t(g[3]) << 16),
                      g[4] | (uint32_t(g[5]) << 16), g[6] | (uint32_t(g[7]) << 16));
    o[1] = make_uint4(g[8] | (uint32_t(g[9]) << 16), g[10] | (uint32_t(g[11]) << 16),
                      g[12] | (uint32_t(g[13]) << 16), g[14] | (uint32_t(g[15]) << 16));
  }
  sh[threadIdx.x] = s;
  __syncthreads();
  for (int o = kNT / 2; o > 0; o >>= 1) {
    if (threadIdx.x < o) sh[threadIdx.x] += sh[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = sh[0];
}

__global__ void k_mse_finish(const float* part, int np, float inv_count, float* loss) {
  // one wave, strided runs, then across the lanes
  float s = 0.f;
  for (int i = threadIdx.x; i < np; i += 64) s += part[i];
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
  if (threadIdx.x == 0) *loss = s * inv_count;
}

__global__ void k_adam(float* p, const float* g, float* m, float* v, int64_t n, float lr_t,
                       float b1, float b2, float eps) {
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += int64_t(gridDim.x) * blockDim.x) {
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] -= lr_t * mi / (sqrtf(vi) + eps);
  }
}

__global__ void k_to_dofs(const float* pred, const uint16_t* feat, int mask_ch, int base_ch,
                          double base_w, int64_t nodes, double scale, double* x) {
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < nodes;
       i += int64_t(gridDim.x) * blockDim.x) {
    const bool fixed = bf2f(feat[i * 16 + mask_ch]) > 0.5f;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      double v = double(pred[i * 16 + c]);
      if (base_ch >= 0) v += base_w * double(bf2f(feat[i * 16 + base_ch + c]));
      x[i * 3 + c] = fixed ? 0.0 : scale * v;
    }
  }
}

__global__ void k_fill0(uint32_t* p, int64_t words) {
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < words;
       i += int64_t(gridDim.x) * blockDim.x)
    p[i] = 0u;
}

inline int grid_for(int64_t work, int cap = 8192) {
  int64_t b = (work + kNT - 1) / kNT;
  if (b < 1) b = 1;
  if (b > cap) b = cap;
  return int(b);
}

template <int VB, int KS>
hipError_t conv_vb(hipStream_t s, const ConvArgs& a) {
  const int nct = a.cout >> 4;
  const int64_t total = int64_t(a.batch) * a.vout.nodes();
  constexpr int64_t per = KS == 1 ? 64 * VB : 16 * VB;  // voxels per workgroup
  const int64_t gx = (total + per - 1) / per;
  if (gx > 0x7fffffff) return hipErrorInvalidValue;
  if (nct % 4 == 0) {
    hipLaunchKernelGGL((k_conv<VB, 4, KS>), dim3(unsigned(gx), nct / 4), dim3(kNT), 0, s, a);
  } else if (nct % 3 == 0) {
    hipLaunchKernelGGL((k_conv<VB, 3, KS>), dim3(unsigned(gx), nct / 3), dim3(kNT), 0, s, a);
  } else if (nct % 2 == 0) {
    hipLaunchKernelGGL((k_conv<VB, 2, KS>), dim3(unsigned(gx), nct / 2), dim3(kNT), 0, s, a);
  } else {
    hipLaunchKernelGGL((k_conv<VB, 1, KS>), dim3(unsigned(gx), nct), dim3(kNT), 0, s, a);
  }
  return hipGetLastError();
}

}  // namespace

hipError_t launch_conv(hipStream_t s, const ConvArgs& a) {
  if (a.cin < 16 || a.cout < 16 || (a.cin & 15) || (a.cout & 15) || (a.in_ld & 3) ||
      (a.in_off & 3) || (a.out_ld & 3) || (a.out_off & 3) || a.batch < 1 ||
      (a.stride != 1 && a.stride != 2) || (!a.out) == (!a.out32) ||
      a.in_off + a.cin > a.in_ld || a.out_off + a.cout > a.out_ld)
    return hipErrorInvalidValue;
  // 64 voxels per wave reuse a weight fragment four times; from about two waves
  // per SIMD of 256 CUs down, the four waves of a workgroup share the voxels, and
  // below that take fewer of them.  us, by `waves`, 64 voxels a wave / 64, 32 and 16
  // shared by four: 4,357 (65x65x33, 64 -> 128 channels) 181 / 173 163 217; 2,178
  // (96 -> 32) 89 / 104 90 121, (16 -> 16) 17 / 15 20 31; 1,106 (32 -> 32) 26 / 19 20
  // 29; 561 (32 -> 32) 24 / 12.0 12.2 17; 289 24 / 10 8.7 11; 149 24 / 9.2 7.6 7.8;
  // 76 24 / 8.3 7.5 6.6.  Within 20 % of the best of them on every pair of channel
  // counts the network has.
  const int64_t total = int64_t(a.batch) * a.vout.nodes();
  const int nct = a.cout >> 4, ct = nct % 4 == 0 ? 4 : nct % 3 == 0 ? 3 : nct % 2 == 0 ? 2 : 1;
  const int64_t waves = total * (nct / ct) / 64;
  if (waves >= 2048) return conv_vb<4, 1>(s, a);
  if (waves >= 512) return conv_vb<4, 4>(s, a);
  if (waves >= 128) return conv_vb<2, 4>(s, a);
  return conv_vb<1, 4>(s, a);
}

size_t conv_fragments(int cin, int cout) {
  // either direction's: slabs are paired along the channels it sums over
  const size_t fwd = size_t((27 * (cin >> 4) + 1) / 2) * (cout >> 4);
  const size_t bwd = size_t((27 * (cout >> 4) + 1) / 2) * (cin >> 4);
  return (fwd > bwd ? fwd : bwd) * 512;
}

namespace {
int wgrad_co_tiles(int cout) {
  const int nco = cout >> 4;
  return nco % 4 == 0 ? 4 : nco % 3 == 0 ? 3 : nco % 2 == 0 ? 2 : 1;
}
}  // namespace

int wgrad_chunks(int64_t voxels, int cin, int cout) {
  // about two workgroups per CU of 256 with the channel blocks, and at least
  // two tiles of voxels each; half / this / twice as many, us with the sum of the
  // parts: 65x33x33, 192 -> 64 channels 260 / 229 / 250, 32 -> 32 38 / 30 / 39; 33^3,
  // 64 -> 128 96 / 88 / 111; up to 17^3 all alike
  const int64_t blocks = int64_t(cin >> 4) * ((cout >> 4) / wgrad_co_tiles(cout));
  const int64_t tiles = (voxels + kWgTile - 1) / kWgTile;
  int64_t c = 512 / blocks;
  if (c > (tiles + 1) / 2) c = (tiles + 1) / 2;
  return int(c < 1 ? 1 : c);
}

hipError_t launch_wgrad(hipStream_t s, const WgradArgs& a, float* dw, float* db) {
  if ((a.cin & 15) || (a.cout & 15) || a.cin < 16 || a.cout < 16 || (a.chunk % kWgTile) ||
      a.nchunk < 1 || (a.x_ld & 3) || (a.x_off & 3) || (a.dz_ld & 3) || (a.dz_off & 3))
    return hipErrorInvalidValue;
  const int64_t total = int64_t(a.batch) * a.vout.nodes();
  if (int64_t(a.nchunk) * a.chunk < total) return hipErrorInvalidValue;
  if ((a.cin >> 4) * (a.cout >> 4) > 48 || a.cin + a.cout > 480) return hipErrorInvalidValue;
  if (db && (a.cout > kNT || kNT % a.cout || !a.bpart)) return hipErrorInvalidValue;
  const int nco = wgrad_co_tiles(a.cout);
  const dim3 g(a.nchunk, a.cin >> 4, (a.cout >> 4) / nco), t(kNT);
  if (nco == 4) hipLaunchKernelGGL(k_wgrad<4>, g, t, 0, s, a);
  else if (nco == 3) hipLaunchKernelGGL(k_wgrad<3>, g, t, 0, s, a);
  else if (nco == 2) hipLaunchKernelGGL(k_wgrad<2>, g, t, 0, s, a);
  else hipLaunchKernelGGL(k_wgrad<1>, g, t, 0, s, a);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const int64_t len = int64_t(27) * a.cin * a.cout;
  const int64_t w = kNT / kRedGroups;
  hipLaunchKernelGGL(k_reduce_parts, dim3(unsigned((len + w - 1) / w)), dim3(kNT), 0, s, a.part,
                     a.nchunk, len, dw);
  if ((e = hipGetLastError()) != hipSuccess || !db) return e;
  hipLaunchKernelGGL(k_reduce_parts, dim3(unsigned((a.cout + w - 1) / w)), dim3(kNT), 0, s, a.bpart,
                     a.nchunk, int64_t(a.cout), db);
  return hipGetLastError();
}

hipError_t launch_arrange(hipStream_t s, const float* w, uint16_t* wf, int cin, int cout,
                          int transposed) {
  if ((cin & 15) || (cout & 15)) return hipErrorInvalidValue;
  const int64_t total = int64_t(conv_fragments(cin, cout));
  hipLaunchKernelGGL(k_arrange, dim3(grid_for(total)), dim3(kNT), 0, s, w, wf, cin, cout, transposed);
  return hipGetLastError();
}

hipError_t launch_act_bwd(hipStream_t s, uint16_t* dy, int dy_ld, int dy_off, const uint16_t* y,
                          int y_ld, int y_off, int64_t voxels, int c, float slope) {
  if ((c & 3) || (dy_ld & 3) || (dy_off & 3) || (y_ld & 3) || (y_off & 3)) return hipErrorInvalidValue;
  const int cq = c >> 2;
  hipLaunchKernelGGL(k_act_bwd, dim3(grid_for(voxels * cq)), dim3(kNT), 0, s, dy, dy_ld, dy_off, y,
                     y_ld, y_off, voxels, cq, slope);
  return hipGetLastError();
}

hipError_t launch_prolong(hipStream_t s, const uint16_t* in, int in_ld, int in_off, Vol vc,
                          uint16_t* out, int out_ld, int out_off, Vol vf, int batch, int c) {
  if ((c & 3) || vf.nx != 2 * vc.nx - 1 || vf.ny != 2 * vc.ny - 1 || vf.nz != 2 * vc.nz - 1)
    return hipErrorInvalidValue;
  const int cq = c >> 2;
  hipLaunchKernelGGL(k_prolong, dim3(grid_for(int64_t(batch) * vf.nodes() * cq)), dim3(kNT), 0, s,
                     in, in_ld, in_off, vc, out, out_ld, out_off, vf, batch, cq);
  return hipGetLastError();
}

hipError_t launch_prolong_bwd(hipStream_t s, const uint16_t* dfine, int f_ld, int f_off, Vol vf,
                              uint16_t* dcoarse, int c_ld, int c_off, Vol vc, int batch, int c) {
  if ((c & 3) || vf.nx != 2 * vc.nx - 1 || vf.ny != 2 * vc.ny - 1 || vf.nz != 2 * vc.nz - 1)
    return hipErrorInvalidValue;
  const int cq = c >> 2;
  hipLaunchKernelGGL(k_prolong_bwd, dim3(grid_for(int64_t(batch) * vc.nodes() * cq)), dim3(kNT), 0,
                     s, dfine, f_ld, f_off, vf, dcoarse, c_ld, c_off, vc, batch, cq);
  return hipGetLastError();
}

hipError_t launch_mse(hipStream_t s, const float* pred, const float* target, int64_t voxels, int c,
                      uint16_t* dpred, float* part, float* loss_dev) {
  if (c < 1 || c > 4) return hipErrorInvalidValue;
  const int nb = grid_for(voxels, 1024);
  hipLaunchKernelGGL(k_mse, dim3(nb), dim3(kNT), 0, s, pred, target, voxels, c, dpred, part);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_mse_finish, dim3(1), dim3(64), 0, s, part, nb, 1.f / float(voxels * c), loss_dev);
  return hipGetLastError();
}

hipError_t launch_adam(hipStream_t s, float* p, const float* g, float* m, float* v, int64_t n,
                       float lr_t, float beta1, float beta2, float eps) {
  hipLaunchKernelGGL(k_adam, dim3(grid_for(n)), dim3(kNT), 0, s, p, g, m, v, n, lr_t, beta1, beta2, eps);
  return hipGetLastError();
}

hipError_t launch_to_dofs(hipStream_t s, const float* pred, const uint16_t* feat, int mask_ch,
                          int base_ch, double base_w, int64_t nodes, double scale, double* x) {
  if (mask_ch < 0 || mask_ch >= 16 || base_ch < -1 || base_ch > 13) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_to_dofs, dim3(grid_for(nodes)), dim3(kNT), 0, s, pred, feat, mask_ch,
                     base_ch, base_w, nodes, scale, x);
  return hipGetLastError();
}

hipError_t launch_fill0(hipStream_t s, void* p, int64_t bytes) {
  if (bytes & 3) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_fill0, dim3(grid_for(bytes / 4)), dim3(kNT), 0, s, static_cast<uint32_t*>(p), bytes / 4);
  return hipGetLastError();
}

}  // namespace nn
}  // namespace gf
