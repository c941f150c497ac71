// Input staging for the MFMA conv path, plus the per-pixel half of the
// SparseFlow prescan and the StaticZero/SparseFlow/DenseKeep route count.
//
// One pass over the fp32 NCHW boundary tensor x[NB][C][H][W] produces:
//   xp   fp16 NHWC x[NB][H][W][Cp] (channels C..Cp-1 zero) — MFMA B operand
//   act  uint32 [NB][H][W]: bit g set iff |x[c]| > thr for some c in
//        channel group g (channels g*GS .. g*GS+GS-1)
//   nnz  count_nonzero(x), published in a count block (cf_count_publish)
//   status |= CF_STATUS_INEXACT_FP16 if some x is not exactly representable
//        in fp16 (the MFMA path multiplies fp16 x by split fp32 weights, so
//        exactness of x is what keeps the contraction fp32-faithful)
// The group-OR per pixel is the channel reduction of the reference prescan
// (catfuse/sparseflow/prescan.py:32-45 _groupwise_amax_last_dim, then
// `> threshold` at :184); the spatial (receptive field, tile) reduction is in
// prescan.hip.  HBM traffic: 4 B read + 2 B (xp) + 4/C B (act) per element.
#include "cf_common.h"

#include <type_traits>

namespace {

constexpr int PX = 64;   // pixels per block
constexpr int CC = 32;   // channels per chunk

// Four consecutive floats at any float's address (one global_load_dwordx4:
// the hardware needs no more than 4-byte alignment).
struct __attribute__((packed, aligned(4))) f32x4u {
  float v[4];
};

// Workgroup: 64 pixels x a run of TC-channel tiles (64, or 32 for copies of one
// 32-channel group).  Bound by HBM; what it needs is bytes in flight, so a tile's
// floats of a thread are loaded together (TC = 64: four 16-byte loads along the
// pixels, two channel pairs of four pixels), and without `act` (whose bits need a
// pixel's every channel in one workgroup) each tile is a workgroup of its own
// (grid z).  A channel pair's halves are one LDS word, in rows of TC / 2 + 1 words a
// pixel: the transposing writes and the row reads both touch every bank alike.
// Measured (MI355X), against one workgroup walking a pixel block's channels
// 32 at a time with 4-byte loads: 128 images of 256 x 14 x 14 33.4 -> 12.1 us,
// of 64 x 56 x 56 (154 MB moved) 61 -> 29.6 us.
template <bool ACT, int TC>
__global__ __launch_bounds__(256) void pack_kernel(
    const float* __restrict__ x, int64_t C, int64_t HW, int64_t Cp, _Float16* __restrict__ xp,
    uint32_t* __restrict__ act, int gs, float thr, unsigned long long* __restrict__ nnz,
    uint32_t* __restrict__ status) {
  typedef _Float16 h2 __attribute__((ext_vector_type(2)));
  constexpr int LD = TC / 2 + 1;   // words of a pixel's row
  constexpr int NI = TC / 32;      // channel pairs of a thread
  // Channels past C neither loaded nor converted: of one group they may be most;
  // in a run of tiles the branch costs more (2 x 2048 x 56 x 56 with `act` 58 -> 65 us).
  constexpr bool SKIP = TC == 32;
  __shared__ uint32_t tile[PX * LD];
  __shared__ uint32_t bits_sh[PX];
  __shared__ unsigned int cnt_sh;
  __shared__ unsigned int inexact_sh;
  const int tid = threadIdx.x;
  const int64_t n = blockIdx.y;
  const int64_t hw0 = (int64_t)blockIdx.x * PX;
  const int p0 = (tid % 16) * 4;   // first of the four pixels of the load phase
  const int cr = tid / 16;         // channel pair of the load phase (and cr + 16)
  const int64_t left = HW - hw0 - p0;  // real pixels from p0 on (may be <= 0)
  if (tid == 0) { cnt_sh = 0; inexact_sh = 0; }
  if (ACT && tid < PX) bits_sh[tid] = 0u;
  uint32_t mybits[4] = {0u, 0u, 0u, 0u};
  unsigned int mycnt = 0;
  bool myinexact = false;
  const float* xn = x + n * C * HW + hw0 + p0;
  __syncthreads();
  for (int64_t c0 = (int64_t)blockIdx.z * TC; c0 < Cp; c0 += (int64_t)gridDim.z * TC) {
    float v[NI][2][4];
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int64_t c = c0 + 2 * (cr + 16 * i) + u;
        const float* src = xn + c * HW;
        if (SKIP && c >= C) {
#pragma unroll
          for (int j = 0; j < 4; ++j) v[i][u][j] = 0.0f;
        } else if (c < C && left >= 4) {
          const f32x4u q = *reinterpret_cast<const f32x4u*>(src);
#pragma unroll
          for (int j = 0; j < 4; ++j) v[i][u][j] = q.v[j];
        } else {
#pragma unroll
          for (int j = 0; j < 4; ++j) v[i][u][j] = (c < C && j < left) ? src[j] : 0.0f;
        }
      }
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int w = cr + 16 * i;
      if (SKIP && c0 + 2 * w >= C) {
#pragma unroll
        for (int j = 0; j < 4; ++j) tile[(p0 + j) * LD + w] = 0u;
        continue;
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        h2 h;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const float f = v[i][u][j];
          h[u] = (_Float16)f;
          myinexact |= ((float)h[u] != f);
          mycnt += (f != 0.0f) ? 1u : 0u;
          if (ACT) {
            // (at most 32 groups of gs channels: c fits 32 bits)
            const uint32_t c = (uint32_t)(c0 + 2 * w + u);
            if (fabsf(f) > thr && c < (uint32_t)C) mybits[j] |= 1u << (c / (uint32_t)gs);
          }
        }
        tile[(p0 + j) * LD + w] = __builtin_bit_cast(uint32_t, h);
      }
    }
    __syncthreads();
    if (xp) {
      // write phase: TC / 8 threads per pixel, 8 channels (16 B) each
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int wp = tid / (TC / 8) + 32 * i, part = tid % (TC / 8);
        if (hw0 + wp < HW && c0 + part * 8 < Cp) {
          const uint32_t* r = &tile[wp * LD + part * 4];
          *reinterpret_cast<uint4*>(xp + ((n * HW + hw0 + wp) * Cp + c0 + part * 8)) =
              make_uint4(r[0], r[1], r[2], r[3]);
        }
      }
    }
    __syncthreads();
  }
  if (ACT) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (mybits[j]) atomicOr(&bits_sh[p0 + j], mybits[j]);
    __syncthreads();
    if (tid < PX && hw0 + tid < HW) act[n * HW + hw0 + tid] = bits_sh[tid];
  }
  if (nnz) {
    // wave-level reduction, then one shared atomic per wave
    unsigned int c = mycnt;
    for (int off = 32; off > 0; off >>= 1) c += __shfl_xor(c, off, 64);
    if ((tid & 63) == 0) atomicAdd(&cnt_sh, c);
  }
  if (myinexact) atomicOr(&inexact_sh, 1u);
  __syncthreads();
  if (tid == 0) {
    if (nnz)
      cf_count_publish(nnz, cnt_sh,
                       blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z),
                       gridDim.x * gridDim.y * gridDim.z);
    if (status && inexact_sh) atomicOr(status, (uint32_t)CF_STATUS_INEXACT_FP16);
  }
}

// The same activity bits and nonzero count from an fp16 NHWC copy that a
// fused conv already wrote (xp[NPIX][Cp], channels >= C zero), so a
// SparseFlow layer whose input carries one needs no fp32 pass.  Sixteen
// lanes per pixel, each reading 16-byte chunks c8 = lane, lane + 16, ... (a
// pixel's channels are one contiguous run, so a 16-lane group reads 256
// contiguous bytes per load); group sizes are multiples of 8, so the 8
// channels of a chunk share one group, and the pixel's bits are OR-reduced
// over its 16 lanes.  Grid-stride over pixels; the count is published with
// one atomic per block.
// Activity bits and nonzero count of an fp16 NHWC copy.  LP lanes share a
// pixel (LP = Cp/8 capped at 16, a power of two: every lane of a wave busy),
// each reading 16-byte chunks of 8 channels; a thread takes two pixels per
// iteration (two loads in flight).  The tests work on the halves' bits: a
// half is nonzero iff its magnitude bits are (so -0 counts as zero, as
// v != 0.0f), and |v| > thr iff its magnitude bits exceed thr_mag (the bits
// of the largest fp16 magnitude <= thr; -1 when thr < 0) and are not a NaN
// (<= 0x7c00), the order of non-negative fp16 values being that of their
// bits.  Each chunk lies in one channel group (gs is a multiple of 8).
template <int LP>
__global__ __launch_bounds__(256) void scan_nhwc_kernel(
    const _Float16* __restrict__ xp, int64_t npix, int Cp, int C, uint32_t* __restrict__ act,
    int gs, int thr_mag, unsigned long long* __restrict__ nnz) {
  typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
  constexpr int PPB = 256 / LP;   // pixels of a block per half-iteration
  __shared__ unsigned int cnt_sh;
  const int tid = threadIdx.x, sub = tid % LP;
  if (tid == 0) cnt_sh = 0;
  __syncthreads();
  unsigned int cnt = 0;
  const int nc8 = Cp / 8;
  for (int64_t p0 = (int64_t)blockIdx.x * 2 * PPB; p0 < npix; p0 += (int64_t)gridDim.x * 2 * PPB) {
    int64_t pp[2];
    uint32_t bits[2] = {0u, 0u};
#pragma unroll
    for (int u = 0; u < 2; ++u) pp[u] = p0 + u * PPB + tid / LP;
    for (int c8 = sub; c8 < nc8; c8 += LP) {
      u32x4 v[2];
#pragma unroll
      for (int u = 0; u < 2; ++u)
        v[u] = pp[u] < npix ? *reinterpret_cast<const u32x4*>(xp + pp[u] * Cp + c8 * 8)
                            : u32x4{0u, 0u, 0u, 0u};
      const int nreal = C - c8 * 8;   // real channels in the chunk (may be <= 0 or >= 8)
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        bool any = false;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const int lo = (int)(v[u][k] & 0x7fffu), hi = (int)((v[u][k] >> 16) & 0x7fffu);
          cnt += (lo != 0 ? 1u : 0u) + (hi != 0 ? 1u : 0u);
          any |= (lo > thr_mag && lo <= 0x7c00 && 2 * k < nreal) ||
                 (hi > thr_mag && hi <= 0x7c00 && 2 * k + 1 < nreal);
        }
        if (any) bits[u] |= 1u << (unsigned)((c8 * 8) / gs);
      }
    }
    // the LP lanes of a pixel share it, so this reduction stays in bounds
#pragma unroll
    for (int u = 0; u < 2; ++u) {
#pragma unroll
      for (int off = LP / 2; off > 0; off >>= 1) bits[u] |= __shfl_xor(bits[u], off, LP);
      if (act && pp[u] < npix && sub == 0) act[pp[u]] = bits[u];
    }
  }
  if (nnz) {
    for (int off = 32; off > 0; off >>= 1) cnt += __shfl_xor(cnt, off, 64);
    if ((tid & 63) == 0) atomicAdd(&cnt_sh, cnt);
    __syncthreads();
    if (tid == 0) cf_count_publish(nnz, cnt_sh, blockIdx.x, gridDim.x);
  }
}

// fp16 NHWC [NB][HW][cp] -> fp32 NCHW [NB][C][HW]: materialises the fp32
// view of a fused conv output that was kept only as its NHWC copy, read where
// its producer left it (desc, nullable: an all-zero copy gives zeros).  What
// reading through the descriptor saves is the launch that filled unwritten
// copies first, 4.5 us of the GPU's time and 5 of the host's.
// XT: the copy's element, fp16 or one byte per channel (uint8_t).
//
// A block moves 64 pixels x 32 channels through LDS (reads: 64-byte runs per
// pixel; writes: 256-byte runs per channel, a wave's 4-byte stores side by
// side), or the wide form below (nhwc_to_nchw says where).
template <typename XT>
__global__ __launch_bounds__(256) void nhwc_to_nchw_kernel(
    const XT* __restrict__ xp_own, const CfOutDesc* __restrict__ desc, float* __restrict__ out,
    int64_t C, int64_t HW, int64_t cp) {
  typedef XT x8 __attribute__((ext_vector_type(8)));
  __shared__ float tile[CC][PX + 1];
  const int tid = threadIdx.x;
  const XT* const xp = cf_copy_source(desc, xp_own);
  const int64_t n = blockIdx.z;
  const int64_t hw0 = (int64_t)blockIdx.x * PX;
  const int64_t c0 = (int64_t)blockIdx.y * CC;
  {
    // read: 4 threads per pixel, 8 channels (16 or 8 bytes) each
    const int px = tid / 4, part = tid % 4;
    x8 v = {};
    if (xp != nullptr && hw0 + px < HW && c0 + part * 8 < cp)
      v = *reinterpret_cast<const x8*>(xp + ((n * HW + hw0 + px) * cp + c0 + part * 8));
#pragma unroll
    for (int j = 0; j < 8; ++j) tile[part * 8 + j][px] = (float)v[j];
  }
  __syncthreads();
  // write: 64 consecutive pixels of one channel per 64 threads
  const int px = tid % PX;
#pragma unroll
  for (int i = 0; i < CC / 4; ++i) {
    const int cl = tid / PX + 4 * i;
    const int64_t c = c0 + cl;
    if (c < C && hw0 + px < HW) out[(n * C + c) * HW + hw0 + px] = tile[cl][px];
  }
}

// The wide form: 64 pixels x 64 channels, the reverse of pack_kernel: a channel
// pair's halves are one word of a pixel's 33-word row; reads are 128-byte runs
// per pixel, writes 16 bytes (four pixels of a channel) a lane.
template <typename XT>
__global__ __launch_bounds__(256) void nhwc_to_nchw_wide_kernel(
    const XT* __restrict__ xp_own, const CfOutDesc* __restrict__ desc, float* __restrict__ out,
    int64_t C, int64_t HW, int64_t cp) {
  typedef XT x8 __attribute__((ext_vector_type(8)));
  typedef _Float16 h2 __attribute__((ext_vector_type(2)));
  constexpr int TC = 64, LD = TC / 2 + 1;
  __shared__ uint32_t tile[PX * LD];
  const int tid = threadIdx.x;
  const XT* const xp = cf_copy_source(desc, xp_own);
  const int64_t n = blockIdx.z;
  const int64_t hw0 = (int64_t)blockIdx.x * PX;
  const int64_t c0 = (int64_t)blockIdx.y * TC;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    // 8 threads per pixel, 8 channels (16 or 8 bytes) each
    const int px = tid / 8 + 32 * i, part = tid % 8;
    x8 v = {};
    if (xp != nullptr && hw0 + px < HW && c0 + part * 8 < cp)
      v = *reinterpret_cast<const x8*>(xp + ((n * HW + hw0 + px) * cp + c0 + part * 8));
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const h2 h = {(_Float16)v[2 * j], (_Float16)v[2 * j + 1]};   // bytes are exact in fp16
      tile[px * LD + part * 4 + j] = __builtin_bit_cast(uint32_t, h);
    }
  }
  __syncthreads();
  const int p0 = (tid % 16) * 4;
  const int64_t left = HW - hw0 - p0;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int w = tid / 16 + 16 * i;
    h2 h[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) h[j] = __builtin_bit_cast(h2, tile[(p0 + j) * LD + w]);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int64_t c = c0 + 2 * w + u;
      if (c >= C) continue;
      float* dst = out + (n * C + c) * HW + hw0 + p0;
      if (left >= 4) {
        f32x4u q;
#pragma unroll
        for (int j = 0; j < 4; ++j) q.v[j] = (float)h[j][u];
        *reinterpret_cast<f32x4u*>(dst) = q;
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (j < left) dst[j] = (float)h[j][u];
      }
    }
  }
}

// Global average pool of an fp16 NHWC copy xp [NB][HW][cp]: out[n][c] =
// (sum over the HW pixels of xp[n][p][c]) * factor, factor = float(1)/HW --
// torch's mean on the GPU (an fp32 sum, then a multiply by float(1)/count).
// The copies this reads hold integers (spikes, SEW sums), whose fp32 sum is
// exact in any order.  Block (n, 512-channel slice); a thread sums two
// adjacent channels (one 4-byte load per pixel, 1 KB per pixel per block).
template <typename XT>
__global__ __launch_bounds__(256) void global_avgpool_nhwc_kernel(
    const XT* __restrict__ xp, const CfOutDesc* desc, float* __restrict__ out, int64_t HW,
    int C, int cp, float factor) {
  // Workgroup: image n, 64 channels; thread (g, j) sums channels c, c + 1
  // (c = 64 * blockIdx.y + 2 j) over pixels g, g + 8, ...; the eight
  // partial sums meet in LDS.  The copy's values are small integers, so
  // every partial sum is exact and the order of the additions does not
  // change the result.
  typedef XT h2 __attribute__((ext_vector_type(2)));
  __shared__ float red[8][64];
  const int64_t n = blockIdx.x;
  const int g = (int)threadIdx.x >> 5, j = (int)threadIdx.x & 31;
  const int c = (int)blockIdx.y * 64 + 2 * j;
  const XT* base = cf_copy_source(desc, xp);   // nullptr: all zero
  float s0 = 0.0f, s1 = 0.0f;
  if (base != nullptr && c < C) {
    const XT* src = base + n * HW * cp + c;
#pragma unroll 4
    for (int64_t p = g; p < HW; p += 8) {
      const h2 v = *reinterpret_cast<const h2*>(src + p * cp);
      s0 += (float)v[0];
      s1 += (float)v[1];
    }
  }
  red[g][2 * j] = s0;
  red[g][2 * j + 1] = s1;
  __syncthreads();
  if (threadIdx.x < 64) {
    const int cc = (int)blockIdx.y * 64 + (int)threadIdx.x;
    float s = 0.0f;
#pragma unroll
    for (int k = 0; k < 8; ++k) s += red[k][threadIdx.x];
    if (cc < C) out[n * C + cc] = s * factor;
  }
}

// Token-major fp32 [NB][P][C] (a transformer's [T, B, N, C] activations)
// -> its fp16 copy [NB][P][cp] (channels C..cp-1 zero), the nonzero count
// (published in a count block) and the exactness status: the staging of a
// fused linear's input, which the matrix-core kernels read as an NHWC image
// of P pixels.  A thread takes U 8-channel chunks a pass (grid-stride).  Bound by
// HBM when large: two chunks, their 16-byte loads in flight together (25,088 rows
// of 384: 22 -> 11.9 us against one chunk in 4-byte loads).  Bound by a launch's
// latency when small: one chunk, whose eight predicated loads are one round
// (681 rows of 5: 4.4 us with two chunks of two load widths, 3.5 so).
template <int U>
__global__ __launch_bounds__(256) void pack_tokens_kernel(
    const float* __restrict__ x, int64_t rows, int C, int cp, _Float16* __restrict__ xp,
    unsigned long long* __restrict__ nnz, uint32_t* __restrict__ status) {
  __shared__ unsigned int cnt_sh;
  __shared__ unsigned int inexact_sh;
  if (threadIdx.x == 0) { cnt_sh = 0; inexact_sh = 0; }
  __syncthreads();
  unsigned int cnt = 0;
  bool inexact = false;
  if constexpr (U == 1) {
    const int nc8 = cp / 8;
    for (int64_t u = (int64_t)blockIdx.x * 256 + threadIdx.x; u < rows * nc8;
         u += (int64_t)gridDim.x * 256) {
      const int64_t r = u / nc8;
      const int c0 = (int)(u % nc8) * 8;
      _Float16 o[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float v = (c0 + j < C) ? x[r * C + c0 + j] : 0.0f;
        const _Float16 hv = (_Float16)v;
        inexact |= ((float)hv != v);
        cnt += (v != 0.0f) ? 1u : 0u;
        o[j] = hv;
      }
      *reinterpret_cast<uint4*>(xp + r * cp + c0) = *reinterpret_cast<const uint4*>(o);
    }
  } else {
    const uint32_t nc8 = (uint32_t)cp / 8u;
    const int64_t units = rows * nc8, step = (int64_t)gridDim.x * 256;
    // (32-bit unit decode wherever it fits: a 64-bit division by a run-time
    // value costs more than the unit's own work)
    const bool small = units + U * step < ((int64_t)1 << 32);
    for (int64_t u0 = (int64_t)blockIdx.x * 256 + threadIdx.x; u0 < units; u0 += U * step) {
      float v[U][8];
      int64_t dst[U];
#pragma unroll
      for (int k = 0; k < U; ++k) {
        const int64_t u = u0 + k * step;
        const bool live = u < units;
        const int64_t r = small ? (int64_t)((uint32_t)u / nc8) : u / nc8;
        const int c0 = (int)(u - r * nc8) * 8;
        dst[k] = live ? r * cp + c0 : -1;
        const float* src = x + r * C + c0;
        if (live && c0 + 8 <= C) {
          const f32x4u q0 = *reinterpret_cast<const f32x4u*>(src);
          const f32x4u q1 = *reinterpret_cast<const f32x4u*>(src + 4);
#pragma unroll
          for (int j = 0; j < 4; ++j) { v[k][j] = q0.v[j]; v[k][4 + j] = q1.v[j]; }
        } else {
#pragma unroll
          for (int j = 0; j < 8; ++j) v[k][j] = (live && c0 + j < C) ? src[j] : 0.0f;
        }
      }
#pragma unroll
      for (int k = 0; k < U; ++k) {
        if (dst[k] < 0) continue;
        _Float16 o[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float f = v[k][j];
          const _Float16 hv = (_Float16)f;
          inexact |= ((float)hv != f);
          cnt += (f != 0.0f) ? 1u : 0u;
          o[j] = hv;
        }
        *reinterpret_cast<uint4*>(xp + dst[k]) = *reinterpret_cast<const uint4*>(o);
      }
    }
  }
  if (nnz) {
    for (int off = 32; off > 0; off >>= 1) cnt += __shfl_xor(cnt, off, 64);
    if ((threadIdx.x & 63) == 0) atomicAdd(&cnt_sh, cnt);
  }
  if (inexact) atomicOr(&inexact_sh, 1u);
  __syncthreads();
  if (threadIdx.x == 0) {
    if (nnz) cf_count_publish(nnz, cnt_sh, blockIdx.x, gridDim.x);
    if (status && inexact_sh) atomicOr(status, (uint32_t)CF_STATUS_INEXACT_FP16);
  }
}

// fp16 [NB][P][cp] -> fp32 [NB][P][C]: the fp32 form of a token-major fused
// output kept only as its fp16 copy.  An element a thread, side by side, or a
// thread takes an 8-channel chunk of a row (one 16-byte load, two 16-byte stores):
// tokens_to_f32 says where.
__global__ __launch_bounds__(256) void tokens_to_f32_kernel(
    const _Float16* __restrict__ xp_own, const CfOutDesc* __restrict__ desc,
    float* __restrict__ out, int64_t rows, int C, int cp) {
  const _Float16* const xp = cf_copy_source(desc, xp_own);   // nullptr: all zero
  const int64_t e0 = (int64_t)blockIdx.x * 256 + threadIdx.x, step = (int64_t)gridDim.x * 256;
  if (xp == nullptr) {
    for (int64_t e = e0; e < rows * C; e += step) out[e] = 0.0f;
    return;
  }
  for (int64_t e = e0; e < rows * C; e += step) {
    const int64_t r = e / C;
    const int c = (int)(e % C);
    out[e] = (float)xp[r * cp + c];
  }
}

__global__ __launch_bounds__(256) void tokens_to_f32_chunks_kernel(
    const _Float16* __restrict__ xp_own, const CfOutDesc* __restrict__ desc,
    float* __restrict__ out, int64_t rows, int C, int cp) {
  const _Float16* const xp = cf_copy_source(desc, xp_own);   // nullptr: all zero
  const uint32_t nc8 = (uint32_t)(C + 7) / 8u;
  const int64_t units = rows * nc8, step = (int64_t)gridDim.x * 256;
  const bool small = units + step < ((int64_t)1 << 32);   // 32-bit unit decode
  // (rows of cp halves are 16-byte aligned where cp is a multiple of 8)
  const bool vec = cp % 8 == 0 && ((uintptr_t)xp & 15) == 0;
  for (int64_t u = (int64_t)blockIdx.x * 256 + threadIdx.x; u < units; u += step) {
    const int64_t r = small ? (int64_t)((uint32_t)u / nc8) : u / nc8;
    const int c0 = (int)(u - r * nc8) * 8;
    const _Float16* src = xp + r * cp + c0;
    float* dst = out + r * C + c0;
    if (vec && c0 + 8 <= C) {
      typedef _Float16 h8 __attribute__((ext_vector_type(8)));
      const h8 h = xp != nullptr ? *reinterpret_cast<const h8*>(src) : h8{};
      f32x4u q0, q1;
#pragma unroll
      for (int j = 0; j < 4; ++j) { q0.v[j] = (float)h[j]; q1.v[j] = (float)h[4 + j]; }
      *reinterpret_cast<f32x4u*>(dst) = q0;
      *reinterpret_cast<f32x4u*>(dst + 4) = q1;
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (c0 + j < C) dst[j] = xp != nullptr ? (float)src[j] : 0.0f;
    }
  }
}

// A plain Linear (no neuron) over a token-major fused output kept only as
// its fp16 copy (a network's last classifier layer after a fused
// Linear-LIF): out[m][o] = bias[o] + sum_k x[m][k] * w[o][k] in fp32, x read
// through the copy's output descriptor (an all-zero copy gives the bias).
// One workgroup per row: its 256 threads take every 256th k (coalesced
// weight rows), OB outputs a pass; the partial sums are reduced in a
// fixed tree (lanes, then waves in order), so the result is deterministic.
// Spike values are small integers; a zero leaves the sums as they are (exact,
// whatever the weight).  Bound by latency: a thread loads the weights of KB
// k's together, beside their spikes (VGG-11's head, 256 rows of 4096 -> 10: 48.6 ->
// 13 us, where each k waited for its own).  At every output pass after the first
// a wave skips the groups of KB k's whose spikes are all zero in it (`live`, a bit
// a group): 32 silent rows of 2048 -> 1000 334 us without, 124 so.  (In the first
// pass a silent row costs what a live one does: 256 rows of 2048 -> 10 6.1 us, where
// looking at the spikes first takes silent ones 5.8 and live ones 7.0.)  OB 4 for a
// last pass of few outputs, KB 1 or 2 for rows of at most 256 or 512: no loads of
// weights that are not used (1024 rows of 2048 -> 1 11.0 -> 6.7 us).
template <int OB, int KB>
__device__ __forceinline__ void linear_tokens_sum(const _Float16* __restrict__ xr,
                                                  const float* __restrict__ w, int K, int no,
                                                  bool mark, bool skip, uint64_t& live,
                                                  float* acc) {
  int g = 0;
  for (int k0 = threadIdx.x; k0 < K; k0 += 256 * KB, ++g) {
    if (skip && g < 64 && ((live >> g) & 1ull) == 0ull) continue;
    float xv[KB], wv[KB][OB];
#pragma unroll
    for (int u = 0; u < KB; ++u) {
      const int k = k0 + 256 * u;
      xv[u] = k < K ? (float)xr[k] : 0.0f;
      // (a row or column beyond the matrix repeats one inside it, unused)
      const float* wk = w + (k < K ? k : k0);
#pragma unroll
      for (int j = 0; j < OB; ++j) wv[u][j] = wk[(size_t)(j < no ? j : 0) * K];
    }
    bool nz = false;
#pragma unroll
    for (int u = 0; u < KB; ++u) {
      nz |= xv[u] != 0.0f;
#pragma unroll
      for (int j = 0; j < OB; ++j) acc[j] = xv[u] != 0.0f ? fmaf(xv[u], wv[u][j], acc[j]) : acc[j];
    }
    if (mark && g < 64 && __any(nz ? 1 : 0)) live |= 1ull << g;
  }
}

constexpr int LT_OB = 16;
template <int KB>
__global__ __launch_bounds__(256) void linear_tokens_kernel(
    const _Float16* __restrict__ xp, const CfOutDesc* __restrict__ desc,
    const float* __restrict__ w, const float* __restrict__ bias, float* __restrict__ out,
    int K, int cp, int O) {
  __shared__ float red[4][LT_OB];
  const int m = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const _Float16* xs = cf_copy_source(desc, xp);
  const _Float16* xr = xs != nullptr ? xs + (size_t)m * cp : nullptr;
  uint64_t live = 0ull;
  auto pass = [&](auto ob_c, int o0) {
    constexpr int OB = decltype(ob_c)::value;
    const float* wo = w + (size_t)o0 * K;
    const int no = O - o0 < OB ? O - o0 : OB;
    float acc[OB];
#pragma unroll
    for (int j = 0; j < OB; ++j) acc[j] = 0.0f;
    // (the first pass marks the live groups for those that follow)
    if (xr != nullptr)
      linear_tokens_sum<OB, KB>(xr, wo, K, no, o0 == 0 && O > LT_OB, o0 > 0, live, acc);
#pragma unroll
    for (int j = 0; j < OB; ++j)
#pragma unroll
      for (int off = 32; off >= 1; off >>= 1) acc[j] += __shfl_xor(acc[j], off, 64);
    if (lane == 0) {
#pragma unroll
      for (int j = 0; j < OB; ++j) red[wave][j] = acc[j];
    }
    __syncthreads();
    if (tid < OB && o0 + tid < O) {
      const float s = ((red[0][tid] + red[1][tid]) + red[2][tid]) + red[3][tid];
      out[(size_t)m * O + o0 + tid] = bias != nullptr ? bias[o0 + tid] + s : s;
    }
    __syncthreads();   // red is rewritten by the next pass
  };
  for (int o0 = 0; o0 < O; o0 += LT_OB) {
    if (O - o0 > 4) pass(std::integral_constant<int, LT_OB>{}, o0);
    else pass(std::integral_constant<int, 4>{}, o0);
  }
}

// Max pooling of an fp16 NHWC copy (the spikes a fused conv wrote):
// out[n][oh][ow][c] = max over the k x k window (stride s, padding p; padded
// positions ignored, as torch's max_pool2d) of xp[n][ih][iw][c].  The max of
// spike values is exact in fp16.  One 8-channel chunk of one output pixel
// per thread; the nonzero count of the output is published (count block).
// KC, SC, PC: the window, stride and padding of the usual pool (3, 2, 1), whose
// nine loads are then in flight together (a window position outside the
// input repeats the centre, which is inside it and changes no maximum); 0: as
// the arguments say.  32 x 112 x 112 x 96: 32 -> 26 us, 32 x 56 x 56 x 192
// 20.6 -> 13.6, 4 x 28 x 28 x 384 8.2 -> 4.6.
template <int KC, int SC, int PC>
__global__ __launch_bounds__(256) void maxpool_nhwc_kernel(
    const _Float16* __restrict__ xp_own, const CfOutDesc* __restrict__ in_desc,
    _Float16* __restrict__ out, CfOutDesc* __restrict__ out_desc, int64_t NB, int H, int W,
    int Ho, int Wo, int cp, int k, int s, int p, unsigned long long* __restrict__ nnz) {
  typedef _Float16 h8 __attribute__((ext_vector_type(8)));
  __shared__ unsigned any_sh[4];
  // the input where its producer left it; an all-zero input pools to an
  // all-zero output, which is then recorded in out_desc instead of written
  const _Float16* const xp = cf_copy_source(in_desc, xp_own);
  if (xp == nullptr && out_desc != nullptr) {
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      if (nnz) nnz[1] = 0ull;
      out_desc->copy = CF_COPY_ZERO;
      out_desc->vstate = 0u;
      out_desc->alias = nullptr;
    }
    return;
  }
  if (out_desc != nullptr && blockIdx.x == 0 && threadIdx.x == 0) {
    out_desc->copy = CF_COPY_WRITTEN;
    out_desc->vstate = 0u;
    out_desc->alias = nullptr;
  }
  const int nc8 = cp / 8;
  const int64_t units = NB * Ho * Wo * nc8;
  // unit decode in 32-bit arithmetic (the host keeps units below 2^31):
  // 64-bit divisions by run-time values cost far more than the pool itself
  const uint32_t HoWo = (uint32_t)(Ho * Wo);
  uint32_t anyw = 0u;
  for (uint32_t u = blockIdx.x * 256u + threadIdx.x; u < (uint32_t)units; u += gridDim.x * 256u) {
    const uint32_t pix = u / (uint32_t)nc8;
    const int c8 = (int)(u - pix * (uint32_t)nc8);
    const uint32_t n32 = pix / HoWo, r = pix - n32 * HoWo;
    const int oh = (int)(r / (uint32_t)Wo), ow = (int)(r - (uint32_t)oh * (uint32_t)Wo);
    const int64_t n = n32;
    h8 m;
    if constexpr (KC != 0) {
      static_assert(PC < KC && SC <= KC, "the window's centre lies inside the input");
      h8 v[KC * KC];
#pragma unroll
      for (int dy = 0; dy < KC; ++dy)
#pragma unroll
        for (int dx = 0; dx < KC; ++dx) {
          int ih = oh * SC - PC + dy, iw = ow * SC - PC + dx;
          if (ih < 0 || ih >= H) ih = oh * SC - PC + KC / 2;
          if (iw < 0 || iw >= W) iw = ow * SC - PC + KC / 2;
          v[dy * KC + dx] =
              xp != nullptr
                  ? *reinterpret_cast<const h8*>(xp + ((n * H + ih) * W + iw) * cp + c8 * 8)
                  : h8{};
        }
      m = v[0];
#pragma unroll
      for (int q = 1; q < KC * KC; ++q)
#pragma unroll
        for (int j = 0; j < 8; ++j) m[j] = v[q][j] > m[j] ? v[q][j] : m[j];
    } else {
    bool first = true;
    for (int dy = 0; dy < k; ++dy) {
      const int ih = oh * s - p + dy;
      if (ih < 0 || ih >= H) continue;
      for (int dx = 0; dx < k; ++dx) {
        const int iw = ow * s - p + dx;
        if (iw < 0 || iw >= W) continue;
        const h8 v = xp != nullptr
                         ? *reinterpret_cast<const h8*>(xp + ((n * H + ih) * W + iw) * cp + c8 * 8)
                         : h8{};
        if (first) {
          m = v;
          first = false;
        } else {
#pragma unroll
          for (int j = 0; j < 8; ++j) m[j] = v[j] > m[j] ? v[j] : m[j];
        }
      }
    }
    }
    const uint4 w = __builtin_bit_cast(uint4, m);
    anyw |= (w.x | w.y | w.z | w.w) & 0x7fff7fffu;
    *reinterpret_cast<h8*>(out + (size_t)pix * cp + c8 * 8) = m;
  }
  if (nnz) {
    const bool any = cf_wg_any(anyw != 0u, any_sh);
    if (threadIdx.x == 0) cf_count_publish(nnz, any ? 1ull : 0ull, blockIdx.x, gridDim.x);
  }
}

__global__ void route_kernel(const unsigned long long* __restrict__ nnz, int64_t numel,
                             double sparse_threshold, int32_t* __restrict__ route) {
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    const unsigned long long k = cf_count_read(nnz);
    int r;
    if (k == 0) r = CF_ROUTE_ZERO;
    else if (1.0 - (double)k / (double)numel > sparse_threshold) r = CF_ROUTE_SPARSE;
    else r = CF_ROUTE_DENSE;
    *route = r;
  }
}

__global__ void zero_u64(unsigned long long* p) { *p = 0ull; }

}  // namespace

CF_API int cf_pack_input(const float* x, int64_t NB, int64_t C, int64_t H, int64_t W,
                         int64_t Cp, void* xp, uint32_t* act, int group_size, float threshold,
                         unsigned long long* nnz, uint32_t* status, void* stream) {
  if (!x || NB < 0 || C <= 0 || H <= 0 || W <= 0) return (int)hipErrorInvalidValue;
  if (xp && (Cp < C || Cp % CC != 0)) return (int)hipErrorInvalidValue;
  if (!xp) Cp = ((C + CC - 1) / CC) * CC;
  if (act && (group_size <= 0 || (C + group_size - 1) / group_size > 32)) return (int)hipErrorInvalidValue;
  if (group_size <= 0) group_size = 32;
  if (NB == 0) return 0;
  if (NB > 65535) return (int)hipErrorInvalidValue;
  const int64_t HW = H * W;
  dim3 grid(cf_blocks(HW, PX), (unsigned)NB, act || Cp > 65535 * 64 ? 1u : cf_blocks(Cp, 64));
  if (nnz && (unsigned long long)grid.x * grid.y * grid.z >= CF_MAX_COUNT_WG)
    grid.z = 1;   // one workgroup walks the channels
  if (nnz && (unsigned long long)grid.x * grid.y >= CF_MAX_COUNT_WG) return (int)hipErrorInvalidValue;
#define CF_PACK(ACT, TC)                                                                          \
  hipLaunchKernelGGL((pack_kernel<ACT, TC>), grid, dim3(256), 0, (hipStream_t)stream, x, C, HW, Cp, \
                     (_Float16*)xp, act, group_size, threshold, nnz, status)
  // (copies of at most 32 channels, 64- / 32-channel tiles: 16 x 3 x 224 x 224 with
  // activity bits 39 / 23.6 us, without 25 / 20.1)
  if (act && Cp <= 32) CF_PACK(true, 32);
  else if (act) CF_PACK(true, 64);
  else if (Cp <= 32) CF_PACK(false, 32);
  else CF_PACK(false, 64);
#undef CF_PACK
  return (int)hipGetLastError();
}

CF_API int cf_scan_nhwc(const void* xp, int64_t NB, int64_t H, int64_t W, int64_t Cp, int64_t C,
                        uint32_t* act, int group_size, float threshold, unsigned long long* nnz,
                        void* stream) {
  if (!xp || NB < 0 || H <= 0 || W <= 0 || C <= 0 || Cp < C || Cp % 8 != 0)
    return (int)hipErrorInvalidValue;
  if (act && (group_size <= 0 || group_size % 8 != 0 || (C + group_size - 1) / group_size > 32))
    return (int)hipErrorInvalidValue;
  if (group_size <= 0) group_size = 32;
  if (threshold != threshold) return (int)hipErrorInvalidValue;   // NaN
  const int64_t npix = NB * H * W;
  if (npix == 0) return 0;
  // bits of the largest fp16 magnitude <= threshold (-1: every value exceeds it)
  int thr_mag = -1;
  if (threshold > 65504.0f) {
    thr_mag = 0x7c00;   // only a larger infinity would exceed it: none
    if (threshold < __builtin_huge_valf()) thr_mag = 0x7bff;
  } else if (threshold == 65504.0f) {
    thr_mag = 0x7bff;
  } else if (threshold >= 0.0f) {
    const _Float16 h = (_Float16)threshold;
    unsigned short b;
    __builtin_memcpy(&b, &h, 2);
    thr_mag = (int)(b & 0x7fffu);
    if ((float)h > threshold) --thr_mag;   // rounded up: the next smaller magnitude
  }
  const int nc8 = (int)(Cp / 8);
  const int lp = nc8 >= 16 ? 16 : (nc8 >= 8 ? 8 : (nc8 >= 4 ? 4 : (nc8 >= 2 ? 2 : 1)));
  const int64_t per_blk = 2 * (256 / lp);
  const int64_t nblk = (npix + per_blk - 1) / per_blk;
  const dim3 grid((unsigned)(nblk < 2048 ? nblk : 2048)), block(256);
  hipStream_t st = (hipStream_t)stream;
  const _Float16* x = (const _Float16*)xp;
  if (lp == 16)
    hipLaunchKernelGGL(scan_nhwc_kernel<16>, grid, block, 0, st, x, npix, (int)Cp, (int)C, act,
                       group_size, thr_mag, nnz);
  else if (lp == 8)
    hipLaunchKernelGGL(scan_nhwc_kernel<8>, grid, block, 0, st, x, npix, (int)Cp, (int)C, act,
                       group_size, thr_mag, nnz);
  else if (lp == 4)
    hipLaunchKernelGGL(scan_nhwc_kernel<4>, grid, block, 0, st, x, npix, (int)Cp, (int)C, act,
                       group_size, thr_mag, nnz);
  else if (lp == 2)
    hipLaunchKernelGGL(scan_nhwc_kernel<2>, grid, block, 0, st, x, npix, (int)Cp, (int)C, act,
                       group_size, thr_mag, nnz);
  else
    hipLaunchKernelGGL(scan_nhwc_kernel<1>, grid, block, 0, st, x, npix, (int)Cp, (int)C, act,
                       group_size, thr_mag, nnz);
  return (int)hipGetLastError();
}

template <typename XT>
static int nhwc_to_nchw(const void* xp, const void* desc, float* out, int64_t NB, int64_t C,
                        int64_t H, int64_t W, int64_t cp, void* stream) {
  if (!xp || !out || NB < 0 || C <= 0 || H <= 0 || W <= 0 || cp < C || cp % 8 != 0 || NB > 65535)
    return (int)hipErrorInvalidValue;
  if (NB == 0) return 0;
  const int64_t HW = H * W;
  // The wide form where its tiles waste no half (an even number of 32-channel
  // groups) and either maps are so small that a tile is mostly channels, or an
  // fp16 copy is so large that the traffic is what bounds it.  Rows of a multiple
  // of 2 KB, or up to 256 bytes less, put the stores of its 16 channels on the same
  // channels of the memory.  Measured after another pass has used the L2 (us, 32
  // channels / wide): 128 x 256 channels of 14 x 14 11.2 / 10.9, 128 x 128 of 28 x 28
  // 16.6 / 14.7, 364 x 48 of 33 x 32 26.0 / 21.7, 30 x 170 of 23 x 31 7.6 / 7.4; but 32 x 384
  // of 14 x 14 5.5 / 6.2, 189 x 64 of 19 x 24 7.3 / 8.9, 32 x 64 of 32 x 32 4.1 / 4.6, 128 x
  // 512 of 7 x 7 6.0 / 6.7, 4096 x 64 of 6 x 5 11.2 / 13.4; one pass after another: 488 x
  // 512 of 2 x 2 8.3 / 6.4, 3906 x 256 of 1 x 1 25 / 14.4, bytes of 128 x 256 of 14 x 14
  // 9.9 / 11.3.
  const int64_t tiles = (HW + PX - 1) / PX * ((C + 63) / 64) * NB;
  const bool wide = (C + CC - 1) / CC % 2 == 0 &&
                    (HW <= 16 ? tiles >= 900
                              : sizeof(XT) == 2 && HW >= 100 && (HW - 1) % 512 < 447 && tiles >= 1050);
  if (wide)
    hipLaunchKernelGGL(nhwc_to_nchw_wide_kernel<XT>,
                       dim3(cf_blocks(HW, PX), (unsigned)((C + 63) / 64), (unsigned)NB), dim3(256),
                       0, (hipStream_t)stream, (const XT*)xp, (const CfOutDesc*)desc, out, C, HW,
                       cp);
  else
    hipLaunchKernelGGL(nhwc_to_nchw_kernel<XT>,
                       dim3(cf_blocks(HW, PX), (unsigned)((C + CC - 1) / CC), (unsigned)NB),
                       dim3(256), 0, (hipStream_t)stream, (const XT*)xp, (const CfOutDesc*)desc, out,
                       C, HW, cp);
  return (int)hipGetLastError();
}

static int tokens_to_f32(const void* xp, const void* desc, float* out, int64_t rows, int64_t C,
                         int64_t cp, void* stream) {
  if (!xp || !out || rows < 0 || C <= 0 || cp < C || rows * cp > ((int64_t)1 << 40))
    return (int)hipErrorInvalidValue;
  if (rows == 0) return 0;
  // Chunks for rows that they fill (after another pass: 4 rows of 512 2.2 -> 1.8 us,
  // 254 of 384 2.4 -> 2.2, 28,661 of 32 3.6 -> 3.0, 50,176 of 384 26 -> 22), but for rows of
  // one (a million of 8 16.2 -> 18.5).  Others cost a second, element-wise round: 784
  // rows of 100 2.6 -> 3.1, 100,000 of 33 6.5 -> 7.2; 50,176 of 257 19.3 -> 17.4.
  const int64_t n = rows * C;
  const bool chunks = C % 8 == 0 ? C >= 16 : C >= 256 && n >= (1 << 23);
  const int64_t units = chunks ? rows * ((C + 7) / 8) : n;
  const int64_t wg = (units + 255) / 256, most = chunks ? 16384 : 4096;
  const dim3 grid((unsigned)(wg < most ? wg : most));
  if (chunks)
    hipLaunchKernelGGL(tokens_to_f32_chunks_kernel, grid, dim3(256), 0, (hipStream_t)stream,
                       (const _Float16*)xp, (const CfOutDesc*)desc, out, rows, (int)C, (int)cp);
  else
    hipLaunchKernelGGL(tokens_to_f32_kernel, grid, dim3(256), 0, (hipStream_t)stream,
                       (const _Float16*)xp, (const CfOutDesc*)desc, out, rows, (int)C, (int)cp);
  return (int)hipGetLastError();
}

CF_API int cf_copy_to_f32(const void* xp, const void* desc, float* out, int64_t NB, int64_t C,
                          int64_t H, int64_t W, int64_t cp, int tokens, void* stream) {
  if (tokens != 0 && tokens != 1) return (int)hipErrorInvalidValue;
  if (tokens) {
    if (NB < 0 || H <= 0 || W <= 0) return (int)hipErrorInvalidValue;
    return tokens_to_f32(xp, desc, out, NB * H * W, C, cp, stream);
  }
  return nhwc_to_nchw<_Float16>(xp, desc, out, NB, C, H, W, cp, stream);
}

CF_API int cf_nhwc_to_nchw(const void* xp, float* out, int64_t NB, int64_t C, int64_t H,
                           int64_t W, int64_t cp, void* stream) {
  return nhwc_to_nchw<_Float16>(xp, nullptr, out, NB, C, H, W, cp, stream);
}

CF_API int cf_nhwc_to_nchw_u8(const void* xp, float* out, int64_t NB, int64_t C, int64_t H,
                              int64_t W, int64_t cp, void* stream) {
  return nhwc_to_nchw<uint8_t>(xp, nullptr, out, NB, C, H, W, cp, stream);
}

template <typename XT>
static int global_avgpool_nhwc(const void* xp, const void* desc, float* out, int64_t NB,
                               int64_t HW, int64_t C, int64_t cp, void* stream) {
  if (!xp || !out || NB < 0 || HW <= 0 || C <= 0 || cp < C || cp % 8 != 0 || NB > INT32_MAX ||
      NB * HW * cp > ((int64_t)1 << 40))
    return (int)hipErrorInvalidValue;
  if (NB == 0) return 0;
  const float factor = 1.0f / (float)HW;
  hipLaunchKernelGGL(global_avgpool_nhwc_kernel<XT>,
                     dim3((unsigned)NB, (unsigned)((C + 63) / 64)), dim3(256), 0,
                     (hipStream_t)stream, (const XT*)xp, (const CfOutDesc*)desc, out, HW, (int)C,
                     (int)cp, factor);
  return (int)hipGetLastError();
}

CF_API int cf_global_avgpool_nhwc(const void* xp, const void* desc, float* out, int64_t NB,
                                  int64_t HW, int64_t C, int64_t cp, void* stream) {
  return global_avgpool_nhwc<_Float16>(xp, desc, out, NB, HW, C, cp, stream);
}

CF_API int cf_global_avgpool_nhwc_u8(const void* xp, const void* desc, float* out, int64_t NB,
                                     int64_t HW, int64_t C, int64_t cp, void* stream) {
  return global_avgpool_nhwc<uint8_t>(xp, desc, out, NB, HW, C, cp, stream);
}

// One-byte copy -> fp16 copy of the same layout (n elements, a multiple of
// 8): for the readers that take fp16 copies only.  Every byte value is exact
// in fp16.
__global__ __launch_bounds__(256) void copy_u8_to_f16_kernel(const uint8_t* __restrict__ src,
                                                             _Float16* __restrict__ dst,
                                                             int64_t n8) {
  typedef uint8_t u8v8 __attribute__((ext_vector_type(8)));
  typedef _Float16 h8v __attribute__((ext_vector_type(8)));
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n8;
       i += (int64_t)gridDim.x * 256) {
    const u8v8 v = *reinterpret_cast<const u8v8*>(src + 8 * i);
    h8v h;
#pragma unroll
    for (int j = 0; j < 8; ++j) h[j] = (_Float16)(float)v[j];
    *reinterpret_cast<h8v*>(dst + 8 * i) = h;
  }
}

CF_API int cf_copy_u8_to_f16(const void* src, void* dst, int64_t n, void* stream) {
  if (!src || !dst || n < 0 || n % 8 != 0) return (int)hipErrorInvalidValue;
  if (n == 0) return 0;
  const int64_t n8 = n / 8;
  const unsigned grid = (unsigned)((n8 + 255) / 256 < 8192 ? (n8 + 255) / 256 : 8192);
  hipLaunchKernelGGL(copy_u8_to_f16_kernel, dim3(grid), dim3(256), 0, (hipStream_t)stream,
                     (const uint8_t*)src, (_Float16*)dst, n8);
  return (int)hipGetLastError();
}

CF_API int cf_pack_tokens(const float* x, int64_t rows, int64_t C, int64_t cp, void* xp,
                          unsigned long long* nnz, uint32_t* status, void* stream) {
  if (!x || !xp || rows < 0 || C <= 0 || cp < C || cp % 8 != 0 || rows * cp > ((int64_t)1 << 40))
    return (int)hipErrorInvalidValue;
  if (rows == 0) return 0;
  const int64_t units = rows * (cp / 8);
  // Two chunks a thread for rows of whole channel groups (after another pass: 4 rows
  // of 512 3.6 -> 3.1 us, 205 of 1536 4.5 -> 4.2, 94,149 of 64 15.3 -> 8.7).  Others have
  // chunks of padding and partial ones, and gain by it only once loads bound the
  // launch: 12,544 rows of 48 (100,352 chunks) 4.4 -> 4.9, of 100 (200,704) 6.5 -> 5.3.
  // (4,096 workgroups hold the card's loads in flight; more only add count-block
  // atomics.)
  if (C % 32 == 0 || (C > 32 && units >= (8 * C >= 7 * cp ? 65536 : 196608)))
    hipLaunchKernelGGL(pack_tokens_kernel<2>,
                       dim3((unsigned)((units + 511) / 512 < 4096 ? (units + 511) / 512 : 4096)),
                       dim3(256), 0, (hipStream_t)stream, x, rows, (int)C, (int)cp, (_Float16*)xp,
                       nnz, status);
  else
    hipLaunchKernelGGL(pack_tokens_kernel<1>,
                       dim3((unsigned)((units + 255) / 256 < 2048 ? (units + 255) / 256 : 2048)),
                       dim3(256), 0, (hipStream_t)stream, x, rows, (int)C, (int)cp, (_Float16*)xp,
                       nnz, status);
  return (int)hipGetLastError();
}

CF_API int cf_tokens_to_f32(const void* xp, float* out, int64_t rows, int64_t C, int64_t cp,
                            void* stream) {
  return tokens_to_f32(xp, nullptr, out, rows, C, cp, stream);
}

CF_API int cf_linear_tokens(const void* xp, const void* desc, const float* w, const float* bias,
                            float* out, int64_t M, int64_t K, int64_t cp, int64_t O,
                            void* stream) {
  if (!xp || !w || !out || M < 0 || M > INT32_MAX || K <= 0 || cp < K || O <= 0 ||
      O > 4096 || K * O > INT32_MAX || (int64_t)M * cp > ((int64_t)1 << 40))
    return (int)hipErrorInvalidValue;
  if (M == 0) return 0;
#define CF_LINEAR(KB)                                                                         \
  hipLaunchKernelGGL(linear_tokens_kernel<KB>, dim3((unsigned)M), dim3(256), 0,               \
                     (hipStream_t)stream, (const _Float16*)xp, (const CfOutDesc*)desc, w, bias, \
                     out, (int)K, (int)cp, (int)O)
  if (K <= 256) CF_LINEAR(1);
  else if (K <= 512) CF_LINEAR(2);
  else CF_LINEAR(4);
#undef CF_LINEAR
  return (int)hipGetLastError();
}

CF_API int cf_maxpool_nhwc(const void* xp, const void* in_desc, void* out, void* out_desc,
                           int64_t NB, int64_t H, int64_t W,
                           int64_t cp, int64_t kernel_size, int64_t stride, int64_t padding,
                           unsigned long long* nz_out, void* stream) {
  if (!xp || !out || NB < 0 || H <= 0 || W <= 0 || cp <= 0 || cp % 8 != 0 || kernel_size <= 0 ||
      stride <= 0 || padding < 0 || 2 * padding > kernel_size || NB * H * W * cp > ((int64_t)1 << 40))
    return (int)hipErrorInvalidValue;
  const int64_t Ho = (H + 2 * padding - kernel_size) / stride + 1;
  const int64_t Wo = (W + 2 * padding - kernel_size) / stride + 1;
  if (Ho <= 0 || Wo <= 0) return (int)hipErrorInvalidValue;
  if (NB == 0) return 0;
  const int64_t units = NB * Ho * Wo * (cp / 8);
  if (units >= ((int64_t)1 << 31)) return (int)hipErrorInvalidValue;   // 32-bit unit indices
  // about one unit a thread (more loads in flight than a grid-stride loop)
  const unsigned grid = (unsigned)((units + 255) / 256 < 65536 ? (units + 255) / 256 : 65536);
  // (floor mode: the centre of a (3, 2, 1) window, row 2 oh and column 2 ow,
  // is inside the input)
  if (kernel_size == 3 && stride == 2 && padding == 1)
    hipLaunchKernelGGL((maxpool_nhwc_kernel<3, 2, 1>), dim3(grid), dim3(256), 0,
                       (hipStream_t)stream, (const _Float16*)xp, (const CfOutDesc*)in_desc,
                       (_Float16*)out, (CfOutDesc*)out_desc, NB, (int)H, (int)W, (int)Ho, (int)Wo,
                       (int)cp, 3, 2, 1, nz_out);
  else
    hipLaunchKernelGGL((maxpool_nhwc_kernel<0, 0, 0>), dim3(grid), dim3(256), 0,
                       (hipStream_t)stream, (const _Float16*)xp, (const CfOutDesc*)in_desc,
                       (_Float16*)out, (CfOutDesc*)out_desc, NB, (int)H, (int)W, (int)Ho, (int)Wo,
                       (int)cp, (int)kernel_size, (int)stride, (int)padding, nz_out);
  return (int)hipGetLastError();
}

// Route word from the nonzero count, exactly the host formula of
// catfuse/sparseflow/ops/st_fusion_conv_bn_lif.py:510-524 evaluated in double.
CF_API int cf_route_from_nnz(const unsigned long long* nnz, int64_t numel,
                             double sparse_threshold, int32_t* route, void* stream) {
  if (!nnz || !route || numel <= 0) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(route_kernel, dim3(1), dim3(64), 0, (hipStream_t)stream, nnz, numel,
                     sparse_threshold, route);
  return (int)hipGetLastError();
}

// Clears a 64-bit device counter with a kernel (graph-capture safe: no memset node).
CF_API int cf_zero_counter(unsigned long long* p, void* stream) {
  if (!p) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(zero_u64, dim3(1), dim3(1), 0, (hipStream_t)stream, p);
  return (int)hipGetLastError();
}

namespace {

// Fills a copy buffer its producer did not write (descriptor ZERO: zeros;
// ALIAS: the aliased copy's bytes); a written copy is left alone.  16-byte
// units, grid-stride.
__global__ __launch_bounds__(256) void resolve_copy_kernel(uint4* __restrict__ buf, int64_t n16,
                                                           const CfOutDesc* desc) {
  const uint32_t st = desc->copy;
  if (st != CF_COPY_ZERO && st != CF_COPY_ALIAS) return;
  const uint4* src = reinterpret_cast<const uint4*>(desc->alias);
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n16;
       i += (int64_t)gridDim.x * 256)
    buf[i] = st == CF_COPY_ALIAS ? src[i] : make_uint4(0u, 0u, 0u, 0u);
}

// v [B][C][HW] from the per-channel potentials when the descriptor says the
// producer kept the state per channel (vstate 1); otherwise v is left alone.
__global__ __launch_bounds__(256) void expand_state_kernel(float* __restrict__ v,
                                                           const float* __restrict__ v_chan,
                                                           const CfOutDesc* desc, int64_t n,
                                                           int C, int64_t HW) {
  if (desc->vstate != 1u) return;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * 256)
    v[i] = v_chan[(int)((i / HW) % C)];
}

}  // namespace

CF_API int cf_resolve_copy(void* buf, int64_t bytes, const void* desc, void* stream) {
  if (!buf || !desc || bytes < 0 || bytes % 16 != 0 || ((uintptr_t)buf & 15) != 0)
    return (int)hipErrorInvalidValue;
  if (bytes == 0) return 0;
  const int64_t n16 = bytes / 16;
  const unsigned nb = cf_blocks(n16, 256), grid = nb < 2048u ? nb : 2048u;
  hipLaunchKernelGGL(resolve_copy_kernel, dim3(grid), dim3(256), 0, (hipStream_t)stream,
                     (uint4*)buf, n16, (const CfOutDesc*)desc);
  return (int)hipGetLastError();
}

CF_API int cf_expand_state(float* v, const float* v_chan, const void* desc, int64_t B, int64_t C,
                           int64_t HW, void* stream) {
  if (!v || !v_chan || !desc || B < 0 || C <= 0 || HW <= 0 || C > INT32_MAX)
    return (int)hipErrorInvalidValue;
  const int64_t n = B * C * HW;
  if (n == 0) return 0;
  const unsigned nb = cf_blocks(n, 256), grid = nb < 2048u ? nb : 2048u;
  hipLaunchKernelGGL(expand_state_kernel, dim3(grid), dim3(256), 0, (hipStream_t)stream, v,
                     v_chan, (const CfOutDesc*)desc, n, (int)C, HW);
  return (int)hipGetLastError();
}
