// Spiking self-attention core with its LIF (Spikformer SSA: Q K^T V * scale,
// then attn_lif), on the matrix cores.
//
// Reference: models/spikformer_github.py:139-160 (SSA.forward: q, k, v are
// spike tensors [T, B, heads, N, dh]; attn = (q @ k^T) * scale; y = attn @ v;
// attn_lif over T).  There is no softmax, so for binary Q, K, V the product
// is evaluated as Q (K^T V):
//   KV = K^T V   dh x dh integers <= N: exact as fp32 sums, then as fp16
//                (N <= 2048) for the second product;
//   Y  = Q KV    N x dh integers <= N * dh: exact in the fp32 accumulators;
//   z  = Y * scale, one rounding; the LIF over T with v in registers.
// The reference's fp32 evaluation rounds attn and every partial sum of
// attn @ v; this one rounds once, so z differs from it by rounding only.
//
// Layouts (token-major, the fp16 NHWC copies of the fused linears): q, k, v
// are fp16 [T*B][N][pitch] with head h at channels off + h*dh .. + dh - 1
// (off = qoff, koff, voff; one concatenated QKV tensor or three tensors);
// out is fp16 [T*B][N][cp_out] with head h at channels h*dh ..; v_in / v_out
// fp32 [B][N][heads*dh].  One workgroup per (b, head), all T steps; dh = 32.
// An input whose count block (nnz) publishes zero takes the zero route: no
// operand reads and no MFMAs, z = 0 (the bits Q (K^T V) * scale has for zero
// operands) into the LIF.
#include "cf_common.h"

namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

constexpr int DH = 32;          // head dim (one MFMA tile edge)
constexpr int NMAX = 256;       // tokens per image this kernel stages (LDS)

struct AttnArgs {
  const _Float16* q;
  const _Float16* k;
  const _Float16* v;
  int qoff, koff, voff, pitch;
  _Float16* out;
  int cp_out;
  const float* v_in;
  float* v_out;
  const unsigned long long* nnz;   // count block of Q, K, V (one tensor), or null
  unsigned long long* nz_out;
  CfOutDesc* out_desc;             // output descriptor (CfOutDesc), or null
  int zero_info;                   // CF_BIAS_* for the LIF on z = 0 (needs out_desc)
  int T, B, N, heads;
  float scale;
  LifParams lif;
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t attn_rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes,
                                           0x00020000);
}

// Every product and sum here is exact (integers), so the order of the sums is
// free and TB time steps run side by side, WPS waves on each: waves WPS t ..
// take step t of the block.  A step's K and V are staged transposed ([d][token],
// two tokens a word, so each MFMA operand is one 16-byte read; rows of NM / 2 + 4
// words spread an operand's 32 rows over all banks).  Each wave sums K^T V
// itself, and its accumulators are the second product's B operand as they
// lie: the k slots of Y = Q (K^T V) are assigned to the rows d a lane holds,
// and Q is read in that order.  The sums then meet in LDS (over the staged
// tokens), and a thread runs the LIF over the block's steps for 8 channels of a
// token and stores 16 bytes a step.  Bound by latency: one round of loads, one
// transpose and two barriers a block.  Four steps a block (TB 4, WPS 2) take
// that once for T = 4: one image (196 tokens, 12 heads) 11.3 us, where a
// workgroup of four waves that took one step after another took 22.6.
// (launch_attention says where one step a block is the faster one.)
template <int NM, int TB, int WPS, int LM>
__global__ __launch_bounds__(64 * TB * WPS) void spike_attention_kernel(AttnArgs a) {
  constexpr int NT = 64 * TB * WPS, KW = NM / 2 + 4, ZLD = DH + 4;
  constexpr int KV_BYTES = 2 * TB * DH * KW * 4, Z_BYTES = TB * NM * ZLD * 4;
  // staged units of a thread (2 tokens x 8 channels; units past NM are not staged)
  constexpr int SU = (2 * NM + 64 * WPS - 1) / (64 * WPS);
  constexpr int MAXT = (NM / 32 + WPS - 1) / WPS;   // 32-token tiles of Y per wave at most
  constexpr int LU = (4 * NM + NT - 1) / NT;        // LIF units of a thread (a token x 8 channels)
  __shared__ __attribute__((aligned(16))) char smem[KV_BYTES > Z_BYTES ? KV_BYTES : Z_BYTES];
  __shared__ unsigned any_sh[TB * WPS];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hi = lane >> 5, col = lane & 31;
  const int ts = wave / WPS, wh = wave % WPS;  // this wave's step of the block, its first tile
  const int N = a.N, C = a.heads * DH;
  const int nks = (N + 15) / 16;            // 16-token MFMA steps of K^T V
  const int ntile = (N + 31) / 32;          // 32-token row tiles of Y
  const bool zero_in = a.nnz != nullptr && cf_count_read(a.nnz) == 0ull;   // uniform
  // An all-zero Q/K/V from the initial state drives every neuron with z = 0:
  // when the caller knows that the LIF never fires on it and holds the
  // final potential, the output is all zero and the state uniform, so
  // workgroup 0 records that in the descriptor and the count, and no
  // workgroup stores anything else.
  if (zero_in && a.v_in == nullptr && a.out_desc != nullptr && (a.zero_info & CF_BIAS_SILENT) &&
      ((a.zero_info & CF_BIAS_VCHAN) || a.v_out == nullptr)) {
    if (blockIdx.x == 0 && tid == 0) {
      if (a.nz_out != nullptr) a.nz_out[1] = 0ull;
      a.out_desc->copy = CF_COPY_ZERO;
      a.out_desc->vstate = (a.zero_info & CF_BIAS_VCHAN) ? 1u : 0u;
      a.out_desc->alias = nullptr;
    }
    return;
  }
  if (a.out_desc != nullptr && blockIdx.x == 0 && tid == 0) {
    a.out_desc->copy = CF_COPY_WRITTEN;
    a.out_desc->vstate = 0u;
    a.out_desc->alias = nullptr;
  }
  // Neighbouring heads (whose 64-byte rows share cache lines) on one XCD.
  const int nwork = a.B * a.heads, xcd = (int)blockIdx.x & 7;
  const int work = xcd * (nwork >> 3) + min(xcd, nwork & 7) + ((int)blockIdx.x >> 3);
  const int b = work / a.heads, h = work % a.heads;

  // membrane potentials: unit i is token tid / 4 + NT / 4 i, channels 8 (tid % 4) ..
  const int ln = tid >> 2, lc = (tid & 3) * 8;
  float v[LU][8];
  const float v0 = lif_initial_v(a.lif);
#pragma unroll
  for (int i = 0; i < LU; ++i) {
    const int n = ln + NT / 4 * i;
    const float* vs = a.v_in + ((size_t)b * N + n) * C + h * DH + lc;
#pragma unroll
    for (int j = 0; j < 8; ++j) v[i][j] = a.v_in != nullptr && n < N ? vs[j] : v0;
  }
  uint32_t* const kT = reinterpret_cast<uint32_t*>(smem) + ts * 2 * DH * KW;   // [d][pair]
  uint32_t* const vT = kT + DH * KW;
  float* const zb = reinterpret_cast<float*>(smem);                            // [t][n][ZLD]
  uint32_t anyw = 0u;

  for (int tb0 = 0; tb0 < a.T; tb0 += TB) {
    const int nst = min(TB, a.T - tb0);
    f32x16 y[MAXT];
#pragma unroll
    for (int i = 0; i < MAXT; ++i) y[i] = f32x16{};
    if (!zero_in) {
      // (steps beyond the last read step 0's rows and are not used)
      const size_t img = (size_t)(ts < nst ? tb0 + ts : 0) * a.B + b;
      const uint32_t bytes = (uint32_t)(((size_t)(N - 1) * a.pitch + DH) * 2);
      const __amdgpu_buffer_rsrc_t rq = attn_rsrc(a.q + img * N * a.pitch + a.qoff + h * DH, bytes);
      const __amdgpu_buffer_rsrc_t rk = attn_rsrc(a.k + img * N * a.pitch + a.koff + h * DH, bytes);
      const __amdgpu_buffer_rsrc_t rv = attn_rsrc(a.v + img * N * a.pitch + a.voff + h * DH, bytes);
      // every load of the block is issued before its first use (rows beyond
      // N read zeros, out of the buffers' range)
      auto off = [&](int n, int c) { return n < N ? (uint32_t)((n * a.pitch + c) * 2) : 0x80000000u; };
      const int g = tid & (64 * WPS - 1);
      u32x4 kx[SU][2], vx[SU][2];
#pragma unroll
      for (int i = 0; i < SU; ++i) {
        const int u = g + 64 * WPS * i, n = (u >> 2) * 2, c = (u & 3) * 8;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          kx[i][e] = __builtin_amdgcn_raw_buffer_load_b128(rk, off(n + e, c), 0, 0);
          vx[i][e] = __builtin_amdgcn_raw_buffer_load_b128(rv, off(n + e, c), 0, 0);
        }
      }
      // Q rows of this wave's tiles: k slots (hi, 0..3) and (hi, 4..7) of MFMA
      // step s are channels 16 s + 4 hi .. + 3 and 16 s + 8 + 4 hi .. + 3
      u32x2 qx[MAXT][2][2];
#pragma unroll
      for (int i = 0; i < MAXT; ++i)
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
          for (int e = 0; e < 2; ++e)
            qx[i][s][e] = __builtin_amdgcn_raw_buffer_load_b64(
                rq, off((wh + WPS * i) * 32 + col, 16 * s + 8 * e + 4 * hi), 0, 0);
#pragma unroll
      for (int i = 0; i < SU; ++i) {
        const int u = g + 64 * WPS * i, pr = u >> 2, c = (u & 3) * 8;
        if (2 * pr < 16 * nks) {
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const uint32_t sel = (j & 1) ? 0x07060302u : 0x05040100u;   // high / low halves
            kT[(c + j) * KW + pr] = __builtin_amdgcn_perm(kx[i][1][j >> 1], kx[i][0][j >> 1], sel);
            vT[(c + j) * KW + pr] = __builtin_amdgcn_perm(vx[i][1][j >> 1], vx[i][0][j >> 1], sel);
          }
        }
      }
      __syncthreads();
      f32x16 kv = {};
      for (int s = 0; s < nks; ++s) {
        const h8 av = *reinterpret_cast<const h8*>(&kT[col * KW + 8 * s + 4 * hi]);
        const h8 bv = *reinterpret_cast<const h8*>(&vT[col * KW + 8 * s + 4 * hi]);
        kv = __builtin_amdgcn_mfma_f32_32x32x16_f16(av, bv, kv, 0, 0, 0);
      }
      h8 kvb[2];   // entries <= N: exact in fp16
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int j = 0; j < 8; ++j) kvb[s][j] = (_Float16)kv[8 * s + j];
#pragma unroll
      for (int i = 0; i < MAXT; ++i)
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          const u32x4 q4 = {qx[i][s][0][0], qx[i][s][0][1], qx[i][s][1][0], qx[i][s][1][1]};
          y[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(h8, q4), kvb[s], y[i], 0,
                                                        0, 0);
        }
      __syncthreads();   // kT and vT are read: the sums take their place
    }
#pragma unroll
    for (int i = 0; i < MAXT; ++i) {
      const int tile = wh + WPS * i;
      if (tile >= ntile) break;
#pragma unroll
      for (int r = 0; r < 16; ++r)
        zb[(ts * NM + tile * 32 + 8 * (r >> 2) + 4 * hi + (r & 3)) * ZLD + col] = y[i][r];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < LU; ++i) {
      const int n = ln + NT / 4 * i;
      if (n >= N) break;
#pragma unroll
      for (int t = 0; t < TB; ++t) {
        if (t >= nst) break;
        const float* zp = &zb[(t * NM + n) * ZLD + lc];
        h8 sp;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float z = zp[j] * a.scale;
          float vv = lif_charge_m<LM>(v[i][j], z, a.lif);
          sp[j] = lif_fire_reset_bit<LM>(vv, a.lif) ? (_Float16)1.0f : (_Float16)0.0f;
          v[i][j] = vv;
        }
        const u32x4 w = __builtin_bit_cast(u32x4, sp);
        anyw |= w[0] | w[1] | w[2] | w[3];
        _Float16* o = a.out + (((size_t)(tb0 + t) * a.B + b) * N + n) * a.cp_out + h * DH + lc;
        if (a.cp_out % 8 == 0 && ((uintptr_t)a.out & 15) == 0) {
          *reinterpret_cast<u32x4*>(o) = w;
        } else {
#pragma unroll
          for (int j = 0; j < 8; ++j) o[j] = sp[j];
        }
      }
    }
    if (tb0 + TB < a.T) __syncthreads();   // the sums are read: the next block stages here
  }
  if (a.v_out) {
#pragma unroll
    for (int i = 0; i < LU; ++i) {
      const int n = ln + NT / 4 * i;
      if (n >= N) break;
      float* vd = a.v_out + ((size_t)b * N + n) * C + h * DH + lc;
#pragma unroll
      for (int j = 0; j < 8; ++j) vd[j] = v[i][j];
    }
  }
  if (a.nz_out) {
    const bool any = __any(anyw != 0u ? 1 : 0) != 0;
    if (lane == 0) any_sh[wave] = any ? 1u : 0u;
    __syncthreads();
    if (tid == 0) {
      unsigned w = 0u;
#pragma unroll
      for (int i = 0; i < TB * WPS; ++i) w |= any_sh[i];
      cf_count_publish(a.nz_out, w ? 1ull : 0ull, blockIdx.x, gridDim.x);
    }
  }
}

// Workgroups of fewer tokens need less LDS, so more share a CU.  Four steps of
// more than 128 tokens take 147 KB, one workgroup a CU: launches of more
// workgroups than CUs then run in rounds, and steps that do not exist (T off 4)
// cost as much as those that do.  They take one step a block, eight waves on it
// (37 KB, four workgroups a CU).  Measured (us, four steps / one step a block),
// 196 tokens: 384 workgroups, T = 1 20.2 / 8.8, 4 26.5 / 21.7, 5 42.3 / 25.1; 1536,
// T = 1 58.1 / 20.9, 2 67.5 / 31.5; 256 tokens, 768, T = 4 49.3 / 37.7; but 256
// workgroups, 196 tokens, T = 4 16.6 / 18.8.  Up to 128 tokens four steps are
// the faster choice at one image and both lie far below what one step after
// another took.
template <int LM>
void launch_attention(const AttnArgs& a, hipStream_t st) {
  const dim3 grid((unsigned)(a.B * a.heads)), block(512);
  const int cus = cf_cu_count() > 0 ? cf_cu_count() : 256;
  if (a.N <= 64) hipLaunchKernelGGL((spike_attention_kernel<64, 4, 2, LM>), grid, block, 0, st, a);
  else if (a.N <= 128)
    hipLaunchKernelGGL((spike_attention_kernel<128, 4, 2, LM>), grid, block, 0, st, a);
  else if (grid.x <= (unsigned)cus)
    hipLaunchKernelGGL((spike_attention_kernel<NMAX, 4, 2, LM>), grid, block, 0, st, a);
  else hipLaunchKernelGGL((spike_attention_kernel<NMAX, 1, 8, LM>), grid, block, 0, st, a);
}

// ---------------------------------------------------------------------------
// Two-pass form for any token count and head dims 32 or 64.
//
// Pass 1 (attn_kv_kernel): one workgroup per (step, image, head) reduces
// K^T V over all N tokens, 256 at a time: the chunk's K and V staged
// transposed in LDS (zero-padded to whole 16-token MFMA steps), the dh x dh
// result as 32 x 32 tiles (dh = 64: one tile per wave over every token;
// dh = 32: the four waves take every fourth 16-token step and their partial
// tiles are summed in LDS).  Every product is 0/1 and every partial sum an
// integer below 2^24, so the fp32 result is exact in any order.  Written to
// the workspace kv [T*B*heads][dh][dh] (row i of K^T, column j of V).
//
// Pass 2 (attn_y_lif_kernel): one workgroup per (image, head, 128-token
// block), all T steps: KV_t is split into two fp16 limbs that are exact
// (hi = KV & ~1023, lo = KV & 1023: integers below 2^16), Y = Q KV_hi +
// Q KV_lo on the matrix cores (every partial sum an integer below 2^24:
// exact), z = Y * scale (one rounding), the LIF with v in registers (wave w:
// tokens 32 w .. 32 w + 31 of the block, dh channels).  The values equal the
// single-pass kernel's (same exact Y, same rounding, same LIF).
constexpr int KV_CHUNK = 256;    // tokens per staged chunk of pass 1
constexpr int Y_TOKENS = 128;    // tokens per workgroup of pass 2

struct AttnKvArgs {
  const _Float16* q;
  const _Float16* k;
  const _Float16* v;
  int qoff, koff, voff, pitch;
  _Float16* out;
  int cp_out;
  const float* v_in;
  float* v_out;
  float* kv;                       // workspace [T*B*heads][dh][dh]
  const unsigned long long* nnz;
  unsigned long long* nz_out;
  CfOutDesc* out_desc;
  int zero_info;
  int T, B, N, heads;
  float scale;
  LifParams lif;
};

// The zero route's elision (as the single-pass kernel): an all-zero Q/K/V
// from the initial state with a silent, caller-held LIF response to z = 0
// records the output as all zero and stores nothing else.
__device__ __forceinline__ bool attn_zero_elided(const AttnKvArgs& a, bool zero_in) {
  return zero_in && a.v_in == nullptr && a.out_desc != nullptr &&
         (a.zero_info & CF_BIAS_SILENT) && ((a.zero_info & CF_BIAS_VCHAN) || a.v_out == nullptr);
}

template <int DHV>
__global__ __launch_bounds__(256) void attn_kv_kernel(AttnKvArgs a) {
  constexpr int KLD = KV_CHUNK + 8;   // row pitch (halves): rows 4 banks apart
  __shared__ __attribute__((aligned(16))) _Float16 kT[DHV][KLD];
  __shared__ __attribute__((aligned(16))) _Float16 vT[DHV][KLD];
  __shared__ __attribute__((aligned(16))) float kvp[DHV == 32 ? 4 : 1][32][33];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hi = lane >> 5, col = lane & 31;
  const int img = blockIdx.x / a.heads, h = blockIdx.x % a.heads;   // img = t * B + b
  const int N = a.N;
  if (a.nnz != nullptr && cf_count_read(a.nnz) == 0ull) return;     // pass 2 takes z = 0
  const _Float16* kb = a.k + (size_t)img * N * a.pitch + a.koff + h * DHV;
  const _Float16* vb = a.v + (size_t)img * N * a.pitch + a.voff + h * DHV;
  // dh = 64: wave (wi, wj) computes the tile KV[32 wi ..][32 wj ..]
  const int wi = DHV == 64 ? (wave >> 1) : 0, wj = DHV == 64 ? (wave & 1) : 0;
  f32x16 acc = {};
  constexpr int PARTS = DHV / 8;                   // 8-channel parts per token
  constexpr int SU = KV_CHUNK * PARTS / 256;       // staged units per thread
  for (int n0 = 0; n0 < N; n0 += KV_CHUNK) {
    const int nc = min(KV_CHUNK, N - n0);
    const int ncp = (nc + 15) & ~15;
    h8 kx[SU], vx[SU];
#pragma unroll
    for (int i = 0; i < SU; ++i) {
      const int u = tid + 256 * i, n = u / PARTS, c = (u % PARTS) * 8;
      kx[i] = h8{};
      vx[i] = h8{};
      if (n < nc) {
        kx[i] = *reinterpret_cast<const h8*>(kb + (size_t)(n0 + n) * a.pitch + c);
        vx[i] = *reinterpret_cast<const h8*>(vb + (size_t)(n0 + n) * a.pitch + c);
      }
    }
    __syncthreads();   // the previous chunk's operand reads are complete
#pragma unroll
    for (int i = 0; i < SU; ++i) {
      const int u = tid + 256 * i, n = u / PARTS, c = (u % PARTS) * 8;
      if (n < ncp) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          kT[c + j][n] = kx[i][j];
          vT[c + j][n] = vx[i][j];
        }
      }
    }
    __syncthreads();
    const int nks = ncp / 16;
    for (int s = (DHV == 32 ? wave : 0); s < nks; s += (DHV == 32 ? 4 : 1)) {
      const int nn = s * 16 + 8 * hi;
      const h8 av = *reinterpret_cast<const h8*>(&kT[32 * wi + col][nn]);   // A[i][n]
      const h8 bv = *reinterpret_cast<const h8*>(&vT[32 * wj + col][nn]);   // B[n][j]
      acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(av, bv, acc, 0, 0, 0);
    }
  }
  float* kvo = a.kv + (size_t)blockIdx.x * DHV * DHV;
  if constexpr (DHV == 64) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int i = 32 * wi + 8 * (r >> 2) + 4 * hi + (r & 3);
      kvo[i * DHV + 32 * wj + col] = acc[r];
    }
  } else {
#pragma unroll
    for (int r = 0; r < 16; ++r) kvp[wave][8 * (r >> 2) + 4 * hi + (r & 3)][col] = acc[r];
    __syncthreads();
    for (int e = tid; e < 32 * 32; e += 256) {
      const int i = e >> 5, j = e & 31;
      kvo[e] = kvp[0][i][j] + kvp[1][i][j] + kvp[2][i][j] + kvp[3][i][j];
    }
  }
}

template <int DHV, int LM>
__global__ __launch_bounds__(256) void attn_y_lif_kernel(AttnKvArgs a) {
  constexpr int NCT = DHV / 32;                       // 32-channel column tiles
  __shared__ __attribute__((aligned(16))) _Float16 kvT[2][DHV][DHV + 8];   // limbs, [j][i]
  __shared__ unsigned any_sh[4];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hi = lane >> 5, col = lane & 31;
  const int nblk = (a.N + Y_TOKENS - 1) / Y_TOKENS;
  const int bh = blockIdx.x / nblk, blk = blockIdx.x % nblk;
  const int b = bh / a.heads, h = bh % a.heads;
  const int N = a.N, C = a.heads * DHV;
  const int tile0 = blk * Y_TOKENS + 32 * wave;       // this wave's first token
  const bool zero_in = a.nnz != nullptr && cf_count_read(a.nnz) == 0ull;
  if (attn_zero_elided(a, zero_in)) {
    if (blockIdx.x == 0 && tid == 0) {
      if (a.nz_out != nullptr) a.nz_out[1] = 0ull;
      a.out_desc->copy = CF_COPY_ZERO;
      a.out_desc->vstate = (a.zero_info & CF_BIAS_VCHAN) ? 1u : 0u;
      a.out_desc->alias = nullptr;
    }
    return;
  }
  if (a.out_desc != nullptr && blockIdx.x == 0 && tid == 0) {
    a.out_desc->copy = CF_COPY_WRITTEN;
    a.out_desc->vstate = 0u;
    a.out_desc->alias = nullptr;
  }
  float v[NCT][16];
#pragma unroll
  for (int ct = 0; ct < NCT; ++ct)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int n = tile0 + 8 * (r >> 2) + 4 * hi + (r & 3);
      float v0 = lif_initial_v(a.lif);
      if (a.v_in && n < N) v0 = a.v_in[((size_t)b * N + n) * C + h * DHV + 32 * ct + col];
      v[ct][r] = v0;
    }
  uint32_t anyw = 0u;
  for (int t = 0; t < a.T; ++t) {
    const size_t img = (size_t)t * a.B + b;
    f32x16 y[NCT];
#pragma unroll
    for (int ct = 0; ct < NCT; ++ct) y[ct] = f32x16{};
    if (!zero_in) {
      // Q rows of this wave's 32 tokens (A operand: row col, k 8 hi ..);
      // rows beyond N read zeros
      const _Float16* qb = a.q + img * N * a.pitch + a.qoff + h * DHV;
      const __amdgpu_buffer_rsrc_t rq =
          attn_rsrc(qb, (uint32_t)(((size_t)(N - 1) * a.pitch + DHV) * 2));
      const int n = tile0 + col;
      const uint32_t qo = n < N ? (uint32_t)(((size_t)n * a.pitch) * 2) : 0x80000000u;
      h8 qr[DHV / 16];
#pragma unroll
      for (int ks = 0; ks < DHV / 16; ++ks)
        qr[ks] = __builtin_bit_cast(
            h8, __builtin_amdgcn_raw_buffer_load_b128(rq, qo + 32 * ks + 16 * hi, 0, 0));
      // KV_t as two exact fp16 limbs, transposed: kvT[limb][j][i] = KV[i][j]
      const float* kvi = a.kv + (img * a.heads + h) * DHV * DHV;
      __syncthreads();   // the previous step's reads of kvT are complete
      for (int e = tid; e < DHV * DHV; e += 256) {
        const int i = e / DHV, j = e % DHV;
        const uint32_t kvv = (uint32_t)kvi[e];          // an integer below 2^16
        kvT[0][j][i] = (_Float16)(float)(kvv & ~1023u);
        kvT[1][j][i] = (_Float16)(float)(kvv & 1023u);
      }
      __syncthreads();
#pragma unroll
      for (int ct = 0; ct < NCT; ++ct)
#pragma unroll
        for (int limb = 0; limb < 2; ++limb)
#pragma unroll
          for (int ks = 0; ks < DHV / 16; ++ks) {
            const h8 bv = *reinterpret_cast<const h8*>(&kvT[limb][32 * ct + col][16 * ks + 8 * hi]);
            y[ct] = __builtin_amdgcn_mfma_f32_32x32x16_f16(qr[ks], bv, y[ct], 0, 0, 0);
          }
    }
    _Float16* ob = a.out + img * N * a.cp_out + h * DHV;
#pragma unroll
    for (int ct = 0; ct < NCT; ++ct)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int nr = tile0 + 8 * (r >> 2) + 4 * hi + (r & 3);
        const float z = y[ct][r] * a.scale;
        float vv = lif_charge_m<LM>(v[ct][r], z, a.lif);
        const bool f = lif_fire_reset_bit<LM>(vv, a.lif);
        v[ct][r] = vv;
        if (nr < N) {
          ob[(size_t)nr * a.cp_out + 32 * ct + col] = f ? (_Float16)1.0f : (_Float16)0.0f;
          anyw |= f ? 1u : 0u;
        }
      }
  }
  if (a.v_out) {
#pragma unroll
    for (int ct = 0; ct < NCT; ++ct)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int n = tile0 + 8 * (r >> 2) + 4 * hi + (r & 3);
        if (n < N) a.v_out[((size_t)b * N + n) * C + h * DHV + 32 * ct + col] = v[ct][r];
      }
  }
  if (a.nz_out) {
    const bool any = cf_wg_any(anyw != 0u, any_sh);
    if (tid == 0) cf_count_publish(a.nz_out, any ? 1ull : 0ull, blockIdx.x, gridDim.x);
  }
}

}  // namespace

CF_API int cf_spike_attention_lif(const void* q, const void* k, const void* v, int64_t qoff,
                                  int64_t koff, int64_t voff, int64_t pitch, void* out,
                                  int64_t cp_out, const float* v_in, float* v_out,
                                  const unsigned long long* nnz, unsigned long long* nz_out,
                                  void* out_desc, int zero_info,
                                  int64_t T, int64_t B, int64_t N,
                                  int64_t heads, int64_t head_dim, double scale, double tau,
                                  double v_th, double v_reset, int hard_reset, int decay_input,
                                  void* stream) {
  if (!q || !k || !v || !out || T <= 0 || B <= 0 || N <= 0 || heads <= 0) return (int)hipErrorInvalidValue;
  if (head_dim != DH || N > NMAX) return (int)hipErrorInvalidValue;
  const int64_t C = heads * head_dim;
  if (pitch % 8 != 0 || qoff % 8 != 0 || koff % 8 != 0 || voff % 8 != 0 || qoff < 0 ||
      koff < 0 || voff < 0 || qoff + C > pitch || koff + C > pitch || voff + C > pitch ||
      cp_out < C || T * B * N * pitch > ((int64_t)1 << 40) || B * heads >= (int64_t)CF_MAX_COUNT_WG ||
      (int64_t)(N - 1) * pitch * 2 + 64 > INT32_MAX)
    return (int)hipErrorInvalidValue;
  if ((zero_info & ~(CF_BIAS_SILENT | CF_BIAS_VCHAN)) != 0 || (zero_info && !out_desc))
    return (int)hipErrorInvalidValue;
  AttnArgs a;
  a.q = (const _Float16*)q; a.k = (const _Float16*)k; a.v = (const _Float16*)v;
  a.qoff = (int)qoff; a.koff = (int)koff; a.voff = (int)voff; a.pitch = (int)pitch;
  a.out = (_Float16*)out; a.cp_out = (int)cp_out; a.v_in = v_in; a.v_out = v_out;
  a.nnz = nnz; a.nz_out = nz_out; a.T = (int)T;
  a.out_desc = (CfOutDesc*)out_desc; a.zero_info = zero_info; a.B = (int)B; a.N = (int)N; a.heads = (int)heads;
  a.scale = (float)scale;
  a.lif = cf_make_lif_params(tau, v_th, v_reset, hard_reset, decay_input);
  const int lm = cf_lif_mode(a.lif);
  hipStream_t st = (hipStream_t)stream;
  if (lm == LM_HARD0_DECAY_P2) launch_attention<LM_HARD0_DECAY_P2>(a, st);
  else if (lm == LM_HARD_DECAY_P2) launch_attention<LM_HARD_DECAY_P2>(a, st);
  else launch_attention<LM_GENERIC>(a, st);
  return (int)hipGetLastError();
}

CF_API int cf_spike_attention_kv_lif(const void* q, const void* k, const void* v, int64_t qoff,
                                     int64_t koff, int64_t voff, int64_t pitch, void* out,
                                     int64_t cp_out, const float* v_in, float* v_out,
                                     float* kv_ws, const unsigned long long* nnz,
                                     unsigned long long* nz_out, void* out_desc, int zero_info,
                                     int64_t T, int64_t B, int64_t N, int64_t heads,
                                     int64_t head_dim, double scale, double tau, double v_th,
                                     double v_reset, int hard_reset, int decay_input,
                                     void* stream) {
  if (!q || !k || !v || !out || !kv_ws || T <= 0 || B <= 0 || N <= 0 || heads <= 0)
    return (int)hipErrorInvalidValue;
  if (head_dim != 32 && head_dim != 64) return (int)hipErrorInvalidValue;
  const int64_t C = heads * head_dim;
  const int64_t nblk = (N + Y_TOKENS - 1) / Y_TOKENS;
  // K^T V entries <= N must stay below 2^16 (two exact fp16 limbs) and Y
  // below 2^24 (exact fp32 sums): N < 65536 / ... head_dim * N < 2^24
  if (N >= 65536 || head_dim * N >= (int64_t)1 << 24) return (int)hipErrorInvalidValue;
  if (pitch % 8 != 0 || qoff % 8 != 0 || koff % 8 != 0 || voff % 8 != 0 || qoff < 0 ||
      koff < 0 || voff < 0 || qoff + C > pitch || koff + C > pitch || voff + C > pitch ||
      cp_out < C || T * B * N * pitch > ((int64_t)1 << 40) ||
      B * heads * nblk >= (int64_t)CF_MAX_COUNT_WG || T * B * heads > INT32_MAX ||
      (int64_t)(N - 1) * pitch * 2 + 128 > INT32_MAX)
    return (int)hipErrorInvalidValue;
  if ((zero_info & ~(CF_BIAS_SILENT | CF_BIAS_VCHAN)) != 0 || (zero_info && !out_desc))
    return (int)hipErrorInvalidValue;
  AttnKvArgs a;
  a.q = (const _Float16*)q; a.k = (const _Float16*)k; a.v = (const _Float16*)v;
  a.qoff = (int)qoff; a.koff = (int)koff; a.voff = (int)voff; a.pitch = (int)pitch;
  a.out = (_Float16*)out; a.cp_out = (int)cp_out; a.v_in = v_in; a.v_out = v_out;
  a.kv = kv_ws; a.nnz = nnz; a.nz_out = nz_out; a.out_desc = (CfOutDesc*)out_desc;
  a.zero_info = zero_info; a.T = (int)T; a.B = (int)B; a.N = (int)N; a.heads = (int)heads;
  a.scale = (float)scale;
  a.lif = cf_make_lif_params(tau, v_th, v_reset, hard_reset, decay_input);
  hipStream_t st = (hipStream_t)stream;
  const dim3 g1((unsigned)(T * B * heads)), g2((unsigned)(B * heads * nblk)), block(256);
  if (head_dim == 64)
    hipLaunchKernelGGL(attn_kv_kernel<64>, g1, block, 0, st, a);
  else
    hipLaunchKernelGGL(attn_kv_kernel<32>, g1, block, 0, st, a);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return (int)e;
  const int lm = cf_lif_mode(a.lif);
#define CF_ATTN_Y(DHV)                                                                         \
  do {                                                                                         \
    if (lm == LM_HARD0_DECAY_P2)                                                               \
      hipLaunchKernelGGL((attn_y_lif_kernel<DHV, LM_HARD0_DECAY_P2>), g2, block, 0, st, a);    \
    else if (lm == LM_HARD_DECAY_P2)                                                           \
      hipLaunchKernelGGL((attn_y_lif_kernel<DHV, LM_HARD_DECAY_P2>), g2, block, 0, st, a);     \
    else                                                                                       \
      hipLaunchKernelGGL((attn_y_lif_kernel<DHV, LM_GENERIC>), g2, block, 0, st, a);           \
  } while (0)
  if (head_dim == 64) CF_ATTN_Y(64);
  else CF_ATTN_Y(32);
#undef CF_ATTN_Y
  return (int)hipGetLastError();
}
