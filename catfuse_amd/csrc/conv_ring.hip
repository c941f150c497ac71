// Fused stride-1 Conv -> BN -> LIF (1x1 without padding, 3x3 with padding 1)
// over flat pixel tiles, both operands streamed through LDS rings.
//
// Tile: 32 * MW output channels x 64 consecutive pixels of the flattened
// (image, row, column) order x a block of 4 time steps.  In the NHWC copies
// such a run is contiguous, and so is everything a 3x3 window needs around
// it (W + 1 pixels more on both sides), so staging is a straight copy, tiles
// cross image borders, and small maps (4x4, 2x2, single pixels) fill a tile
// with several images.  What a tap reads outside its own image is replaced by
// a zero pixel: a 9-bit mask per lane selects it.
//
// Pipeline: a stage is one filter tap of one 32-channel chunk (3x3) or one
// chunk (1x1).  Weight fragments and pixels are copied global -> LDS without
// passing registers, several stages ahead (3x3 pixels two chunks), and a wave
// waits only for the copies of the next stage (s_waitcnt vmcnt of what was
// issued since), so it never waits for a load it has just issued; one tap or
// one chunk ahead in registers (conv_halo.hip) is what bounds launches of few
// workgroups, whose waves have no neighbours to hide a wait behind.  The
// fragments of a stage are read from LDS while the stage before it is
// multiplied, and every read and copy is issued between two matrix
// instructions.  512 -> 512 channels, 3x3 on 7x7, one image: 54 us
// (conv_halo.hip) -> 35 with the reads in a row after the barrier -> 27, of
// which 15.4 are the longest chain of matrix instructions and 9 the launch, the
// first copies and the epilogue.
//
// MW = 1: 32 channels; the four waves are 2 pixel halves x 2 pairs of time
// steps: twice the workgroups and half the chain of matrix instructions of a
// 64-channel tile.  MW = 2: 64 channels; 2 pixel halves x 2 channel halves.
//
// Accumulation order per output element: chunk-major, then tap, then the
// two 16-channel halves, hi limb then lo limb, as conv_halo.hip and
// conv_mfma.hip: the results are theirs bit for bit.
#include "cf_mfma.h"

namespace {

struct RingArgs {
  const _Float16* x;      // [T][rows][Cp], rows = B * H * W
  const _Float16* w;      // fragment-major limbs (cf_wfrag_index)
  const float* alpha;
  const float* beta;
  const float* v_in;      // [B][Cout][H * W] (pooled: of the pooled map), nullable
  float* v_out;
  _Float16* out;          // [T][rows][cp_out] (pooled: a quarter of the rows)
  int cp_out;
  const _Float16* id;     // spike-valued identity [T][rows][cp_id], nullable
  int cp_id;
  const unsigned long long* nnz;   // as HaloArgs (conv_halo.hip)
  unsigned long long* nz_out;
  const CfOutDesc* x_desc;
  const CfOutDesc* id_desc;
  CfOutDesc* out_desc;
  int bias_info;
  const unsigned long long* id_nnz;
  int T, rows, H, W, Cp, Cout, Coutp;
  int ntiles, ncb;        // pixel tiles, channel blocks
  int cb_major;           // neighbouring workgroups share channels, not pixels
  LifParams lif;
};

template <int V>
struct RingInt {
  static constexpr int v = V;
};

template <int N>
__device__ __forceinline__ void wait_vm() {
  static_assert(N >= 0 && N < 64, "vmcnt");
  asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory");
}
__device__ __forceinline__ void ring_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// NPX: staged pixels of a step (3x3: at least 64 + 2 W + 3, the last one the
// zero pixel; 1x1: 64).  NX: slots of the pixel ring, each the pixels of one
// chunk (3x3: three, or two for layers of at most two chunks, which are then
// both staged before the first tap: maps too wide for three slots) or of two
// (1x1: 128-byte runs of a pixel's channels, a whole cache line, where a chunk
// alone is half of one).  NW: slots of the weight ring (3x3: nine, a tap's slot
// is its number).
template <int K, int MW, int NPX, int NX, int NW>
struct RingGeom {
  static constexpr int KK = K * K, TB = 4;
  static constexpr int PB = K == 3 ? 64 : 128;    // bytes of a staged pixel
  static constexpr int WB = MW * 4096;            // weights of a stage (bytes)
  static constexpr int XT = NPX * PB;             // staged pixels of a step (bytes)
  static constexpr int XB = TB * XT;              // of a slot
  static constexpr int LDS = NX * XB + NW * WB;
  static constexpr int DX = NX - 1, DW = NW - 1;  // slots a copy is issued ahead
  static constexpr int XL = XT / 1024;            // 1 KB copies of a step's pixels
  static constexpr int TW = 2 / MW, TPW = 2 * MW; // groups of time steps, steps a wave
  static constexpr int NT = K == 3 ? 256 : 320;   // threads (1x1: a fifth wave copies weights)
};

template <int K, int MW, int NPX, int NX, int NW, int LM, bool POOL>
__global__ __launch_bounds__((RingGeom<K, MW, NPX, NX, NW>::NT), 1)
void conv_ring_kernel(const RingArgs a) {
  using G = RingGeom<K, MW, NPX, NX, NW>;
  constexpr int KK = G::KK, TB = G::TB, WB = G::WB, XT = G::XT, XB = G::XB, XL = G::XL;
  constexpr int DX = G::DX, DW = G::DW, PB = G::PB;
  constexpr int TPW = G::TPW, TW = G::TW, BM = 32 * MW;
  constexpr int NG = 4 / TW;                // groups of 4 channels a lane finishes
  static_assert(K == 1 || (K == 3 && NW == 9 && (NX == 2 || (NX == 3 && XL <= 9))),
                "3x3: one slot a tap");
  static_assert(NPX % 16 == 0 && (K == 3 || NPX == 64), "staged pixels");
  __shared__ __attribute__((aligned(16))) char smem[G::LDS];
  __shared__ __attribute__((aligned(16))) float bn_s[2][BM];
  __shared__ unsigned any_sh[5];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // wave: pixel half, channel half (MW = 2), group of time steps
  const int wn = wave & 1, wc = MW == 2 ? wave >> 1 : 0, wt = MW == 2 ? 0 : wave >> 1;
  const int hi = lane >> 5;
  const int HW = a.H * a.W;

  // Route and sources, as halo_body (conv_halo.hip): a zero count or an
  // all-zero copy takes StaticZero; copies are read where their descriptors
  // say.
  const unsigned long long* const zp = reinterpret_cast<const unsigned long long*>(&g_halo_zero);
  const CfOutDesc* const zdesc = reinterpret_cast<const CfOutDesc*>(&g_halo_zero);
  const unsigned long long in_count = *(a.nnz != nullptr ? a.nnz + 1 : zp);
  const unsigned long long id_count = *(a.id_nnz != nullptr ? a.id_nnz + 1 : zp);
  const CfOutDesc xd = *(a.x_desc != nullptr ? a.x_desc : zdesc);
  const CfOutDesc idd = *(a.id_desc != nullptr ? a.id_desc : zdesc);
  const _Float16* const xsrc = xd.copy == CF_COPY_ZERO    ? nullptr
                               : xd.copy == CF_COPY_ALIAS ? (const _Float16*)xd.alias
                                                          : a.x;
  const bool zero = (a.nnz != nullptr && in_count == 0ull) || xsrc == nullptr;
  const _Float16* const id = a.id == nullptr             ? nullptr
                             : idd.copy == CF_COPY_ZERO  ? nullptr
                             : idd.copy == CF_COPY_ALIAS ? (const _Float16*)idd.alias
                                                         : a.id;
  // StaticZero from the initial state with a silent bias response: the
  // output is all zero, or the identity's copy; only the descriptor and the
  // count are stored (workgroup 0).
  if (zero && a.v_in == nullptr && a.out_desc != nullptr && (a.bias_info & CF_BIAS_SILENT) != 0 &&
      ((a.bias_info & CF_BIAS_VCHAN) != 0 || a.v_out == nullptr) &&
      (id == nullptr || (a.id_desc != nullptr && a.cp_id == a.cp_out))) {
    if (blockIdx.x == 0 && tid == 0) {
      if (a.nz_out != nullptr)
        a.nz_out[1] = id != nullptr && (a.id_nnz == nullptr || id_count != 0ull) ? 1ull : 0ull;
      a.out_desc->copy = id != nullptr ? CF_COPY_ALIAS : CF_COPY_ZERO;
      a.out_desc->vstate = (a.bias_info & CF_BIAS_VCHAN) != 0 ? 1u : 0u;
      a.out_desc->alias = id;
    }
    return;
  }

  // Work item: workgroup L runs on XCD L % 8, which takes a contiguous range
  // of items, so neighbours share an L2.
  const int nwork = a.ntiles * a.ncb;
  const int xcd = (int)blockIdx.x & 7;
  const int work = xcd * (nwork >> 3) + min(xcd, nwork & 7) + ((int)blockIdx.x >> 3);
  const int cb = a.cb_major ? work / a.ntiles : work % a.ncb;
  const int tile = a.cb_major ? work - cb * a.ntiles : work / a.ncb;
  const int P0 = tile * 64, cout0 = cb * BM;
  const int nch = a.Cp / KC;
  if (tid < BM) {
    bn_s[0][tid] = a.alpha[cout0 + tid];
    bn_s[1][tid] = a.beta[cout0 + tid];
  }

  // This lane's pixel (accumulator column lane % 32 of its wave's half): its
  // image, position and, for 3x3, the taps that stay inside the image.
  const int n = wn * 32 + (lane & 31);
  const int p = P0 + n;
  const bool p_ok = p < a.rows;
  const int img = p / HW, pix = p - img * HW;
  const int py = pix / a.W, px = pix - py * a.W;
  uint32_t taps_in = 0u;
  if (K == 3 && p_ok) {
    const uint32_t r = (py > 0 ? 1u : 0u) | 2u | (py + 1 < a.H ? 4u : 0u);
    const uint32_t c = (px > 0 ? 1u : 0u) | 2u | (px + 1 < a.W ? 4u : 0u);
#pragma unroll
    for (int kh = 0; kh < 3; ++kh) taps_in |= ((r >> kh) & 1u ? c : 0u) << (3 * kh);
  }

  // Weight copy f of a stage's 4 * MW: a fragment of 1 KB, in the slot as
  // [32-channel tile][limb][16-channel half].
  const int k16s = a.Cp / 16;
  const cf_v4i wr = halo_rsrc_v4(a.w + (size_t)(cout0 / 32) * KK * k16s * 512, 0x7fffffffu);
  const uint32_t limb_bytes = (uint32_t)a.Coutp * KK * (uint32_t)a.Cp * 2u;
  const unsigned smem0 = lds_addr(smem);
  const unsigned ring0 = smem0 + NX * XB;
  auto issue_w = [&](int f, int ch, int tap, int slot) {
    const uint32_t voff = ch < nch ? (uint32_t)lane * 16u : HALO_OOB;
    const uint32_t so = (uint32_t)(((f >> 2) * KK + tap) * k16s + ch * 2 + (f & 1)) * 1024u +
                        ((f >> 1) & 1 ? limb_bytes : 0u);
    lds_buf_copy16_at(wr, voff, __builtin_amdgcn_readfirstlane(ch < nch ? so : 0u),
                      __builtin_amdgcn_readfirstlane(ring0 + slot * WB + f * 1024));
  };
  // 1x1: the weights are wave 4's alone.  Loads complete in order, so a wave
  // that waits for pixels (from the L2, where the layer before left them) would
  // also wait for the weights it issued before them, which a network's pass
  // brings from further away; a wave of their own keeps DW stages of them in
  // flight (64 rows of 4096 -> 4096 38.3 -> 34.6 us; with 13 stages of weights
  // but two pairs of pixels ahead instead of 5 and three, 39.8).  Its barriers
  // are those of the other waves, one for one.
  if constexpr (K == 1) {
    if (wave == 4) {
      for (int tb0 = 0; tb0 < a.T; tb0 += TB) {
        if (!zero) {
#pragma unroll
          for (int s = 0; s < DW; ++s)
#pragma unroll
            for (int f = 0; f < 4 * MW; ++f) issue_w(f, s, 0, s);
          wait_vm<(DW - 1) * 4 * MW>();
          ring_barrier();
          int wd = DW;
          for (int ch = 0; ch < nch; ++ch) {
            wait_vm<(DW - 2) * 4 * MW>();
            ring_barrier();
#pragma unroll
            for (int f = 0; f < 4 * MW; ++f) issue_w(f, ch + DW, 0, wd);
            wd = wd == NW - 1 ? 0 : wd + 1;
          }
        }
        wait_vm<0>();
        __syncthreads();
        if (MW == 1) {      // the exchange of sums
          __syncthreads();
          __syncthreads();
        }
        __syncthreads();    // the staged output
        if (tb0 + TB < a.T) __syncthreads();
      }
      if (a.nz_out != nullptr) cf_wg_any(false, any_sh);
      return;
    }
  }
  // Pixel copy i of step `wave` of the block: 1 KB, 1024 / PB pixels.  A
  // pixel's 16-byte parts are stored in the order part ^ swizzle (3x3: pixel /
  // 4 % 4, 1x1: pixel / 2 % 8), which spreads the 16 lanes of a fragment read
  // (any 16 consecutive pixels) over all banks.
  constexpr int LPP = PB / 16, PPC = 64 / LPP;     // lanes a pixel, pixels a copy
  const int ext = K == 3 ? a.W + 1 : 0;            // staged pixels before the tile's first
  const int npx = 64 + 2 * ext;                    // real staged pixels
  const int g0 = P0 - ext + lane / LPP;            // pixel of copy 0
  cf_v4i xr;
  bool live = false;                               // the step this wave copies exists
  auto issue_x = [&](int ch, int i, int buf) {
    const int g = g0 + PPC * i, q = lane / LPP + PPC * i;
    const int part = (lane % LPP) ^ (K == 3 ? (q >> 2) & 3 : (q >> 1) & 7);
    const bool ok = live & (ch + part / 4 < nch) & (g >= 0) & (g < a.rows) & (q < npx);
    const uint32_t voff = ok ? (uint32_t)(g * a.Cp * 2 + part * 16) : HALO_OOB;
    lds_buf_copy16_at(xr, voff, __builtin_amdgcn_readfirstlane(ch < nch ? ch * (KC * 2) : 0),
                      __builtin_amdgcn_readfirstlane(smem0 + buf * XB + wave * XT + i * 1024));
  };

  // Fragments in two register sets: a stage's are read from LDS while the
  // stage before it is multiplied.
  f16v acc[TPW];
  h8 ah[2][2], al[2][2], bb[2][2][TPW];
  // The reads of a stage's fragments, RD in all, one by one: for each
  // 16-channel half the hi limb, the steps' pixels, the lo limb; weights from
  // `slot`, pixels from `buf` at `tap` (1x1: half `tap` of the slot's channels).
  constexpr int RD = 2 * (TPW + 2);
  struct Src {
    const char* w;
    const char* x;
    int part;
  };
  auto frag_src = [&](int slot, int buf, int tap) {
    Src r;
    r.w = smem + NX * XB + slot * WB + wc * 4096 + lane * 16;
    int pl = n;
    if constexpr (K == 3) {
      pl = n + (tap / 3) * a.W + tap % 3;
      pl = (taps_in >> tap) & 1u ? pl : NPX - 1;
    }
    r.x = smem + buf * XB + wt * TPW * XT + pl * PB;
    r.part = (K == 3 ? hi ^ ((pl >> 2) & 3) : (4 * tap + hi) ^ ((pl >> 1) & 7)) << 4;
    return r;
  };
  auto read_frag = [&](const Src& r, int set, int k) {
    const int ks = k / (TPW + 2), q = k % (TPW + 2);
    if (q == 0) ah[set][ks] = *reinterpret_cast<const h8*>(r.w + ks * 1024);
    else if (q <= TPW)
      bb[set][ks][q - 1] =
          *reinterpret_cast<const h8*>(r.x + (q - 1) * XT + (r.part ^ (ks * 32)));
    else al[set][ks] = *reinterpret_cast<const h8*>(r.w + 2048 + ks * 1024);
  };
  auto read_frags = [&](int set, int slot, int buf, int tap) {
    const Src r = frag_src(slot, buf, tap);
#pragma unroll
    for (int k = 0; k < RD; ++k) read_frag(r, set, k);
  };
  // Matrix instruction m of a stage's MF (16-channel half, limb, step).
  constexpr int MF = 4 * TPW;
  auto mfma = [&](int set, int m) {
    const int ks = m / (2 * TPW), limb = m / TPW & 1, t = m % TPW;
    acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(limb ? al[set][ks] : ah[set][ks],
                                                    bb[set][ks][t], acc[t], 0, 0, 0);
  };
  // One stage: its matrix instructions from register set `set`, each followed
  // by a part of the stage's other work, so that all of it issues under them
  // (a wave issues in order: reads in a row would hold back the matrix
  // instructions behind them).  After the first one, `sync` publishes the
  // next stage; then its fragments are read into the other set (`src` gives
  // the addresses), and the NC copies of a later stage are issued.
  auto run_stage = [&](auto set_c, auto nc_c, auto&& sync, auto&& src, auto&& copy) {
    constexpr int set = decltype(set_c)::v, NC = decltype(nc_c)::v;
    __builtin_amdgcn_sched_barrier(0);
    mfma(set, 0);
    __builtin_amdgcn_sched_barrier(0);
    sync();
    const Src r = src();
#pragma unroll
    for (int m = 1; m < MF; ++m) {
      // reads spread over instructions 1 .. MF - 2, the copies after them
#pragma unroll
      for (int k = (m - 1) * RD / (MF - 2); k < m * RD / (MF - 2) && k < RD; ++k)
        read_frag(r, set ^ 1, k);
#pragma unroll
      for (int c = (m - 1) * NC / (MF - 1); c < m * NC / (MF - 1); ++c) copy(c);
      __builtin_amdgcn_sched_barrier(0);
      mfma(set, m);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // Potentials of this lane's channels, in registers from block to block.
  // (Pooled: of the pooled pixel whose top-left conv pixel this lane holds.)
  const int gq = wt * NG;                          // first group of four channels
  const int col = wc * 32 + 8 * gq + 4 * hi;       // its first channel in the block
  const int HWs = POOL ? HW / 4 : HW;
  const bool s_ok = p_ok && (!POOL || ((px | py) & 1) == 0);
  const int spix = POOL ? (py >> 1) * (a.W >> 1) + (px >> 1) : pix;
  float v[NG * 4];
  {
    const float v0 = lif_initial_v(a.lif);
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int c = cout0 + col + 8 * g + j;
        v[4 * g + j] = a.v_in != nullptr && s_ok && c < a.Cout
                           ? a.v_in[((size_t)img * a.Cout + c) * HWs + spix] : v0;
      }
  }

  uint32_t anyw = 0u;
  for (int tb0 = 0; tb0 < a.T; tb0 += TB) {
    const int nst = min(TB, a.T - tb0);
#pragma unroll
    for (int t = 0; t < TPW; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[t][r] = 0.0f;

    if (!zero) {
      live = wave < nst;
      xr = halo_rsrc_v4(xsrc + (size_t)(live ? tb0 + wave : 0) * a.rows * a.Cp, 0x7fffffffu);
      if constexpr (K == 3) {
        // every wave copies: the pixels of step `wave`, MW weight fragments
#pragma unroll
        for (int i = 0; i < XL; ++i) issue_x(0, i, 0);
#pragma unroll
        for (int tap = 0; tap < DW; ++tap)
#pragma unroll
          for (int i = 0; i < MW; ++i) issue_w(wave * MW + i, 0, tap, tap);
#pragma unroll
        for (int i = 0; i < XL; ++i) issue_x(1, i, 1);
        wait_vm<(DW - 1) * MW + XL>();             // chunk 0's pixels, tap 0's weights
        ring_barrier();
        read_frags(0, 0, 0, 0);
        int b0 = 0, b1 = 1, b2 = 2;                // buffers of chunks ch, ch + 1, ch + 2
        auto step = [&](auto tap_c, auto set_c, int ch) {
          constexpr int tap = decltype(tap_c)::v;
          constexpr int nt = tap == 8 ? 0 : tap + 1;
          // The next stage's weights were issued DW - 1 steps ago: what came
          // after them may still be in flight (DW - 2 steps' copies).
          constexpr int nx = [] {
            int c = 0;
            for (int k = 1; k <= DW - 2; ++k) c += NX == 3 && (tap + 9 - k) % 9 < XL ? 1 : 0;
            return c;
          }();
          constexpr int XC = NX == 3 && tap < XL ? 1 : 0;
          run_stage(
              set_c, RingInt<XC + MW>{},
              [&] {
                wait_vm<(DW - 2) * MW + nx>();
                ring_barrier();
              },
              [&] { return frag_src(nt, tap == 8 ? b1 : b0, nt); },
              [&](int c) {
                const int f = wave * MW + c - XC;
                if (c < XC) issue_x(ch + 2, tap, b2);
                else if (tap == 0) issue_w(f, ch, 8, 8);
                else issue_w(f, ch + 1, tap - 1, tap - 1);
              });
        };
        // (nine stages a chunk: the register sets swap roles every chunk)
        auto chunk = [&](auto set_c, int ch) {
          constexpr int e = decltype(set_c)::v, o = e ^ 1;
          step(RingInt<0>{}, RingInt<e>{}, ch); step(RingInt<1>{}, RingInt<o>{}, ch);
          step(RingInt<2>{}, RingInt<e>{}, ch); step(RingInt<3>{}, RingInt<o>{}, ch);
          step(RingInt<4>{}, RingInt<e>{}, ch); step(RingInt<5>{}, RingInt<o>{}, ch);
          step(RingInt<6>{}, RingInt<e>{}, ch); step(RingInt<7>{}, RingInt<o>{}, ch);
          step(RingInt<8>{}, RingInt<e>{}, ch);
          const int b = b0;
          b0 = b1; b1 = NX == 3 ? b2 : b; b2 = b;
        };
        for (int ch = 0; ch < nch; ch += 2) {
          chunk(RingInt<0>{}, ch);
          if (ch + 1 < nch) chunk(RingInt<1>{}, ch + 1);
        }
      } else {
        // Stage s issues half (s % 2: pixels 0-31 or 32-63) of the chunk pair
        // DX pairs ahead: XH copies a wave.
        constexpr int XH = XL / 2;
#pragma unroll
        for (int c = 0; c < DX * XL; ++c) issue_x(c / XL * 2, c % XL, c / XL);
        wait_vm<(DX - 1) * XL>();                  // pair 0
        ring_barrier();
        read_frags(0, 0, 0, 0);
        // ring slots: pair of stage ch + 1, pair being copied, weights of
        // stage ch + 1
        int x1 = 0, xd = DX, w1 = 1 % NW;
        auto step = [&](auto set_c, int ch) {
          constexpr int odd = decltype(set_c)::v;   // ch % 2
          if (odd) x1 = x1 == NX - 1 ? 0 : x1 + 1;
          run_stage(
              set_c, RingInt<XH>{},
              [&] {
                // an odd stage is followed by the next pair, whose second half
                // was issued 2 DX - 2 stages ago
                if (odd) wait_vm<(2 * DX - 3) * XH>();
                ring_barrier();
              },
              [&] { return frag_src(w1, x1, odd ^ 1); },
              [&](int c) { issue_x((ch & ~1) + 2 * DX, odd * XH + c, xd); });
          if (odd) xd = xd == NX - 1 ? 0 : xd + 1;
          w1 = w1 == NW - 1 ? 0 : w1 + 1;
        };
        for (int ch = 0; ch < nch; ch += 2) {
          step(RingInt<0>{}, ch);
          if (ch + 1 < nch) step(RingInt<1>{}, ch + 1);
        }
      }
    }

    // Epilogue.  LDS is reused once every copy has landed and every wave has
    // read its last fragments.
    wait_vm<0>();
    __syncthreads();
    // The sums of this lane's channels at every step, z[t][4 g + j].  MW = 1:
    // a wave holds 2 steps of all 16 rows of its lanes and finishes 8 rows at
    // all 4 steps, so the two waves of a tile swap halves.
    float z[TB][NG * 4];
    if constexpr (MW == 2) {
#pragma unroll
      for (int t = 0; t < TB; ++t)
#pragma unroll
        for (int q = 0; q < 16; ++q) z[t][q] = acc[t][q];
    } else {
      float* const xch = reinterpret_cast<float*>(smem) + wn * 2 * 16 * 64 + lane;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int q = 0; q < 8; ++q)
          xch[((wt ^ 1) * 16 + t * 8 + q) * 64] = wt ? acc[t][q] : acc[t][8 + q];
      __syncthreads();
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          const float own = wt ? acc[t][8 + q] : acc[t][q];
          const float other = xch[(wt * 16 + t * 8 + q) * 64];
          z[t][q] = wt ? other : own;
          z[2 + t][q] = wt ? own : other;
        }
      if (!POOL) __syncthreads();                  // the output staging reuses the words
    }
    if constexpr (POOL) {
      // BN -> AvgPool2d(2, 2) -> LIF: the window of an even pixel (W is a
      // power of two up to 16, so its two rows lie in this wave's 32 pixels) is
      // lanes l, l + 1, l + W, l + W + 1; summed in cf_avgpool2x2_lif's order
      const int rows_s = a.rows / 4;
#pragma unroll
      for (int t = 0; t < TB; ++t) {
        if (t >= nst) break;
        const __amdgpu_buffer_rsrc_t ro =
            halo_rsrc(a.out + (size_t)(tb0 + t) * rows_s * a.cp_out,
                      (uint32_t)(rows_s * a.cp_out * 2));
#pragma unroll
        for (int g = 0; g < NG; ++g) {
          h4 sp;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const int c = col + 8 * g + j;
            const float zz = __builtin_fmaf(z[t][4 * g + j], bn_s[0][c], bn_s[1][c]);
            const float z01 = __shfl_down(zz, 1, 64);
            const float z10 = __shfl_down(zz, a.W, 64);
            const float z11 = __shfl_down(zz, a.W + 1, 64);
            const float zp2 = (((zz + z01) + z10) + z11) * 0.25f;
            float vv = lif_charge_m<LM>(v[4 * g + j], zp2, a.lif);
            sp[j] = lif_fire_reset_bit<LM>(vv, a.lif) ? (_Float16)1.0f : (_Float16)0.0f;
            v[4 * g + j] = vv;
          }
          const bool ok = s_ok && cout0 + col + 8 * g < a.Cout;
          const u32x2 pw = __builtin_bit_cast(u32x2, sp);
          anyw |= ok ? (pw[0] | pw[1]) : 0u;
          __builtin_amdgcn_raw_buffer_store_b64(
              pw, ro,
              ok ? (uint32_t)(((img * HWs + spix) * a.cp_out + cout0 + col + 8 * g) * 2) : HALO_OOB,
              0, 0);
        }
      }
    } else {
      // Copy-out chunks of this thread: 16 bytes (8 channels) of a pixel, CPI
      // a step; the identity's matching chunk is loaded before the LIF and
      // added in packed fp16 (exact for the small integers both hold).
      constexpr int CH8 = BM / 8, OLD = BM + 8;
      constexpr int CPI = 64 * CH8 / 256;          // chunks of this thread a step
      _Float16* const ost = reinterpret_cast<_Float16*>(smem);
      static_assert(TB * 64 * OLD * 2 <= G::LDS, "output staging");
      uint32_t co[CPI], ci[CPI];
      u32x4 idc[TB][CPI];
#pragma unroll
      for (int i = 0; i < CPI; ++i) {
        const int c = tid + 256 * i, pp = P0 + c / CH8, ch0 = cout0 + c % CH8 * 8;
        const bool ok = pp < a.rows && ch0 < a.cp_out;
        co[i] = ok ? (uint32_t)((pp * a.cp_out + ch0) * 2) : HALO_OOB;
        ci[i] = ok ? (uint32_t)((pp * a.cp_id + ch0) * 2) : HALO_OOB;
      }
#pragma unroll
      for (int t = 0; t < TB; ++t) {
        const bool have = id != nullptr && t < nst;
        const __amdgpu_buffer_rsrc_t ri =
            halo_rsrc(have ? id + (size_t)(tb0 + t) * a.rows * a.cp_id : (const _Float16*)zp,
                      have ? (uint32_t)(a.rows * a.cp_id * 2) : 0u);
#pragma unroll
        for (int i = 0; i < CPI; ++i)
          idc[t][i] = __builtin_amdgcn_raw_buffer_load_b128(ri, ci[i], 0, 0);
      }
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        const float4 al4 = *reinterpret_cast<const float4*>(&bn_s[0][col + 8 * g]);
        const float4 be4 = *reinterpret_cast<const float4*>(&bn_s[1][col + 8 * g]);
        const float alv[4] = {al4.x, al4.y, al4.z, al4.w};
        const float bev[4] = {be4.x, be4.y, be4.z, be4.w};
#pragma unroll
        for (int t = 0; t < TB; ++t) {
          if (t >= nst) break;
          h4 sp;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const float zz = __builtin_fmaf(z[t][4 * g + j], alv[j], bev[j]);
            float vv = lif_charge_m<LM>(v[4 * g + j], zz, a.lif);
            sp[j] = lif_fire_reset_bit<LM>(vv, a.lif) ? (_Float16)1.0f : (_Float16)0.0f;
            v[4 * g + j] = vv;
          }
          *reinterpret_cast<h4*>(&ost[(t * 64 + n) * OLD + col + 8 * g]) = sp;
        }
      }
      __syncthreads();
#pragma unroll
      for (int t = 0; t < TB; ++t) {
        if (t >= nst) break;
        const __amdgpu_buffer_rsrc_t ro =
            halo_rsrc(a.out + (size_t)(tb0 + t) * a.rows * a.cp_out,
                      (uint32_t)(a.rows * a.cp_out * 2));
#pragma unroll
        for (int i = 0; i < CPI; ++i) {
          const int c = tid + 256 * i;
          const h8 sp = *reinterpret_cast<const h8*>(&ost[(t * 64 + c / CH8) * OLD + c % CH8 * 8]);
          const u32x4 o = __builtin_bit_cast(u32x4, sp + __builtin_bit_cast(h8, idc[t][i]));
          anyw |= co[i] != HALO_OOB ? (o[0] | o[1] | o[2] | o[3]) : 0u;
          __builtin_amdgcn_raw_buffer_store_b128(o, ro, co[i], 0, CF_CPOL_NT);
        }
      }
    }
    if (tb0 + TB < a.T) __syncthreads();   // the next block's copies reuse the LDS
  }
  if (a.v_out != nullptr) {
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int c = cout0 + col + 8 * g + j;
        if (s_ok && c < a.Cout) a.v_out[((size_t)img * a.Cout + c) * HWs + spix] = v[4 * g + j];
      }
  }
  if (a.nz_out != nullptr) {
    // magnitude bits only (-0.0 counts as zero)
    const bool any = cf_wg_any((anyw & 0x7fff7fffu) != 0u, any_sh);
    if (tid == 0) cf_count_publish(a.nz_out, any ? 1ull : 0ull, blockIdx.x, gridDim.x);
  }
  if (a.out_desc != nullptr && blockIdx.x == 0 && tid == 0) {
    a.out_desc->copy = CF_COPY_WRITTEN;
    a.out_desc->vstate = 0u;
    a.out_desc->alias = nullptr;
  }
}

template <int K, int MW, int NPX, int NX, int NW>
hipError_t launch_ring(const RingArgs& a, bool pool, hipStream_t st) {
  const dim3 grid((unsigned)(a.ntiles * a.ncb)), block(RingGeom<K, MW, NPX, NX, NW>::NT);
#define CF_RING(LMV, POOLV) \
  hipLaunchKernelGGL((conv_ring_kernel<K, MW, NPX, NX, NW, LMV, POOLV>), grid, block, 0, st, a)
  const int lm = cf_lif_mode(a.lif);
  if (pool) {
    if constexpr (K == 3 && NX == 3) {             // (pooled maps are at most 16 wide)
      if (lm == LM_HARD0_DECAY_P2) CF_RING(LM_HARD0_DECAY_P2, true);
      else if (lm == LM_HARD_DECAY_P2) CF_RING(LM_HARD_DECAY_P2, true);
      else CF_RING(LM_GENERIC, true);
    } else {
      return hipErrorInvalidValue;
    }
  } else if (lm == LM_HARD0_DECAY_P2) CF_RING(LM_HARD0_DECAY_P2, false);
  else if (lm == LM_HARD_DECAY_P2) CF_RING(LM_HARD_DECAY_P2, false);
  else CF_RING(LM_GENERIC, false);
#undef CF_RING
  return hipGetLastError();
}

}  // namespace

// Runs one conv of the cf_conv_mfma argument list here when this kernel
// covers it and is the faster one; returns false (nothing launched) otherwise,
// else sets *rc (launch false: only says which).  (Called with the arguments
// cf_conv_mfma has checked, no tile masks.)
bool cf_conv_ring(int* rc, const void* x, const void* w_packed, const float* alpha,
                  const float* beta, const float* v_in, float* v_out, void* out_nhwc,
                  int64_t cp_out, const void* identity_nhwc, int64_t cp_id,
                  const unsigned long long* nnz, unsigned long long* nz_out, const void* x_desc,
                  const void* id_desc, void* out_desc, int bias_info,
                  const unsigned long long* id_nnz, int64_t T, int64_t B, int64_t Cp,
                  int64_t Cout, int64_t Coutp, int64_t H, int64_t W, int64_t k, bool pool,
                  const LifParams& lif, bool launch, hipStream_t st) {
  const int64_t rows = B * H * W, KK = k * k;
  if (cp_out != (Cout + 31) / 32 * 32 || (identity_nhwc && (cp_id % 8 != 0 || cp_id < cp_out || pool)) ||
      (Cout % 32 != 0 && (pool || !cf_lif_silent_at_rest(lif))))
    return false;   // (channels past Cout are written as they come: zeros)
  if ((((uintptr_t)x | (uintptr_t)w_packed | (uintptr_t)out_nhwc | (uintptr_t)identity_nhwc) & 15))
    return false;
  if (T > 4 && !v_out) return false;
  // 32-bit indices of the outputs, 31-bit byte offsets within a step's copies
  // and the packed weights
  if (T * rows * Cout > INT32_MAX || 8 * rows * Cp > INT32_MAX || 4 * Coutp * KK * Cp > INT32_MAX ||
      rows * cp_out * 2 > INT32_MAX || rows * (identity_nhwc ? cp_id : 0) * 2 > INT32_MAX)
    return false;
  if (k == 3 && (W > 62 || (W > 30 && Cp > 2 * KC))) return false;
  if (pool && (k != 3 || !(W == 2 || W == 4 || W == 8 || W == 16) || H % 2 != 0)) return false;
  RingArgs a;
  a.x = (const _Float16*)x; a.w = (const _Float16*)w_packed; a.alpha = alpha; a.beta = beta;
  a.v_in = v_in; a.v_out = v_out; a.out = (_Float16*)out_nhwc; a.cp_out = (int)cp_out;
  a.id = (const _Float16*)identity_nhwc; a.cp_id = (int)cp_id; a.nnz = nnz; a.nz_out = nz_out;
  a.x_desc = (const CfOutDesc*)x_desc; a.id_desc = (const CfOutDesc*)id_desc;
  a.out_desc = (CfOutDesc*)out_desc; a.bias_info = bias_info; a.id_nnz = id_nnz;
  a.T = (int)T; a.rows = (int)rows; a.H = (int)H; a.W = (int)W; a.Cp = (int)Cp;
  a.Cout = (int)Cout; a.Coutp = (int)Coutp;
  a.ntiles = (int)((rows + 63) / 64);
  a.lif = lif;
  // What neighbouring workgroups share should be the larger operand.
  a.cb_major = 4 * Cout * KK * Cp > 8 * rows * Cp;
  const int64_t cus = cf_cu_count() > 0 ? cf_cu_count() : 256;
  const int64_t n32 = a.ntiles * ((Cout + 31) / 32), n64 = a.ntiles * (Coutp / 64);
  int mw = 1;
  if (k == 3) {
    // One workgroup per CU at a time (its LDS), so a launch takes whole
    // rounds of about 9 us + 0.125 us a (chunk, tap) stage.  conv_halo.hip's
    // 8x8 tiles of 64 channels take 8 us + 0.33 us a stage for up to one
    // workgroup per CU, and as much more for every further one.  Measured
    // (us here / there, T = 4, SEW and VGG maps): 512 channels 7x7, 1 image
    // 27 / 54, 16 31 / 57, 32 (two rounds) 61 / 67; 4x4, 64 images 33 / 96;
    // 2x2, 64 27 / 91; 256 channels 14x14, 1 18 / 31, 8 21 / 34, 16 (two
    // rounds) 39.4 / 38.7; 128 channels 28x28, 1 14 / 20, 8 (two) 28 / 23; 64
    // channels 56x56, 1 (two slots of pixels) 12.6 / 16.
    const int64_t stages = 9 * (Cp / KC);
    const int64_t halo_wg = B * ((H + 7) / 8) * ((W + 7) / 8) * (Coutp / 64);
    const int64_t here = (n32 + cus - 1) / cus * (9000 + 125 * stages);
    const int64_t there = 8000 + 330 * stages * (halo_wg > cus ? halo_wg : cus) / cus;
    if (here >= there) return false;
  } else {
    // One round only: a launch of more workgroups overlaps one's epilogue with
    // another's loads in conv_halo.hip, which here waits for the LDS.
    // 32-channel tiles where they fit the round, else 64-channel ones.
    // Measured (us, 32 / 64 channels here / there, T = 4): 64 rows of 4096 ->
    // 4096 35 / 51 / 87; 196 rows 1536 -> 384 18 / 25 / 34, 384 -> 1152 11 /
    // 14 / 15; 1,568 rows 1536 -> 384 36 (300 workgroups) / 26 / 39; 784 rows
    // 384 -> 1152 22 (468) / 16 / 20, 384 -> 1536 30 (624) / 28 (312) / 21.
    if (n32 > cus && n64 > cus) return false;
    // Few chunks do not pay for filling the rings.  Up to four steps (more take
    // conv_halo.hip two blocks), here / there: 32 -> 32 channels, 784 rows, T = 1
    // 6.4 / 5.6, 2 6.6 / 6.2, 3 1.01 of it, 4 0.96; 64 -> 64 T = 1 6.6 / 6.1, 2 1.02
    // of it, 3 0.97; 96 1.01, 0.96.  64-channel tiles where conv_halo.hip has its
    // one round too: 1,568 rows, 96 -> 512 T = 1 8.7 / 7.3, 192 1.05 of it, 224 1.02,
    // 256 0.99, T = 4 1.10, 1.00, 0.98, 0.94; where it has two (1,470 rows -> 704, 7x7
    // maps) as 32-channel ones: 96 channels T = 1 1.02, 2 0.98.  (Maps below 4x4
    // take the general kernel instead, two to ten times as long.)
    if (T <= 4 && H >= 4 && W >= 4) {
      const int64_t nch = Cp / KC;
      const int64_t halo_wg = B * ((H + 7) / 8) * ((W + 7) / 8) * (Coutp / 64);
      if (nch + T < 5 || (n32 > cus && halo_wg <= cus && nch < (T < 4 ? 7 : 6)))
        return false;
    }
    mw = n32 <= cus ? 1 : 2;
  }
  a.ncb = mw == 2 ? (int)(Coutp / 64) : (int)((Cout + 31) / 32);
  if (nz_out && (unsigned long long)a.ntiles * a.ncb >= CF_MAX_COUNT_WG) return false;
  if (!launch) return true;
  if (k == 3)
    *rc = (int)(W <= 14   ? launch_ring<3, 1, 96, 3, 9>(a, pool, st)
                : W <= 30 ? launch_ring<3, 1, 128, 3, 9>(a, pool, st)
                          : launch_ring<3, 1, 192, 2, 9>(a, pool, st));
  else if (mw == 1)
    *rc = (int)launch_ring<1, 1, 64, 4, 6>(a, pool, st);
  else
    *rc = (int)launch_ring<1, 2, 64, 3, 7>(a, pool, st);
  return true;
}
