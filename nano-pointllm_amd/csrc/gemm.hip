// Prefill-regime W8A8 GEMM (M > 64, or M > 32 with N > 12288 and K > 4096):
// y = epi(xq @ wq^T) with int8 MFMA.
//
// Replaces the prefill/mixed projections (llama/paged_attention.py:1349-1352,
// 1488; llama/lightweight_runner.py:320-404) for the int8 contract of
// integer_linear_per_output_reference (nanopointllm/compression/w8a8.py:118-139).
//
// These kernels take what gemm_pipe_choice (gemm_pipe.hip) leaves: products of
// fewer than 16 k-blocks (K <= 960), at most 64 rows, and those whose tiles
// there would not fill three fifths of the CUs.  The last two take only the
// 32x32, 64x32, 64x64 and two-per-CU 128x128 tiles; the others below (112x256
// weights-direct, 112x96, 128x96, 128x192, 128x224, 128x256, 256x256 and 128x128
// with one per CU) serve K <= 960 alone.
//
// Design (MFMA-bound), chosen by measurement on MI355X (gemm_kernel; the
// weights-direct gemm_wd_kernel further below keeps the weights out of LDS):
//   * v_mfma_i32_16x16x64_i8.  Its operand is exactly one packed 16x64
//     fragment (lane l holds 16 bytes of row l%16), read with one contiguous
//     ds_read_b128.  On random int8 data it sustains more than the 32x32x32
//     form: 3.3 against 3.0 POPS from LDS alone, and 15-25% more in this
//     kernel on LLaMA-7B shapes (the matrix pipes slow down with the
//     data-dependent switching of their inputs).
//   * Every wavefront owns a BR x BC grid of 16x16 output blocks; the
//     workgroup tile is a WM x WN grid of wavefronts: 128x256 (8 wavefronts
//     of 64x64) when there are enough such tiles to fill every CU twice, else
//     128x128 (16 wavefronts of 32x32), else 64x64 (4 wavefronts of 32x32,
//     4 workgroups per CU) when 128x128 tiles would not cover every CU; past
//     64 rows, 64x32 (4 wavefronts of 32x16) when those fill one round; and
//     112x96 (14 wavefronts of 16x48) or 128x96 (8 of 32x48), one per CU,
//     when one round of those fills the CUs.  The full rule is at launch_t.
//   * Both operands are in the packed 16x64 tile layout, so a k-step (64) of
//     the workgroup tile is (BM + BN)/16 fragments of 1 KiB.  Each wavefront
//     copies its share with global_load_lds_dwordx4 straight into a 3- or
//     4-stage LDS ring (lane l lands at slot base + 16*l, the fragment layout),
//     keeping STG - 1 k-steps in flight; explicit vmcnt waits and one barrier
//     per k-step order the ring.
//   * Workgroups are mapped XCD-major: consecutive tiles of the same weight
//     column block land on the same XCD and share its L2.
#include "gemm_tile.h"

namespace w8a8 {

namespace {

// WM x WN wavefronts, each owning BR x BC blocks of 16x16 (BM = 16 WM BR,
// BN = 16 WN BC), with an STG-deep LDS ring whose stages hold KT k-blocks
// (64 K each) of both operands.
// The second launch bound is waves per SIMD: OCC workgroups of WM x WN
// wavefronts over the CU's 4 SIMDs, so the register budget admits OCC
// workgroups per CU.
template <int WM, int WN, int BR, int BC, int STG, int OCC, int KT, int EPI, typename TY,
          typename TH>
__global__ __launch_bounds__(WM * WN * 64, OCC * WM * WN / 4) void gemm_kernel(GemmParams p) {
  constexpr int NW = WM * WN;
  constexpr int BMF = WM * BR;  // 16-row activation tiles per k-block
  constexpr int BNF = WN * BC;  // 16-row weight tiles per k-block
  constexpr int F = BMF + BNF;
  constexpr int FS = F * KT;    // fragments per stage
  // Fragment copies per wave per stage: LPW for the first FS - (LPW-1) NW
  // waves, LPW - 1 for the rest.
  constexpr int LPW = (FS + NW - 1) / NW;
  using Scales = TileScales<EPI, 16 * BMF, 16 * BNF>;
  constexpr int kRing = STG * FS * 1024;
  // One array for the ring and the scales: the compiler takes LDS-DMA into
  // one object to be finished by its own wait before it reads another.
  __shared__ i32x4 smem[(kRing + sizeof(Scales)) / 16];
  auto lds = reinterpret_cast<i32x4 (*)[FS][64]>(smem);
  Scales& scales = *reinterpret_cast<Scales*>(smem + kRing / 16);

  // XCD-major tile mapping: workgroup b runs on XCD b % 8.
  const int b = blockIdx.x;
  const int tile = (b % kXcds) * p.per_xcd + b / kXcds;
  if (tile >= p.tiles) return;
  const int mb0 = (tile % p.tiles_m) * BMF;
  const int nb0 = (tile / p.tiles_m) * BNF;

  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int wm = wave / WN;
  const int wn = wave % WN;
  const int KB = p.KB;
  const int NS = static_cast<int>(ceil_div(KB, KT));  // ring stages over K

  // Fragment f = q*NW + wave of a stage is k-block f / F of the stage; of
  // that k-block, g = f % F < BMF are activation blocks mb0 + g, the rest
  // weight blocks nb0 + g - BMF.  Blocks past the operand are clamped to its
  // last block: their products only reach accumulator rows or columns that
  // the epilogue never stores.  K-blocks past KB (the last stage of a K that
  // is not a multiple of 64 KT) reload block KB - 1 and are not multiplied.
  const bool full = (LPW - 1) * NW + wave < FS;  // wave-uniform
  const i32x4* src[LPW];
  int kk_of[LPW];
#pragma unroll
  for (int q = 0; q < LPW; ++q) {
    const int f = min(q * NW + wave, FS - 1);
    const int g = f % F;
    kk_of[q] = f / F;
    if (g < BMF) {
      src[q] = p.a + static_cast<int64_t>(min(mb0 + g, p.MB - 1)) * KB * 64 + lane;
    } else {
      src[q] = p.w + static_cast<int64_t>(min(nb0 + g - BMF, p.NB - 1)) * KB * 64 + lane;
    }
  }
  auto issue = [&](int stage, int slot) {
#pragma unroll
    for (int q = 0; q < LPW; ++q)
      if (q < LPW - 1 || full) {
        const int kb = min(stage * KT + kk_of[q], KB - 1);
        __builtin_amdgcn_global_load_lds(
            static_cast<const void*>(src[q] + static_cast<int64_t>(kb) * 64),
            (lds_void*)(&lds[slot][q * NW + wave][0]), 16, 0, 0);
      }
  };

  i32x4 acc[BR][BC];
#pragma unroll
  for (int i = 0; i < BR; ++i)
#pragma unroll
    for (int j = 0; j < BC; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[i][j][r] = 0;

  scales.template load<NW>(p, mb0, nb0, wave, lane);

#pragma unroll
  for (int s = 0; s < STG - 1; ++s)
    if (s < NS) issue(s, s);

  for (int st = 0; st < NS; ++st) {
    // Stage st has landed once only the later stages' loads may remain.
    if (st + STG - 2 < NS) {
      if (full) {
        wait_vmcnt<LPW * (STG - 2)>();
      } else {
        wait_vmcnt<(LPW - 1) * (STG - 2)>();
      }
    } else {
      wait_vmcnt<0>();
    }
    ring_barrier();
    // Every wave has finished reading the slot of stage st-1: refill it.
    if (st + STG - 1 < NS) issue(st + STG - 1, (st + STG - 1) % STG);
    const int slot = st % STG;
#pragma unroll
    for (int kk = 0; kk < KT; ++kk) {
      if (KT == 1 || st * KT + kk < KB) {
        i32x4 af[BR], bf[BC];
#pragma unroll
        for (int i = 0; i < BR; ++i) af[i] = lds[slot][kk * F + wm * BR + i][lane];
#pragma unroll
        for (int j = 0; j < BC; ++j) bf[j] = lds[slot][kk * F + BMF + wn * BC + j][lane];
#pragma unroll
        for (int i = 0; i < BR; ++i)
#pragma unroll
          for (int j = 0; j < BC; ++j) acc[i][j] = mfma_16x16x64(bf[j], af[i], acc[i][j]);
      }
    }
  }

  if (NS == 0) {  // K = 0: no stage's barrier has stood behind the scales' copies
    wait_vmcnt<0>();
    ring_barrier();
  }
  constexpr bool kHoist = OCC * NW / 4 <= 4;  // at least 128 registers
  store_tile<WM, WN, BR, BC, kRing, EPI, TY, TH, false, kHoist>(p, acc, wm, wn, mb0, nb0, lane, smem,
                                                               scales);
}

// Weights-direct GEMM: NW wavefronts, each owning all A 16-row activation
// blocks of the tile and B 16-row weight blocks of its own (tile 16A x
// 16 NW B).  A weight fragment is used by exactly one wavefront, so it goes
// from global memory straight into registers (the packed fragment is the
// MFMA operand image) through a ring of D + 1 register sets, D k-blocks ahead;
// only the activation fragments, which every wavefront reads, pass through
// LDS: buffer_load ... lds copies into an S-slot ring, and each wavefront
// reads k-block t+1 into registers during k-block t's MFMAs.  Per k-block a
// wavefront reads A KiB from LDS for A x B MFMAs, against (BR + BC) KiB for
// BR x BC in gemm_kernel.  One barrier per k-block.
template <int NW, int A, int B, int D, int EPI, typename TY, typename TH>
__global__ __launch_bounds__(NW * 64, NW / 4) void gemm_wd_kernel(GemmParams p) {
  static_assert(D >= 2 && NW % 4 == 0, "prefetch depth and wavefront count");
  constexpr int S = D <= 2 ? 2 : (D <= 4 ? 4 : 8);  // ring slots: a power of two >= D
  constexpr int BS = D + 1;                          // weight register sets
  constexpr int LPW = (A + NW - 1) / NW;             // activation copies per wavefront
  constexpr int BM = 16 * A;
  constexpr int BN = 16 * NW * B;
  constexpr bool kHalfCols = EPI == kEpiSilu || EPI == kEpiSiluQ8;
  constexpr int kRing = S * A * 1024;
  constexpr int kOut = BM * (kHalfCols ? BN / 2 : BN) * static_cast<int>(sizeof(TY));
  constexpr int kLds = kRing > kOut ? kRing : kOut;
  using Scales = TileScales<EPI, BM, BN>;
  // One array, as in gemm_kernel.
  __shared__ i32x4 lds[(kLds + sizeof(Scales)) / 16];
  Scales& scales = *reinterpret_cast<Scales*>(lds + kLds / 16);
  auto ring = reinterpret_cast<i32x4 (*)[A][64]>(lds);

  const int b = blockIdx.x;
  const int tile = (b % kXcds) * p.per_xcd + b / kXcds;
  if (tile >= p.tiles) return;
  const int mb0 = (tile % p.tiles_m) * A;
  const int nb0 = (tile / p.tiles_m) * (NW * B);
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int KB = p.KB;

  // Activation block q * NW + wave of the tile (clamped to the last block:
  // its products reach only rows the epilogue never stores).
  const bool full = (LPW - 1) * NW + wave < A;
  const __amdgpu_buffer_rsrc_t arsrc = dma_rsrc(p.a + static_cast<int64_t>(mb0) * KB * 64);
  uint32_t aoff[LPW];
#pragma unroll
  for (int q = 0; q < LPW; ++q) {
    const int f = min(q * NW + wave, A - 1);
    aoff[q] = static_cast<uint32_t>((min(mb0 + f, p.MB - 1) - mb0) * KB * 1024 + lane * 16);
  }
  const i32x4* bsrc[B];
#pragma unroll
  for (int j = 0; j < B; ++j)
    bsrc[j] = p.w + static_cast<int64_t>(min(nb0 + wave * B + j, p.NB - 1)) * KB * 64 + lane;

  i32x4 breg[BS][B];
  i32x4 af[2][A];
  i32x4 acc[A][B];
#pragma unroll
  for (int i = 0; i < A; ++i)
#pragma unroll
    for (int j = 0; j < B; ++j) acc[i][j] = i32x4{0, 0, 0, 0};

  auto issue = [&](int kb, auto set_c) __attribute__((always_inline)) {
    constexpr int set = decltype(set_c)::value;
#pragma unroll
    for (int q = 0; q < LPW; ++q)
      if (q < LPW - 1 || full)
        dma16(arsrc, &ring[kb & (S - 1)][q * NW + wave][0], aoff[q] + static_cast<uint32_t>(kb) * 1024);
#pragma unroll
    for (int j = 0; j < B; ++j) breg[set][j] = bsrc[j][static_cast<int64_t>(kb) * 64];
  };
  // Loads per wavefront per k-block.
  constexpr int kLoadsFull = LPW + B;
  constexpr int kLoadsPart = LPW - 1 + B;

  scales.template load<NW>(p, mb0, nb0, wave, lane);
  static_for<D>([&](auto i) __attribute__((always_inline)) {
    if (decltype(i)::value < KB) issue(decltype(i)::value, i);
  });
  // k-block 0 has landed once only k-blocks 1 .. D-1 may be in flight.
  if (D - 1 < KB) {
    if (full) wait_vmcnt<kLoadsFull * (D - 1)>(); else wait_vmcnt<kLoadsPart * (D - 1)>();
  } else {
    wait_vmcnt<0>();
  }
  ring_barrier_tracked();
#pragma unroll
  for (int i = 0; i < A; ++i) af[0][i] = ring[0][i][lane];

  // k-block kb: make kb+1's activations visible and read them, refill the
  // slot and register set kb+1 leaves behind with k-block kb+D, then kb's
  // MFMAs.  STEADY: kb + 1 < KB is known.
  auto step = [&](int kb, auto set_c, auto cur_c, auto steady_c) __attribute__((always_inline)) {
    constexpr int set = decltype(set_c)::value;
    constexpr int nset = (set + D) % BS;
    constexpr int cur = decltype(cur_c)::value;
    constexpr bool steady = decltype(steady_c)::value;
    if (steady || kb + 1 < KB) {
      // k-block kb+1 has landed once only kb+2 .. kb+D-1 may be in flight.
      if (kb + D - 1 < KB) {
        if (full) wait_vmcnt<kLoadsFull * (D - 2)>(); else wait_vmcnt<kLoadsPart * (D - 2)>();
      } else {
        wait_vmcnt<0>();
      }
      ring_barrier_tracked();
      // Slot (kb+D) & (S-1) held k-block kb+D-S <= kb-1, read before the barrier.
      if (kb + D < KB) issue(kb + D, std::integral_constant<int, nset>{});
#pragma unroll
      for (int i = 0; i < A; ++i) af[cur ^ 1][i] = ring[(kb + 1) & (S - 1)][i][lane];
    }
#pragma unroll
    for (int i = 0; i < A; ++i)
#pragma unroll
      for (int j = 0; j < B; ++j) acc[i][j] = mfma_16x16x64(breg[set][j], af[cur][i], acc[i][j]);
  };
  // Unrolled by U, a multiple of the register-set count and of 2, so every
  // set and buffer index is static.
  constexpr int U = (BS % 2 == 0) ? BS : 2 * BS;
  int kb = 0;
  for (; kb + U < KB; kb += U) {
    static_for<U>([&](auto i) __attribute__((always_inline)) {
      constexpr int I = decltype(i)::value;
      step(kb + I, std::integral_constant<int, I % BS>{}, std::integral_constant<int, I % 2>{},
           std::true_type{});
    });
  }
  static_for<U>([&](auto i) __attribute__((always_inline)) {
    constexpr int I = decltype(i)::value;
    if (kb + I < KB)
      step(kb + I, std::integral_constant<int, I % BS>{}, std::integral_constant<int, I % 2>{},
           std::false_type{});
  });

  store_tile<1, NW, A, B, kLds, EPI, TY, TH>(p, acc, 0, wave, mb0, nb0, lane, lds, scales);
}

// Launches the weights-direct kernel for the problem in p.
template <int NW, int A, int B, int D, int EPI, typename TY, typename TH>
hipError_t launch_wd(GemmParams p, hipStream_t st) {
  const int64_t tiles_m = ceil_div(p.MB, A);
  const int64_t tiles = tiles_m * ceil_div(p.NB, NW * B);
  if (tiles == 0) return hipSuccess;
  if (ceil_div(tiles, kXcds) * kXcds > INT32_MAX) return hipErrorInvalidConfiguration;
  p.tiles_m = static_cast<int>(tiles_m);
  p.tiles = static_cast<int>(tiles);
  p.per_xcd = static_cast<int>(ceil_div(tiles, kXcds));
  hipLaunchKernelGGL((gemm_wd_kernel<NW, A, B, D, EPI, TY, TH>), dim3(p.per_xcd * kXcds),
                     dim3(NW * 64), 0, st, p);
  return hipGetLastError();
}

// Launches one tile configuration for the problem in p (tile counts are
// filled in here).
template <int WM, int WN, int BR, int BC, int STG, int OCC, int KT, int EPI, typename TY,
          typename TH>
hipError_t launch_cfg(GemmParams p, hipStream_t st) {
  const int64_t tiles_m = ceil_div(p.MB, WM * BR);
  const int64_t tiles = tiles_m * ceil_div(p.NB, WN * BC);
  if (tiles == 0) return hipSuccess;
  if (ceil_div(tiles, kXcds) * kXcds > INT32_MAX) return hipErrorInvalidConfiguration;
  p.tiles_m = static_cast<int>(tiles_m);
  p.tiles = static_cast<int>(tiles);
  p.per_xcd = static_cast<int>(ceil_div(tiles, kXcds));
  hipLaunchKernelGGL((gemm_kernel<WM, WN, BR, BC, STG, OCC, KT, EPI, TY, TH>),
                     dim3(p.per_xcd * kXcds), dim3(WM * WN * 64), 0, st, p);
  return hipGetLastError();
}

// Tile configurations, chosen by tile count.  Measured on MI355X, random data,
// cold weights, LLaMA-7B projections (K = 4096 and 11008) at M = 256..2048,
// which the pipelined tiles have since taken from all but the 32x32, 64x32, 64x64
// and two-per-CU 128x128 ones: the figures below order the ring tiles among
// themselves, and the projections named are no longer what they run.  A launch is fastest
// when its tiles fill one round of workgroup slots (2 per CU) as closely as
// possible, and when several rounds are needed, with the widest tile:
//   * first the one-workgroup-per-CU tiles taken when one round of them fills
//     the CUs (gemm_tile_choice): 112x256 weights-direct (gemm_wd_kernel;
//     N = 12288 at M = 449..560), then 112x96 and 128x96 (N = 4096 at
//     M = 465..640);
//   * past 64 rows (M > 64), 64x32 tiles (4 waves of 32x16, a 3-stage ring of
//     four k-blocks, 2 workgroups per CU) when they fit in one round and
//     number at least half the CUs: O and down at M = 65..128 13-16% faster
//     than the tiles below, 4-10% at M = 160..256, N = 2048 14%; beyond one
//     round (N = 8192 past M = 128) they lose;
//   * 128x128 tiles, when they fit in one round: 16 waves of 32x32, a
//     4-stage ring of one k-block (64 K), 2 workgroups per CU, when there
//     are more of them than CUs; else (one tile per CU or less, where every
//     k-step's barrier and memory latency is exposed) ring stages of several
//     k-blocks cut the barriers and keep more bytes in flight: 64x64 (4 waves
//     of 32x32, a 2-stage ring of four k-blocks, 2 per CU) when those tiles
//     fit in one round, else 128x128 with a 4-stage ring of two k-blocks,
//     one per CU (8-14% faster on O and down at M = 560..1024, 15-20% at
//     M = 384, with weights streamed from HBM).  With at most one 64x64 tile
//     per CU, 32x32 tiles of one wave (a 3-stage ring of four k-blocks, 3 per
//     CU by LDS) spread the work over more CUs when they fit in one round:
//     9-13% faster on QKV at M = 64;
//   * else the widest of 128x192, 128x224 and 128x256 whose tiles still fit
//     in one round, trying the narrowest first (8 waves of 32x96, 32x112 or
//     64x64, 3-stage ring): N = 22016 at M = 560 in 495 tiles of 128x224 was
//     8% faster than in 430 of 128x256;
//   * else (several rounds) 128x256, except just past one round of those
//     (1 to 1.25 tiles per slot), where the few tiles of the second round cost
//     more than the wider tile saves and 128x128 is kept, and except from two
//     full rounds of 256x256 tiles (one per CU, 16 waves of 64x64, 2-stage
//     ring of two k-blocks) when those add no row padding: the square tile
//     reads a third fewer operand bytes per MAC (2048 x 22016 x 4096: 1.94
//     against 1.71 POPS; 8192^3: 2.03 against 1.99), while at 1.3-1.5 rounds
//     it gains nothing.
template <int EPI, typename TY, typename TH>
hipError_t launch_t(const GemmParams& p, hipStream_t st) {
  switch (gemm_tile_choice(p.MB, p.NB, cu_count())) {
    case kGemmTinyDeep:
      return launch_cfg<1, 1, 2, 2, 3, 4, 4, EPI, TY, TH>(p, st);
    case kGemmSmallDeep:
      return launch_cfg<2, 2, 2, 2, 2, 2, 4, EPI, TY, TH>(p, st);
    case kGemmBigDeep:
      return launch_cfg<4, 4, 2, 2, 4, 1, 2, EPI, TY, TH>(p, st);
    case kGemmBig:
      return launch_cfg<4, 4, 2, 2, 4, 2, 1, EPI, TY, TH>(p, st);
    case kGemmW192:
      return launch_cfg<4, 2, 2, 6, 3, 2, 1, EPI, TY, TH>(p, st);
    case kGemmW224:
      return launch_cfg<4, 2, 2, 7, 3, 2, 1, EPI, TY, TH>(p, st);
    case kGemmW256Sq:
      return launch_cfg<4, 4, 4, 4, 2, 1, 2, EPI, TY, TH>(p, st);
    case kGemmMid:
      return launch_cfg<2, 2, 2, 1, 3, 2, 4, EPI, TY, TH>(p, st);
    case kGemmWd7x2:
      return launch_wd<8, 7, 2, 4, EPI, TY, TH>(p, st);
    case kGemmT112x96:
      return launch_cfg<7, 2, 1, 3, 3, 1, 3, EPI, TY, TH>(p, st);
    case kGemmT128x96:
      return launch_cfg<4, 2, 2, 3, 2, 1, 4, EPI, TY, TH>(p, st);
    default:
      return launch_cfg<2, 4, 4, 4, 3, 2, 1, EPI, TY, TH>(p, st);
  }
}

struct RingLaunch {
  template <int EPI, typename TY, typename TH>
  static hipError_t launch(const GemmParams& p, hipStream_t st) {
    return launch_t<EPI, TY, TH>(p, st);
  }
};

}  // namespace

int gemm_tile_choice(int64_t MB, int64_t NB, int64_t cus) {
  // The 112 x 256 weights-direct tile when one round of it (one workgroup per
  // CU) fills at least 85% of the CUs with at least 85% of the tile rows in
  // use (N = 12288 at M = 449..560).  A 144 x 64 weights-direct tile for
  // N = 4096 at the same M measured slower than the 128 x 128 deep ring
  // (K = 4096 27.2 vs 23.5 us, K = 11008 59.6 vs 51.3 us with the fp16
  // epilogue), so those keep the LDS-ring tiles.
  if (MB > 4) {
    const int64_t tm = ceil_div(MB, 7);
    const int64_t tiles = tm * ceil_div(NB, 16);
    if (tiles <= cus && 100 * tiles >= 85 * cus && 100 * MB >= 85 * tm * 7) return kGemmWd7x2;
  }
  // Narrow tiles (96 columns) when one round of them, at least four tile rows
  // deep, fills at least 80% of the CUs with at least 85% of the tile rows in
  // use: N = 4096 at M = 465..640, where 128x128 tiles leave 96 of 256 CUs
  // idle.  Measured at M = 560 (fp16 epilogue, K = 4096 and 11008, before the
  // pipelined tiles took those): 112x96 20.8 against 23.6 us and 48.1 against
  // 58.5; at M = 567 (36 row blocks) 128x96 21.6 against 23.8 us.  The 14 wavefronts of
  // 112x96 each own a 16-row strip.
  if (MB > 4) {
    auto one_round = [&](int64_t rows, int64_t cols) {
      const int64_t tm = ceil_div(MB, rows);
      const int64_t tiles = tm * ceil_div(NB, cols);
      return tm >= 4 && tiles <= cus && 100 * tiles >= 80 * cus && 100 * MB >= 85 * tm * rows;
    };
    if (one_round(7, 6)) return kGemmT112x96;
    if (one_round(8, 6)) return kGemmT128x96;
  }
  const int64_t slots = cus * 2;
  const int64_t tiles_m = ceil_div(MB, 8);  // 128-row tiles
  const int64_t big_tiles = tiles_m * ceil_div(NB, 8);
  if (big_tiles <= slots) {
    const int64_t mid_tiles = ceil_div(MB, 4) * ceil_div(NB, 2);
    if (MB > 4 && 2 * mid_tiles >= cus && mid_tiles <= slots) return kGemmMid;
    if (big_tiles > cus) return kGemmBig;
    const int64_t small_tiles = ceil_div(MB, 4) * ceil_div(NB, 4);
    if (small_tiles <= cus && ceil_div(MB, 2) * ceil_div(NB, 2) <= 3 * cus) return kGemmTinyDeep;
    if (small_tiles <= slots) return kGemmSmallDeep;
    return kGemmBigDeep;
  }
  if (tiles_m * ceil_div(NB, 12) <= slots) return kGemmW192;
  if (tiles_m * ceil_div(NB, 14) <= slots) return kGemmW224;
  const int64_t wide_tiles = tiles_m * ceil_div(NB, 16);
  const bool short_second_round = wide_tiles > slots && wide_tiles * 100 < slots * 125;
  if (short_second_round) return kGemmBig;
  const int64_t sq_tiles_m = ceil_div(MB, 16);
  if (sq_tiles_m * ceil_div(NB, 16) >= 2 * cus && sq_tiles_m * 2 == tiles_m) return kGemmW256Sq;
  return kGemmW256;
}

hipError_t launch_gemm(const LinearOperands& op, hipStream_t st) {
  const GemmParams p = gemm_params(op);
  if (p.MB == 0 || p.NB == 0) return hipSuccess;
  const int pipe = gemm_pipe_choice(p.MB, p.NB, p.KB, cu_count());
  if (pipe != kPipeNone) return launch_gemm_pipe(op, pipe, st);
  return gemm_dispatch<RingLaunch>(op, p, st);
}

}  // namespace w8a8
