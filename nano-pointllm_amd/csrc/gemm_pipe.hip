// Prefill-regime W8A8 GEMM on pipelined tiles: the shapes that gemm_pipe_choice
// gives a tile (16 k-blocks or more, so K > 960; more than 64 rows; tiles for
// three fifths of the CUs);
// the others stay on gemm.hip's ring kernels.
//
// Replaces the prefill/mixed projections (llama/paged_attention.py:1349-1352,
// 1488; llama/lightweight_runner.py:320-404) for the int8 contract of
// integer_linear_per_output_reference (nanopointllm/compression/w8a8.py:118-139).
#include "gemm_tile.h"

namespace w8a8 {

namespace {

// Pipelined GEMM: WM x WN wavefronts (8, or 4), one workgroup per CU, each
// wavefront BR x BC 16x16 blocks (tile 16 WM BR x 16 WN BC), an S-slot LDS ring of single
// k-blocks (64 K) and one barrier per k-block.
//   * Each wavefront keeps the fragments of its shorter side of a k-block in
//     registers (`held`, double-buffered: read up to a k-block before its
//     MFMAs) and passes the longer side's through R registers (`strm`, read R
//     fragments ahead: a quarter of a k-block on the 352-wide tiles, a third on
//     192 x 288, half on 256 x 256, a whole one on the others), also across the
//     barriers: no MFMA waits for an LDS read issued right behind a barrier.  (gemm_kernel reads a k-block's fragments after
//     its barrier, so all wavefronts read at once while the matrix pipes idle.)
//   * The k-loop has no branch: operand copies past the last k-block re-read it
//     into slots that nothing reads, and wavefronts without a share of their
//     own copy the last fragment again (the same bytes to the same place), so
//     every wait is a fixed count and the compiler schedules whole k-blocks.
//   * Copies are LDS-DMA buffer loads with the k-block as scalar offset, issued
//     between the MFMAs.
// What bounds it: the k-loop runs at 1.62 thousand shader cycles a k-block on
// 256 x 352 (1.41 of them MFMA), 1.27 (1.02) on 256 x 256, 0.50 (0.26) on
// 128 x 128, where the operands, cold and shared by a few CUs, arrive at 55 to 70
// GB/s per CU; with every CU busy the shader clock falls from 2.4 to 1.7-2.0 GHz
// (power: with zero operands it stays at 2.4).  Two k-blocks per barrier, deeper
// rings and other orders of the LDS reads all measured the same or slower.
template <int WM, int WN, int BR, int BC, int S, int R, int EPI, typename TY, typename TH>
__global__ __launch_bounds__(WM * WN * 64, WM * WN / 4) void gemm_pipe_kernel(GemmParams p) {
  constexpr int NW = WM * WN;
  constexpr int BMF = WM * BR;             // 16-row activation tiles per k-block
  constexpr int BNF = WN * BC;             // 16-row weight tiles per k-block
  constexpr int F = BMF + BNF;
  constexpr int LPW = (F + NW - 1) / NW;   // fragment copies per wavefront and k-block
  constexpr bool kHoldB = BC <= BR;
  constexpr int NH = kHoldB ? BC : BR;     // held fragments
  constexpr int NS = kHoldB ? BR : BC;     // streamed fragments
  // At k-block kb's barrier kb and kb + 1 are in the ring, kb - 1's slot is
  // free, and the S - 3 slots between are being filled.
  static_assert(S >= 3 && NW % 4 == 0 && R <= NS && LPW <= NS, "ring shape");
  using Scales = TileScales<EPI, 16 * BMF, 16 * BNF>;
  constexpr int kRing = S * F * 1024;
  __shared__ i32x4 smem[(kRing + sizeof(Scales)) / 16];  // one array, as in gemm_kernel
  auto lds = reinterpret_cast<i32x4 (*)[F][64]>(smem);
  Scales& scales = *reinterpret_cast<Scales*>(smem + kRing / 16);

  const int b = blockIdx.x;
  const int tile = (b % kXcds) * p.per_xcd + b / kXcds;
  if (tile >= p.tiles) return;
  const int mb0 = (tile % p.tiles_m) * BMF;
  const int nb0 = (tile / p.tiles_m) * BNF;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / WN;
  const int wn = wave % WN;
  const int KB = p.KB;

  // Fragment g < BMF of a k-block is activation block mb0 + g, the others
  // weight block nb0 + g - BMF, clamped to the operand's last block (products
  // that the epilogue never stores).
  const i32x4* src[LPW];
  int frag[LPW];
#pragma unroll
  for (int q = 0; q < LPW; ++q) {
    const int g = min(q * NW + wave, F - 1);
    frag[q] = g;
    src[q] = g < BMF ? p.a + static_cast<int64_t>(min(mb0 + g, p.MB - 1)) * KB * 64
                     : p.w + static_cast<int64_t>(min(nb0 + g - BMF, p.NB - 1)) * KB * 64;
  }
  auto copy = [&](int kb, int slot, int q) __attribute__((always_inline)) {
    dma16(dma_rsrc(src[q]), &lds[slot][frag[q]][0], lane * 16, kb * 1024);
  };

  i32x4 acc[BR][BC];
#pragma unroll
  for (int i = 0; i < BR; ++i)
#pragma unroll
    for (int j = 0; j < BC; ++j) acc[i][j] = i32x4{0, 0, 0, 0};

  scales.template load<NW>(p, mb0, nb0, wave, lane);
#pragma unroll
  for (int s = 0; s < S - 1; ++s)
#pragma unroll
    for (int q = 0; q < LPW; ++q) copy(min(s, KB - 1), s, q);
  wait_vmcnt<LPW * (S - 2)>();  // k-block 0
  ring_barrier_tracked();
  const int hoff = kHoldB ? BMF + wn * BC : wm * BR;
  const int soff = kHoldB ? wm * BR : BMF + wn * BC;
  i32x4 held[2][NH], strm[R];
#pragma unroll
  for (int j = 0; j < NH; ++j) held[0][j] = lds[0][hoff + j][lane];
#pragma unroll
  for (int i = 0; i < R; ++i) strm[i] = lds[0][soff + i][lane];

  int slot = 0;       // of k-block kb
  int fill = S - 1;   // of k-block kb + S - 1
  // k-block kb, the I-th of an unrolled group: streamed fragment i sits in
  // register (I NS + i) % R, the held ones in set I % 2.
  auto step = [&](int kb, auto idx) __attribute__((always_inline)) {
    constexpr int I = decltype(idx)::value;
    constexpr int cur = I % 2;
    const int next = slot + 1 == S ? 0 : slot + 1;
    const int fkb = min(kb + S - 1, KB - 1);
    // k-block kb + 1 has landed, and every wavefront has read kb - 1 (its
    // MFMAs, issued above, waited for the reads), whose slot is refilled.
    wait_vmcnt<LPW * (S - 3)>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    static_for<NS>([&](auto ic) __attribute__((always_inline)) {
      constexpr int i = decltype(ic)::value;
      constexpr int reg = (I * NS + i) % R;
#pragma unroll
      for (int q = i * LPW / NS; q < (i + 1) * LPW / NS; ++q) copy(fkb, fill, q);
#pragma unroll
      for (int j = 0; j < NH; ++j) {
        if constexpr (kHoldB) {
          acc[i][j] = mfma_16x16x64(held[cur][j], strm[reg], acc[i][j]);
        } else {
          acc[j][i] = mfma_16x16x64(strm[reg], held[cur][j], acc[j][i]);
        }
      }
      // The fragment R ahead takes the register just used; past the last
      // k-block these reads bring stale bytes that no MFMA takes.
      strm[reg] = i + R < NS ? lds[slot][soff + i + R][lane] : lds[next][soff + i + R - NS][lane];
#pragma unroll
      for (int j = i * NH / NS; j < (i + 1) * NH / NS; ++j)
        held[cur ^ 1][j] = lds[next][hoff + j][lane];
      __builtin_amdgcn_sched_barrier(0);
    });
    slot = next;
    fill = fill + 1 == S ? 0 : fill + 1;
  };
  // Unrolled until the register sets repeat.
  constexpr int U = (2 * NS) % R == 0 ? 2 : 2 * R;
  int kb = 0;
  for (; kb + U <= KB; kb += U)
    static_for<U>([&](auto i) __attribute__((always_inline)) { step(kb + decltype(i)::value, i); });
  static_for<U>([&](auto i) __attribute__((always_inline)) {
    if (kb + decltype(i)::value < KB) step(kb + decltype(i)::value, i);
  });

  wait_vmcnt<0>();  // copies past the last k-block, before the epilogue reuses the ring
  store_tile<WM, WN, BR, BC, kRing, EPI, TY, TH, true, false>(p, acc, wm, wn, mb0, nb0, lane, smem,
                                                              scales);
}

// Launches a pipelined tile for the problem in p.
template <int WM, int WN, int BR, int BC, int S, int R, int EPI, typename TY, typename TH>
hipError_t launch_pipe(GemmParams p, hipStream_t st) {
  const int64_t tiles_m = ceil_div(p.MB, WM * BR);
  const int64_t tiles = tiles_m * ceil_div(p.NB, WN * BC);
  if (ceil_div(tiles, kXcds) * kXcds > INT32_MAX) return hipErrorInvalidConfiguration;
  p.tiles_m = static_cast<int>(tiles_m);
  p.tiles = static_cast<int>(tiles);
  p.per_xcd = static_cast<int>(ceil_div(tiles, kXcds));
  hipLaunchKernelGGL((gemm_pipe_kernel<WM, WN, BR, BC, S, R, EPI, TY, TH>),
                     dim3(p.per_xcd * kXcds), dim3(WM * WN * 64), 0, st, p);
  return hipGetLastError();
}

struct PipeLaunch {
  template <int EPI, typename TY, typename TH>
  static hipError_t launch(const GemmParams& p, hipStream_t st, int tile) {
    switch (tile) {
      case kPipe256x352:
        return launch_pipe<4, 2, 4, 11, 4, 3, EPI, TY, TH>(p, st);
      case kPipe256x256:
        return launch_pipe<4, 2, 4, 8, 4, 4, EPI, TY, TH>(p, st);
      case kPipe256x192:
        return launch_pipe<4, 2, 4, 6, 5, 6, EPI, TY, TH>(p, st);
      case kPipe256x128:
        return launch_pipe<4, 2, 4, 4, 6, 4, EPI, TY, TH>(p, st);
      case kPipe192x288:
        return launch_pipe<4, 2, 3, 9, 5, 3, EPI, TY, TH>(p, st);
      case kPipe192x160:
        return launch_pipe<4, 2, 3, 5, 7, 5, EPI, TY, TH>(p, st);
      case kPipe192x352:
        return launch_pipe<4, 2, 3, 11, 4, 3, EPI, TY, TH>(p, st);
      case kPipe128x128:
        return launch_pipe<2, 4, 4, 2, 9, 4, EPI, TY, TH>(p, st);
      case kPipe128x96:
        return launch_pipe<4, 2, 2, 3, 9, 3, EPI, TY, TH>(p, st);
      case kPipe128x64:
        return launch_pipe<4, 2, 2, 2, 13, 2, EPI, TY, TH>(p, st);
      case kPipe64x64:
        return launch_pipe<2, 2, 2, 2, 16, 2, EPI, TY, TH>(p, st);
      default:
        return hipErrorInvalidValue;
    }
  }
};

}  // namespace

// The pipelined tile whose rounds over the CUs take least, by the time of one
// of its k-steps with all CUs busy (nanoseconds, measured at K = 4096 and
// 11008: the wider the tile, the less per product).  So packed QKV takes
// 192x160 at 560 rows (231 tiles, 33.4 us; 35.2 on the weights-direct tile)
// and 256x192 at 2048 (two full rounds, 91 us against 104 for 128x256), gate/up
// 192x288 at 560 (52.7 against 63.9 for 128x224), 192x352 at 768 (61.9 against
// 68.2 for 256x352) and 256x352 at 1024 and 2048 (82 against 105, 153 against 179),
// O and down 64x64 at 201 (13.4 / 28.4 against 14.5 / 32.7 on the ring), 128x64 at
// 350 (16.1 / 36.3 against 16.7 / 40.7), 128x96 at 560 (16.8 / 38.0 against 20.4 /
// 49 for the ring's 112x96 and 18.6 / 41.3 for 128x128), 128x128 at 1024 (51 against
// 57 for the ring of 16 wavefronts) and 256x128 at 2048 (34 / 77 against 38 / 99).
// Taken where the tiles fill three fifths of the CUs; below that the smaller
// ring tiles cover more of them (down at 100 rows: 27.0 against 28.0 us on 64x64).
// From 16 k-blocks: filling a ring of up to 16 is a large part of a shorter
// product (2048 x 12288 x 512 21.4 on the ring against 22.0, 560 x 4096 x 768 6.8
// against 7.0).  One line for all sizes is not the best one: products of several
// rounds gain earlier (2048 x 22016 x 768 59.8 on the ring against 52.0).
int gemm_pipe_choice(int64_t MB, int64_t NB, int64_t KB, int64_t cus) {
  struct Tile {
    GemmPipe id;
    int mb, nb, step_ns;
  };
  static constexpr Tile kTiles[] = {
      {kPipe256x352, 16, 22, 880}, {kPipe192x352, 12, 22, 740}, {kPipe256x256, 16, 16, 670},
      {kPipe192x288, 12, 18, 600}, {kPipe256x192, 16, 12, 560}, {kPipe256x128, 16, 8, 435},
      {kPipe192x160, 12, 10, 400}, {kPipe128x128, 8, 8, 275},   {kPipe128x96, 8, 6, 240},
      {kPipe128x64, 8, 4, 205},    {kPipe64x64, 4, 4, 160},
  };
  if (MB <= 4 || KB < 16 || KB >= (int64_t{1} << 20)) return kPipeNone;
  int best = kPipeNone;
  int64_t best_ns = 0, best_tiles = 0;
  for (const Tile& t : kTiles) {
    const int64_t tiles = ceil_div(MB, t.mb) * ceil_div(NB, t.nb);
    const int64_t ns = ceil_div(tiles, cus) * t.step_ns;
    if (best == kPipeNone || ns < best_ns) {
      best = t.id;
      best_ns = ns;
      best_tiles = tiles;
    }
  }
  return 5 * best_tiles >= 3 * cus ? best : kPipeNone;
}

hipError_t launch_gemm_pipe(const LinearOperands& op, int tile, hipStream_t st) {
  return gemm_dispatch<PipeLaunch>(op, gemm_params(op), st, tile);
}

}  // namespace w8a8
