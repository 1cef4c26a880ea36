// Prefill-regime W8A8 GEMM (M > 64, or M > 32 with N > 12288 and K > 4096):
// y = epi(xq @ wq^T) with int8 MFMA.
//
// Replaces the prefill/mixed projections (llama/paged_attention.py:1349-1352,
// 1488; llama/lightweight_runner.py:320-404) for the int8 contract of
// integer_linear_per_output_reference (nanopointllm/compression/w8a8.py:118-139).
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
#include "w8a8_internal.h"

#include <utility>

namespace w8a8 {

namespace {

struct GemmParams {
  const i32x4* a;
  const float* sx;
  const i32x4* w;
  const float* sw;
  const float* bias;
  void* y;
  int64_t ldy;
  float out_scale;
  const uint32_t* rq_mult;
  const int32_t* rq_shift;
  const int32_t* rq_bias;
  float* absmax_parts;  // kEpiSilu: [M][NB] per-block row |h|max (nullable)
  // kEpiDequant with 16-bit outputs (nullable): the residual rows added to them.
  const void* res;
  int64_t ld_res;
  int M;
  int N;
  int MB;
  int NB;
  int KB;
  int tiles_m;
  int tiles;
  int per_xcd;
};

constexpr int kXcds = 8;

typedef __attribute__((address_space(3))) void lds_void;

// C layout: lane l, register r holds row 4(l/16) + r of the first operand and
// row l%16 of the second.  The kernels pass the weights first, so a lane holds
// four consecutive outputs of one activation row.
__device__ inline i32x4 mfma_16x16x64(i32x4 a, i32x4 b, i32x4 c) {
  return __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, c, 0, 0, 0);
}

// Waits until at most n of this wave's vector-memory loads (the LDS-DMA
// fragment copies) are outstanding.  gfx9 s_waitcnt: vmcnt in bits [3:0] and
// [15:14], expcnt [6:4] and lgkmcnt [11:8] left at their maxima.
template <int n>
__device__ inline void wait_vmcnt() {
  static_assert(n >= 0 && n < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((n & 15) | ((n >> 4) << 14) | (7 << 4) | (15 << 8));
}

// Workgroup barrier for the LDS ring.  The wave's own LDS reads complete
// first (lgkmcnt(0)), so a later LDS-DMA write into the slot they read cannot
// overtake them; unlike __syncthreads it does not drain outstanding loads.
__device__ inline void ring_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// N consecutive elements as one LDS or global access.
template <typename T, int N>
struct alignas(sizeof(T) * N) Pack {
  T v[N];
};

// The epilogue's operands of one workgroup tile in LDS: row scales and, per
// column, the weight scale and bias (or the integer requant's multiplier,
// shift and bias).  Copied by LDS-DMA before the first operand fragments, so
// they have landed with them and the epilogue waits for no memory access.
// Addresses past the operands are clamped to their last element.
template <int EPI, int BM, int BN>
struct TileScales {
  static constexpr bool kRows = EPI != kEpiI32 && EPI != kEpiRequant;
  static constexpr int kCols = EPI == kEpiI32       ? 0
                               : EPI == kEpiRequant ? 3
                                                    : (EPI == kEpiBf16Exact ? 1 : 2);
  static constexpr int kRowsPad = kRows ? (BM + 63) / 64 * 64 : 4;
  static constexpr int kColsPad = (BN + 63) / 64 * 64;
  alignas(16) float sx[kRowsPad];
  alignas(16) float col[kCols > 0 ? kCols : 1][kCols > 0 ? kColsPad : 4];

  // Called by every wavefront of the workgroup before its first ring load.
  template <int NW>
  __device__ inline void load(const GemmParams& p, int mb0, int nb0, int wave, int lane) {
    auto copy = [&](float* dst, const void* src, int64_t first, int64_t last) {
      int64_t i = first + lane;
      i = i < last ? i : last;
      __builtin_amdgcn_global_load_lds(static_cast<const float*>(src) + i, (lds_void*)dst, 4, 0, 0);
    };
    if constexpr (kRows) {
      for (int c = wave; c < kRowsPad / 64; c += NW)
        copy(sx + 64 * c, p.sx, static_cast<int64_t>(mb0) * 16 + 64 * c, p.M - 1);
    }
    if constexpr (kCols > 0) {
      // Wavefronts from the last on, so that few hold both kinds of copies.
      for (int c = NW - 1 - wave; c < kCols * kColsPad / 64; c += NW) {
        const int k = c / (kColsPad / 64);
        float* const dst = &col[0][0] + 64 * c;
        const void* src = p.sw;
        if constexpr (EPI == kEpiRequant) {
          src = k == 0 ? static_cast<const void*>(p.rq_mult)
                       : (k == 1 ? static_cast<const void*>(p.rq_shift) : p.rq_bias);
        } else if (k == 1) {
          src = p.bias;
        }
        if (src != nullptr) {
          copy(dst, src, static_cast<int64_t>(nb0) * 16 + 64 * (c % (kColsPad / 64)), p.N - 1);
        } else {
          // No bias: -0 changes no binary32 value it is added to, the zeros'
          // signs included.
          dst[lane] = EPI == kEpiRequant ? 0.0f : -0.0f;
        }
      }
    }
  }
};

// Stores a workgroup's output tile through the epilogue EPI: a WM x WN grid
// of wavefronts, each holding BR x BC 16x16 blocks of int32 accumulators.
// Register r of block (i, j) in lane l holds tile row 16(wm BR + i) + l%16
// and tile column 16(wn BC + j) + 4(l/16) + r: four consecutive columns of one
// row (the weights are the MFMA's first operand).  A lane therefore needs one
// row scale per i and four column scales per j (from LDS, TileScales), and
// packs its four (or with SiLU, whose gate/up pairs are adjacent columns, two)
// outputs itself.
//
// 32-bit outputs leave as 16-byte stores.  16- and 8-bit outputs pass through
// the operand ring's LDS at `stage` and leave as 16-byte chunks of whole tile
// rows, in passes of as many row blocks per wavefront as STAGE_BYTES hold.
// The LDS row stride is an odd multiple of 16 bytes: the 16 rows a wavefront
// writes at once then start in different banks.
//
// Bound by VALU work and stores: 12 thousand shader cycles for a 256 x 256
// binary16 tile of 8 wavefronts, 5.6 for 128 x 256, 25 with SiLU on 256 x 256.
// With a row per register instead (a row scale per accumulator, each loaded
// from memory behind a bounds check, and 2-byte LDS writes) these took 32,
// 16.6 and 47.  A 2048 x 22016 x 4096 SiLU product went from 191 to 177 us.
// ROOMY: the kernel has registers for residual chunks beside its accumulators.
template <int WM, int WN, int BR, int BC, int STAGE_BYTES, int EPI, typename TY, typename TH,
          bool ROOMY = false>
__device__ inline void store_tile(const GemmParams& p, i32x4 (&acc)[BR][BC], int wm, int wn,
                                  int mb0, int nb0, int lane, void* stage,
                                  const TileScales<EPI, 16 * WM * BR, 16 * WN * BC>& ts) {
  using Scales = TileScales<EPI, 16 * WM * BR, 16 * WN * BC>;
  constexpr int BN = 16 * WN * BC;
  constexpr bool kHalfCols = EPI == kEpiSilu || EPI == kEpiSiluQ8;  // one output per gate/up pair
  constexpr int OW = kHalfCols ? 2 : 4;                             // outputs per lane and block
  constexpr int BNO = kHalfCols ? BN / 2 : BN;
  constexpr int kOutBytes = static_cast<int>(sizeof(TY));
  constexpr bool kStage = kOutBytes < 4;
  constexpr int kRowBytes = BNO * kOutBytes;
  constexpr int kStride = (kRowBytes / 16 | 1) * 16;
  static_assert(kRowBytes % 16 == 0, "tile rows are whole 16-byte chunks");
  constexpr int kFit = STAGE_BYTES / (WM * 16 * kStride);
  constexpr int IPP = !kStage || kFit > BR ? BR : kFit;  // row blocks per wavefront and pass
  static_assert(IPP >= 1, "a pass holds at least one row block per wavefront");

  const int quad = lane >> 4;
  const int64_t m0 = static_cast<int64_t>(mb0) * 16;
  const int64_t n0 = static_cast<int64_t>(nb0) * 16;
  // This lane's row of block i and first column of block j, in the tile.
  auto row_of = [&](int i) { return 16 * (wm * BR + i) + (lane & 15); };
  auto col_of = [&](int j) { return 16 * (wn * BC + j) + 4 * quad; };

  [[maybe_unused]] float sx[BR];
  if constexpr (Scales::kRows) {
#pragma unroll
    for (int i = 0; i < BR; ++i) sx[i] = ts.sx[row_of(i)];
  }
  // Column operands k of block column j.
  auto cols = [&](int k, int j) __attribute__((always_inline)) {
    return *reinterpret_cast<const Pack<float, 4>*>(&ts.col[k][col_of(j)]);
  };
  struct Cols {
    Pack<float, 4> c[Scales::kCols > 0 ? Scales::kCols : 1];
  };
  auto cols_of = [&](int j) __attribute__((always_inline)) {
    Cols c;
    if constexpr (Scales::kCols > 0) {
#pragma unroll
      for (int k = 0; k < Scales::kCols; ++k) c.c[k] = cols(k, j);
    }
    return c;
  };

  // The lane's outputs of block (i, j).
  auto outputs = [&](int i, int j, const Cols& cj) __attribute__((always_inline)) {
    Pack<TY, OW> o;
    const i32x4 a = acc[i][j];
    if constexpr (kHalfCols) {
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        float gu[2];
#pragma unroll
        for (int c = 0; c < 2; ++c)
          gu[c] = to_f32(from_f32<TH>(
              dequant1b(a[2 * e + c], sx[i], cj.c[0].v[2 * e + c], true, cj.c[1].v[2 * e + c])));
        const TH h = from_f32<TH>(silu_mul<TH>(gu[0], gu[1]));
        if constexpr (EPI == kEpiSilu) {
          o.v[e] = h;
        } else {
          o.v[e] = static_cast<int8_t>(quant1(to_f32(h), p.out_scale));
        }
      }
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if constexpr (EPI == kEpiI32) {
          o.v[r] = a[r];
        } else if constexpr (EPI == kEpiDequant) {
          o.v[r] = from_f32<TY>(dequant1b(a[r], sx[i], cj.c[0].v[r], true, cj.c[1].v[r]));
        } else if constexpr (EPI == kEpiRequant) {
          o.v[r] = static_cast<int8_t>(requant1(
              a[r], __builtin_bit_cast(int32_t, cj.c[2].v[r]),
              __builtin_bit_cast(uint32_t, cj.c[0].v[r]), __builtin_bit_cast(int32_t, cj.c[1].v[r])));
        } else {
          static_assert(EPI == kEpiBf16Exact, "epilogue");
          o.v[r] = __builtin_bit_cast(
              TY, dequant_bf16_exact(a[r], f16_bits(sx[i]), f16_bits(cj.c[0].v[r])));
        }
      }
    }
    return o;
  };

  const bool vec_ok =
      ((reinterpret_cast<uintptr_t>(p.y) | static_cast<uintptr_t>(p.ldy * kOutBytes)) & 15) == 0;
  if constexpr (!kStage) {
#pragma unroll
    for (int j = 0; j < BC; ++j) {
      const Cols cj = cols_of(j);
#pragma unroll
      for (int i = 0; i < BR; ++i) {
        const int64_t m = m0 + row_of(i);
        const int64_t n = n0 + col_of(j);
        const Pack<TY, 4> o = outputs(i, j, cj);
        if (m < p.M && n < p.N) {
          TY* const dst = static_cast<TY*>(p.y) + m * p.ldy + n;
          if (vec_ok && n + 4 <= p.N) {
            *reinterpret_cast<Pack<TY, 4>*>(dst) = o;
          } else {
            for (int r = 0; r < 4; ++r)
              if (n + r < p.N) dst[r] = o.v[r];
          }
        }
      }
    }
  } else {
    char* const st = static_cast<char*>(stage);
    constexpr int EV = 16 / kOutBytes;    // outputs per 16-byte chunk
    constexpr int CPR = kRowBytes / 16;   // chunks per tile row
    constexpr int NT = WM * WN * 64;
    constexpr int RPP = NT / CPR;         // rows per sweep; threads past RPP * CPR idle
    static_assert(RPP >= 1, "a sweep covers at least one tile row");
    const int64_t n_out_total = kHalfCols ? p.N / 2 : p.N;
    const int64_t n0_out = kHalfCols ? n0 / 2 : n0;
    const int crow = static_cast<int>(threadIdx.x) / CPR;
    const int cchunk = static_cast<int>(threadIdx.x) % CPR;
    const int64_t nc = n0_out + cchunk * EV;  // this thread's first output column
    // Output row of tile-local row `row` of the pass over blocks i0 .. i0 + ni.
    auto out_row = [&](int row, int i0, int ni) {
      return m0 + 16 * (row / (16 * ni) * BR + i0) + row % (16 * ni);
    };
    // Residual add, y = dtype(dtype(dequant) + res); with ROOMY the pass's
    // residual chunks (up to 8 per thread) are requested before its arithmetic.
    // It spares O and down of a prefill layer a pass over their rows (three
    // trips through memory).
    constexpr bool kRes = EPI == kEpiDequant && kOutBytes == 2;
    constexpr int kSweeps = (WM * 16 * IPP + RPP - 1) / RPP;
    constexpr bool kEarly = kRes && ROOMY && kSweeps <= 8;
    const bool res_vec = kRes && p.res != nullptr && nc + EV <= n_out_total &&
                         ((reinterpret_cast<uintptr_t>(p.res) |
                           static_cast<uintptr_t>(p.ld_res * kOutBytes)) & 15) == 0;
    [[maybe_unused]] Pack<TY, EV> early[kEarly ? kSweeps : 1];
#pragma unroll
    for (int i0 = 0; i0 < BR; i0 += IPP) {
      const int ni = BR - i0 < IPP ? BR - i0 : IPP;  // compile-time after unrolling
      if constexpr (kEarly) {
        if (res_vec) {
#pragma unroll
          for (int t = 0; t < kSweeps; ++t) {
            const int row = t * RPP + crow;
            const int64_t m = out_row(row, i0, ni);
            const bool ok = crow < RPP && row < WM * 16 * ni && m < p.M;
            early[t] = *reinterpret_cast<const Pack<TY, EV>*>(
                static_cast<const TY*>(p.res) + (ok ? m : 0) * p.ld_res + nc);
          }
        }
      }
      ring_barrier();  // the ring's (or the last pass's) readers are done
#pragma unroll
      for (int j = 0; j < BC; ++j) {
        const Cols cj = cols_of(j);
#pragma unroll
        for (int i = i0; i < i0 + ni; ++i) {
          const Pack<TY, OW> o = outputs(i, j, cj);
          const int row = 16 * (wm * ni + i - i0) + (lane & 15);
          const int col = kHalfCols ? col_of(j) / 2 : col_of(j);
          *reinterpret_cast<Pack<TY, OW>*>(st + row * kStride + col * kOutBytes) = o;
          if constexpr (EPI == kEpiSilu) {
            if (p.absmax_parts != nullptr) {
              // The row's 8 outputs of packed block nb lie in the four lanes
              // l%16 + 16q.
              float v = fmaxf(fabsf(to_f32(o.v[0])), fabsf(to_f32(o.v[1])));
              v = fmaxf(v, __shfl_xor(v, 16));
              v = fmaxf(v, __shfl_xor(v, 32));
              const int64_t m = m0 + row_of(i);
              const int64_t nb = static_cast<int64_t>(nb0) + wn * BC + j;
              if (quad == 0 && m < p.M && nb < p.NB) p.absmax_parts[m * p.NB + nb] = v;
            }
          }
        }
      }
      ring_barrier();
      const int rows = WM * 16 * ni;
#pragma unroll
      for (int base = 0; base < rows; base += RPP) {
        const int row = base + crow;
        const int64_t m = out_row(row, i0, ni);
        const int64_t n = nc;
        if (crow < RPP && row < rows && m < p.M && n < n_out_total) {
          TY* const dst = static_cast<TY*>(p.y) + m * p.ldy + n;
          Pack<TY, EV>& out = *reinterpret_cast<Pack<TY, EV>*>(st + row * kStride + cchunk * 16);
          if constexpr (kRes) {
            if (p.res != nullptr) {
              const TY* const r = static_cast<const TY*>(p.res) + m * p.ld_res + n;
              Pack<TY, EV> o = out;
              if (res_vec) {
                Pack<TY, EV> a;
                if constexpr (kEarly) {
                  a = early[base / RPP];
                } else {
                  a = *reinterpret_cast<const Pack<TY, EV>*>(r);
                }
#pragma unroll
                for (int e = 0; e < EV; ++e) o.v[e] = add_rounded(o.v[e], a.v[e]);
              } else {
                for (int e = 0; e < EV; ++e)
                  if (n + e < n_out_total) o.v[e] = add_rounded(o.v[e], r[e]);
              }
              out = o;
            }
          }
          const TY* const src = out.v;
          if (vec_ok && n + EV <= n_out_total) {
            *reinterpret_cast<i32x4*>(dst) = *reinterpret_cast<const i32x4*>(src);
          } else {
            for (int e = 0; e < EV; ++e)
              if (n + e < n_out_total) dst[e] = src[e];
          }
        }
      }
    }
  }
}

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

  store_tile<WM, WN, BR, BC, kRing, EPI, TY, TH>(p, acc, wm, wn, mb0, nb0, lane, smem, scales);
}

// Workgroup barrier with the wave's LDS reads complete, through the builtin
// s_waitcnt, so the compiler's own wait insertion knows they are (an inline
// asm wait is opaque to it, and it would then wait for the newer reads of
// the next k-block too).  The empty asm statements keep LDS accesses on
// their side of the barrier.
__device__ inline void ring_barrier_tracked() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0); vmcnt and expcnt at their maxima
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// f(integral_constant<int, I>) for I = 0 .. N-1, unrolled at compile time.
template <typename F, int... I>
__device__ inline void static_for_impl(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ inline void static_for(F&& f) {
  static_for_impl(f, std::make_integer_sequence<int, N>{});
}

__device__ inline __amdgpu_buffer_rsrc_t dma_rsrc(const void* base) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, 0x7fffffff, 0x00020000);
}

// 16 bytes per lane from the buffer at voffset + soffset (wave-uniform) into
// LDS at lds + 16 * lane (buffer_load_dwordx4 ... lds).
__device__ inline void dma16(__amdgpu_buffer_rsrc_t r, void* lds, uint32_t voffset,
                             uint32_t soffset = 0) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void*)lds, 16, voffset, soffset, 0, 0);
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

// Pipelined GEMM: WM x WN = 8 wavefronts, one workgroup per CU, each wavefront
// BR x BC 16x16 blocks (tile 16 WM BR x 16 WN BC), an S-slot LDS ring of single
// k-blocks (64 K) and one barrier per k-block.
//   * Each wavefront keeps the fragments of its shorter side of a k-block in
//     registers (`held`, double-buffered) and passes the longer side's through
//     R registers (`strm`), every fragment read from LDS about a k-block before
//     its MFMAs, also across the barriers: no MFMA waits for an LDS read
//     issued behind a barrier.  (gemm_kernel reads a k-block's fragments after
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
  store_tile<WM, WN, BR, BC, kRing, EPI, TY, TH, true>(p, acc, wm, wn, mb0, nb0, lane, smem, scales);
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

// Tile configurations, chosen by tile count (measured on MI355X, random data,
// cold weights, LLaMA-7B projections at M = 256..2048).  A launch is fastest
// when its tiles fill one round of workgroup slots (2 per CU) as closely as
// possible, and when several rounds are needed, with the widest tile:
//   * first the one-workgroup-per-CU tiles taken when one round of them fills
//     the CUs (gemm_tile_choice): 112x256 weights-direct (gemm_wd_kernel,
//     packed QKV at M = 449..560), then 112x96 and 128x96 (O and down at
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
//     64x64, 3-stage ring): 128x224 takes gate/up at M = 560 in 495 tiles,
//     8% faster than 430 tiles of 128x256;
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
  switch (gemm_pipe_choice(p.MB, p.NB, p.KB, cu_count())) {
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
    case kPipe128x128:
      return launch_pipe<2, 4, 4, 2, 9, 4, EPI, TY, TH>(p, st);
    default:
      break;
  }
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

}  // namespace

// The pipelined tile whose rounds over the CUs take least, by the time of one
// of its k-steps with all CUs busy (nanoseconds, measured at K = 4096 and
// 11008: the wider the tile, the less per product).  So packed QKV takes
// 192x160 at 560 rows (231 tiles, 33.4 us; 35.2 on the weights-direct tile)
// and 256x192 at 2048 (two full rounds, 91 us against 104 for 128x256), gate/up
// 192x288 at 560 (52.7 against 63.9 for 128x224) and 256x352 at 1024 and 2048
// (82 against 105, 153 against 179), O and down 128x128 at 560 (18.6 / 41.5
// against 20.4 / 49 for 112x96) and 1024 (51 against 57 for the ring of 16
// wavefronts) and 256x128 at 2048 (34 / 77 against 38 / 99).
// Taken where the tiles fill three fifths of the CUs; below that the smaller
// ring tiles cover more of them, and below 16 k-blocks filling the ring (up to
// 8) would be a large part of the work.
int gemm_pipe_choice(int64_t MB, int64_t NB, int64_t KB, int64_t cus) {
  struct Tile {
    GemmPipe id;
    int mb, nb, step_ns;
  };
  static constexpr Tile kTiles[] = {
      {kPipe256x352, 16, 22, 880}, {kPipe256x256, 16, 16, 670}, {kPipe192x288, 12, 18, 600},
      {kPipe256x192, 16, 12, 560}, {kPipe256x128, 16, 8, 435},  {kPipe192x160, 12, 10, 400},
      {kPipe128x128, 8, 8, 275},
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

int gemm_tile_choice(int64_t MB, int64_t NB, int64_t cus) {
  // The 112 x 256 weights-direct tile when one round of it (one workgroup per
  // CU) fills at least 85% of the CUs with at least 85% of the tile rows in
  // use (the packed QKV at M = 449..560).  A 144 x 64 weights-direct tile for
  // O and down at the same M measured slower than the 128 x 128 deep ring
  // (27.2 vs 23.5 us and 59.6 vs 51.3 us with the fp16 epilogue), so those
  // keep the LDS-ring tiles.
  if (MB > 4) {
    const int64_t tm = ceil_div(MB, 7);
    const int64_t tiles = tm * ceil_div(NB, 16);
    if (tiles <= cus && 100 * tiles >= 85 * cus && 100 * MB >= 85 * tm * 7) return kGemmWd7x2;
  }
  // Narrow tiles (96 columns) when one round of them, at least four tile rows
  // deep, fills at least 80% of the CUs with at least 85% of the tile rows in
  // use: O and down (N = 4096) at M = 465..640, where 128x128 tiles leave 96
  // of 256 CUs idle.  Measured at M = 560 (fp16 epilogue): 112x96 takes O in
  // 20.8 against 23.6 us and down in 48.1 against 58.5 us; at M = 567 (36
  // row blocks) 128x96 takes O in 21.6 against 23.8 us.  The 14 wavefronts of
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
  GemmParams p;
  p.a = reinterpret_cast<const i32x4*>(op.a);
  p.sx = op.sx;
  p.w = reinterpret_cast<const i32x4*>(op.w);
  p.sw = op.sw;
  p.bias = op.bias;
  p.y = op.y;
  p.ldy = op.ldy;
  p.out_scale = op.out_scale;
  p.rq_mult = op.rq_mult;
  p.rq_shift = op.rq_shift;
  p.rq_bias = op.rq_bias;
  p.absmax_parts = op.absmax_parts;
  p.res = op.res;
  p.ld_res = op.ld_res;
  p.M = static_cast<int>(op.M);
  p.N = static_cast<int>(op.N);
  p.MB = static_cast<int>(ceil_div(op.M, kTileRows));
  p.NB = static_cast<int>(ceil_div(op.N, kTileRows));
  p.KB = static_cast<int>(ceil_div(op.K, kTileK));
  p.tiles_m = p.tiles = p.per_xcd = 0;
  if (p.MB == 0 || p.NB == 0) return hipSuccess;
  switch (op.epi) {
    case kEpiI32:
      return launch_t<kEpiI32, int32_t, float>(p, st);
    case kEpiDequant:
      if (op.y_dtype == kF16) return launch_t<kEpiDequant, __half, float>(p, st);
      if (op.y_dtype == kBF16) return launch_t<kEpiDequant, __hip_bfloat16, float>(p, st);
      if (op.y_dtype == kF32) return launch_t<kEpiDequant, float, float>(p, st);
      return hipErrorInvalidValue;
    case kEpiSilu:
      if (op.y_dtype == kF16) return launch_t<kEpiSilu, __half, __half>(p, st);
      if (op.y_dtype == kBF16) return launch_t<kEpiSilu, __hip_bfloat16, __hip_bfloat16>(p, st);
      return hipErrorInvalidValue;
    case kEpiSiluQ8:
      if (op.h_dtype == kF16) return launch_t<kEpiSiluQ8, int8_t, __half>(p, st);
      if (op.h_dtype == kBF16) return launch_t<kEpiSiluQ8, int8_t, __hip_bfloat16>(p, st);
      return hipErrorInvalidValue;
    case kEpiRequant:
      return launch_t<kEpiRequant, int8_t, float>(p, st);
    case kEpiBf16Exact:
      return launch_t<kEpiBf16Exact, __hip_bfloat16, float>(p, st);
    default:
      return hipErrorInvalidValue;
  }
}

}  // namespace w8a8
