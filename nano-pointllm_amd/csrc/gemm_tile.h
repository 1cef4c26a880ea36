// The int8 GEMM kernels' common parts (gemm.hip, gemm_pipe.hip): parameters, waits
// and LDS-DMA copies, the epilogue's operands in LDS and the epilogue itself.
#pragma once

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
// The outputs pass through the operand ring's LDS at `stage` and leave as
// 16-byte chunks of whole tile rows, in passes of as many row blocks per
// wavefront as STAGE_BYTES hold.  The LDS row stride is an odd multiple of 16
// bytes: the 16 rows a wavefront writes at once then start in different banks.
// 32-bit outputs too: stored from the registers, 64 bytes (half a line) of 16
// rows at a time, int32 calls of 2048 x 22016 x 768 took 103 us, 1024 x 12288 x
// 512 24.5 and 560 x 12288 x 4096 38.9; through LDS 75.5, 16.9 and 31.6.
//
// Bound by VALU work and stores: 12 thousand shader cycles for a 256 x 256
// binary16 tile of 8 wavefronts, 5.6 for 128 x 256, 25 with SiLU on 256 x 256.
// With a row per register instead (a row scale per accumulator, each loaded
// from memory behind a bounds check, and 2-byte LDS writes) these took 32,
// 16.6 and 47.  A 2048 x 22016 x 4096 SiLU product went from 191 to 177 us.
// ROOMY: the kernel has registers for residual chunks beside its accumulators.
// HOIST: and for the integer requant's twelve column operands of a block column,
// read once for all its rows (1024 x 22016 x 768 40.5 us, 42.7 where they are read
// for each block; on the 128 x 128 ring tile of 64 registers they spill, 2048 x
// 4096 x 768 29 us against 21).
template <int WM, int WN, int BR, int BC, int STAGE_BYTES, int EPI, typename TY, typename TH,
          bool ROOMY = false, bool HOIST = true>
__device__ inline void store_tile(const GemmParams& p, i32x4 (&acc)[BR][BC], int wm, int wn,
                                  int mb0, int nb0, int lane, void* stage,
                                  const TileScales<EPI, 16 * WM * BR, 16 * WN * BC>& ts) {
  using Scales = TileScales<EPI, 16 * WM * BR, 16 * WN * BC>;
  constexpr int BN = 16 * WN * BC;
  constexpr bool kHalfCols = EPI == kEpiSilu || EPI == kEpiSiluQ8;  // one output per gate/up pair
  constexpr int OW = kHalfCols ? 2 : 4;                             // outputs per lane and block
  constexpr int BNO = kHalfCols ? BN / 2 : BN;
  constexpr int kOutBytes = static_cast<int>(sizeof(TY));
  constexpr int kRowBytes = BNO * kOutBytes;
  constexpr int kStride = (kRowBytes / 16 | 1) * 16;
  static_assert(kRowBytes % 16 == 0, "tile rows are whole 16-byte chunks");
  constexpr int kFit = STAGE_BYTES / (WM * 16 * kStride);
  constexpr int IPP = kFit > BR ? BR : kFit;  // row blocks per wavefront and pass
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
  constexpr bool kHoist = EPI != kEpiRequant || HOIST;
  struct Cols {
    Pack<float, 4> c[Scales::kCols > 0 ? Scales::kCols : 1];
  };
  auto cols_of = [&](int j) __attribute__((always_inline)) {
    Cols c;
    if constexpr (Scales::kCols > 0 && kHoist) {
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
          const auto col = [&](int k) {
            return kHoist ? cj.c[k].v[r] : ts.col[k][col_of(j) + r];
          };
          o.v[r] = static_cast<int8_t>(
              requant1(a[r], __builtin_bit_cast(int32_t, col(2)), __builtin_bit_cast(uint32_t, col(0)),
                       __builtin_bit_cast(int32_t, col(1))));
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
      if constexpr (EPI == kEpiRequant) __builtin_amdgcn_sched_barrier(0);
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

inline GemmParams gemm_params(const LinearOperands& op) {
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
  return p;
}

// L::launch<EPI, TY, TH>(p, extra..., st) for the call's epilogue and types.
template <typename L, typename... Extra>
hipError_t gemm_dispatch(const LinearOperands& op, const GemmParams& p, hipStream_t st,
                         Extra... extra) {
  switch (op.epi) {
    case kEpiI32:
      return L::template launch<kEpiI32, int32_t, float>(p, st, extra...);
    case kEpiDequant:
      if (op.y_dtype == kF16) return L::template launch<kEpiDequant, __half, float>(p, st, extra...);
      if (op.y_dtype == kBF16) return L::template launch<kEpiDequant, __hip_bfloat16, float>(p, st, extra...);
      if (op.y_dtype == kF32) return L::template launch<kEpiDequant, float, float>(p, st, extra...);
      return hipErrorInvalidValue;
    case kEpiSilu:
      if (op.y_dtype == kF16) return L::template launch<kEpiSilu, __half, __half>(p, st, extra...);
      if (op.y_dtype == kBF16) return L::template launch<kEpiSilu, __hip_bfloat16, __hip_bfloat16>(p, st, extra...);
      return hipErrorInvalidValue;
    case kEpiSiluQ8:
      if (op.h_dtype == kF16) return L::template launch<kEpiSiluQ8, int8_t, __half>(p, st, extra...);
      if (op.h_dtype == kBF16) return L::template launch<kEpiSiluQ8, int8_t, __hip_bfloat16>(p, st, extra...);
      return hipErrorInvalidValue;
    case kEpiRequant:
      return L::template launch<kEpiRequant, int8_t, float>(p, st, extra...);
    case kEpiBf16Exact:
      return L::template launch<kEpiBf16Exact, __hip_bfloat16, float>(p, st, extra...);
    default:
      return hipErrorInvalidValue;
  }
}

}  // namespace

}  // namespace w8a8
