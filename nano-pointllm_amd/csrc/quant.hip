// Per-row symmetric int8 quantization and 16x64 tile packing.
//
// quant_rows_kernel restates, per row r of a [rows, K] matrix:
//   scale_from_absmax  (nanopointllm/compression/w8a8.py:46-50)
//   quantize_symmetric (nanopointllm/compression/w8a8.py:33-43)
// It serves both per-token activation quantization
// (dynamic_per_token_activation_qdq, w8a8.py:106-115) and per-output weight
// quantization (per_output_weight_qdq, w8a8.py:53-62): both are "one scale per
// row of a row-major matrix".
#include "w8a8_internal.h"

#include <type_traits>

namespace w8a8 {

namespace {

constexpr int kQuantThreads = 256;
// Rows up to kQuantThreads * 8 * REG elements are held in registers between
// the absmax pass and the quantize pass (one global read); REG (1, 2, 4 or
// 8 chunks of 8 elements per thread) is the smallest that covers the row.
constexpr int kRegChunksMax = 8;

// Quantizes one value with the row scale s.  The division-free form needs a
// 16-bit input and a binary16-representable scale (always true for dynamic
// scales; checked per row for caller scales); otherwise divide.
template <typename TX>
__device__ inline int32_t quant_elem(float x, float s, float r, bool fast) {
  if constexpr (sizeof(TX) == 2) {
    if (fast) return quant1_h(x, s, r);
  }
  return quant1(x, s);
}

// Writes 8 quantized values of row `row` starting at column k0.
template <bool PACKED>
__device__ inline void store8(int8_t* __restrict__ q, int64_t row, int64_t k0, int64_t ldq,
                              int64_t ncols_out, int vec_out, int64_t KB, const int32_t (&qi)[8]) {
  u32x2 word = {pack4_i8(qi[0], qi[1], qi[2], qi[3]), pack4_i8(qi[4], qi[5], qi[6], qi[7])};
  if constexpr (PACKED) {
    *reinterpret_cast<u32x2*>(q + packed_offset(row, k0, KB)) = word;
  } else {
    // Row-major: columns K..ncols_out-1 are written as zeros.
    int8_t* dst = q + row * ldq + k0;
    const int nw = static_cast<int>(ncols_out - k0 < 8 ? ncols_out - k0 : 8);
    if (vec_out && nw == 8) {
      *reinterpret_cast<u32x2*>(dst) = word;
    } else {
      for (int j = 0; j < nw; ++j) dst[j] = static_cast<int8_t>(qi[j]);
    }
  }
}

// Loads the REG 8-element chunks (tid + c * NT) of a row whose elements are
// 16-byte aligned, K % 8 == 0: range-checked raw buffer loads, all issued
// before any is used (zeros past K, and for a null row).  A load under a
// branch per chunk would wait for each before issuing the next.
template <typename TX, int REG, int NT>
__device__ inline void load_row_chunks(const TX* row, int64_t K, int tid, float (&v)[REG][8]) {
  constexpr int kWords = sizeof(TX) == 4 ? 2 : 1;
  const __amdgpu_buffer_rsrc_t d = raw_rsrc(row, static_cast<int>(K * sizeof(TX)));
  u32x4 raw[REG][kWords];
#pragma unroll
  for (int c = 0; c < REG; ++c) {
    const int off = (tid + c * NT) * 8 * static_cast<int>(sizeof(TX));
#pragma unroll
    for (int w = 0; w < kWords; ++w) raw[c][w] = load16(d, off + 16 * w);
  }
#pragma unroll
  for (int c = 0; c < REG; ++c) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if constexpr (sizeof(TX) == 4) {
        v[c][j] = __uint_as_float(raw[c][j >> 2][j & 3]);
      } else {
        const uint32_t w = raw[c][0][j >> 1];
        v[c][j] = bits_to_f32<TX>(j & 1 ? w >> 16 : w & 0xffffu);
      }
    }
  }
}

// One workgroup per row.  The row (8 elements per thread-chunk) is read once
// into registers when it fits (REG), reduced to |x|max for a dynamic scale
// (or the caller's scale is read), then quantized and written either as a
// row-major int8 row or as the row's slots of the packed tiles.  For packed
// output the grid covers ceil(rows/16)*16 rows and every row writes all
// ceil(K/64)*64 columns, so tile padding is zero-filled.
template <typename TX, bool PACKED, bool DYNAMIC, int REG, int NT>
__global__ __launch_bounds__(NT) void quant_rows_kernel(
    const TX* __restrict__ x, int64_t ldx, int64_t rows, int64_t K, int vec_in,
    const float* __restrict__ scale_in, int64_t scale_stride, int8_t* __restrict__ q,
    int64_t ldq, int64_t ncols_out, int vec_out, int64_t KB, float* __restrict__ scales_out) {
  __shared__ float red[NT / 64];
  const int64_t row = PACKED ? packed_row_of(blockIdx.x, gridDim.x) : blockIdx.x;
  const int tid = threadIdx.x;
  const bool live = row < rows;
  const TX* xr = x + (live ? row : 0) * ldx;
  const int64_t nchunk_in = (K + 7) / 8;
  const int64_t nchunk_out = PACKED ? KB * 8 : (ncols_out + 7) / 8;

  float v[REG > 0 ? REG : 1][8];
  if constexpr (REG > 0) {
    if (vec_in) {
      load_row_chunks<TX, REG, NT>(live ? xr : nullptr, K, tid, v);
    } else {
#pragma unroll
      for (int c = 0; c < REG; ++c) {
        const int64_t k0 = (tid + static_cast<int64_t>(c) * NT) * 8;
        const int64_t rem = K - k0;
        if (live && rem > 0) {
          load8(xr + k0, v[c], false, static_cast<int>(rem < 8 ? rem : 8));
        } else {
#pragma unroll
          for (int j = 0; j < 8; ++j) v[c][j] = 0.0f;
        }
      }
    }
  }

  float s = 1.0f;
  if constexpr (DYNAMIC) {
    float amax = 0.0f;
    if constexpr (REG > 0) {
#pragma unroll
      for (int c = 0; c < REG; ++c)
#pragma unroll
        for (int j = 0; j < 8; ++j) amax = fmaxf(amax, fabsf(v[c][j]));
    } else if (live) {
      for (int64_t c = tid; c < nchunk_in; c += NT) {
        float t[8];
        const int64_t k0 = c * 8;
        load8(xr + k0, t, vec_in != 0, static_cast<int>(K - k0 < 8 ? K - k0 : 8));
#pragma unroll
        for (int j = 0; j < 8; ++j) amax = fmaxf(amax, fabsf(t[j]));
      }
    }
    amax = wave_max_abs(amax);
    if ((tid & 63) == 0) red[tid >> 6] = amax;
    __syncthreads();
    amax = red[0];
#pragma unroll
    for (int w = 1; w < NT / 64; ++w) amax = fmaxf(amax, red[w]);
    s = scale_from_absmax(amax);
  } else {
    if (live) s = scale_in[row * scale_stride];
  }
  const float r = 1.0f / s;
  const bool fast = DYNAMIC || __half2float(__float2half_rn(s)) == s;
  if (live && tid == 0 && scales_out != nullptr) scales_out[row] = s;

  if constexpr (REG > 0) {
#pragma unroll
    for (int c = 0; c < REG; ++c) {
      const int64_t chunk = tid + static_cast<int64_t>(c) * NT;
      if (chunk < nchunk_out) {
        const int64_t k0 = chunk * 8;
        int32_t qi[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) qi[j] = quant_elem<TX>(v[c][j], s, r, fast);
        store8<PACKED>(q, row, k0, ldq, ncols_out, vec_out, KB, qi);
      }
    }
  } else {
    for (int64_t c = tid; c < nchunk_out; c += NT) {
      const int64_t k0 = c * 8;
      const int64_t rem = K - k0;
      const int valid = live ? static_cast<int>(rem <= 0 ? 0 : (rem < 8 ? rem : 8)) : 0;
      float t[8];
      if (valid > 0) {
        load8(xr + k0, t, vec_in != 0, valid);
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) t[j] = 0.0f;
      }
      int32_t qi[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) qi[j] = (j < valid) ? quant_elem<TX>(t[j], s, r, fast) : 0;
      store8<PACKED>(q, row, k0, ldq, ncols_out, vec_out, KB, qi);
    }
  }
}

// Second phase of the two-phase per-token requantization (one workgroup per
// row): the producing epilogue left the row's |x|max split over nparts
// partial maxima, parts[row * nparts + i]; their max gives the binary16
// scale (scale_from_absmax, w8a8.py:46-50) without a reduction over x, and
// the row is quantized (quantize_symmetric, w8a8.py:33-43) into row-major q.
// The row's chunks (REG per thread, or a second pass when REG is 0) are
// requested before the partials, so both reads are in flight together.
template <typename TX, int REG, int NT>
__global__ __launch_bounds__(NT) void quant_rows_parts_kernel(
    const TX* __restrict__ x, int64_t ldx, int64_t K, int vec_in,
    const float* __restrict__ parts, int64_t nparts, int8_t* __restrict__ q, int64_t ldq,
    int vec_out, float* __restrict__ scales_out) {
  __shared__ float red[NT / 64];
  const int64_t row = blockIdx.x;
  const int tid = threadIdx.x;
  const TX* xr = x + row * ldx;
  const int64_t nchunk = (K + 7) / 8;
  float v[REG > 0 ? REG : 1][8];
  if constexpr (REG > 0) {
    if (vec_in) {
      load_row_chunks<TX, REG, NT>(xr, K, tid, v);
    } else {
#pragma unroll
      for (int c = 0; c < REG; ++c) {
        const int64_t k0 = (tid + static_cast<int64_t>(c) * NT) * 8;
        const int64_t rem = K - k0;
        if (rem > 0) {
          load8(xr + k0, v[c], false, static_cast<int>(rem < 8 ? rem : 8));
        } else {
#pragma unroll
          for (int j = 0; j < 8; ++j) v[c][j] = 0.0f;
        }
      }
    }
  }
  const float* pr = parts + row * nparts;
  float amax = 0.0f;
  for (int64_t i = tid; i < nparts; i += NT) amax = fmaxf(amax, pr[i]);
  amax = wave_max_abs(amax);
  if ((tid & 63) == 0) red[tid >> 6] = amax;
  __syncthreads();
  amax = red[0];
#pragma unroll
  for (int w = 1; w < NT / 64; ++w) amax = fmaxf(amax, red[w]);
  const float s = scale_from_absmax(amax);
  const float r = 1.0f / s;
  if (tid == 0) scales_out[row] = s;
  if constexpr (REG > 0) {
#pragma unroll
    for (int c = 0; c < REG; ++c) {
      const int64_t chunk = tid + static_cast<int64_t>(c) * NT;
      if (chunk < nchunk) {
        const int64_t k0 = chunk * 8;
        const int valid = static_cast<int>(K - k0 < 8 ? K - k0 : 8);
        int32_t qi[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) qi[j] = (j < valid) ? quant_elem<TX>(v[c][j], s, r, true) : 0;
        store8<false>(q, row, k0, ldq, K, vec_out, 0, qi);
      }
    }
  } else {
    for (int64_t c = tid; c < nchunk; c += NT) {
      const int64_t k0 = c * 8;
      const int valid = static_cast<int>(K - k0 < 8 ? K - k0 : 8);
      float t[8];
      load8(xr + k0, t, vec_in != 0, valid);
      int32_t qi[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) qi[j] = (j < valid) ? quant_elem<TX>(t[j], s, r, true) : 0;
      store8<false>(q, row, k0, ldq, K, vec_out, 0, qi);
    }
  }
}

// |x|max over the LPG lanes of a power-of-two group (every lane active; all
// its lanes end with the result).  Within a row of 16 the partners come from
// DPP quad permutations and mirrors (a mirror pairs each lane with one of the
// other half, which holds that half's maximum after the levels below), past
// it from the permlane swaps of wave_butterfly.
template <int LPG>
__device__ inline float group_max_abs(float v) {
  constexpr int kQuadXor1 = 0xb1, kQuadXor2 = 0x4e, kRowHalfMirror = 0x141, kRowMirror = 0x140;
  auto dpp = [&](auto ctrl) {
    const uint32_t u = __builtin_amdgcn_update_dpp(0u, __float_as_uint(v), decltype(ctrl)::value,
                                                   0xf, 0xf, false);
    v = fmaxf(v, __uint_as_float(u));
  };
  if constexpr (LPG >= 2) dpp(std::integral_constant<int, kQuadXor1>{});
  if constexpr (LPG >= 4) dpp(std::integral_constant<int, kQuadXor2>{});
  if constexpr (LPG >= 8) dpp(std::integral_constant<int, kRowHalfMirror>{});
  if constexpr (LPG >= 16) dpp(std::integral_constant<int, kRowMirror>{});
  if constexpr (LPG >= 32) {
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  }
  if constexpr (LPG >= 64) {
    const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  }
  return v;
}

// Quantize-dequantize outputs of one 8-column chunk: int8 values (q nullable)
// and q * s rounded to the input type, the columns below K.
struct QdqOut {
  int8_t* q;
  int64_t ldq;
  void* deq;
  int64_t ldd;
  int vec_q, vec_d;
};

template <typename TX>
__device__ inline void qdq_store8(const QdqOut& o, int64_t row, int64_t k0, int valid,
                                  const float (&v)[8], float s, float r) {
  int32_t qi[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) qi[j] = quant_elem<TX>(v[j], s, r, true);
  if (o.q != nullptr) {
    int8_t* dst = o.q + row * o.ldq + k0;
    if (o.vec_q && valid >= 8) {
      *reinterpret_cast<u32x2*>(dst) =
          u32x2{pack4_i8(qi[0], qi[1], qi[2], qi[3]), pack4_i8(qi[4], qi[5], qi[6], qi[7])};
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (j < valid) dst[j] = static_cast<int8_t>(qi[j]);
    }
  }
  float d[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) d[j] = __fmul_rn(static_cast<float>(qi[j]), s);
  TX* dst = static_cast<TX*>(o.deq) + row * o.ldd + k0;
  if (o.vec_d && valid >= 8) {
    if constexpr (sizeof(TX) == 2) {
      *reinterpret_cast<u32x4*>(dst) = u32x4{pack2_bits<TX>(d[0], d[1]), pack2_bits<TX>(d[2], d[3]),
                                             pack2_bits<TX>(d[4], d[5]), pack2_bits<TX>(d[6], d[7])};
    } else {
#pragma unroll
      for (int h = 0; h < 2; ++h)
        reinterpret_cast<u32x4*>(dst)[h] =
            u32x4{__float_as_uint(d[4 * h]), __float_as_uint(d[4 * h + 1]),
                  __float_as_uint(d[4 * h + 2]), __float_as_uint(d[4 * h + 3])};
    }
  } else {
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (j < valid) dst[j] = from_f32<TX>(d[j]);
  }
}

// Quantize-dequantize with one scale per row and group of 8 LPG columns
// (groupwise_weight_qdq, w8a8.py:65-91): LPG adjacent lanes hold a group, one
// 8-column chunk each, so a group's scale takes log2(LPG) lane exchanges and
// the matrix is read and written once.  Bound: HBM (2 bytes in, 3 out per
// 16-bit weight): 4096 x 11008 bfloat16 in groups of 128 takes 44.5 us, 5.1
// TB/s (a large copy reaches 4.8, read and written); a workgroup per group (quantization
// alone 230 us) and torch's elementwise passes behind it took 602.
template <typename TX, int LPG>
__global__ __launch_bounds__(kQuantThreads) void qdq_groups_kernel(
    const TX* __restrict__ x, int64_t ldx, int64_t K, int vec_in, int groups, int blocks_per_row,
    QdqOut out, float* __restrict__ scales_out) {
  const int64_t row = blockIdx.x / blocks_per_row;
  const int chunk =
      static_cast<int>(blockIdx.x % blocks_per_row) * kQuantThreads + static_cast<int>(threadIdx.x);
  const int64_t k0 = static_cast<int64_t>(chunk) * 8;
  const int valid = static_cast<int>(K - k0 <= 0 ? 0 : (K - k0 < 8 ? K - k0 : 8));
  float v[8];
  load8(x + row * ldx + k0, v, vec_in != 0, valid);
  float amax = 0.0f;
#pragma unroll
  for (int j = 0; j < 8; ++j) amax = fmaxf(amax, fabsf(v[j]));
  amax = group_max_abs<LPG>(amax);
  const float s = scale_from_absmax(amax);
  const float r = 1.0f / s;
  if (valid > 0) {
    if (chunk % LPG == 0) scales_out[row * groups + chunk / LPG] = s;
    qdq_store8<TX>(out, row, k0, valid, v, s, r);
  }
}

// Quantize-dequantize with one workgroup per (row, group): whole rows
// (dynamic_per_token_activation_qdq, per_output_weight_qdq) and the group
// sizes the kernel above does not take.  The group stays in REG chunks per
// thread between the absmax and the outputs (REG 0: it is read twice).
// Latency-bound at activation sizes: 560 x 4096 bfloat16 as a call takes 15.2
// us, mostly the host's, against 31.2 for quant_rows_kernel (4.8 us) and three
// elementwise passes (20 us).  Few long rows are bound by what one CU keeps in
// flight, hence the four chunks at a time: one row of 2 million bfloat16 takes
// 290 us (a chunk at a time on 512 threads 599, the separate kernels 366).
template <typename TX, int REG, int NT>
__global__ __launch_bounds__(NT) void qdq_rows_kernel(const TX* __restrict__ x, int64_t ldx,
                                                      int64_t K, int64_t group, int vec_in,
                                                      int groups, QdqOut out,
                                                      float* __restrict__ scales_out) {
  __shared__ float red[NT / 64];
  const int64_t row = blockIdx.x / groups;
  const int64_t c0 = static_cast<int64_t>(blockIdx.x % groups) * group;
  const int64_t n = K - c0 < group ? K - c0 : group;  // columns of this group
  const int tid = threadIdx.x;
  const TX* xr = x + row * ldx + c0;
  out.q = out.q != nullptr ? out.q + c0 : nullptr;
  out.deq = static_cast<TX*>(out.deq) + c0;
  const int64_t nchunk = (n + 7) / 8;
  auto valid_of = [&](int64_t k0) { return static_cast<int>(n - k0 <= 0 ? 0 : (n - k0 < 8 ? n - k0 : 8)); };
  // REG 0: f(k0, valid columns, values) for each of the thread's chunks, four
  // whole ones at a time so that their loads are in flight together.
  [[maybe_unused]] auto each_chunk = [&](auto&& f) __attribute__((always_inline)) {
    int64_t c = tid;
    auto whole = [&](auto vec) __attribute__((always_inline)) {
      for (; c + 3 * NT < n / 8; c += 4 * NT) {
        float t[4][8];
#pragma unroll
        for (int u = 0; u < 4; ++u) load8(xr + (c + u * NT) * 8, t[u], decltype(vec)::value, 8);
#pragma unroll
        for (int u = 0; u < 4; ++u) f((c + u * NT) * 8, 8, t[u]);
      }
    };
    if (vec_in) whole(std::true_type{}); else whole(std::false_type{});
    for (; c < nchunk; c += NT) {
      const int valid = valid_of(c * 8);
      float t[8];
      load8(xr + c * 8, t, vec_in != 0, valid);
      f(c * 8, valid, t);
    }
  };
  float v[REG > 0 ? REG : 1][8];
  float amax = 0.0f;
  if constexpr (REG > 0) {
    if (vec_in) {
      load_row_chunks<TX, REG, NT>(xr, n, tid, v);
    } else {
#pragma unroll
      for (int c = 0; c < REG; ++c) {
        const int64_t k0 = (tid + static_cast<int64_t>(c) * NT) * 8;
        load8(xr + k0, v[c], false, valid_of(k0));
      }
    }
#pragma unroll
    for (int c = 0; c < REG; ++c)
#pragma unroll
      for (int j = 0; j < 8; ++j) amax = fmaxf(amax, fabsf(v[c][j]));
  } else {
    each_chunk([&](int64_t, int, const float(&t)[8]) __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < 8; ++j) amax = fmaxf(amax, fabsf(t[j]));
    });
  }
  amax = wave_max_abs(amax);
  if constexpr (NT > 64) {
    if ((tid & 63) == 0) red[tid >> 6] = amax;
    __syncthreads();
    amax = red[0];
#pragma unroll
    for (int w = 1; w < NT / 64; ++w) amax = fmaxf(amax, red[w]);
  }
  const float s = scale_from_absmax(amax);
  const float r = 1.0f / s;
  if (tid == 0) scales_out[blockIdx.x] = s;
  if constexpr (REG > 0) {
#pragma unroll
    for (int c = 0; c < REG; ++c) {
      const int64_t k0 = (tid + static_cast<int64_t>(c) * NT) * 8;
      const int valid = valid_of(k0);
      if (valid > 0) qdq_store8<TX>(out, row, k0, valid, v[c], s, r);
    }
  } else {
    each_chunk([&](int64_t k0, int valid, const float(&t)[8]) __attribute__((always_inline)) {
      qdq_store8<TX>(out, row, k0, valid, t, s, r);
    });
  }
}

// Packs a row-major int8 [rows, K] matrix into 16x64 tiles.  One thread per
// 16-byte lane slot.  layout 1 maps packed row p to source row p/2 (p even)
// or rows/2 + p/2 (p odd): the gate/up "interleave" order of
// _pack_gateup_tensors (llama/lightweight_runner.py:81-92) applied to a
// split-packed [gate; up] source.
__global__ __launch_bounds__(256) void pack_rows_kernel(const int8_t* __restrict__ src,
                                                         int64_t rows, int64_t K, int64_t ld,
                                                         int layout, int vec, int64_t KB,
                                                         int64_t nslots,
                                                         int8_t* __restrict__ dst) {
  const int64_t slot = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (slot >= nslots) return;
  const int64_t tile = slot >> 6;
  const int lane = static_cast<int>(slot & 63);
  const int64_t rb = tile / KB;
  const int64_t kb = tile - rb * KB;
  const int64_t prow = rb * 16 + (lane & 15);
  const int64_t k0 = kb * 64 + (lane >> 4) * 16;
  u32x4 out = {0u, 0u, 0u, 0u};
  if (prow < rows && k0 < K) {
    int64_t srow = prow;
    if (layout == 1) srow = (prow & 1) ? (rows / 2 + (prow >> 1)) : (prow >> 1);
    const int8_t* p = src + srow * ld + k0;
    const int64_t valid = K - k0 < 16 ? K - k0 : 16;
    if (vec && valid == 16) {
      out = *reinterpret_cast<const u32x4*>(p);
    } else {
      uint8_t b[16];
#pragma unroll
      for (int j = 0; j < 16; ++j) b[j] = (j < valid) ? static_cast<uint8_t>(p[j]) : 0u;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        out[j] = static_cast<uint32_t>(b[4 * j]) | (static_cast<uint32_t>(b[4 * j + 1]) << 8) |
                 (static_cast<uint32_t>(b[4 * j + 2]) << 16) |
                 (static_cast<uint32_t>(b[4 * j + 3]) << 24);
      }
    }
  }
  reinterpret_cast<u32x4*>(dst)[slot] = out;
}

// Weight rows of up to kPackSources row-major matrices, in packed row order:
// one after another, or (interleave) packed row p from row p / 2 of matrix
// p % 2 (the gate/up order of pack_rows_kernel's layout 1).
struct QuantPackSrc {
  const void* x[kPackSources];
  int64_t ld[kPackSources];
  int64_t end[kPackSources];  // rows of this matrix and those before it
  int interleave;
  int vec;  // 16-byte aligned rows, K % 8 == 0
};

// Per-output weight quantization straight into the packed tiles: one
// workgroup per 16-row tile block, one wavefront per row.  The row stays in
// REG 16-byte chunks per lane (as stored, so 16-bit weights take 4 registers
// per 8 columns) between the absmax and the quantization; REG 0 reads it
// twice, and takes unaligned rows too.  Every pass of 1024 columns goes through LDS, so that each wavefront
// writes one whole 1 KiB tile: a row's own 8-byte pieces lie 256 bytes apart
// in the tiles, and rows on different XCDs would write every line in parts.
// The LDS copy of a 256-byte tile quarter is padded by 16 bytes: a
// wavefront's 64 pieces of one row then spread over all banks.  Bound: HBM
// (2 bytes in, 1 out per 16-bit weight): gate and up of 11008 x 4096 binary16
// take 56 us with the call, 4.8 TB/s; concatenating them (136 us), quantizing
// rows (46), packing (33) and interleaving the scales (5) took 215.
template <typename TX, int REG>
__global__ __launch_bounds__(1024) void quant_pack_rows_kernel(QuantPackSrc src, int64_t rows,
                                                               int64_t K, int KB,
                                                               int8_t* __restrict__ dst,
                                                               float* __restrict__ scales) {
  constexpr int kWords = static_cast<int>(sizeof(TX)) / 2;  // 16-byte loads per 8 columns
  constexpr int kQuarter = 256 + 16;
  constexpr int kPassTiles = 16;
  __shared__ u32x4 buf[2][kPassTiles * 4 * kQuarter / 16];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t prow = static_cast<int64_t>(blockIdx.x) * 16 + wave;
  const bool live = prow < rows;
  int m = 0;
  int64_t srow = 0;
  if (live) {
    if (src.interleave) {
      m = static_cast<int>(prow & 1);
      srow = prow >> 1;
    } else {
      while (prow >= src.end[m]) ++m;
      srow = prow - (m > 0 ? src.end[m - 1] : 0);
    }
  }
  const TX* xr = live ? static_cast<const TX*>(src.x[m]) + srow * src.ld[m] : nullptr;
  const __amdgpu_buffer_rsrc_t rs = raw_rsrc(xr, static_cast<int>(K * sizeof(TX)));
  // Chunk c of the lane: columns 8 (64 c + lane), zeros past K.
  auto fetch_vec = [&](int c, u32x4(&raw)[kWords]) {
    const int off = (c * 64 + lane) * 8 * static_cast<int>(sizeof(TX));
#pragma unroll
    for (int w = 0; w < kWords; ++w) raw[w] = load16(rs, off + 16 * w);
  };
  auto fetch_elems = [&](int c, u32x4(&raw)[kWords]) {
    const int64_t k0 = (static_cast<int64_t>(c) * 64 + lane) * 8;
    const int64_t left = live ? K - k0 : 0;
#pragma unroll
    for (int w = 0; w < kWords; ++w) raw[w] = u32x4{0u, 0u, 0u, 0u};
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (j < left) {
        if constexpr (sizeof(TX) == 4) {
          raw[j >> 2][j & 3] = __builtin_bit_cast(uint32_t, xr[k0 + j]);
        } else {
          raw[0][j >> 1] |= static_cast<uint32_t>(__builtin_bit_cast(uint16_t, xr[k0 + j]))
                            << (16 * (j & 1));
        }
      }
    }
  };
  auto fetch = [&](int c, u32x4(&raw)[kWords]) {
    if (src.vec) fetch_vec(c, raw); else fetch_elems(c, raw);
  };
  auto elem = [&](const u32x4(&raw)[kWords], int j) {
    if constexpr (sizeof(TX) == 4) {
      return __uint_as_float(raw[j >> 2][j & 3]);
    } else {
      const uint32_t w = raw[0][j >> 1];
      return bits_to_f32<TX>(j & 1 ? w >> 16 : w & 0xffffu);
    }
  };
  const int chunks = (KB + 7) / 8;
  u32x4 v[REG > 0 ? REG : 1][kWords];
  float amax = 0.0f;
  auto max_of = [&](const u32x4(&raw)[kWords]) {
#pragma unroll
    for (int j = 0; j < 8; ++j) amax = fmaxf(amax, fabsf(elem(raw, j)));
  };
  if constexpr (REG > 0) {
#pragma unroll
    for (int c = 0; c < REG; ++c) fetch_vec(c, v[c]);
#pragma unroll
    for (int c = 0; c < REG; ++c) {
      max_of(v[c]);
      // Opaque to the compiler from here, so that it converts the elements
      // again instead of keeping 8 binary32 values a chunk.
#pragma unroll
      for (int w = 0; w < kWords; ++w) asm volatile("" : "+v"(v[c][w]));
    }
  } else {
    for (int c = 0; c < chunks; ++c) {
      fetch(c, v[0]);
      max_of(v[0]);
    }
  }
  const float s = scale_from_absmax(wave_max_abs(amax));
  const float r = 1.0f / s;
  if (live && lane == 0) scales[prow] = s;

  int8_t* const out = dst + static_cast<int64_t>(blockIdx.x) * KB * kTileBytes;
  auto put = [&](const u32x4(&raw)[kWords], int half, int8_t* lds) {
    int32_t qi[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) qi[j] = quant_elem<TX>(elem(raw, j), s, r, true);
    // Tile 8 half + lane / 8 of the pass, quarter (lane % 8) / 2, slot of row `wave`.
    *reinterpret_cast<u32x2*>(lds + ((8 * half + (lane >> 3)) * 4 + ((lane & 7) >> 1)) * kQuarter +
                              wave * 16 + (lane & 1) * 8) =
        u32x2{pack4_i8(qi[0], qi[1], qi[2], qi[3]), pack4_i8(qi[4], qi[5], qi[6], qi[7])};
  };
  // Pass i: columns [1024 i, 1024 i + 1024).  Two LDS buffers: a wavefront
  // that fills pass i + 2's has passed barrier i + 1, behind every read of
  // pass i.
  auto flush = [&](int i, const int8_t* lds) {
    __syncthreads();
    const int kb = i * kPassTiles + wave;
    if (kb < KB)
      *reinterpret_cast<u32x4*>(out + static_cast<int64_t>(kb) * kTileBytes + lane * 16) =
          *reinterpret_cast<const u32x4*>(lds + (wave * 4 + (lane >> 4)) * kQuarter + (lane & 15) * 16);
  };
  if constexpr (REG > 0) {
    static_assert(REG % 2 == 0, "a pass takes two chunks");
#pragma unroll
    for (int i = 0; i < REG / 2; ++i) {
      if (2 * i < chunks) {
        int8_t* lds = reinterpret_cast<int8_t*>(buf[i & 1]);
        put(v[2 * i], 0, lds);
        put(v[2 * i + 1], 1, lds);
        flush(i, lds);
      }
    }
  } else {
    for (int i = 0; 2 * i < chunks; ++i) {
      int8_t* lds = reinterpret_cast<int8_t*>(buf[i & 1]);
      u32x4 second[kWords];
      fetch(2 * i, v[0]);
      fetch(2 * i + 1, second);
      put(v[0], 0, lds);
      put(second, 1, lds);
      flush(i, lds);
    }
  }
}

// Row-major int8 copy [rows, K] -> [rows, ldd] with zero columns K..ldd-1.
// One thread per 16-byte destination chunk.
__global__ __launch_bounds__(256) void pad_rows_kernel(const int8_t* __restrict__ src,
                                                        int64_t rows, int64_t K, int64_t ld,
                                                        int8_t* __restrict__ dst, int64_t ldd) {
  const int64_t chunks_per_row = ldd / 16;
  const int64_t idx = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (idx >= rows * chunks_per_row) return;
  const int64_t r = idx / chunks_per_row;
  const int64_t k0 = (idx - r * chunks_per_row) * 16;
  uint8_t b[16];
#pragma unroll
  for (int j = 0; j < 16; ++j) b[j] = (k0 + j < K) ? static_cast<uint8_t>(src[r * ld + k0 + j]) : 0u;
  u32x4 out;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    out[j] = static_cast<uint32_t>(b[4 * j]) | (static_cast<uint32_t>(b[4 * j + 1]) << 8) |
             (static_cast<uint32_t>(b[4 * j + 2]) << 16) | (static_cast<uint32_t>(b[4 * j + 3]) << 24);
  }
  *reinterpret_cast<u32x4*>(dst + r * ldd + k0) = out;
}

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
inline bool aligned8(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 7u) == 0; }

template <typename TX, bool PACKED, bool DYN, int REG, int NT>
void quant_launch_reg(dim3 g, hipStream_t st, const TX* x, int64_t ldx, int64_t rows,
                      int64_t K, int vec_in, const float* scale_in, int64_t scale_stride,
                      int8_t* q, int64_t ldq, int64_t ncols_out, int vec_out, int64_t KB,
                      float* scales_out) {
  hipLaunchKernelGGL((quant_rows_kernel<TX, PACKED, DYN, REG, NT>), g, dim3(NT), 0, st, x, ldx,
                     rows, K, vec_in, scale_in, scale_stride, q, ldq, ncols_out, vec_out, KB,
                     scales_out);
}

template <typename TX, bool PACKED, bool DYN, int NT>
void quant_launch_nt(dim3 g, hipStream_t st, int64_t chunks, const TX* x, int64_t ldx,
                     int64_t rows, int64_t K, int vec_in, const float* scale_in,
                     int64_t scale_stride, int8_t* q, int64_t ldq, int64_t ncols_out,
                     int vec_out, int64_t KB, float* scales_out) {
  const int64_t per = ceil_div(chunks, NT);
#define W8A8_QUANT_REG(R)                                                                     \
  quant_launch_reg<TX, PACKED, DYN, R, NT>(g, st, x, ldx, rows, K, vec_in, scale_in,          \
                                           scale_stride, q, ldq, ncols_out, vec_out, KB,      \
                                           scales_out)
  if (per <= 1)
    W8A8_QUANT_REG(1);
  else if (per <= 2)
    W8A8_QUANT_REG(2);
  else if (per <= 4)
    W8A8_QUANT_REG(4);
  else if (per <= kRegChunksMax)
    W8A8_QUANT_REG(kRegChunksMax);
  else
    W8A8_QUANT_REG(0);
#undef W8A8_QUANT_REG
}

// Few rows (decode) leave most of the GPU idle, so each row's latency is what
// counts: wide rows then get up to 1024 threads (16 wavefronts share each
// CU's SIMDs and hide each other's load latency).  Many rows keep 256
// threads per row.
template <typename TX, bool PACKED, bool DYN>
void quant_launch(dim3 g, hipStream_t st, int64_t chunks, const TX* x, int64_t ldx,
                  int64_t rows, int64_t K, int vec_in, const float* scale_in,
                  int64_t scale_stride, int8_t* q, int64_t ldq, int64_t ncols_out, int vec_out,
                  int64_t KB, float* scales_out) {
  if constexpr (!PACKED) {
    if (rows <= kGemvMaxRows && chunks > kQuantThreads) {
      if (chunks > 2 * kQuantThreads)
        return quant_launch_nt<TX, PACKED, DYN, 4 * kQuantThreads>(
            g, st, chunks, x, ldx, rows, K, vec_in, scale_in, scale_stride, q, ldq, ncols_out,
            vec_out, KB, scales_out);
      return quant_launch_nt<TX, PACKED, DYN, 2 * kQuantThreads>(
          g, st, chunks, x, ldx, rows, K, vec_in, scale_in, scale_stride, q, ldq, ncols_out,
          vec_out, KB, scales_out);
    }
  }
  quant_launch_nt<TX, PACKED, DYN, kQuantThreads>(g, st, chunks, x, ldx, rows, K, vec_in,
                                                  scale_in, scale_stride, q, ldq, ncols_out,
                                                  vec_out, KB, scales_out);
}

template <typename TX>
hipError_t quant_dispatch(const TX* x, int64_t ldx, int64_t rows, int64_t K,
                          const float* scale_in, int64_t scale_stride, int8_t* q, int64_t ldq,
                          int64_t ncols_out, bool packed, float* scales_out, hipStream_t st) {
  const int vec_in = aligned16(x) && (ldx % 8 == 0) && (K % 8 == 0);
  const int vec_out = aligned8(q) && (ldq % 8 == 0);
  const int64_t KB = ceil_div(K, kTileK);
  const int64_t grid = packed ? ceil_div(rows, kTileRows) * kTileRows : rows;
  if (grid == 0) return hipSuccess;
  const int64_t chunks = packed ? KB * 8 : ceil_div(ncols_out > K ? ncols_out : K, 8);
  const bool dyn = scale_in == nullptr;
  dim3 g(static_cast<unsigned>(grid));
  if (packed) {
    if (dyn)
      quant_launch<TX, true, true>(g, st, chunks, x, ldx, rows, K, vec_in, scale_in,
                                   scale_stride, q, ldq, ncols_out, vec_out, KB, scales_out);
    else
      quant_launch<TX, true, false>(g, st, chunks, x, ldx, rows, K, vec_in, scale_in,
                                    scale_stride, q, ldq, ncols_out, vec_out, KB, scales_out);
  } else {
    if (dyn)
      quant_launch<TX, false, true>(g, st, chunks, x, ldx, rows, K, vec_in, scale_in,
                                    scale_stride, q, ldq, ncols_out, vec_out, KB, scales_out);
    else
      quant_launch<TX, false, false>(g, st, chunks, x, ldx, rows, K, vec_in, scale_in,
                                     scale_stride, q, ldq, ncols_out, vec_out, KB, scales_out);
  }
  return hipGetLastError();
}

}  // namespace

hipError_t launch_quant_rows(const void* x, int x_dtype, int64_t ldx, int64_t rows, int64_t K,
                             const float* scale_in, int64_t scale_stride, int8_t* q,
                             int64_t ldq, int64_t ncols_out, bool packed, float* scales_out,
                             hipStream_t st) {
  switch (x_dtype) {
    case kF32:
      return quant_dispatch(static_cast<const float*>(x), ldx, rows, K, scale_in, scale_stride,
                            q, ldq, ncols_out, packed, scales_out, st);
    case kF16:
      return quant_dispatch(static_cast<const __half*>(x), ldx, rows, K, scale_in, scale_stride,
                            q, ldq, ncols_out, packed, scales_out, st);
    case kBF16:
      return quant_dispatch(static_cast<const __hip_bfloat16*>(x), ldx, rows, K, scale_in,
                            scale_stride, q, ldq, ncols_out, packed, scales_out, st);
    default:
      return hipErrorInvalidValue;
  }
}

// Register chunks per lane: aligned rows of up to 512 REG columns are read once.
template <typename TX>
hipError_t quant_pack_dispatch(const QuantPackSrc& src, int64_t rows, int64_t K, int8_t* dst,
                               float* scales, hipStream_t st) {
  const int64_t KB = ceil_div(K, kTileK);
  const dim3 g(static_cast<unsigned>(ceil_div(rows, kTileRows)));
#define W8A8_QUANT_PACK(R)                                                                     \
  hipLaunchKernelGGL((quant_pack_rows_kernel<TX, R>), g, dim3(1024), 0, st, src, rows, K,      \
                     static_cast<int>(KB), dst, scales)
  if (!src.vec)
    W8A8_QUANT_PACK(0);
  else if (K <= 4 * 512)
    W8A8_QUANT_PACK(4);
  else if (K <= 8 * 512)
    W8A8_QUANT_PACK(8);
  else if (sizeof(TX) == 2 && K <= 16 * 512)
    W8A8_QUANT_PACK(sizeof(TX) == 2 ? 16 : 0);
  else if (sizeof(TX) == 2 && K <= 22 * 512)
    W8A8_QUANT_PACK(sizeof(TX) == 2 ? 22 : 0);
  else
    W8A8_QUANT_PACK(0);
#undef W8A8_QUANT_PACK
  return hipGetLastError();
}

template <typename TX, int NT>
void qdq_rows_launch(dim3 g, hipStream_t st, const TX* x, int64_t ldx, int64_t K, int64_t group,
                     int vec_in, int groups, const QdqOut& out, float* scales) {
  const int64_t per = ceil_div(group < K ? group : K, 8 * NT);
#define W8A8_QDQ_REG(R)                                                                          \
  hipLaunchKernelGGL((qdq_rows_kernel<TX, R, NT>), g, dim3(NT), 0, st, x, ldx, K, group, vec_in, \
                     groups, out, scales)
  if (per <= 1)
    W8A8_QDQ_REG(1);
  else if (per <= 2)
    W8A8_QDQ_REG(2);
  else if (per <= 4)
    W8A8_QDQ_REG(4);
  else if (per <= kRegChunksMax)
    W8A8_QDQ_REG(kRegChunksMax);
  else
    W8A8_QDQ_REG(0);
#undef W8A8_QDQ_REG
}

// qdq_groups_kernel counts a row's chunks and groups in 32 bits (the 2^30 and
// fewer of this K leave room for its last workgroup's idle lanes); the other
// kernel's columns are 64-bit throughout.
constexpr int64_t kQdqGroupsMaxK = int64_t{1} << 33;

// Groups of 8, 16, .. 512 columns run on qdq_groups_kernel; other groups take
// a workgroup each: one wavefront up to 512 columns, 256 threads past that, 512
// where up to 2048 workgroups leave the CUs room for them, and 1024 where there
// are at most two workgroups per CU of more columns than 512 threads hold in
// registers (one row of 70000 bfloat16 15.2 us a call, 18.2 on 512 threads;
// 64 rows 15.1 against 21.7).
template <typename TX>
hipError_t qdq_dispatch(const TX* x, int64_t ldx, int64_t rows, int64_t K, int64_t group,
                        const QdqOut& o, float* scales, hipStream_t st) {
  const int64_t groups = ceil_div(K, group);
  QdqOut out = o;
  const bool cols8 = K % 8 == 0 && group % 8 == 0;
  const int vec_in = cols8 && aligned16(x) && ldx % 8 == 0;
  out.vec_q = cols8 && aligned8(o.q) && o.ldq % 8 == 0;
  out.vec_d = cols8 && aligned16(o.deq) && o.ldd % 8 == 0;
  const int64_t lanes = group / 8;
  if (group % 8 == 0 && lanes <= 64 && (lanes & (lanes - 1)) == 0 && groups > 1 &&
      K <= kQdqGroupsMaxK) {
    const int64_t bpr = ceil_div(groups * lanes, kQuantThreads);
    if (rows * bpr > INT32_MAX) return hipErrorInvalidConfiguration;
#define W8A8_QDQ_LPG(L)                                                                        \
  case L:                                                                                      \
    hipLaunchKernelGGL((qdq_groups_kernel<TX, L>), dim3(static_cast<unsigned>(rows * bpr)),    \
                       dim3(kQuantThreads), 0, st, x, ldx, K, vec_in, static_cast<int>(groups), \
                       static_cast<int>(bpr), out, scales);                                    \
    break
    switch (lanes) {
      W8A8_QDQ_LPG(1);
      W8A8_QDQ_LPG(2);
      W8A8_QDQ_LPG(4);
      W8A8_QDQ_LPG(8);
      W8A8_QDQ_LPG(16);
      W8A8_QDQ_LPG(32);
      W8A8_QDQ_LPG(64);
    }
#undef W8A8_QDQ_LPG
    return hipGetLastError();
  }
  if (rows * groups > INT32_MAX) return hipErrorInvalidConfiguration;
  const dim3 g(static_cast<unsigned>(rows * groups));
  const int64_t n = group < K ? group : K;
  const int ng = static_cast<int>(groups);
  if (n <= 512)
    qdq_rows_launch<TX, 64>(g, st, x, ldx, K, group, vec_in, ng, out, scales);
  else if (rows * groups <= 2 * cu_count() && n > 8 * kRegChunksMax * 2 * kQuantThreads)
    qdq_rows_launch<TX, 4 * kQuantThreads>(g, st, x, ldx, K, group, vec_in, ng, out, scales);
  else if (rows * groups <= 2048 && n > 8 * kQuantThreads)
    qdq_rows_launch<TX, 2 * kQuantThreads>(g, st, x, ldx, K, group, vec_in, ng, out, scales);
  else
    qdq_rows_launch<TX, kQuantThreads>(g, st, x, ldx, K, group, vec_in, ng, out, scales);
  return hipGetLastError();
}

template <typename TX, int NT>
void quant_parts_launch(dim3 g, hipStream_t st, int64_t chunks, const TX* x, int64_t ldx,
                        int64_t K, int vec_in, const float* parts, int64_t nparts, int8_t* q,
                        int64_t ldq, int vec_out, float* scales) {
  const int64_t per = ceil_div(chunks, NT);
#define W8A8_PARTS_REG(R)                                                                     \
  hipLaunchKernelGGL((quant_rows_parts_kernel<TX, R, NT>), g, dim3(NT), 0, st, x, ldx, K,       \
                     vec_in, parts, nparts, q, ldq, vec_out, scales)
  if (per <= 1)
    W8A8_PARTS_REG(1);
  else if (per <= 2)
    W8A8_PARTS_REG(2);
  else if (per <= 4)
    W8A8_PARTS_REG(4);
  else if (per <= kRegChunksMax)
    W8A8_PARTS_REG(kRegChunksMax);
  else
    W8A8_PARTS_REG(0);
#undef W8A8_PARTS_REG
}

template <typename TX>
hipError_t quant_parts_dispatch(const TX* x, int64_t ldx, int64_t rows, int64_t K,
                                const float* parts, int64_t nparts, int8_t* q, int64_t ldq,
                                float* scales, hipStream_t st) {
  const int vec_in = aligned16(x) && (ldx % 8 == 0) && (K % 8 == 0);
  const int vec_out = aligned8(q) && (ldq % 8 == 0);
  const int64_t chunks = ceil_div(K, 8);
  const dim3 g(static_cast<unsigned>(rows));
  // Few rows (decode) get wide workgroups, as in quant_launch.
  if (rows <= kGemvMaxRows && chunks > 2 * kQuantThreads)
    quant_parts_launch<TX, 4 * kQuantThreads>(g, st, chunks, x, ldx, K, vec_in, parts, nparts, q,
                                              ldq, vec_out, scales);
  else if (rows <= kGemvMaxRows && chunks > kQuantThreads)
    quant_parts_launch<TX, 2 * kQuantThreads>(g, st, chunks, x, ldx, K, vec_in, parts, nparts, q,
                                              ldq, vec_out, scales);
  else
    quant_parts_launch<TX, kQuantThreads>(g, st, chunks, x, ldx, K, vec_in, parts, nparts, q,
                                          ldq, vec_out, scales);
  return hipGetLastError();
}

hipError_t launch_quant_rows_parts(const void* x, int x_dtype, int64_t ldx, int64_t rows,
                                   int64_t K, const float* parts, int64_t nparts, int8_t* q,
                                   int64_t ldq, float* scales_out, hipStream_t st) {
  if (rows == 0) return hipSuccess;
  switch (x_dtype) {
    case kF32:
      return quant_parts_dispatch(static_cast<const float*>(x), ldx, rows, K, parts, nparts, q,
                                  ldq, scales_out, st);
    case kF16:
      return quant_parts_dispatch(static_cast<const __half*>(x), ldx, rows, K, parts, nparts, q,
                                  ldq, scales_out, st);
    case kBF16:
      return quant_parts_dispatch(static_cast<const __hip_bfloat16*>(x), ldx, rows, K, parts,
                                  nparts, q, ldq, scales_out, st);
    default:
      return hipErrorInvalidValue;
  }
}

hipError_t launch_qdq_rows(const void* x, int x_dtype, int64_t ldx, int64_t rows, int64_t K,
                           int64_t group, int8_t* q, int64_t ldq, void* deq, int64_t ldd,
                           float* scales_out, hipStream_t st) {
  if (rows == 0 || K == 0) return hipSuccess;
  const QdqOut out{q, ldq, deq, ldd, 0, 0};
  switch (x_dtype) {
    case kF32:
      return qdq_dispatch(static_cast<const float*>(x), ldx, rows, K, group, out, scales_out, st);
    case kF16:
      return qdq_dispatch(static_cast<const __half*>(x), ldx, rows, K, group, out, scales_out, st);
    case kBF16:
      return qdq_dispatch(static_cast<const __hip_bfloat16*>(x), ldx, rows, K, group, out,
                          scales_out, st);
    default:
      return hipErrorInvalidValue;
  }
}

hipError_t launch_quant_pack_rows(const void* const* x, const int64_t* ld, const int64_t* x_rows,
                                  int n_src, int x_dtype, int64_t K, bool interleave, int8_t* dst,
                                  float* scales, hipStream_t st) {
  QuantPackSrc src{};
  src.interleave = interleave ? 1 : 0;
  src.vec = K % 8 == 0;
  const int64_t per16 = x_dtype == kF32 ? 4 : 8;  // elements of 16 bytes
  int64_t rows = 0;
  for (int i = 0; i < n_src; ++i) {
    rows += x_rows[i];
    src.x[i] = x[i];
    src.ld[i] = ld[i];
    src.end[i] = rows;
    if (x_rows[i] > 0 && (!aligned16(x[i]) || ld[i] % per16 != 0)) src.vec = 0;
  }
  switch (x_dtype) {
    case kF32:
      return quant_pack_dispatch<float>(src, rows, K, dst, scales, st);
    case kF16:
      return quant_pack_dispatch<__half>(src, rows, K, dst, scales, st);
    case kBF16:
      return quant_pack_dispatch<__hip_bfloat16>(src, rows, K, dst, scales, st);
    default:
      return hipErrorInvalidValue;
  }
}

hipError_t launch_pack_rows(const int8_t* src, int64_t rows, int64_t K, int64_t ld, int layout,
                            int8_t* dst, hipStream_t st) {
  const int64_t KB = ceil_div(K, kTileK);
  const int64_t nslots = ceil_div(rows, kTileRows) * KB * kTileVec;
  if (nslots == 0) return hipSuccess;
  const int vec = aligned16(src) && (ld % 16 == 0);
  const int64_t blocks = ceil_div(nslots, 256);
  hipLaunchKernelGGL(pack_rows_kernel, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, st,
                     src, rows, K, ld, layout, vec, KB, nslots, dst);
  return hipGetLastError();
}

hipError_t launch_pad_rows(const int8_t* src, int64_t rows, int64_t K, int64_t ld, int8_t* dst,
                           int64_t ldd, hipStream_t st) {
  const int64_t total = rows * (ldd / 16);
  if (total == 0) return hipSuccess;
  hipLaunchKernelGGL(pad_rows_kernel, dim3(static_cast<unsigned>(ceil_div(total, 256))), dim3(256),
                     0, st, src, rows, K, ld, dst, ldd);
  return hipGetLastError();
}

}  // namespace w8a8
