// MXFP8 re-quantisation of the bf16 weights the optimizer step has just refreshed.
//
// Replaces `_quant_mxfp8_w` and `_quant_mxfp8_w_cm` (ancora/kernels/quant.py:60-100), which the
// reference launches from the next forward once the step has set its dirty flags
// (ancora/model/resident_train.py:190-199, 354-357). Per block of 32 consecutive K and per
// column: amax of |w|, E8M0 scale byte = (biased fp32 exponent of amax) - 7 (0 below 7), element
// = E4M3FN(w / 2^(byte-127)), round to nearest even: a product with a power of two, exact, and the hardware's
// conversion. Where a column holds something else than ordinary numbers (amax below 2^-96, infinities, NaN) the same in
// integer arithmetic on the bf16 bit patterns: an element with biased exponent eb and 7-bit mantissa m becomes the E4M3
// number with biased exponent e = eb - byte + 7 and mantissa m rounded to 3 bits (carry into e),
// or, for e <= 0, the multiple of 2^-9 nearest to 1.m * 2^(e-7). (That arithmetic for every element, 13 instructions
// against 4, took as long as the memory: the 28 weights of four layers 40.5 -> 32.6 us, 5.9 TB/s, column-major
// 45.9 -> 37.3, one layer of 512 10.6 -> 6.2.)
//
// HBM-bound byte work: 2 B read, 1 + 1/32 B written per element. A lane loads 16 rows x 8 columns
// with 16-byte loads; the stores of either output layout fill whole 128-byte lines: row-major
// (K,N) rows of 8 bytes per lane over 16 lanes, or column-major (N,K) 16 bytes per lane and
// column, the 8 lanes that hold the 128 rows of the tile completing the line.
#include "common.h"

namespace {

constexpr int kThreads = 256;
constexpr int kRows = 32;          // scale block along K
constexpr int kHalf = 16;          // rows of it held by one lane

// E4M3FN byte (without sign) of the bf16 magnitude `a` (15 bits) scaled by 2^(127-byte);
// adj = (7 - byte) << 7.
__device__ __forceinline__ uint32_t e4m3_general(uint32_t a, int adj) {
  if (a >= 0x7F80u) return 0x7Fu;                  // Inf / NaN
  if (a < 0x80u) return 0u;                        // zero and bf16 subnormals
  const int t = (int)a + adj;                      // (e << 7) | m
  if (t >= 128) return (uint32_t)(t + 7 + ((t >> 4) & 1)) >> 4;
  const int sh = 5 - (t >> 7);                     // bits of the 8-bit significand to drop (>= 5)
  if (sh >= 10) return 0u;
  const uint32_t sig = 0x80u | (a & 0x7Fu);
  return (sig + (1u << (sh - 1)) - 1u + ((sig >> sh) & 1u)) >> sh;
}

__device__ __forceinline__ float lo_half(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float hi_half(uint32_t w) { return __uint_as_float(w & 0xFFFF0000u); }
// Four E4M3FN bytes of floats below 464 in magnitude: v_cvt_pk_fp8_f32, round to nearest even, subnormal results, the
// sign of zero kept.
__device__ __forceinline__ uint32_t e4m3_four(float a, float b, float c, float d) {
  return (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(c, d, __builtin_amdgcn_cvt_pk_fp8_f32(a, b, 0, false), true);
}

// Wavefront tile: 64 rows x 128 columns (row-major output) or 128 rows x 64 columns (column-major
// output). A lane holds 16 rows x 8 columns, i.e. half a scale block; the two halves sit in lanes
// `lane` and `lane ^ kPartner` and exchange their column maxima.
// With `table` set the launch covers n weights, tile0 their first wavefront tiles: a weight of a 1024-wide
// layer is 2 .. 6 MB, 1 us of HBM traffic in a launch of 10 us, so a refresh of 28 weights one by one ran at 0.7
// TB/s (275 us).
template <bool CM>
__global__ void __launch_bounds__(kThreads, 4)
k_quant_mxfp8_w(anc_quant_desc_t d, const anc_quant_desc_t *__restrict__ table, int n, int64_t tiles) {
  constexpr int kColGroups = CM ? 8 : 16;          // lanes across the columns (8 columns each)
  constexpr int kTileCols = kColGroups * 8, kTileRows = (64 / kColGroups) * kHalf;
  const int lane = threadIdx.x & 63;
  int64_t tile = (int64_t)blockIdx.x * (kThreads / 64) + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  if (tile >= tiles) return;                                      // whole wavefront
  if (table != nullptr) {
    int lo = 0, hi = n - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (table[mid].tile0 <= tile) lo = mid; else hi = mid - 1;
    }
    d = table[lo];
    tile -= d.tile0;
  }
  const uint16_t *__restrict__ w = (const uint16_t *)d.w;
  uint8_t *__restrict__ fp8 = (uint8_t *)d.fp8, *__restrict__ sc = (uint8_t *)d.scale;
  const int K = d.K, N = d.N;
  const int tn = N / kTileCols, tk = K / kTileRows;
  const int cb = (int)(tile % tn);
  const int rb = (int)((tile / tn) % tk);
  const int64_t e = tile / ((int64_t)tn * tk);
  const int hb = lane / kColGroups, half = hb & 1;                // half-block of this lane
  const int kb = rb * (kTileRows / kRows) + (hb >> 1);            // scale block along K
  const int col0 = cb * kTileCols + (lane % kColGroups) * 8;
  const int row0 = kb * kRows + half * kHalf;
  const uint16_t *src = w + (e * K + row0) * N + col0;

  anc_u32x4 v[kHalf];
#pragma unroll
  for (int r = 0; r < kHalf; ++r) v[r] = anc_ld_stream((const anc_u32x4 *)(src + (int64_t)r * N));

  // amax per column as the maximum of the 15-bit magnitudes (same order as the values), two
  // columns per packed 16-bit max
  typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
  u16x2 am2[4] = {{0, 0}, {0, 0}, {0, 0}, {0, 0}};
#pragma unroll
  for (int r = 0; r < kHalf; ++r) {
    const uint32_t q[4] = {v[r].x, v[r].y, v[r].z, v[r].w};
#pragma unroll
    for (int h = 0; h < 4; ++h) {
      const uint32_t m = q[h] & 0x7FFF7FFFu;
      am2[h] = __builtin_elementwise_max(am2[h], __builtin_bit_cast(u16x2, m));
    }
  }
  uint32_t amax[8];
#pragma unroll
  for (int h = 0; h < 4; ++h) {
    uint32_t m = __builtin_bit_cast(uint32_t, am2[h]);
    const uint32_t o = (uint32_t)__shfl_xor((int)m, kColGroups, 64);
    m = __builtin_bit_cast(uint32_t, __builtin_elementwise_max(am2[h], __builtin_bit_cast(u16x2, o)));
    amax[2 * h] = m & 0xFFFFu;
    amax[2 * h + 1] = m >> 16;
  }
  uint32_t byte[8];
  float by[8];            // the scale's reciprocal, 2^(127 - byte)
  bool plain = true;      // every column: zeros, or finite with a scale byte high enough that what has a zero exponent
                          // field (2^-126 and less) scales to 2^-23 and less, which rounds to zero
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const uint32_t ea = amax[j] >> 7;
    byte[j] = ea >= 7u ? ea - 7u : 0u;
    by[j] = __uint_as_float((254u - byte[j]) << 23);
    plain = plain && (amax[j] == 0u || (ea != 255u && byte[j] >= 24u));
  }

  // scale bytes, from the lane that holds the first half of the block
  if (half == 0) {
    if constexpr (!CM) {
      const anc_u32x2 s2 = {byte[0] | (byte[1] << 8) | (byte[2] << 16) | (byte[3] << 24),
                            byte[4] | (byte[5] << 8) | (byte[6] << 16) | (byte[7] << 24)};
      anc_st_stream((anc_u32x2 *)(sc + (e * (K / kRows) + kb) * N + col0), s2);
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) sc[(e * N + col0 + j) * (int64_t)(K / kRows) + kb] = (uint8_t)byte[j];
    }
  }

  if constexpr (!CM) {
    // row-major: 8 bytes per row
#pragma unroll
    for (int r = 0; r < kHalf; ++r) {
      const uint32_t q[4] = {v[r].x, v[r].y, v[r].z, v[r].w};
      uint32_t o[2] = {0u, 0u};
      if (plain) {
#pragma unroll
        for (int h = 0; h < 2; ++h) o[h] = e4m3_four(lo_half(q[2 * h]) * by[4 * h], hi_half(q[2 * h]) * by[4 * h + 1],
                                                     lo_half(q[2 * h + 1]) * by[4 * h + 2], hi_half(q[2 * h + 1]) * by[4 * h + 3]);
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const uint32_t w = (j & 1) ? (q[j >> 1] >> 16) : (q[j >> 1] & 0xFFFFu);
          o[j >> 2] |= (e4m3_general(w & 0x7FFFu, (7 - (int)byte[j]) * 128) | ((w >> 8) & 0x80u)) << (8 * (j & 3));
        }
      }
      anc_st_stream((anc_u32x2 *)(fp8 + (e * K + row0 + r) * N + col0), anc_u32x2{o[0], o[1]});
      __builtin_amdgcn_sched_barrier(0);          // one row at a time: keeps the live set small
    }
  } else {
    // column-major: 16 bytes (the lane's 16 rows) per column
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      uint32_t o[4] = {0, 0, 0, 0};
      auto at = [&](int r) { const uint32_t q[4] = {v[r].x, v[r].y, v[r].z, v[r].w}; return q[j >> 1]; };
      if (plain) {
        auto x = [&](int r) { return ((j & 1) ? hi_half(at(r)) : lo_half(at(r))) * by[j]; };
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = e4m3_four(x(4 * i), x(4 * i + 1), x(4 * i + 2), x(4 * i + 3));
      } else {
#pragma unroll
        for (int r = 0; r < kHalf; ++r) {
          const uint32_t w = (j & 1) ? (at(r) >> 16) : (at(r) & 0xFFFFu);
          o[r >> 2] |= (e4m3_general(w & 0x7FFFu, (7 - (int)byte[j]) * 128) | ((w >> 8) & 0x80u)) << (8 * (r & 3));
        }
      }
      const anc_u32x4 o4 = {o[0], o[1], o[2], o[3]};
      anc_st_stream((anc_u32x4 *)(fp8 + (e * N + col0 + j) * (int64_t)K + row0), o4);
      __builtin_amdgcn_sched_barrier(0);          // one column at a time
    }
  }
}

}  // namespace

static int launch_quant(const anc_quant_desc_t &d, const anc_quant_desc_t *table, int n, int64_t tiles, int col_major,
                        hipStream_t s) {
  const int64_t blocks = (tiles + kThreads / 64 - 1) / (kThreads / 64);
  ANC_REQUIRE(blocks < (1ll << 31), "anc_quant_mxfp8_w: too large");
  AncProfScope prof(ANC_PROF_MISC, s);
  if (col_major) hipLaunchKernelGGL((k_quant_mxfp8_w<true>), dim3((unsigned)blocks), dim3(kThreads), 0, s, d, table, n, tiles);
  else           hipLaunchKernelGGL((k_quant_mxfp8_w<false>), dim3((unsigned)blocks), dim3(kThreads), 0, s, d, table, n, tiles);
  ANC_LAUNCH_CHECK();
  return ANC_OK;
}

extern "C" int64_t anc_quant_mxfp8_num_tiles(int64_t E, int64_t K, int64_t N) {
  if (E <= 0 || K <= 0 || N <= 0 || K % 128 != 0 || N % 128 != 0 || K >= (1ll << 31) || N >= (1ll << 31)) {
    anc_set_error("anc_quant_mxfp8_num_tiles: K=%lld and N=%lld must be positive multiples of 128", (long long)K, (long long)N);
    return -1;
  }
  return E * (K * N / 8192);                                      // 64x128 or 128x64 per wavefront
}

extern "C" int anc_quant_mxfp8_w(uint64_t w_bf16, uint64_t fp8_out, uint64_t scale_out, int64_t E,
                                 int64_t K, int64_t N, int col_major, uint64_t stream) {
  ANC_REQUIRE(w_bf16 && fp8_out && scale_out && E > 0, "anc_quant_mxfp8_w: bad arguments");
  ANC_REQUIRE(K > 0 && N > 0 && K % 128 == 0 && N % 128 == 0,
              "anc_quant_mxfp8_w: K=%lld and N=%lld must be positive multiples of 128", (long long)K,
              (long long)N);
  ANC_REQUIRE(K < (1ll << 31) && N < (1ll << 31), "anc_quant_mxfp8_w: dimension too large");
  ANC_REQUIRE(((w_bf16 | fp8_out) & 15) == 0 && (scale_out & 7) == 0,
              "anc_quant_mxfp8_w: w and fp8_out must be 16-byte, scale_out 8-byte aligned");
  const anc_quant_desc_t d{w_bf16, fp8_out, scale_out, 0, (int32_t)K, (int32_t)N};
  return launch_quant(d, nullptr, 0, anc_quant_mxfp8_num_tiles(E, K, N), col_major, anc_stream(stream));
}

extern "C" int anc_quant_mxfp8_w_multi(uint64_t desc_table, int32_t n_weights, int64_t total_tiles, int col_major,
                                       uint64_t stream) {
  ANC_REQUIRE(desc_table != 0 && (desc_table & 7) == 0 && n_weights > 0, "anc_quant_mxfp8_w_multi: empty descriptor table");
  ANC_REQUIRE(total_tiles > 0, "anc_quant_mxfp8_w_multi: bad total_tiles");
  return launch_quant(anc_quant_desc_t{}, (const anc_quant_desc_t *)desc_table, (int)n_weights, total_tiles, col_major,
                      anc_stream(stream));
}
