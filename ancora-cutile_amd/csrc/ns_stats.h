// What the gates' statistics of a matrix are made of (ns.hip says what they are for): shared by the kernels of their own and by the
// launch of B = b A + c A A that carries them for one matrix.
#pragma once
#include "ns_common.h"
#include "reduce.h"

// 16-byte loads in flight per lane: all that a lane has of a 1024x1024 matrix, M^2 / 2^17. Of a larger one that is no multiple of
// 1024 the loads behind the last whole eight (two of 1152x1152, seven of 1408x1408) come one at a time. (One at a time, behind a test for the end: 5.3 -> 4.6 us for one such
// matrix, 19.3 -> 17.3 for 48, 5.8 TB/s; with loads that the caches keep instead of streamed ones 34.9.)
constexpr int kCondAhead = 8;
// Part b of the matrices' squares of Fh, for thread 0 of 256.
__device__ __forceinline__ double cond_part(const uint16_t *Fh, int M, int b, double *wave_sum) {
  const int64_t per = (int64_t)M * M / kCondParts;
  const uint16_t *src = Fh + (int64_t)b * per;
  double acc = 0.0;
  const int n = (int)(per / anc_reduce::kRun);                           // (per: a multiple of 256)
  int v = (int)threadIdx.x;
  auto add = [&](anc_u32x4 r) {                              // run_sumsq of eight elements
    const uint32_t w[4] = {r.x, r.y, r.z, r.w};
    float s = 0.0f;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float x0 = __uint_as_float(w[k] << 16), x1 = __uint_as_float(w[k] & 0xFFFF0000u);
      s = s + x0 * x0;
      s = s + x1 * x1;
    }
    acc = acc + (double)s;
  };
  for (; v + (kCondAhead - 1) * anc_reduce::kThreads < n; v += kCondAhead * anc_reduce::kThreads) {
    anc_u32x4 r[kCondAhead];
#pragma unroll
    for (int k = 0; k < kCondAhead; ++k) r[k] = anc_ld_stream((const anc_u32x4 *)src + v + k * anc_reduce::kThreads);
#pragma unroll
    for (int k = 0; k < kCondAhead; ++k) add(r[k]);
  }
  for (; v < n; v += anc_reduce::kThreads) add(anc_ld_stream((const anc_u32x4 *)src + v));
  acc = anc_wave_sum_f64(acc);
  if ((threadIdx.x & 63) == 0) wave_sum[threadIdx.x >> 6] = acc;
  __syncthreads();
  double t = wave_sum[0];
#pragma unroll
  for (int w = 1; w < anc_reduce::kThreads / 64; ++w) t = t + wave_sum[w];
  return t;
}

struct WideRule {
  double near_lo, lo, hi;    // in units of the proxy N * ||offdiag(A0)||^2; near_lo == lo: no near range
  double near_diff;          // > 0: in the near range the gate takes a matrix whose proxy exceeds its column
                             // concentration by more than this; 0: the kColcFrac rule there as above the band
};
// kBulkShare: outlier columns keep the cheap gates while the other columns still hold a few
// thousandths of the mass (1 % of the columns x100: 1e-2 of it, 8e-4 .. 1.6e-3 with those gates);
// beyond that the bulk's directions drown in the rounding of the outliers (x300: share 1e-3, 1.4e-3
// .. 1.9e-3; x1000: 1e-4, 3.6e-3 .. 4.0e-3; x3000: 5.2e-3 .. 5.8e-3) and only every residual
// term from iteration 1 on recovers them (8e-5 .. 2.9e-4).
// kColcFrac: a matrix keeps the cheap gates only if its column norms explain its proxy (colc at least
// 0.85 of it: pure outlier columns and scaled columns read 1.00 .. 1.01). Anything less is a
// mixture (a low-rank signal WITH outlier columns: 3.5e-3 at a ratio of 0.28 and 6.6e-3 at 0.5 with
// the cheap gates at 1024x3072, 1e-4 .. 2e-4 with every residual term) or has its mass in directions
// that are not columns at all (near-duplicate rows: ratio 0.5 .. 0.75).
constexpr double kColcFrac = 0.85, kBulkShare = 3e-3;
// sum of a matrix's partial sums, called by whole wavefronts
__device__ __forceinline__ double cond_sum(const double *parts) { return anc_wave_sum_f64(parts[threadIdx.x & 63]); }
static_assert(kCondParts == 64, "a partial sum per lane");
__device__ __host__ __forceinline__ bool wants_colstat(const WideRule &r, double p) {
  return p >= r.hi || (p > r.near_lo && p <= r.lo);
}
constexpr int kColBlock = 64;       // columns per block of k_ns_colstat (measured: 64 -> 92 us, 256 -> 104 us
                                    // per Qwen3-0.6B step: more blocks beat longer row pieces)
constexpr int kColLanes = kColBlock / 8, kColRowGroups = anc_reduce::kThreads / kColLanes;
constexpr int kColRowStep = 4;      // every fourth row: the thresholds are coarse (a quarter of the proxy; 1.3
                                    // against 1.0 and 1.9+), a quarter of the rows places a matrix as well as all
                                    // of them (flat columns read 1 + 8/M more) and costs a quarter of the bytes
static_assert(kColBlock % 64 == 0 && kColBlock <= anc_reduce::kThreads, "k_ns_colstat: whole wavefronts of one lane per column in the final sum");
struct ColLds {
  double colsum[kColRowGroups][kColBlock], wave_sum[2][kColBlock / 64];
};
// (sum c^2, sum c^4) of a part's columns, for thread 0 of 256
__device__ __forceinline__ void col_part(const uint16_t *X, int M, int N, int part, ColLds &lds, double &t2, double &t4) {
  // lane (rg, cg): columns part*64 + 8*cg .. +7 (one 16-byte load per row), rows 4 rg, 4 (rg + 32), ...
  const int cg = (int)threadIdx.x % kColLanes, rg = (int)threadIdx.x / kColLanes;
  const int j = part * kColBlock + 8 * cg;
  double c[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  if (j < N) {
    const uint16_t *src = X + j;
#pragma unroll 8
    for (int i = kColRowStep * rg; i < M; i += kColRowStep * kColRowGroups) {
      const anc_u32x4 w = *(const anc_u32x4 *)(src + (int64_t)i * N);
      const uint32_t u[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const double x0 = (double)__uint_as_float(u[k] << 16), x1 = (double)__uint_as_float(u[k] & 0xFFFF0000u);
        c[2 * k] = c[2 * k] + x0 * x0;
        c[2 * k + 1] = c[2 * k + 1] + x1 * x1;
      }
    }
  }
#pragma unroll
  for (int k = 0; k < 8; ++k) lds.colsum[rg][8 * cg + k] = c[k];
  __syncthreads();
  if (threadIdx.x < kColBlock) {               // one lane per column: the row groups in order
    double c2 = lds.colsum[0][threadIdx.x];
#pragma unroll
    for (int r = 1; r < kColRowGroups; ++r) c2 = c2 + lds.colsum[r][threadIdx.x];
    const double s2 = anc_wave_sum_f64(c2), s4 = anc_wave_sum_f64(c2 * c2);
    if ((threadIdx.x & 63) == 0) { lds.wave_sum[0][threadIdx.x >> 6] = s2; lds.wave_sum[1][threadIdx.x >> 6] = s4; }
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    t2 = lds.wave_sum[0][0];
    t4 = lds.wave_sum[1][0];
#pragma unroll
    for (int w = 1; w < kColBlock / 64; ++w) { t2 = t2 + lds.wave_sum[0][w]; t4 = t4 + lds.wave_sum[1][w]; }
  }
}
// The wide gate's decision on matrix e, from its proxy's sum and, where that asks for them, the column norms
__device__ __forceinline__ bool is_wide(const WideRule &r, int N, int parts, const double *c, double sum) {
  const double p = sum * (double)N;
  if (p > r.lo && p < r.hi) return true;
  if (!wants_colstat(r, p)) return false;
  double s2 = c[0], s4 = c[1], lightest = c[0];
#pragma unroll 16
  for (int i = 1; i < parts; ++i) {
    const double x2 = c[2 * i], x4 = c[2 * i + 1];
    s2 = s2 + x2;
    s4 = s4 + x4;
    lightest = x2 < lightest ? x2 : lightest;
  }
  const double colc = s2 > 0.0 ? (double)N * s4 / (s2 * s2) : 1.0;
  // outlier columns: the share of the mass outside them, from the lightest block of columns
  const double bulk = s2 > 0.0 ? (double)parts * lightest / s2 : 1.0;
  if (p < r.hi && r.near_diff > 0.0) return p - colc > r.near_diff;
  return colc < kColcFrac * p || (p >= r.hi && bulk < kBulkShare);
}

// The statistics of one matrix as workgroups of 256 threads: kCondParts for the proxy, then one per 64 columns, whether the proxy will
// ask for them or not (nobody knows it yet). The last to arrive decides. `arrived` is 0 before the launch.
struct NsStatOne {
  const uint16_t *Fh, *Xh;
  double *condpart, *cond, *colpart;
  int32_t *flag, *arrived;
  int M, N, parts;
  WideRule rule;
};
__device__ __forceinline__ void stat_block(const NsStatOne &s, int b, void *lds) {
  if (b < kCondParts) {
    const double t = cond_part(s.Fh, s.M, b, (double *)lds);
    if (threadIdx.x == 0) s.condpart[b] = t;
  } else {
    double t2, t4;
    col_part(s.Xh, s.M, s.N, b - kCondParts, *(ColLds *)lds, t2, t4);
    if (threadIdx.x == 0) { s.colpart[2 * (b - kCondParts)] = t2; s.colpart[2 * (b - kCondParts) + 1] = t4; }
  }
  if (threadIdx.x >= 64) return;
  int before = 0;
  if (threadIdx.x == 0) before = __hip_atomic_fetch_add(s.arrived, 1, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
  if (__builtin_amdgcn_readfirstlane(before) != kCondParts + s.parts - 1) return;
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  const double sum = cond_sum(s.condpart);
  if (threadIdx.x == 0) {
    s.cond[0] = sum;
    s.flag[0] = is_wide(s.rule, s.N, s.parts, s.colpart, sum) ? 1 : 0;
  }
}
struct NsStatArgs : NsGemmArgs<1> {
  int tiles_only;            // workgroups before the statistics'
  NsStatOne stat;
};
constexpr int64_t kStatTiles = 256, kStatCols = 12288;       // tiles of a launch that leaves CUs over, columns it reads (measured in ns.hip)
