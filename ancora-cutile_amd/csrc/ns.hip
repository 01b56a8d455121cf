// Batched Newton-Schulz / Polar-Express chain for gfx950.
// Replaces `newton_schulz_resident[_e]` and the kernels they launch
// (ancora/kernels/muon_ns.py:68-174, 245-283, 293-406, 430-468); numpy form
// ancora/optim/muon.py:67-80 and tests/kernels/_probe_polar_express_device.py:27-34.
//
// Per matrix X (M,N), M <= N:  X /= ||X||_F + eps;  steps x { A = X X^T;
//   B = b A + c A A;  X = a X + B X }.
//
// Precision design (bf16 modes). The reference stores X, A and B as bf16 between the
// GEMMs, which leaves it about 6e-3 (relative Frobenius) from the fp32 numpy result.
// Here the iterate is carried between steps as a bf16 pair X = Xh + Xl (Xh = bf16(x),
// Xl = bf16(x - Xh): 16 significant bits, 4 bytes per element like fp32 but directly usable
// as matrix-core operands), and the diagonals of A and B -- the entries that approach 1 and
// b+c while the off-diagonal part goes to zero -- never pass through bf16:
//   A = dA + F    dA = diag(A) kept as an fp32 vector, F = off-diagonal part
//   A A = dA^2 + dA F + F dA + F F       only F F is a matrix-core product (bf16 F)
//   B = dB + Boff                        likewise
//   B X = dB (.) X + Boff X              dB (.) X is an fp32 row scaling in the epilogue
// Xh alone is the matrix-core operand of the early iterations. Where the shape needs it (see
// split_plan below) late iterations add the residual products: A gets Xh Xl^T + Xl Xh^T and
// B X gets Boff Xl as extra accumulation terms of the same tile. The symmetric products are
// "NT" (both operands K-contiguous rows of X or F); B X reads the iterate as (k, n) tiles
// and transposes inside LDS reads, so no transposed copy of X exists. Every matrix the chain
// writes for itself is in panel layout (32-column panels, see NsGemm); the input pair is row-major. The
// fp32 input is read once (normalisation) and the fp32 result written once (last step).
//
// Determinism: one workgroup owns one output tile (64 to 256 wide) and its whole K loop, terms in
// a fixed order, K tiles in ascending order; no split-K. Atomics only count the workgroups of a gate's statistic that are done
// (k_ns_colstat, stat_block): whoever comes last adds the partial sums in their fixed order. A matrix's result
// does not depend on the batch size E or on its position in the batch. Symmetric outputs
// (A, B) are multiplied in the 64x64 blocks on and below the diagonal, whatever the launch's tiles, and mirrored;
// without residual terms that is bit-identical to computing both halves (same products, same order, and an epilogue
// that is symmetric in (i,j)). With residual terms the two cross products Xh Xl^T and
// Xl Xh^T enter one accumulator in a fixed order, so elements computed directly inside a
// diagonal block differ from their mirror images in the last bits; nothing depends on it.
//
// The products run on the tiles of ns_gemm_big.hip (256 wide) and ns_gemm_tile.hip (128 and 64 wide), chosen per
// launch by the number of tiles (pick_tile); the bits are the same on all of them.
#include <algorithm>
#include <cfloat>
#include <vector>

#include "ns_stats.h"
#include "ns_common.h"

namespace {

using namespace anc_reduce;

// ---------------------------------------------------------------- fp32 validation GEMM
// 128x128x16 tiles, v_mfma_f32_32x32x2_f32: every product and every sum in fp32.
constexpr int BM = 128, BN = 128, kGemmThreads = 256;
constexpr int FK = 16, FPITCH = 20, FNPITCH = 132;

struct NsGemmF32 {
  const float *A;          // (E, Mo, K) rows of the output
  const float *B;          // NT: (E, No, K);  NN: (E, K, No)
  int K, nn;
  int64_t strideA, strideB;
  int Mo, No;              // output dims per matrix
  float ca, cb, cc;
  const float *D;          // epilogue operand, same shape as the output (may be null)
  float *out;
  int epi;
};

__global__ void __launch_bounds__(kGemmThreads, 2) k_ns_gemm_f32(NsGemmF32 p) {
  __shared__ __attribute__((aligned(16))) float sA[BM * FPITCH];
  __shared__ __attribute__((aligned(16))) float sB[BM * FPITCH > FK * FNPITCH ? BM * FPITCH : FK * FNPITCH];
  const int tiles_m = p.Mo / BM, tiles_n = p.No / BN;
  const int L = xcd_remap((int)blockIdx.x, (int)gridDim.x);
  const int e = L / (tiles_m * tiles_n), t = L % (tiles_m * tiles_n);
  const int tm = t / tiles_n, tn = t % tiles_n;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int K = p.K;

  f32x16 acc[2][2];
#pragma unroll
  for (int bi = 0; bi < 2; ++bi)
#pragma unroll
    for (int bj = 0; bj < 2; ++bj)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[bi][bj][r] = 0.0f;

  const float *Ae = p.A + (int64_t)e * p.strideA + (int64_t)(tm * BM) * K;
  const float *Be = p.B + (int64_t)e * p.strideB;
  for (int k0 = 0; k0 < K; k0 += FK) {
    // A tile: 128 rows x 16 k, 4 lanes per row
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int row = (tid >> 2) + 64 * i, kq = (tid & 3) * 4;
      *(anc_f32x4 *)&sA[row * FPITCH + kq] = *(const anc_f32x4 *)(Ae + (int64_t)row * K + k0 + kq);
    }
    if (!p.nn) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int row = (tid >> 2) + 64 * i, kq = (tid & 3) * 4;
        *(anc_f32x4 *)&sB[row * FPITCH + kq] =
            *(const anc_f32x4 *)(Be + (int64_t)(tn * BN + row) * K + k0 + kq);
      }
    } else {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int kr = (tid >> 5) + 8 * i, c4 = (tid & 31) * 4;
        *(anc_f32x4 *)&sB[kr * FNPITCH + c4] =
            *(const anc_f32x4 *)(Be + (int64_t)(k0 + kr) * p.No + tn * BN + c4);
      }
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < FK / 2; ++kk) {
      float a[2], b[2];
      const int kx = kk * 2 + (lane >> 5);
#pragma unroll
      for (int bi = 0; bi < 2; ++bi) a[bi] = sA[(wm * 64 + bi * 32 + (lane & 31)) * FPITCH + kx];
#pragma unroll
      for (int bj = 0; bj < 2; ++bj)
        b[bj] = p.nn ? sB[kx * FNPITCH + wn * 64 + bj * 32 + (lane & 31)]
                     : sB[(wn * 64 + bj * 32 + (lane & 31)) * FPITCH + kx];
#pragma unroll
      for (int bi = 0; bi < 2; ++bi)
#pragma unroll
        for (int bj = 0; bj < 2; ++bj)
          acc[bi][bj] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[bi], b[bj], acc[bi][bj], 0, 0, 0);
    }
    __syncthreads();
  }
  const int64_t base = (int64_t)e * p.Mo * p.No;
#pragma unroll
  for (int bi = 0; bi < 2; ++bi)
#pragma unroll
    for (int bj = 0; bj < 2; ++bj)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int gi = tm * BM + wm * 64 + bi * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
        const int gj = tn * BN + wn * 64 + bj * 32 + (lane & 31);
        const int64_t o = base + (int64_t)gi * p.No + gj;
        const float v = acc[bi][bj][r];
        float y;
        if (p.epi == EPI_GRAM)      y = v;
        else if (p.epi == EPI_BMAT) y = p.cb * p.D[o] + p.cc * v;
        else                        y = p.ca * p.D[o] + v;
        p.out[o] = y;
      }
}

// ------------------------------------------------------------------ Frobenius prologue
template <int GD, typename T>
__global__ void __launch_bounds__(kThreads)
k_fro_partials(const T *__restrict__ X, int64_t mn, int nchunks, double *__restrict__ partials) {
  const int64_t e = (int64_t)blockIdx.x / nchunks, c = (int64_t)blockIdx.x % nchunks;
  chunk_partial<GD>((const void *)(X + e * mn), mn, c, partials + blockIdx.x);
}

// One block per matrix: lane t adds partials t, t+256, ... in order; butterfly; 4 wavefronts in order.
// Lane 0 returns the sum of squares.
__device__ __forceinline__ double fro_sum(const double *p, int nchunks) {
  __shared__ double wave_sum[kThreads / 64];
  double acc = 0.0;
  for (int i = threadIdx.x; i < nchunks; i += kThreads) acc = acc + p[i];
  acc = anc_wave_sum_f64(acc);
  if ((threadIdx.x & 63) == 0) wave_sum[threadIdx.x >> 6] = acc;
  __syncthreads();
  double t = wave_sum[0];
#pragma unroll
  for (int w = 1; w < kThreads / 64; ++w) t = t + wave_sum[w];
  return t;
}
__global__ void __launch_bounds__(kThreads)
k_fro_finalize(const double *__restrict__ partials, int nchunks, float eps, float *__restrict__ recip) {
  const double t = fro_sum(partials + (int64_t)blockIdx.x * nchunks, nchunks);
  if (threadIdx.x == 0) recip[blockIdx.x] = 1.0f / ((float)sqrt(t) + eps);
}

// The same for the bf16 pairs of up to kMaxGroups batches in one launch. The first step multiplies the input as it
// is, A = scale^2 * (U U^T), so U has to lie where neither those products nor scale^2 leave the fp32 range: a matrix
// whose sum of squares is outside 2^-100 .. 2^100 is multiplied in place by the power of two 2^k that brings ||U||
// into [1, 2), and its reciprocal carries 2^-k, so the first step sees the same scale*U as without. (Exact but for
// elements 2^-126 of the norm and less, which become subnormal.) Partial sums that are not finite, from runs of
// squares added up in fp32, are replaced by a sum over the matrix itself. One launch instead of two per batch: 7
// batches of a small model took 52 us of launches here.
struct NsPrologue {
  int n;
  int blocks[kMaxGroups];            // matrices per batch
  int nchunks[kMaxGroups];
  const double *partials[kMaxGroups];
  float *recip[kMaxGroups];
  uint16_t *Uh[kMaxGroups], *Ul[kMaxGroups];       // Ul null: a bf16 input without a low half,
  uint32_t *zero16[kMaxGroups];                    // whose substitute this kernel clears
  int32_t *arrived[kMaxGroups];                    // (E) cleared, see NsStatOne
  int64_t mn[kMaxGroups];
};
// Sum of squares of one matrix, every square and sum in fp64: lane t adds the 8-element vectors t, t+256, ... in
// order; butterfly; 4 wavefronts in order. `lo` null: no low half.
__device__ __forceinline__ double pair_sum(const uint16_t *hi, const uint16_t *lo, int64_t mn) {
  __shared__ double wave_sum[kThreads / 64];
  double acc = 0.0;
  for (int64_t o = (int64_t)threadIdx.x * 8; o < mn; o += (int64_t)kThreads * 8)
    for (int i = 0; i < 8; ++i) {
      const double x = (double)anc_bf16_bits_to_f32(hi[o + i]) + (lo == nullptr ? 0.0 : (double)anc_bf16_bits_to_f32(lo[o + i]));
      acc = acc + x * x;
    }
  acc = anc_wave_sum_f64(acc);
  if ((threadIdx.x & 63) == 0) wave_sum[threadIdx.x >> 6] = acc;
  __syncthreads();
  double t = wave_sum[0];
#pragma unroll
  for (int w = 1; w < kThreads / 64; ++w) t = t + wave_sum[w];
  return t;
}
__global__ void __launch_bounds__(kThreads) k_pair_prologue(NsPrologue a, float eps) {
  int e = (int)blockIdx.x, q = 0;
  while (q + 1 < a.n && e >= a.blocks[q]) { e -= a.blocks[q]; ++q; }
  double t = fro_sum(a.partials[q] + (int64_t)e * a.nchunks[q], a.nchunks[q]);
  const int64_t mn = a.mn[q];
  if (!(t <= DBL_MAX)) t = pair_sum(a.Uh[q] + (int64_t)e * mn, a.Ul[q] == nullptr ? nullptr : a.Ul[q] + (int64_t)e * mn, mn);
  int k = 0;
  if (t > 0.0 && t <= DBL_MAX && !(t >= 0x1p-100 && t <= 0x1p100)) k = -ilogb(sqrt(t));
  const float r = 1.0f / ((float)ldexp(sqrt(t), k) + ldexpf(eps, k));       // (of the matrix times 2^k)
  if (threadIdx.x == 0) { a.recip[q][e] = r; a.arrived[q][e] = 0; }
  if (a.Ul[q] == nullptr && e == 0 && threadIdx.x < 4) a.zero16[q][threadIdx.x] = 0u;
  if (k == 0) return;                // (uniform over the block)
  for (int64_t o = (int64_t)threadIdx.x * 8; o < mn; o += (int64_t)kThreads * 8) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (h && a.Ul[q] == nullptr) break;
      uint16_t *p = (h ? a.Ul[q] : a.Uh[q]) + (int64_t)e * mn + o;
      anc_u32x4 w = *(const anc_u32x4 *)p;
      uint32_t u[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float lo = ldexpf(__uint_as_float(u[i] << 16), k), hi = ldexpf(__uint_as_float(u[i] & 0xFFFF0000u), k);
        u[i] = (__float_as_uint(lo) >> 16) | (__float_as_uint(hi) & 0xFFFF0000u);
      }
      *(anc_u32x4 *)p = anc_u32x4{u[0], u[1], u[2], u[3]};
    }
  }
}

// Normalisation X * recip[e]. With Xh == null the fp32 matrix is scaled in place (fp32 chain,
// steps == 0); otherwise X is left alone and the scaled iterate leaves as the bf16 pair
// Xh = bf16(x), Xl = bf16(x - Xh), both (M,N) row-major. 8 elements per lane.
__global__ void __launch_bounds__(kThreads)
k_ns_prep(float *__restrict__ X, const float *__restrict__ recip, int64_t mn, int64_t total8,
          uint16_t *__restrict__ Xh, uint16_t *__restrict__ Xl) {
  const int64_t i8 = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (i8 >= total8) return;
  const int64_t o = i8 * 8;
  const float rc = recip[o / mn];
  const anc_f32x4 x0 = anc_ld_stream((const anc_f32x4 *)(X + o));
  const anc_f32x4 x1 = anc_ld_stream((const anc_f32x4 *)(X + o + 4));
  const float xs[8] = {x0.x * rc, x0.y * rc, x0.z * rc, x0.w * rc, x1.x * rc, x1.y * rc, x1.z * rc, x1.w * rc};
  if (Xh == nullptr) {
    const anc_f32x4 y0 = {xs[0], xs[1], xs[2], xs[3]}, y1 = {xs[4], xs[5], xs[6], xs[7]};
    *(anc_f32x4 *)(X + o) = y0;
    *(anc_f32x4 *)(X + o + 4) = y1;
    return;
  }
  uint32_t h[8], l[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    h[k] = anc_bf16_rne_bits(xs[k]) & 0xFFFFu;
    l[k] = anc_bf16_rne_bits(xs[k] - anc_bf16_bits_to_f32(h[k])) & 0xFFFFu;
  }
  const anc_u32x4 ho = {h[0] | (h[1] << 16), h[2] | (h[3] << 16), h[4] | (h[5] << 16), h[6] | (h[7] << 16)};
  const anc_u32x4 lo = {l[0] | (l[1] << 16), l[2] | (l[3] << 16), l[4] | (l[5] << 16), l[6] | (l[7] << 16)};
  anc_st_stream((anc_u32x4 *)(Xh + o), ho);
  anc_st_stream((anc_u32x4 *)(Xl + o), lo);
}

// ------------------------------------------------------------------ conditioning proxy
// ||offdiag(A)||_F^2 of the first iteration's A = X X^T (||X||_F = 1, so tr A = 1): 1/N for a
// matrix with independent entries whatever its row scaling, N/r - N/M for one whose mass sits
// in r directions that are spread over the rows (outlier columns). Read from Fh (bf16, zero
// diagonal). kCondParts blocks per matrix, each over M*M/kCondParts consecutive elements: lane t
// takes the 8-element vectors t, t+256, ..., adds their squares left to right in fp32, widens to
// fp64; butterfly over the wavefront; the 4 wavefront sums in order. k_ns_colstat and k_ns_classify_order combine the
// kCondParts partial sums by the same butterfly (one wavefront, a part per lane); whichever decides leaves the sum for
// the products to read. (64 parts: a single 1024x1024 matrix in 8 parts took 36 us, latency of a
// few wavefronts.)
struct NsCondArgs {
  int n;
  int blocks[kMaxGroups];
  const uint16_t *Fh[kMaxGroups];
  double *out[kMaxGroups];
  int32_t *arrived[kMaxGroups];      // (E) cleared for k_ns_colstat<true>, or null
  int M[kMaxGroups];
};
__global__ void __launch_bounds__(kThreads) k_ns_cond(NsCondArgs a) {
  __shared__ double wave_sum[kThreads / 64];
  int b = (int)blockIdx.x, q = 0;
  while (q + 1 < a.n && b >= a.blocks[q]) { b -= a.blocks[q]; ++q; }
  const double t = cond_part(a.Fh[q], a.M[q], b, wave_sum);  // b = e * kCondParts + part
  if (threadIdx.x == 0) {
    a.out[q][b] = t;
    if (a.arrived[q] != nullptr && b % kCondParts == 0) a.arrived[q][b / kCondParts] = 0;
  }
}

// ------------------------------------------------------------------ column statistic, classification
// The proxy cannot tell a few huge COLUMNS (N/r of them: 1 % of the columns x100 reads 100 whatever
// N) from a low-rank signal over weak noise (rank 32: N/32), and the two need different plans: the
// first meets the bar with the cheap gates, the second only with every residual term (rank 32 plus
// 10 % noise at 1024x2048: 2.9e-3 against 1.4e-4). What separates them is where the mass sits among
// the columns: colc = N * sum_j c_j^4 / (sum_j c_j^2)^2 over the column norms c_j of the input
// (taken over every fourth row) is N/r for r outlier columns (equal to the proxy) and 1.0 .. 1.5
// for anything rotationally spread.
// The same statistic separates, just below the band, scaled columns (colc = proxy: the low gate
// suffices) from a spectrum with a gap (colc = 1: near-duplicate rows, 2.4e-3 at 1024x1024 without
// the wide gate's terms, 4.6e-4 with).
// k_ns_colstat: one block per 64 columns of a matrix; 8 lanes cover a 128-byte row piece with
// 16-byte loads, the 32 row groups walk the M rows (fp64 sums of squares: the pair entries run on
// unnormalised input) and are added in order through LDS; the block leaves (sum c^2, sum c^4) of
// its columns (one wavefront's butterfly). A block returns at
// once unless the matrix's proxy asks for the statistic. Then the partial sums are added in order and the flag is written that
// every later product reads: DECIDE, by the matrix's first block where nobody asks and by the last to arrive where it does;
// otherwise by k_ns_classify_order, for batches that a gated launch takes in another order. (A launch of its own, one wavefront per
// matrix, was almost all start and end. Keller's coefficients, us per chain with it / without, every matrix asking: 1 x (1536,1536) 323.3 /
// 320.0, 3 x (1024,1024) 270.3 / 266.9, 2 x (1024,3072) 385.5 / 382.0, 16 x (1024,1024) 907.0 / 906.2, 28 x (1024,3072) 3303 / 3310, 48 x (1024,1024) 2330 /
// 2331: from 16 matrices on level, although each of the asking blocks releases and acquires at the agent's scope.)
__device__ __forceinline__ int anc_wave_sum_i32(int v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}
// First of E matrices in run x of the eight that a launch's sequence is cut into
__device__ __forceinline__ int anc_run_start(int x, int E) { return (int)(((int64_t)x * E + kXcds - 1) / kXcds); }
struct NsColArgs {
  int n;
  int blocks[kMaxGroups];          // colstat: E * parts, classify: E
  double *sum[kMaxGroups];         // (E) the proxy's sum, for the products to read
  const uint16_t *Xh[kMaxGroups];  // (E, M, N) row-major
  const double *cond[kMaxGroups];  // (E, kCondParts)
  double *part[kMaxGroups];        // (E, parts, 2)
  int32_t *flag[kMaxGroups];       // (E) or null (no wide gate)
  int32_t *order[kMaxGroups];      // (E) or null
  int32_t *arrived[kMaxGroups];    // (E) blocks of k_ns_colstat<true> whose partial sums are written
  double gate[kMaxGroups];         // matrices whose sum exceeds it take a gate's terms some time
  int M[kMaxGroups], N[kMaxGroups], parts[kMaxGroups];
  WideRule rule[kMaxGroups];
};
__device__ __forceinline__ bool wide_at(const NsColArgs &a, int q, int e, double sum) {
  return is_wide(a.rule[q], a.N[q], a.parts[q], a.part[q] + (int64_t)e * a.parts[q] * 2, sum);
}
template <bool DECIDE>
__global__ void __launch_bounds__(kThreads) k_ns_colstat(NsColArgs a) {
  __shared__ ColLds lds;
  int b = (int)blockIdx.x, q = 0;
  while (q + 1 < a.n && b >= a.blocks[q]) { b -= a.blocks[q]; ++q; }
  const int e = b / a.parts[q], part = b % a.parts[q];
  const int M = a.M[q], N = a.N[q];
  const double sum = cond_sum(a.cond[q] + (int64_t)e * kCondParts);
  if (!wants_colstat(a.rule[q], sum * (double)N)) {
    if (DECIDE && part == 0 && threadIdx.x == 0) {
      a.sum[q][e] = sum;
      a.flag[q][e] = wide_at(a, q, e, sum) ? 1 : 0;
    }
    return;
  }
  double t2, t4;
  col_part(a.Xh[q] + (int64_t)e * M * N, M, N, part, lds, t2, t4);
  if (threadIdx.x == 0) {
    double *out = a.part[q] + ((int64_t)e * a.parts[q] + part) * 2;
    out[0] = t2;
    out[1] = t4;
    if constexpr (DECIDE) {
      if (__hip_atomic_fetch_add(a.arrived[q] + e, 1, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) == a.parts[q] - 1) {
        a.sum[q][e] = sum;
        a.flag[q][e] = wide_at(a, q, e, sum) ? 1 : 0;
      }
    }
  }
}
// One block per batch: the wide gate's flag per matrix, and the order in which the launches of a gated
// iteration take the matrices. A matrix that takes a gate's terms has three times the products of one that does not;
// such matrices lie together (the tall weights of a stack) and a launch's sequence is cut into eight runs, one per XCD,
// so they are dealt over the runs in turn, each run's first. (Qwen3-0.6B set, 59 of 196 matrices gated, A = X X^T of
// iteration 2: 1114 -> 729 us, for 1 to 3 us.)
constexpr int kClassifyThreads = 1024, kMaxOrdered = 8192;
__global__ void __launch_bounds__(kClassifyThreads) k_ns_classify_order(NsColArgs a) {
  constexpr int kWaves = kClassifyThreads / 64, kAhead = 4;
  __shared__ uint8_t heavy[kMaxOrdered];
  __shared__ int count[kWaves];
  const int q = (int)blockIdx.x, E = a.blocks[q], wave = (int)(threadIdx.x >> 6), lane = (int)(threadIdx.x & 63);
  for (int e0 = wave; e0 < E; e0 += kWaves * kAhead) {
    double parts[kAhead];
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      const int e = e0 + i * kWaves;
      parts[i] = e < E ? a.cond[q][(int64_t)e * kCondParts + lane] : 0.0;
    }
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      const int e = e0 + i * kWaves;
      if (e >= E) break;
      const double sum = anc_wave_sum_f64(parts[i]);
      if (lane == 0) a.sum[q][e] = sum;
    }
  }
  __syncthreads();
  for (int e = (int)threadIdx.x; e < E; e += kClassifyThreads) {      // (a matrix per lane)
    const double sum = a.sum[q][e];
    const bool wide = a.flag[q] != nullptr && wide_at(a, q, e, sum);
    if (a.flag[q] != nullptr) a.flag[q][e] = wide ? 1 : 0;
    if (e < kMaxOrdered) heavy[e] = wide || sum > a.gate[q] ? 1 : 0;
  }
  __syncthreads();
  int32_t *order = a.order[q];
  if (order == nullptr) return;
  if (E > kMaxOrdered) {
    for (int e = (int)threadIdx.x; e < E; e += kClassifyThreads) order[e] = e;
    return;
  }
  int mine = 0;
  for (int e = (int)threadIdx.x; e < E; e += kClassifyThreads) mine += heavy[e];
  mine = anc_wave_sum_i32(mine);
  if (lane == 0) count[wave] = mine;
  __syncthreads();
  int n_heavy = 0;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) n_heavy += count[w];
  const int f = E / kXcds;                                            // every run begins with a matrix in f places or f + 1
  int before = 0;                                                     // heavy ones of the chunks before
  for (int at = 0; at < E; at += kClassifyThreads) {
    const int e = at + (int)threadIdx.x;
    const bool h = e < E && heavy[e] != 0;
    const uint64_t m = __ballot(h);
    __syncthreads();
    if (lane == 0) count[wave] = __popcll(m);
    __syncthreads();
    int hb = before + __popcll(m & ((1ull << lane) - 1));
    for (int w = 0; w < kWaves; ++w) { hb += w < wave ? count[w] : 0; before += count[w]; }
    if (e >= E) continue;
    const int s = h ? hb : n_heavy + (e - hb);                        // its place among all, heavy ones first
    int x = s % kXcds, y = s / kXcds;
    if (s >= kXcds * f) {                                             // the runs with one more, in turn
      int left = s - kXcds * f;
      y = f;
      for (x = 0; x < kXcds; ++x)
        if (anc_run_start(x + 1, E) - anc_run_start(x, E) > f && left-- == 0) break;
    }
    order[anc_run_start(x, E) + y] = e;
  }
}

// ------------------------------------------------------------------------- workspace
struct Carve {
  uint64_t base;
  int64_t off = 0;
  explicit Carve(uint64_t b) : base(b) {}
  template <typename T> T *take(int64_t count) {
    T *p = (T *)(base + (uint64_t)off);
    off += (count * (int64_t)sizeof(T) + 255) / 256 * 256;
    return p;
  }
};

// Which iterations carry bf16 residual operands. Rounding X to bf16 costs about 1e-3 of
// relative Frobenius error per late iteration on square Gaussian inputs (less on wide
// ones, more on small ones); measured against the fp32 numpy chain, 5 Polar-Express steps:
//   no residuals         1024x1024 2.2e-3   1024x2048 1.4e-3   1024x3072 1.2e-3   256x256 2.8e-3
//   X in the last two    1024x1024 1.4e-3                                         256x256 2.4e-3
//   X, F, B in last three 1024x1024 7e-5                                          256x256 3e-4
// The plan depends on (M, N, steps) only, never on the batch.
struct SplitPlan {
  int x_from;    // first iteration whose A and B X products add the residual of X for every matrix
  int fb_from;   // first iteration whose A A and B X products add the residuals of F and Boff
  // Conditioning gates. In iteration k < x_from with gate_tau[k] > 0, a matrix whose proxy
  // N * ||offdiag(A0)||_F^2 exceeds gate_tau[k] adds the residual of X to A = X X^T and, with bit k
  // of gate_bx set, to X = a X + B X as well.
  static constexpr int kGateIters = 8;
  float gate_tau[kGateIters];
  unsigned gate_bx;
  // The wide gate: a matrix whose proxy lies in (wide_lo, wide_hi), or outside it with a column
  // statistic that says so (is_wide), adds the residual of X to A = X X^T from iteration
  // wide_gram_from on and the residuals of X, F and Boff to all three products from iteration
  // wide_all_from on. wide_hi == 0: no such gate.
  float wide_lo, wide_hi, wide_near;   // wide_near: start of the near range below the band (== wide_lo: none)
  float wide_near_diff;                // see WideRule::near_diff
  int wide_gram_from, wide_all_from;
  // No fp32 copy of A except for the matrices the wide gate flags: B = b A + c A A takes the
  // off-diagonal entries of A from the bf16 Fh it multiplies anyway. Costs 3 .. 8 % of accuracy where
  // N >= 2M (independent entries 1.36e-3 -> 1.41e-3 at 1024x2048 and 1.16e-3 -> 1.20e-3 at 1024x3072,
  // 1 % of the columns x100 1.58e-3 -> 1.66e-3 and 1.15e-3 -> 1.24e-3) and saves 6 of the 13 bytes
  // per element of A an iteration moves; N < 2M keeps the copy (the column-scaled probe input at
  // 1024x1024 would go from 1.85e-3 to 2.10e-3).
  bool drop_a32;
  // The low half of the iterate as one byte per element wherever it is never a matrix-core operand
  // (NsGemm::l8_in): the matrices that take no gate, and for a gated one every iterate but those its
  // gated products read. 3 instead of 4 bytes per element read and written by X = a X + B X; the
  // numpy model of this chain puts the cost at the fourth digit (1.4077e-3 -> 1.4074e-3 at
  // 1024x2048, 1.1997e-3 -> 1.1985e-3 at 1024x3072). The result itself moves by 1.2e-3: the chain
  // turns any perturbation of its iterate, this one of 2^-16 per element included, into another
  // realisation of its own rounding error (an exact low half moves it as far). Measured: X = a X +
  // B X 4.85 -> 4.69 ms per step of Qwen3-0.6B, 2.0 GB less HBM traffic.
  bool low8;
  bool gated(int k) const { return k >= 0 && k < kGateIters && k < x_from && gate_tau[k] > 0.0f; }
  bool wide() const { return wide_hi > 0.0f; }
  bool wide_gram(int k) const { return wide() && k >= wide_gram_from && k < x_from; }
  bool wide_all(int k) const { return wide() && k >= wide_all_from && k < fb_from; }
  bool any_gate(int steps) const {
    if (wide()) return true;
    for (int k = 0; k < steps; ++k) if (gated(k)) return true;
    return false;
  }
};
// The proxy is 1.0 for a matrix with independent entries whatever its row scaling (1.2 with 1 %
// of the rows x100), 1.7 for columns scaled over 0.1..3, about 100 with 1 % of the columns x100.
//   kTauHard: inputs whose Frobenius mass sits in a few directions spread over all rows (a
//     gradient with a few outlier columns: the transposed iterate of a tall weight with outlier
//     rows). Rounding X to bf16 then costs the small directions their signal in A = X X^T while the
//     large ones converge: 1% of the columns x100 gives 2.2e-3 at 1024x3072 and 3.8e-3 at
//     1024x1024 without the extra terms of iterations 1-2, 1.2e-3 and 8e-4 with them. Row outliers,
//     whose mass lands on the exact fp32 diagonal of A, need nothing (5e-4 .. 7e-4).
//   kTauPlain: N < 2M runs the residual of X in both X-products of the last two iterations; a
//     matrix with independent entries needs them in the last one only (1.66e-3 against 1.41e-3 at
//     1024x1024, 5.3e-4 either way with outlier rows), the column-scaled case needs both (1.85e-3
//     against 2.09e-3). So the first of the two is gated low. Between the two thresholds square
//     matrices were still within 4 % of the bar (columns scaled over 0.03..3, proxy 1.79: 1.93e-3;
//     log-normal column scales, sigma 0.45, proxy 2.2: 1.79e-3), so iteration 2 carries the same
//     two terms behind the same gate: 1.48e-3 and 1.25e-3.
//   kTauWideLo .. kTauWideHi: inputs whose spectrum is spread over decades, or with many moderately
//     large columns. Measured proxies (1024x1024 / 1024x3072): log-uniform spectrum over one decade
//     1.4 / 4.0, 1.5 decades 2.4 / 7.4, two 3.6 / 11.3, three 5.8 / 19.4; 10 % of the columns x10 8.4;
//     against 1 % of the columns x100 100, x1000 102, a rank-32 signal over noise 32 / 95, a
//     power-law spectrum 146 / 437. In the band the plan above leaves 2.5e-3 .. 4.2e-3 (every operand
//     rounding of the later iterations counts: the small singular values are still far from 1);
//     with all residuals in all products from iteration 2 on 1.0e-4 .. 4.8e-4, from iteration 1 on
//     (what runs) 2e-5 .. 8e-5. Above the band the gates above suffice for outlier columns (8e-4 ..
//     1.4e-3; only outliers x1000 miss the bar, with or without these terms at 1024x1024).
//   Outside the band the column statistic decides (k_ns_colstat): a matrix whose column
//     concentration explains less than kColcFrac of its proxy is not a matrix of outlier or scaled
//     columns. Above the band that is a low-rank signal over weak noise or a steep spectrum, alone
//     or mixed with outlier columns (rank 32 + 10 % noise at 1024x2048 / 1024x3072, proxy 65 / 97:
//     2.9e-3 with the gates above, 1.4e-4 with the wide gate's terms; + 1 % noise 5.0e-3 -> 2.5e-4);
//     just below it (kTauWideNear .. kTauWideLo, N < 2M only) a gap in the spectrum with flat
//     column norms (a fraction of near-duplicate rows: proxy 1.55 / 1.7 / 1.8 / 2.0 gives 1.44e-3 /
//     1.74e-3 / 1.98e-3 / 2.4e-3 with the low gate, 3e-5 .. 5e-5 with these terms), while scaled
//     columns (concentration = proxy) stay with the low gate.
//   The wide gate's terms start at iteration 1: from iteration 2 the low-rank cases above stay at
//     1.5e-3 .. 2.7e-3.
//   N >= 2M carries no residual term in its plan and has no low gate: an input whose spectrum has
//     a gap with flat column norms (a fraction of near-duplicate rows, proxy 1 + twice that fraction
//     times N/M) would leave the bar between proxy 1.2 and the band: 1024x2048 reads 1.80e-3 at
//     proxy 1.15, 2.15e-3 at 1.3, 2.8e-3 at 1.6, 4.6e-3 at 2.3 (1024x3072: 1.57e-3, 1.91e-3, 2.5e-3,
//     3.7e-3) with the plan alone. What decides is the part of the proxy the column norms do not
//     explain: with the columns of such a matrix scaled by exp(sigma z), sigma 0 .. 0.4 (proxy up to
//     2.5), the error stays a function of proxy - colc alone (0.10: 1.67e-3 .. 1.76e-3, 0.19: 1.90e-3
//     .. 1.94e-3, 0.29: 2.12e-3 .. 2.15e-3, 0.5: 2.5e-3 .. 2.6e-3 at 1024x2048), where the ratio
//     colc / proxy moves from 0.78 to 0.87. So the near range of these shapes starts at
//     kTauWideNear2M and takes a matrix with proxy - colc > kNearDiff2M (the wide gate's terms: 1e-5
//     .. 5e-5). Independent entries, outlier rows, scaled or outlier columns and heavy tails read
//     proxy - colc < 0.01. (A cheaper gate for the range -- the residual of X in both X-products of
//     iterations 2 .. 4, 6e-4 .. 1.4e-3 in the numpy model of this chain -- was built and taken out
//     again: a GPU fault in the test run that carried it, cause not found.)
constexpr float kTauWideNear2M = 1.15f, kNearDiff2M = 0.15f;
constexpr float kTauHard = 2.5f, kTauPlain = 1.3f, kTauWideLo = 2.5f, kTauWideHi = 40.0f, kTauWideNear = 1.5f;
SplitPlan split_plan(int64_t M, int64_t N, int mode, int steps) {
  SplitPlan sp{};
  sp.x_from = sp.fb_from = steps;
  if (mode == ANC_NS_BF16_X3) {
    // every product with the residuals of both operands' bf16 roundings, in every iteration:
    // about 1e-5 on every input tried, three times the matrix-core work
    sp.x_from = sp.fb_from = 0;
    return sp;
  }
  if (mode == ANC_NS_BF16_LATE3 && M >= 1024) {
    // For coefficients that do not drive the singular values to 1 (Keller's quintic leaves them in
    // 0.7 .. 1.2, so offdiag(A) never becomes small and every operand rounding stays first-order:
    // the gated plan below gives 3.7e-3 at 1024x1024 and 2.8e-3 at 1024x3072 there). Every matrix,
    // no gates of its own: the residual of X from iteration 2 on, those of F and Boff from
    // iteration 3 on. All three from iteration 2: 6e-5 / 3e-5 for 2.2 times the plain chain; all
    // three in the last two iterations only: 2.2e-3 at 1024x1024. M < 1024 runs a heavier plan
    // in either mode (below).
    // From a fixed iteration on whatever the chain's length (Keller's iterates do not settle, so a
    // longer chain keeps adding first-order roundings: with the last three iterations only, 6 steps
    // gave 3.1e-3 and 8 steps 8.9e-3 at 1024x1024), and the last three of a shorter one.
    sp.x_from = sp.fb_from = steps >= 5 ? 2 : (steps > 3 ? steps - 3 : 0);
    // The residuals of F and Boff can start one iteration after that of X: 8e-4 at 1024x1024
    // (independent entries, scaled columns, outlier columns alike) and 4e-4 .. 7.5e-4 at 1024x3072
    // for 2.05 instead of 2.2 times the plain chain's work. (F and Boff first and X later, or the
    // last two iterations only: 2.0e-3 .. 2.3e-3.)
    if (steps >= 5) sp.fb_from = sp.x_from + 1;
    // and the matrices the wide gate flags (below) start one iteration earlier, as they do under
    // Polar Express: a rank-32 signal over 1 % noise is 2.1e-3 at 1024x1024 with the terms from
    // iteration 2 and 3e-4 from iteration 1
    if (sp.x_from > 1) {
      sp.wide_lo = kTauWideLo; sp.wide_hi = kTauWideHi;
      sp.wide_near = N < 2 * M ? kTauWideNear : kTauWideLo;
      sp.wide_gram_from = 1; sp.wide_all_from = 1;
    }
    return sp;
  }
  if (mode != ANC_NS_BF16 && mode != ANC_NS_BF16_LATE3) return sp;
  // The first iterations are insensitive (the singular values are still far below 1, so
  // B X is a small correction to a X); residuals start at a fixed iteration index.
  if (M >= 1024) {
    sp.drop_a32 = mode == ANC_NS_BF16 && N >= 2 * M;
    sp.low8 = sp.drop_a32;
    if (steps >= 2) {                         // terms from iteration 1 to the end, whatever the length
                                              // (cond 1e3 without: 6 steps 4.4e-3 .. 7e-3, 8 steps 6e-3 .. 1.8e-2)
      sp.wide_lo = kTauWideLo; sp.wide_hi = kTauWideHi;
      sp.wide_near = N < 2 * M ? kTauWideNear : kTauWideLo;
      if (mode == ANC_NS_BF16 && N >= 2 * M) { sp.wide_near = kTauWideNear2M; sp.wide_near_diff = kNearDiff2M; }
      sp.wide_gram_from = 1; sp.wide_all_from = 1;
    }
    if (N < 2 * M) {
      sp.x_from = steps - 2 < 3 ? steps - 2 : 3;
      sp.gate_tau[1] = sp.gate_tau[2] = kTauHard;
      if (steps == 5) {                       // the schedule the low gate was measured on
        sp.gate_tau[2] = sp.gate_tau[3] = kTauPlain;
        sp.gate_bx = (1u << 2) | (1u << 3);
        sp.x_from = 4;
      }
    } else {
      // N >= 2M: iteration 2 alone (1 % of the columns x100 without it: 1024x2048 1.6e-3 .. 1.7e-3,
      // 1024x2560 1.8e-3, 1536x3072 2.1e-3, 1024x3072 2.2e-3, 2048x4096 2.2e-3, 4096x8192 2.3e-3;
      // with it 1.0e-3 .. 1.2e-3). One rule for every such shape.
      sp.gate_tau[2] = kTauHard;
      // a chain shorter than the 5 steps this was measured on ends before iteration 2's term has
      // paid off (3 steps at 1024x3072: 2.3e-3, 2 steps 2.7e-3): iteration 1 as well
      if (steps < 5) sp.gate_tau[1] = kTauHard;
    }
  } else {
    // Small matrices average fewer rounding errors per element and cost next to nothing: all
    // residuals from iteration 1 on, from iteration 0 below M = 256, no gates. With them from
    // iteration 2 (relative Frobenius error, Polar Express / Keller): 128x128 condition number 1e3
    // 4.0e-3 / 2.8e-3, columns scaled 0.1..3 under Keller 2.5e-3, 128x384 and 256x512 condition
    // number 1e3 5.5e-3 / 4.0e-3 and 2.4e-3 / 1.8e-3, 512x1024 with 1 % of the columns x100
    // 4.4e-3; from iteration 1: at most 1.0e-3 on all of these from M = 256 on; 128x128 with one
    // column x100 still 4.8e-3, 1e-5 from iteration 0.
    const int from = M < 256 ? 0 : 1;
    sp.x_from = sp.fb_from = steps - 3 < from ? steps - 3 : from;
  }
  if (sp.x_from < 0) sp.x_from = 0;
  if (sp.fb_from < 0) sp.fb_from = 0;
  return sp;
}

struct Plan {
  int nchunks;
  bool split;
  SplitPlan sp;
  uint16_t *Fl, *Bl;
  double *partials;
  float *recip;
  uint32_t *zero16;      // 16 zero bytes: the low half of a bf16 input
  anc_muon_desc_t *desc; // one weight's descriptor (anc_muon_resident_step)
  double *condpart;      // (E, kCondParts) partial sums of the conditioning proxy, bf16 modes
  double *cond;          // (E) the proxy
  double *colpart;       // (E, col_parts, 2) column statistic, plans with a wide gate
  int32_t *wide_flag;    // (E) the wide gate's decision
  int32_t *order;        // (E) the order of the matrices in launches with gated products
  int col_parts;
  // bf16 modes
  uint16_t *Xh[2], *Xl[2];
  float *A32, *dA, *dB;
  uint16_t *Fh, *Bh;
  // fp32 mode
  float *Af, *Bf, *Yf;
  int64_t bytes;
};

Plan make_plan(uint64_t base, int64_t E, int64_t M, int64_t N, int mode, int steps) {
  Plan pl{};
  Carve c(base);
  pl.nchunks = (int)((M * N + ANC_GN_CHUNK - 1) / ANC_GN_CHUNK);
  pl.sp = split_plan(M, N, mode, steps);
  pl.split = pl.sp.x_from < steps;
  pl.partials = c.take<double>(E * ((M * N + 4095) / 4096));   // (the momentum kernel's blocks; chunks are twice as long)
  pl.zero16 = c.take<uint32_t>(4);
  pl.desc = c.take<anc_muon_desc_t>(1);
  pl.recip = c.take<float>(E);
  if (mode == ANC_NS_FP32) {
    pl.Af = c.take<float>(E * M * M);
    pl.Bf = c.take<float>(E * M * M);
    pl.Yf = c.take<float>(E * M * N);
  } else {
    for (int i = 0; i < 2; ++i) {
      pl.Xh[i] = c.take<uint16_t>(E * M * N);
      pl.Xl[i] = c.take<uint16_t>(E * M * N);
    }
    pl.A32 = c.take<float>(E * M * M);
    pl.Fh = c.take<uint16_t>(E * M * M);
    pl.Bh = c.take<uint16_t>(E * M * M);
    if (pl.sp.fb_from < steps || pl.sp.wide()) {
      pl.Fl = c.take<uint16_t>(E * M * M);
      pl.Bl = c.take<uint16_t>(E * M * M);
    }
    pl.dA = c.take<float>(E * M);
    pl.dB = c.take<float>(E * M);
    pl.condpart = c.take<double>(E * kCondParts);
    pl.cond = c.take<double>(E);
    pl.order = c.take<int32_t>(E);
    if (pl.sp.wide()) {
      pl.col_parts = (int)((N + kColBlock - 1) / kColBlock);
      pl.colpart = c.take<double>(E * pl.col_parts * 2);
      pl.wide_flag = c.take<int32_t>(E);
    }
  }
  pl.bytes = c.off;
  return pl;
}

constexpr int kTileFlags = ANC_NS_TILE128 | ANC_NS_FORCE_T64 | ANC_NS_FORCE_T128 | ANC_NS_FORCE_T256;

int check_shape(int64_t E, int64_t M, int64_t N, int mode, const char *who) {
  ANC_REQUIRE(E > 0 && M > 0 && N > 0, "%s: E, M, N must be positive", who);
  ANC_REQUIRE(M % 128 == 0 && N % 128 == 0, "%s: (M,N)=(%lld,%lld) must be multiples of 128", who,
              (long long)M, (long long)N);
  ANC_REQUIRE(M <= N, "%s: M=%lld > N=%lld; pass tall matrices transposed", who, (long long)M,
              (long long)N);
  ANC_REQUIRE(mode == ANC_NS_BF16 || mode == ANC_NS_FP32 || mode == ANC_NS_BF16_FAST || mode == ANC_NS_BF16_X3 ||
                  mode == ANC_NS_BF16_LATE3,
              "%s: unknown mode %d", who, mode);
  ANC_REQUIRE(E * (M / 128) * (N / 128) < (1ll << 30) && E * M * N < (1ll << 40),
              "%s: batch too large", who);
  return ANC_OK;
}

void add_prologue(NsPrologue &a, const Plan &pl, uint64_t Uh, uint64_t Ul, uint64_t fro, int64_t n_partials, int64_t E,
                  int64_t mn) {
  const int q = a.n++;
  a.blocks[q] = (int)E;
  a.nchunks[q] = (int)n_partials;
  a.partials[q] = (const double *)fro;
  a.recip[q] = pl.recip;
  a.Uh[q] = (uint16_t *)Uh;
  a.Ul[q] = (uint16_t *)Ul;
  a.zero16[q] = pl.zero16;
  a.arrived[q] = pl.order;
  a.mn[q] = mn;
}
int launch_prologue(const NsPrologue &a, float eps, hipStream_t s) {
  int64_t blocks = 0;
  for (int q = 0; q < a.n; ++q) blocks += a.blocks[q];
  ANC_REQUIRE(blocks < (1ll << 31), "Newton-Schulz chain: too many matrices");
  AncProfScope prof(ANC_PROF_NS_FRO, s);
  hipLaunchKernelGGL(k_pair_prologue, dim3((unsigned)blocks), dim3(kThreads), 0, s, a, eps);
  ANC_LAUNCH_CHECK();
  return ANC_OK;
}

// One problem of a chain launch: a batch of E (M,N) matrices with its workspace plan.
struct ChainProb {
  Plan pl;
  const uint16_t *inH, *inL;   // the input bf16 pair
  int nxt;                     // which pair of the plan receives the first step's output
  const float *scale0;         // per-matrix factor the first step applies to its input, or null
  float *X32;                  // fp32 result (may overlay the input pair when steps >= 2)
  uint16_t *X16;               // or bf16 result (may overlay inH when steps >= 2)
  int64_t E, M, N;
  const anc_muon_desc_t *upd;  // or: the weights (E entries) the last step updates in its epilogue
};

// Tiles of a launch, from the number of tiles it has (symmetric products: those on and below the diagonal), problems
// weighted by their K against the longest (a launch ends with its longest tiles; short ones fill gaps). A CU takes
// operand bytes into LDS at one rate whatever the tile, so small tiles finish first while they find idle CUs and lose,
// by the bytes they fetch more often, once every CU has several; large ones lose where the last of them have the chip
// to themselves. With residual terms a K tile brings three products, so small tiles hold out longer, and what counts
// is how many rounds the 128-wide ones make: one per CU (symmetric products) or two (X = a X + B X), or just over that.
// Measured, us per chain with the product on 64 / 128 / 256-wide tiles (tiles of 64, of 128):
//   A and B, mostly one term       3 x (1024,1024) 238 / 261 / 424 (408, 108), 4 x 291 / 280 / 440 (544, 144), 10 x 527 / 503 / 572
//               (1360, 360), 14 x (1024,2048) 901 / 791 / 853 (1904, 504), 16 x (1024,1024) 755 / 704 / 686 (2176, 576)
//   residual terms                 16 x (512,1536) 444 / 458 (576, 160), 20 x 544 / 542 (720, 200), 14 x (640,1792) 655 / 615
//               (770, 210), 16 x (640,640) 407 / 386 (880, 240), 9 x (896,896) 514 / 492 (945, 252), 18 x (640,1792) 773 / 849
//               (990, 270), 16 x (768,768) 559 / 588 (1248, 336), 24 x (640,640) 540 / 531 (1320, 360), 20 x (768,768) 672 / 639
//               (1560, 420)
//   just over one round of 256-wide tiles    26 x (1024,1024) 393 / 334 / 387 (5 launches alone; 260 of them), 48 x (768,768)
//               555 / 465 / 522 (288), 33 x (1024,1024) 520 / 449 / 437 (330)
//   X = a X + B X, mostly one term 1 x (1024,2048) 163 / 171 (512, 128), 1 x (1536,1536) 281 / 275 (576, 144), 1 x (1024,3072) 199 /
//               193 (768, 192), 3 x (1152,1152) 307 / 290 (972, 243), 5 x (1024,1024) 313 / 309 /
//               326 (1280, 320), 6 x (1024,2048) 437 / 395 / 401 (3072, 768), 14 x (1024,1024) 653 / 595 / 584
//               (3584, 896), 8 x (1024,2048) 596 / 528 / 506 (4096, 1024)
//   residual terms                 12 x (640,640) 329 / 334 (1200, 300), 6 x (896,896) 389 / 401 (1176, 294), 24 x (512,512) 345 / 338 /
//               381 (1536, 384), 12 x (768,768) 459 / 435 / 492 (1728, 432), 30 x (384,768) 346 / 353 (2160, 540), 24 x (640,640)
//               549 / 530 (2400, 600), 16 x (512,1536) 476 / 441 / 483 (3072, 768), 24 x 647 / 605 / 682 (4608, 1152), 30 x 809 /
//               777 / 799 (5760, 1440), 24 x (768,1536) 1324 / 1145 / 1147 (6912, 1728)
//   just over one round of large tiles       18 x (1024,1024) 811 / 774 / 786 (4608), 20 x 890 / 825 / 809 (5120)
//   with the update of the weight, the whole step of one: (1024,2048) 167.5 / 172.2 (512), (1024,2304) 185.7 / 182.2 (576), (1536,1536) 279.8 /
//               285.1 (576), (1024,2560) 191.0 / 187.0, (1280,2048) 221.5 / 225.5 (640), (1280,2304) 230.4 / 235.3 (720), (1024,3072) 199.8 /
//               200.1 (768), (1024,3328) 210.1 / 207.0 (832): level to 2 % from 512 to 832 tiles, and one line in between
// What the lines and the 64x64 blocks on the diagonal, with a second store below them, cost against earlier lines and whole
// 256-wide blocks: batches of (128,128) 1 .. 3.5 % (12: 77.8 -> 80.5, 40: 82.4 -> 84.3, 100: 121.0 -> 124.2), 4 x (256,256) 87.8 -> 89.1. Launches
// of 257 .. 330 workgroups are level on one card and 1 .. 5 % slower on another (28 x (256,256) 137.4 -> 136.9, 130.6 -> 137.2; 14 x (384,384) 163.7 ->
// 161.9, 153.8 -> 155.8; 8 x (512,512) 174.8 -> 175.9, 160.8 -> 165.0). The rest gains (20 x (256,256) 125.7 -> 110.8, 60 x (512,512) 767 -> 757,
// 20 x (1024,1024) 871 -> 827; 565 batches of 1 .. 60 matrices of 23 shapes 5.7 % in the mean).
int pick_tile(int epi, const NsGemm *ps, const int64_t *Es, int n) {
  double longest = 0.0, t64 = 0.0, t128 = 0.0, t256 = 0.0, several = 0.0;
  for (int k = 0; k < n; ++k) longest = ps[k].K > longest ? (double)ps[k].K : longest;
  for (int k = 0; k < n; ++k) {
    const double m = (double)(ps[k].M / 64), h = (double)(ps[k].M / 128), q = (double)ps[k].M / 256.0;
    const double w = (double)Es[k] * ((double)ps[k].K / longest);
    const double t = w * (epi == EPI_BX ? m * (double)(ps[k].N / 64) : m * (m + 1.0) / 2.0);
    t64 += t;
    t128 += epi == EPI_BX ? t / 4.0 : w * (h * (h + 1.0) / 2.0);
    t256 += w * (q * (q + 1.0) / 2.0);
    if (ps[k].nterms > 1) several += t;
  }
  const bool terms = several > 0.5 * t64;
  if (epi != EPI_BX) {
    if (terms ? t128 <= 205.0 || (t128 > 256.0 && t128 <= 345.0) : t64 <= 520.0) return 64;
    return t64 <= 2050.0 || (t256 > 256.0 && t256 <= 306.0) ? 128 : 256;
  }
  if (terms ? t128 <= 345.0 || (t128 > 512.0 && t128 <= 580.0) : t64 <= (ps[0].upd != nullptr ? 780.0 : 540.0)) return 64;
  return t64 <= (terms && longest < 1024.0 ? 7000.0 : 3500.0) || (t64 > 4096.0 && t64 <= 4900.0) ? 128 : 256;
}

// The same for the bare product of weight gradients. Its K is a batch of tokens: short ones are bound by the
// output, which small tiles spread best, long ones by operands that leave the L2; and a launch lasts as long as the CU with
// the most tiles, of which it takes three 64-wide or 128x64 ones at once, two 128-wide, one 256-wide. Measured, us on tiles of
// 64 / 128x64 / 128 / 256, written (in brackets: added up):
//   tiles of 64      256 tokens             512 tokens             768 tokens             1024 tokens            2048 tokens
//   288              5.5/6.2/7.1/11.0       6.7/7.1/8.3/13.1       8.0/7.8/9.5/15.0       9.2/8.6/10.6/16.8      15.6/13.5/16.1/26.9
//                    (5.7/6.4/7.3/12.0)     (6.9/7.3/8.5/14.0)     (8.1/8.2/9.8/16.1)     (9.3/9.1/11.2/18.5)    (16.8/14.5/17.1/29.3)
//   432              5.8/6.6/7.4/11.2       6.8/7.2/8.3/13.1       7.8/7.9/9.5/14.9       9.2/9.0/10.9/16.9      16.6/14.3/16.4/27.5
//                    (6.0/6.9/7.6/12.3)     (7.0/7.8/8.9/14.4)     (8.4/8.8/10.3/17.0)    (10.6/10.3/11.9/19.5)  (18.5/15.6/17.7/30)
//   512              6.1/6.9/7.6/11.5       7.0/7.4/8.4/13.1       7.9/8.2/9.5/14.9       9.1/9.1/10.9/16.9      17.9/14.5/16.5/28.0
//                    (6.5/7.1/7.9/12.1)     (7.2/7.9/9.1/14.0)     (8.1/8.8/10.4/16.1)    (9.6/10.0/12.1/18.6)   (19.1/15.7/18.0/31)
//   640              6.3/7.0/7.6/11.7       8.5/8.6/9.5/13.3       12.8/13.7/11.0/14.9    16.4/17.3/12.8/16.9    27.7/29.0/19.3/27.7
//                    (7.3/8.3/8.3/12.3)     (11.5/12.2/11.1/15.9)  (15.1/15.7/12.8/17.8)  (18.2/18.8/14.4/20.1)  (29.7/30/21.0/31)
//   768              6.9/7.3/7.9/11.6       8.8/8.5/9.3/13.1       10.8/10.6/10.5/14.8    13.9/14.6/12.1/17.3    25.1/26.3/17.9/27.8
//                    (7.1/8.2/8.5/14.1)     (9.8/10.4/10.1/16.7)   (13.1/13.8/12.2/19.4)  (16.3/17.0/13.9/21.9)  (26.8/27.5/19.8/32)
//   896              8.3/7.8/8.1/11.5       10.5/9.4/10.0/13.2     13.0/11.2/11.4/15.0    16.1/15.4/12.9/17.6    27.5/26.4/19.4/27.9
//                    (8.8/8.8/8.9/14.6)     (11.9/11.1/10.9/17.9)  (15.4/14.8/13.1/20.3)  (18.3/17.5/14.9/22.9)  (30/27.9/21.2/33)
//   1056             9.0/9.8/10.0/11.5      12.2/13.1/13.7/13.3    15.9/16.8/16.3/15.1    19.9/21.0/21.0/17.7    35/37/35/27.8
//                    (10.3/10.6/11.8/15.3)  (14.8/15.9/16.4/18.4)  (18.7/20.4/20.2/20.6)  (22.9/24.3/23.7/23.2)  (38/40/37/33)
//   1344             10.2/10.4/11.1/11.5    14.7/13.4/14.1/13.8    18.8/17.1/16.8/16.1    23.4/21.7/20.9/18.6    41/39/35/28.8
//                    (12.7/12.3/12.8/16.9)  (18.0/16.4/16.7/19.6)  (22.8/20.6/20.3/22.0)  (27.7/24.6/23.7/24.9)  (46/41/37/35)
//   1536             10.5/11.9/12.0/12.7    14.6/13.6/14.0/14.8    20.4/19.0/17.0/17.0    25.2/23.3/20.7/19.4    44/40/35/30
//                    (14.8/14.5/14.1/17.6)  (20.0/18.3/17.3/20.2)  (24.5/22.0/20.4/22.8)  (29.7/25.7/23.7/25.8)  (50/42/37/37)
// (up to 256 tiles of 64 those are fastest at every length: 128 of them at 1504 tokens 6.7 / 10.4 / 13.2 / 20.8. Beyond 640 tokens
// and 1024 tiles with gradients added up, smaller tiles would be up to 16 % ahead of 256-wide ones; 512 at 1024 tokens, added up, lose
// 4 % on 128x64.) The lines in between: 448 tokens 704 tiles 8.0 / 8.2 / 8.6 / 12.5, 832 9.5 / 8.6 / 9.3 / 12.4, 1152 11.5 / 12.2 / 13.0 / 12.7;
// 640 tokens 640 tiles 10.3 / 10.9 / 10.3 / 14.0, added up 13.4 / 14.2 / 12.1 / 16.7, 960 tiles 12.6 / 10.9 / 11.1 / 14.2.
// Calls of several weights have the lines of one. Seven weights in 1008 tiles 352 tokens 10.6 / 10.1 / 10.3 / 11.6, added up 12.7 / 11.9 / 11.8 /
// 17.1; two in 1024 tiles 9.0 / 9.5 / 9.7 / 11.9 (12.6 / 11.5 / 11.9 / 17.1), four 9.7 / 9.3 / 10.0 / 12.0 (12.3 / 11.5 / 11.8 / 17.9); seven in 1152
// tiles 11.8 / 12.0 / 13.1 / 12.0 (14.8 / 14.3 / 14.9 / 18.1), in 1248 at 256 tokens 10.2 / 10.9 / 11.8 / 11.1 (13.8 / 13.0 / 13.9 / 17.5); added up
// at 512 tokens 1056 tiles 15.2 / 16.4 / 15.5 / 18.9, seven weights in 1248 17.7 / 16.7 / 16.8 / 20.4.
int pick_tile_plain(const NsGemm *ps, const int64_t *Es, int n) {
  double longest = 0.0, t64 = 0.0;
  bool adds = false;
  for (int k = 0; k < n; ++k) {
    longest = ps[k].K > longest ? (double)ps[k].K : longest;
    adds = adds || (ps[k].plain_sum && ps[k].A32 != nullptr);
  }
  for (int k = 0; k < n; ++k) t64 += (double)Es[k] * (ps[k].M / 64) * (ps[k].N / 64) * ((double)ps[k].K / longest);
  if (t64 <= 512.0) return t64 <= 256.0 || longest <= (adds && t64 > 352.0 ? 900.0 : 768.0) ? 64 : kTile128x64;
  if (longest > 640.0) return t64 <= 1024.0 ? 128 : 256;
  // beyond 1024 tiles of 64, 128x64 ones no longer fit in two rounds of one per CU
  const bool third = t64 > 1024.0 && t64 <= (adds ? 1070.0 : 1300.0);
  if (longest <= 448.0) {
    if (t64 <= 768.0 || third) return 64;
    if (t64 <= (adds && longest > 192.0 ? 1450.0 : 1536.0)) return kTile128x64;
  } else {
    if ((t64 <= 640.0 && !(adds && longest > 576.0)) || third) return 64;
    if ((t64 <= 1024.0 && !adds) || (t64 > 768.0 && t64 <= 990.0) || (t64 > 1300.0 && t64 <= (adds || longest > 544.0 ? 1450.0 : 1536.0)))
      return kTile128x64;
  }
  return t64 <= (adds ? 3000.0 : 2000.0) ? 128 : 256;
}

// What leaves a launch past the caches (NsGemm::stream_out): the caches are left to the operands of the tiles still to
// come, but the next launch finds nothing there.
// The next iterate, on 128-wide tiles. A bf16 pair of about three times what the L2s hold (32 MiB) pushes operands out of
// them; of a smaller one A = X X^T finds enough there, and 64-wide tiles of that product read every row so often that
// they want it there at any size. Up to M = 256 a column panel of the iterate has two readers at most and nothing is
// gained. Measured, us per chain, kept / past the caches:
//   38 MB       12 x (512,1536) on 128-wide tiles 447 / 478, 24 x (384,1024) 375 / 393
//   79 .. 85    48 x (640,640) 1060 / 1035, 24 x (640,1280) 821 / 842, 16 x (1152,1152) 979 / 988
//   96 .. 118   30 x (896,896) 1480 / 1460, 60 x (640,640) 1252 / 1233, 100 x (384,768) 998 / 978
//   127 .. 159  30 x (640,1792) 1243 / 1211, 80 x (384,1152) 1000 / 959, 10 x (1408,2816) 1464 / 1440, 20 x (1408,1408) 2024 / 1990,
//               24 x (1152,1152) 1451 / 1450, 12 x (1152,2304) 1063 / 1071
//   M <= 256    300 x (256,256) 786 / 763, 200 x (256,768) 1073 / 1082, 600 x (128,256) 580 / 587
//   A on 64-wide tiles   12 x (512,1536) 356 / 360, 60 x (384,768) 560 / 581, 18 x (640,1792) 755 / 803
// The next iterate, on 256-wide tiles: kept where A = X X^T does not run on 256-wide ones, which is where few matrices
// are wide, and reads the high halves only: 12 x (1024,2048) 678 / 705, 12 x (1024,3072) 923 / 949, 6 x (1536,4096) 1174 / 1205;
// on 256-wide ones 12 x (1536,1536) 1282 / 1252, 24 x (1024,3072) 1589 / 1565, 40 x (1024,1024) 1542 / 1522; both halves
// 40 x (512,1536) 1018 / 1011, 20 x (768,2304) 1436 / 1429.
// A and B on 256-wide tiles: kept up to 24 Mi elements. 16 x (1024,1024) 667 / 684, 20 x (1024,1024) 793 / 815, 24 x (1024,1024)
// 899 / 900, 24 x (1024,2048) 1134 / 1153; 32 x (1024,1024) 1338 / 1335, 40 x (1024,1024) 1539 / 1522, 12 x (1536,1536) 1264 / 1252.
// The fp32 copy of A that B reads on 128-wide tiles, from 22 Mi elements on: 42 x (640,640) (16 Mi) 888 / 891, 30 x (896,896) (23 Mi)
// 1434 / 1421, 60 x (640,640) (23 Mi) 1208 / 1198, 24 x (1152,1152) (30 Mi) 1353 / 1308; 12 x (768,768) 419 / 430.
constexpr int64_t kStreamPair = 90 << 20, kKeepSquare = 24 << 20, kKeepA32 = 22 << 20;

// What a mode's tile flags ask for (0: nothing).
int forced_tile(int flags) {
  return (flags & ANC_NS_FORCE_T64) ? 64 : (flags & (ANC_NS_FORCE_T128 | ANC_NS_TILE128)) ? 128
         : (flags & ANC_NS_FORCE_T256) ? 256 : 0;
}

WideRule wide_rule(const SplitPlan &sp) {
  return WideRule{(double)sp.wide_near, (double)sp.wide_lo, (double)sp.wide_hi, (double)sp.wide_near_diff};
}

// steps x { A = X X^T; B = b A + c A A; X = a X + B X } on n problems side by side: every
// product of a step is ONE launch over all problems (problems in the order given; put the
// longest K first). First step's output goes to pair `nxt` of each plan, later steps ping-pong;
// the last step writes the fp32 results. `flags`: the tile flags of the mode.
int run_bf16_chain(ChainProb *cp, int n, int steps, const float *coef, int flags, hipStream_t s,
                   const NsUpdate *upd = nullptr) {
  const int force = forced_tile(flags);
  const uint16_t *curH[kMaxGroups], *curL[kMaxGroups];
  int nxt[kMaxGroups];
  int64_t Es[kMaxGroups];
  for (int q = 0; q < n; ++q) { curH[q] = cp[q].inH; curL[q] = cp[q].inL; nxt[q] = cp[q].nxt; Es[q] = cp[q].E; }
  bool want_cond = false;      // some later iteration gates a product on the proxy
  for (int q = 0; q < n; ++q) want_cond = want_cond || cp[q].pl.sp.any_gate(steps);
  for (int q = 0; q < n; ++q)  // (the statistics' buffers come with the wide gate)
    ANC_REQUIRE(!cp[q].pl.sp.any_gate(steps) || cp[q].pl.sp.wide(), "Newton-Schulz chain: a plan with gates has the wide one");
  // the matrices are dealt over the launches' runs (k_ns_classify_order) where a gate picks some of several
  auto ordered = [&](int q) {
    bool gated = false;
    for (int j = 1; j < steps; ++j) gated = gated || cp[q].pl.sp.gated(j);
    return gated && cp[q].E > 1;
  };
  double l8_cur[kMaxGroups];   // the proxy bound the current iterate's 8-bit low halves were written with (0: none)
  for (int q = 0; q < n; ++q) l8_cur[q] = 0.0;
  for (int k = 0; k < steps; ++k) {
    const bool last = k + 1 == steps;
    NsGemm ga[kMaxGroups], gb[kMaxGroups], gx[kMaxGroups];
    for (int q = 0; q < n; ++q) {
      const Plan &pl = cp[q].pl;
      const int64_t M = cp[q].M, N = cp[q].N, mn = M * N;
      const bool split = k >= pl.sp.x_from;        // X residual terms
      const bool split_fb = k >= pl.sp.fb_from;    // F and Boff residual terms
      // a property of the shape: whether 256-wide tiles fit, and with them 8-bit low halves of the iterate
      const bool wide256 = !(flags & ANC_NS_TILE128) && M % 256 == 0 && N % 256 == 0;
      NsGemm g{};
      g.M = (int)M; g.N = (int)N;
      g.fits256 = wide256 ? 1 : 0;
      g.A32 = pl.A32; g.Fh = pl.Fh; g.dA = pl.dA; g.Bh = pl.Bh; g.dB = pl.dB;
      if (pl.sp.drop_a32) {
        // the first iteration runs before the classification: nobody is flagged yet
        g.a32_gated = 1;
        g.a32_flag = (k > 0 && pl.sp.wide()) ? pl.wide_flag : nullptr;
      }
      g.Fl = split_fb ? pl.Fl : nullptr;
      g.Bl = split_fb ? pl.Bl : nullptr;
      g.ca = coef[3 * k]; g.cb = coef[3 * k + 1]; g.cc = coef[3 * k + 2];
      g.scale = (k == 0) ? cp[q].scale0 : nullptr;
      g.x_panel = k > 0 ? 1 : 0;                   // the input pair is row-major as the caller left it
      // the wide gate of this iteration (a band of the proxy; the proxy is N * sum, hence the / N)
      const bool wide_g = pl.sp.wide_gram(k);      // implies !split
      const bool wide_a = pl.sp.wide_all(k);       // implies !split_fb
      auto set_wide = [&](NsGemm &w, int nterms_wide) {
        w.wide_flag = pl.wide_flag;
        w.nterms_wide = nterms_wide;
      };
      // A = X X^T
      ga[q] = g;
      ga[q].A[0] = ga[q].B[0] = curH[q];
      ga[q].A[1] = ga[q].B[1] = curL[q];
      ga[q].nterms = split ? 3 : 1;
      const bool gated = pl.sp.gated(k);           // implies !split
      if (gated) {
        ga[q].cond = pl.cond;
        ga[q].cond_thresh = (double)pl.sp.gate_tau[k] / (double)N;
        ga[q].order = ordered(q) ? pl.order : nullptr;
        ga[q].nterms_hard = 3;
      }
      if (wide_g) set_wide(ga[q], 3);
      if (wide_a) {                                // the residual of F, for the matrices in the band only
        set_wide(ga[q], split ? 0 : 3);
        ga[q].Fl = pl.Fl;
        ga[q].lo_gated = 1;
      }
      ga[q].K = (int)N; ga[q].strideA = mn; ga[q].strideB = mn;
      // B = b A + c A A
      gb[q] = g;
      gb[q].A[0] = gb[q].B[0] = pl.Fh;
      gb[q].A[1] = gb[q].B[1] = pl.Fl;
      gb[q].nterms = split_fb ? 3 : 1;
      if (wide_a) {
        set_wide(gb[q], 3);
        gb[q].Bl = pl.Bl;
        gb[q].lo_gated = 1;
      }
      gb[q].K = (int)M; gb[q].strideA = M * M; gb[q].strideB = M * M;
      // X = a X + B X
      gx[q] = g;
      gx[q].A[0] = pl.Bh; gx[q].B[0] = curH[q];
      gx[q].A[1] = pl.Bl; gx[q].B[1] = curL[q];
      // (a plan never splits F and Boff before X: Bl alone does not occur)
      gx[q].nterms = split_fb ? 3 : split ? 2 : 1;
      if (gated && ((pl.sp.gate_bx >> k) & 1u) && !split_fb) {
        gx[q].cond = pl.cond;
        gx[q].cond_thresh = (double)pl.sp.gate_tau[k] / (double)N;
        gx[q].order = ordered(q) ? pl.order : nullptr;
        gx[q].nterms_hard = 2;
      }
      if (wide_a) set_wide(gx[q], 3);
      gx[q].K = (int)M; gx[q].strideA = M * M; gx[q].strideB = mn;
      gx[q].Xh = curH[q]; gx[q].Xl = curL[q];
      gx[q].Yh = last ? nullptr : pl.Xh[nxt[q]];
      gx[q].Yl = last ? nullptr : pl.Xl[nxt[q]];
      gx[q].lo_zero = (k == 0 && cp[q].inL == nullptr) ? 1 : 0;
      if (gx[q].lo_zero) gx[q].Xl = (const uint16_t *)pl.zero16;
      gx[q].X32 = (last && cp[q].upd == nullptr) ? cp[q].X32 : nullptr;
      gx[q].X16 = (last && cp[q].upd == nullptr) ? cp[q].X16 : nullptr;
      gx[q].upd = last ? cp[q].upd : nullptr;
      // The next iterate's low half is one byte for the matrices whose low half no product of the
      // next iteration multiplies: every matrix outside the wide gate if that iteration has no gate,
      // those below its gate if it has one, none if its plan splits X for everybody.
      double l8_next = 0.0;
      if (wide256 && pl.sp.low8 && !last && pl.sp.any_gate(steps) && k + 1 < pl.sp.x_from)
        l8_next = pl.sp.gated(k + 1) ? (double)pl.sp.gate_tau[k + 1] / (double)N : 1e300;
      gx[q].l8_cond = pl.cond;
      gx[q].l8_wide = pl.sp.wide() ? pl.wide_flag : nullptr;
      gx[q].l8_in = l8_cur[q];
      gx[q].l8_out = l8_next;
      l8_cur[q] = l8_next;
    }
    // (on the last step too, where nobody reads on: one kernel for all steps)
    NsGemm next[kMaxGroups];                 // the product that reads the next iterate
    int64_t pair = 0, square = 0;
    bool terms = false;
    for (int q = 0; q < n; ++q) {
      next[q] = ga[q];
      next[q].nterms = k + 1 >= cp[q].pl.sp.x_from ? 3 : 1;
      terms = terms || next[q].nterms > 1;
      if (cp[q].M > 256) pair += Es[q] * cp[q].M * cp[q].N * 4;
      square += Es[q] * cp[q].M * cp[q].M;
    }
    const int reader = force != 0 ? force : pick_tile(EPI_GRAM, next, Es, n);
    for (int q = 0; q < n; ++q) {
      gx[q].stream_out = (reader != 64 && pair >= kStreamPair ? kStream128 : 0) | (reader == 256 || terms ? kStream256 : 0);
      ga[q].stream_out = gb[q].stream_out = square > kKeepSquare ? kStream256 : 0;
      if (square > kKeepA32) gb[q].stream_out |= kStream128;
    }
    {
      AncProfScope prof(ANC_PROF_NS_GRAM, s);
      if (int rc = anc_ns_gemm_multi(EPI_GRAM, ga, Es, n, force, s)) return rc;
    }
    // One matrix whose B = b A + c A A runs on 64-wide tiles that leave CUs over: the statistics are workgroups of that launch. The column
    // statistic is read there whether the proxy asks for it or not: beyond kStatCols columns matrices that do not lose by it what those
    // that do gain by the launches.
    // us per chain, beside B / in launches of their own, plain matrices (with 1 % of the columns x100, which ask for it):
    //   Keller     (1024,1024) 139.9 / 144.0 (139.4 / 148.9), (1152,1152) 173.9 / 178.2 (173.7 / 182.6), (1280,1280) 190.5 / 194.1 (191.0 / 199.0),
    //              (1408,1408) 216.8 / 223.3 (217.0 / 228.0), (1024,3072) 236.2 / 239.7 (236.4 / 245.4), (1408,5632) 476.1 / 481.6 (481.3 / 488.1),
    //              (1024,8192) 430.3 / 430.1 (433.7 / 440.3), (1280,8192) 573.0 / 573.9 (577.1 / 584.3), (1408,8192) 678.1 / 677.2 (680.9 / 691.0),
    //              (1024,12288) 605.7 / 603.0 (610.2 / 616.6), (1152,12288) 755.4 / 750.8 (759.6 / 764.1), (1408,12288) 991.6 / 990.2 (997.5 /
    //              1003.8); (1024,14336) 742.1 / 739.1 (749.1 / 753.1), (1024,16384) 827.5 / 820.1 (832.8 / 837.5), (1024,65536) 3117 / 3086
    //              (3143 / 3141)
    //   Polar Express  (1024,1024) 126.2 / 130.6 (131.4 / 141.0), (1152,2432) 173.8 / 176.9 (180.5 / 188.6), (1408,1408) 179.5 / 185.4 (203.6 / 214.6)
    // Matrices whose next iterate has 8-bit low halves (Polar Express, N >= 2M) keep launches of their own, though nothing asks for that:
    // (1024,3072) 177.0 there, 173.4 beside B, (1024,8192) 303.5, 303.8.
    NsStatOne beside{};
    const bool with_b = k == 0 && want_cond && n == 1 && Es[0] == 1 && cp[0].scale0 != nullptr && !(gx[0].l8_out > 0.0) &&
                        !ordered(0) && (cp[0].M / 64) * (cp[0].M / 64 + 1) / 2 <= kStatTiles && cp[0].N <= kStatCols &&
                        (force != 0 ? force : pick_tile(EPI_BMAT, gb, Es, n)) == 64;
    if (with_b) {
      const Plan &pl = cp[0].pl;
      beside = NsStatOne{pl.Fh, cp[0].inH, pl.condpart, pl.cond, pl.colpart, pl.wide_flag, pl.order, (int)cp[0].M, (int)cp[0].N, pl.col_parts,
                         wide_rule(pl.sp)};
    } else if (k == 0 && want_cond) {
      // the proxy of every problem that gates a later product, from the Fh this launch wrote
      NsCondArgs ca{};
      int blocks = 0;
      bool any_ordered = false;
      for (int q = 0; q < n; ++q) any_ordered = any_ordered || (cp[q].pl.sp.any_gate(steps) && ordered(q));
      for (int q = 0; q < n; ++q) {
        if (!cp[q].pl.sp.any_gate(steps)) continue;
        ca.arrived[ca.n] = any_ordered ? nullptr : cp[q].pl.order;       // (no order: its place counts arrivals)
        ca.Fh[ca.n] = cp[q].pl.Fh; ca.out[ca.n] = cp[q].pl.condpart; ca.M[ca.n] = (int)cp[q].M;
        ca.blocks[ca.n] = (int)(cp[q].E * kCondParts);
        blocks += ca.blocks[ca.n];
        ++ca.n;
      }
      AncProfScope prof(ANC_PROF_NS_FRO, s);
      hipLaunchKernelGGL(k_ns_cond, dim3((unsigned)blocks), dim3(kThreads), 0, s, ca);
      ANC_LAUNCH_CHECK();
      // the wide gate's decision per matrix, from the proxy and, where it asks, the column norms
      NsColArgs cs{}, cf{};
      int cs_blocks = 0;
      for (int q = 0; q < n; ++q) {
        const Plan &pl = cp[q].pl;
        if (!pl.sp.any_gate(steps)) continue;
        const int i = cs.n;
        cs.Xh[i] = cp[q].inH; cs.cond[i] = pl.condpart; cs.sum[i] = pl.cond; cs.part[i] = pl.colpart; cs.flag[i] = pl.wide_flag;
        cs.gate[i] = 1e300;
        for (int j = 1; j < steps; ++j)
          if (pl.sp.gated(j)) cs.gate[i] = std::min(cs.gate[i], (double)pl.sp.gate_tau[j] / (double)cp[q].N);
        cs.order[i] = ordered(q) ? pl.order : nullptr;
        cs.arrived[i] = any_ordered ? nullptr : pl.order;
        cs.M[i] = (int)cp[q].M; cs.N[i] = (int)cp[q].N; cs.parts[i] = pl.col_parts;
        cs.rule[i] = wide_rule(pl.sp);
        cs.blocks[i] = (int)(cp[q].E * pl.col_parts);
        cs_blocks += cs.blocks[i];
        ++cs.n;
      }
      if (any_ordered) hipLaunchKernelGGL((k_ns_colstat<false>), dim3((unsigned)cs_blocks), dim3(kThreads), 0, s, cs);
      else             hipLaunchKernelGGL((k_ns_colstat<true>), dim3((unsigned)cs_blocks), dim3(kThreads), 0, s, cs);
      ANC_LAUNCH_CHECK();
      if (any_ordered) {
        cf = cs;
        for (int i = 0, q = 0; q < n; ++q)
          if (cp[q].pl.sp.any_gate(steps)) cf.blocks[i++] = (int)cp[q].E;
        hipLaunchKernelGGL(k_ns_classify_order, dim3((unsigned)cf.n), dim3(kClassifyThreads), 0, s, cf);
        ANC_LAUNCH_CHECK();
      }
    }
    {
      AncProfScope prof(ANC_PROF_NS_BMAT, s);
      if (with_b) {
        if (int rc = anc_ns_gemm_tile_multi(EPI_BMAT, gb, Es, 1, s, 64, false, nullptr, false, &beside)) return rc;
      } else if (int rc = anc_ns_gemm_multi(EPI_BMAT, gb, Es, n, force, s)) return rc;
    }
    {
      AncProfScope prof(last && upd != nullptr ? ANC_PROF_NS_BX_UPD : ANC_PROF_NS_BX, s);
      if (int rc = anc_ns_gemm_multi(EPI_BX, gx, Es, n, force, s, last ? upd : nullptr)) return rc;
    }
    for (int q = 0; q < n; ++q) {
      curH[q] = cp[q].pl.Xh[nxt[q]]; curL[q] = cp[q].pl.Xl[nxt[q]];
      nxt[q] ^= 1;
    }
  }
  return ANC_OK;
}

}  // namespace

static int pair_multi_impl(const char *who, const anc_ns_problem_t *probs, int32_t n_probs,
                           const uint64_t *desc_tables, const NsUpdate *upd, int steps, const float *coef,
                           float eps, int mode, uint64_t stream);

int anc_ns_gemm_multi(int epi, const NsGemm *ps, const int64_t *Es, int n, int force, hipStream_t s,
                      const NsUpdate *upd) {
  ANC_REQUIRE(n >= 1 && n <= kMaxGroups, "Newton-Schulz chain: 1..%d problems per launch", kMaxGroups);
  bool any_upd = false, all_upd = true;
  for (int k = 0; k < n; ++k) { any_upd = any_upd || ps[k].upd != nullptr; all_upd = all_upd && ps[k].upd != nullptr; }
  ANC_REQUIRE(any_upd == all_upd && (!any_upd || upd != nullptr),
              "Newton-Schulz chain: the fused update applies to every problem of a launch or to none");
  // B is symmetric and stored in full, so X = a X + B X can fetch its tile by rows k (256-byte rows) as
  // well as by rows m (64-byte row pieces). Measured per 5 launches: 84 x (1024, 3072) 4.12
  // against 4.27 ms, 208 x (1024, 1024) 3.37 against 3.56 ms, but 64 x (512, 512) 0.238 against
  // 0.212 ms: by rows k from M = 1024 on. The two ways read the same values except inside the
  // diagonal blocks of a B that descends from an A = X X^T with residual terms: there
  // element (i, j) and element (j, i) add the same products in a different order and may differ
  // in the last bit. So the way of reading is a property of the problem's shape, never of what
  // it shares a call with: a call with problems of both kinds becomes two launches.
  // Where 256-wide tiles are the choice, problems whose dims do not allow them get a launch of their own.
  NsGemm part[kMaxGroups];
  int64_t pe[kMaxGroups];
  bool done[2] = {false, false};
  for (int pass = 0; pass < 4; ++pass) {
    const bool by_rows = epi == EPI_BX && (pass & 1) == 0, wide = pass < 2;
    auto collect = [&](bool all) {
      int m = 0;
      for (int k = 0; k < n; ++k) {
        if (epi == EPI_BX ? (ps[k].M >= 1024) != by_rows : (pass & 1) != 0) continue;
        if (!all && (ps[k].fits256 != 0) != wide) continue;
        part[m] = ps[k];
        pe[m++] = Es[k];
      }
      return m;
    };
    const auto pick = [&](int m) { return force ? force : pick_tile(epi, part, pe, m); };
    const auto narrow = [](int tile) { return tile == 256 ? 128 : tile; };
    const NsUpdate *u = any_upd ? upd : nullptr;
    const int m_wide = collect(false);
    if (wide) {
      if (m_wide > 0 && pick(m_wide) == 256) {
        if (int rc = anc_ns_gemm_big_multi(epi, part, pe, m_wide, s, by_rows, u)) return rc;
      } else if (const int m = collect(true)) {
        if (int rc = anc_ns_gemm_tile_multi(epi, part, pe, m, s, narrow(pick(m)), by_rows, u, false)) return rc;
        done[pass & 1] = true;
      }
    } else if (m_wide > 0 && !done[pass & 1]) {
      if (int rc = anc_ns_gemm_tile_multi(epi, part, pe, m_wide, s, narrow(pick(m_wide)), by_rows, u, false)) return rc;
    }
  }
  return ANC_OK;
}

int anc_ns_gemm_plain(const NsGemm *ps, const int64_t *Es, int n, hipStream_t s, bool a_transposed) {
  ANC_REQUIRE(n >= 1 && n <= kMaxGroups, "anc_ns_gemm_plain: 1..%d problems per launch", kMaxGroups);
  const int tile = pick_tile_plain(ps, Es, n);
  if (tile == 256) return anc_ns_gemm_big_plain(ps, Es, n, s, a_transposed);
  return anc_ns_gemm_tile_multi(EPI_BX, ps, Es, n, s, tile, a_transposed, nullptr, true);
}

extern "C" int64_t anc_ns_workspace_bytes(int64_t E, int64_t M, int64_t N, int mode) {
  mode &= ~kTileFlags;
  if (check_shape(E, M, N, mode, "anc_ns_workspace_bytes")) return -1;
  // sized for any step count: with steps >= 3 every optional buffer of the mode's plan is present
  // (the longer of a long and a 5-step chain's plans, should the two ever differ)
  const int64_t a = make_plan(0, E, M, N, mode, 64).bytes, b = make_plan(0, E, M, N, mode, 5).bytes;
  return a > b ? a : b;
}

// FLOPs of a symmetric M x M product, per unit of K, counted in blocks on or below the diagonal: 256x256 where both
// dims are multiples of 256 and ANC_NS_TILE128 is not set, else 128x128: M^2 + 256 M or M^2 + 128 M. The kernels multiply
// 64x64 blocks, M^2 + 64 M (see anc_optim.h).
static double sym_tile_flops(int64_t M, int64_t N, bool force_small) {
  const double ts = (!force_small && M % 256 == 0 && N % 256 == 0) ? 256.0 : 128.0;
  const double t = (double)M / ts;
  return t * (t + 1) / 2 * 2.0 * ts * ts;
}

// Matrix-core work of one chain call: `executed` counts the terms multiplied (residual terms too), of symmetric products
// the blocks of sym_tile_flops,
// `dense` is the textbook steps*(4 M^2 N + 2 M^3) per matrix.
extern "C" int anc_ns_flops(int64_t E, int64_t M, int64_t N, int steps, int mode,
                            double *executed, double *dense) {
  const int flags = mode & kTileFlags;
  mode &= ~kTileFlags;
  if (int rc = check_shape(E, M, N, mode, "anc_ns_flops")) return rc;
  ANC_REQUIRE(executed != nullptr && dense != nullptr && steps >= 0, "anc_ns_flops: bad arguments");
  const double m = (double)M, n = (double)N, e = (double)E;
  *dense = e * steps * (4.0 * m * m * n + 2.0 * m * m * m);
  if (mode == ANC_NS_FP32) { *executed = *dense; return ANC_OK; }
  const SplitPlan sp = split_plan(M, N, mode, steps);
  const double sym = sym_tile_flops(M, N, (flags & ANC_NS_TILE128) != 0);
  double ex = 0.0;
  for (int k = 0; k < steps; ++k) {
    const bool sx = k >= sp.x_from, sfb = k >= sp.fb_from;
    ex += sym * (sx ? 3 : 1) * n;                                        // A = X X^T
    ex += sym * (sfb ? 3 : 1) * m;                                       // B = b A + c A A
    ex += 2.0 * m * n * (1 + (sx ? 1 : 0) + (sfb ? 1 : 0)) * m;          // X = a X + B X
  }
  *executed = e * ex;
  return ANC_OK;
}

extern "C" int anc_ns_product_flops(int64_t E, int64_t M, int64_t N, int steps, int mode, int k, int product,
                                    double *executed) {
  const int flags = mode & kTileFlags;
  mode &= ~kTileFlags;
  if (int rc = check_shape(E, M, N, mode, "anc_ns_product_flops")) return rc;
  ANC_REQUIRE(executed != nullptr && steps > 0 && k >= 0 && k < steps && product >= 0 && product <= 2,
              "anc_ns_product_flops: bad arguments");
  const double m = (double)M, n = (double)N;
  if (mode == ANC_NS_FP32) {
    *executed = (double)E * (product == 1 ? 2.0 * m * m * m : 2.0 * m * m * n);
    return ANC_OK;
  }
  const SplitPlan sp = split_plan(M, N, mode, steps);
  const bool sx = k >= sp.x_from, sfb = k >= sp.fb_from;
  const double sym = sym_tile_flops(M, N, (flags & ANC_NS_TILE128) != 0);
  double ex;
  if (product == 0)      ex = sym * (sx ? 3 : 1) * n;
  else if (product == 1) ex = sym * (sfb ? 3 : 1) * m;
  else                   ex = 2.0 * m * n * (1 + (sx ? 1 : 0) + (sfb ? 1 : 0)) * m;
  *executed = (double)E * ex;
  return ANC_OK;
}

// Of the last chain call on this workspace: how many matrices took extra terms through a
// conditioning gate, and the matrix-core work all of them together add to anc_ns_flops' `executed`.
// Synchronises `stream`, then reads the proxy's partial sums back and takes the kernels' decisions.
extern "C" int anc_ns_hard_info(uint64_t workspace, int64_t E, int64_t M, int64_t N, int mode, int steps,
                                int32_t *n_gated, double *extra_flops, uint64_t stream) {
  const int flags = mode & kTileFlags;
  mode &= ~kTileFlags;
  if (int rc = check_shape(E, M, N, mode, "anc_ns_hard_info")) return rc;
  ANC_REQUIRE(n_gated != nullptr && extra_flops != nullptr && workspace != 0 && steps >= 0,
              "anc_ns_hard_info: bad arguments");
  *n_gated = 0;
  *extra_flops = 0.0;
  if (mode == ANC_NS_FP32) return ANC_OK;
  const Plan pl = make_plan(workspace, E, M, N, mode, steps);
  if (!pl.sp.any_gate(steps)) return ANC_OK;
  std::vector<double> host((size_t)E);
  ANC_HIP(hipStreamSynchronize(anc_stream(stream)));
  ANC_HIP(hipMemcpy(host.data(), pl.cond, host.size() * sizeof(double), hipMemcpyDeviceToHost));
  std::vector<int32_t> wide((size_t)E, 0);
  if (pl.sp.wide())
    ANC_HIP(hipMemcpy(wide.data(), pl.wide_flag, wide.size() * sizeof(int32_t), hipMemcpyDeviceToHost));
  const double gram_extra = 2.0 * sym_tile_flops(M, N, (flags & ANC_NS_TILE128) != 0) * (double)N;     // two more terms
  const double bx_extra = 2.0 * (double)M * (double)M * (double)N;                   // one more term
  for (int64_t e = 0; e < E; ++e) {
    const double t = host[(size_t)e];
    bool any = false;
    const bool in_band = wide[(size_t)e] != 0;
    for (int k = 0; k < steps; ++k) {
      if (in_band) {                    // the wide gate takes precedence over the others
        const bool sx = k >= pl.sp.x_from;
        if (pl.sp.wide_gram(k)) { *extra_flops += gram_extra; any = true; }
        if (pl.sp.wide_all(k)) {
          *extra_flops += 2.0 * sym_tile_flops(M, N, (flags & ANC_NS_TILE128) != 0) * (double)M + (sx ? 1.0 : 2.0) * bx_extra;
          any = true;
        }
        continue;
      }
      if (!pl.sp.gated(k) || !(t > (double)pl.sp.gate_tau[k] / (double)N)) continue;
      any = true;
      *extra_flops += gram_extra + (((pl.sp.gate_bx >> k) & 1u) ? bx_extra : 0.0);
    }
    if (any) ++*n_gated;
  }
  return ANC_OK;
}

extern "C" int anc_ns_batched(uint64_t X, int64_t E, int64_t M, int64_t N, int steps,
                              const float *coef, float eps, int mode, uint64_t workspace,
                              int64_t workspace_bytes, uint64_t stream) {
  const int flags = mode & kTileFlags;
  mode &= ~kTileFlags;
  if (int rc = check_shape(E, M, N, mode, "anc_ns_batched")) return rc;
  ANC_REQUIRE(X != 0 && (X & 15) == 0, "anc_ns_batched: X must be a 16-byte aligned device pointer");
  ANC_REQUIRE(steps >= 0 && steps <= 64 && (steps == 0 || coef != nullptr),
              "anc_ns_batched: steps=%d out of range or null coefficients", steps);
  ANC_REQUIRE(workspace != 0 && (workspace & 255) == 0, "anc_ns_batched: workspace must be 256-byte aligned");
  const Plan pl = make_plan(workspace, E, M, N, mode, steps);
  ANC_REQUIRE(workspace_bytes >= pl.bytes, "anc_ns_batched: workspace holds %lld bytes, %lld needed",
              (long long)workspace_bytes, (long long)pl.bytes);
  hipStream_t s = anc_stream(stream);
  float *X32 = (float *)X;
  const int64_t mn = M * N;

  // ---- X /= ||X||_F + eps
  { AncProfScope prof(ANC_PROF_NS_FRO, s); hipLaunchKernelGGL((k_fro_partials<ANC_F32, float>), dim3((unsigned)(E * pl.nchunks)), dim3(kThreads), 0, s, X32, mn,
                     pl.nchunks, pl.partials); }
  ANC_LAUNCH_CHECK();
  { AncProfScope prof(ANC_PROF_NS_FRO, s); hipLaunchKernelGGL(k_fro_finalize, dim3((unsigned)E), dim3(kThreads), 0, s, pl.partials, pl.nchunks,
                     eps, pl.recip); }
  ANC_LAUNCH_CHECK();
  const int64_t total8 = E * mn / 8;
  const unsigned prep_grid = (unsigned)((total8 + kThreads - 1) / kThreads);

  if (mode == ANC_NS_FP32) {
    { AncProfScope prof(ANC_PROF_NS_PREP, s); hipLaunchKernelGGL(k_ns_prep, dim3(prep_grid), dim3(kThreads), 0, s, X32, pl.recip, mn, total8,
                       (uint16_t *)nullptr, (uint16_t *)nullptr); }
    ANC_LAUNCH_CHECK();
    float *cur = X32, *nxt = pl.Yf;
    const unsigned g_mm = (unsigned)(E * (M / BM) * (M / BN)), g_mn = (unsigned)(E * (M / BM) * (N / BN));
    for (int k = 0; k < steps; ++k) {
      const float a = coef[3 * k], b = coef[3 * k + 1], c = coef[3 * k + 2];
      NsGemmF32 g{};
      g.A = cur; g.B = cur; g.K = (int)N; g.nn = 0; g.strideA = mn; g.strideB = mn;
      g.Mo = (int)M; g.No = (int)M; g.out = pl.Af; g.epi = EPI_GRAM;
      { AncProfScope prof(ANC_PROF_NS_GEMM_F32, s); hipLaunchKernelGGL(k_ns_gemm_f32, dim3(g_mm), dim3(kGemmThreads), 0, s, g); }
      ANC_LAUNCH_CHECK();
      NsGemmF32 h{};
      h.A = pl.Af; h.B = pl.Af; h.K = (int)M; h.nn = 0; h.strideA = M * M; h.strideB = M * M;
      h.Mo = (int)M; h.No = (int)M; h.cb = b; h.cc = c; h.D = pl.Af; h.out = pl.Bf; h.epi = EPI_BMAT;
      { AncProfScope prof(ANC_PROF_NS_GEMM_F32, s); hipLaunchKernelGGL(k_ns_gemm_f32, dim3(g_mm), dim3(kGemmThreads), 0, s, h); }
      ANC_LAUNCH_CHECK();
      NsGemmF32 y{};
      y.A = pl.Bf; y.B = cur; y.K = (int)M; y.nn = 1; y.strideA = M * M; y.strideB = mn;
      y.Mo = (int)M; y.No = (int)N; y.ca = a; y.D = cur; y.out = nxt; y.epi = EPI_BX;
      { AncProfScope prof(ANC_PROF_NS_GEMM_F32, s); hipLaunchKernelGGL(k_ns_gemm_f32, dim3(g_mn), dim3(kGemmThreads), 0, s, y); }
      ANC_LAUNCH_CHECK();
      float *tmp = cur; cur = nxt; nxt = tmp;
    }
    if (cur != X32)
      ANC_HIP(hipMemcpyAsync(X32, cur, (size_t)(E * mn) * sizeof(float), hipMemcpyDeviceToDevice, s));
    return ANC_OK;
  }

  // ---- bf16 matrix-core chain
  if (steps == 0) {
    { AncProfScope prof(ANC_PROF_NS_PREP, s); hipLaunchKernelGGL(k_ns_prep, dim3(prep_grid), dim3(kThreads), 0, s, X32, pl.recip, mn, total8,
                       (uint16_t *)nullptr, (uint16_t *)nullptr); }
    ANC_LAUNCH_CHECK();
    return ANC_OK;
  }
  { AncProfScope prof(ANC_PROF_NS_PREP, s); hipLaunchKernelGGL(k_ns_prep, dim3(prep_grid), dim3(kThreads), 0, s, X32, pl.recip, mn, total8,
                     pl.Xh[0], pl.Xl[0]); }
  ANC_LAUNCH_CHECK();
  ChainProb cp{pl, pl.Xh[0], pl.Xl[0], 1, nullptr, X32, nullptr, E, M, N, nullptr};
  return run_bf16_chain(&cp, 1, steps, coef, flags, s);
}

// The chain on bf16 matrices in place. The input is its own high half, exactly; there is no low half, no
// widened copy, no scaling pass (the first step's epilogues carry the scale) and the last epilogue rounds. Against
// widen + anc_ns_batched + round, 24 x (1024, 2048) drop 200 us of conversion passes. A plan that splits
// the first iteration (M < 256, ANC_NS_BF16_X3) multiplies residuals there, so it gets a cleared low half.
extern "C" int anc_ns_batched_bf16(uint64_t X, int64_t E, int64_t M, int64_t N, int steps, const float *coef,
                                   float eps, int mode, uint64_t workspace, int64_t workspace_bytes,
                                   uint64_t stream) {
  const int flags = mode & kTileFlags;
  mode &= ~kTileFlags;
  if (int rc = check_shape(E, M, N, mode, "anc_ns_batched_bf16")) return rc;
  ANC_REQUIRE(mode != ANC_NS_FP32, "anc_ns_batched_bf16: bf16 modes only");
  ANC_REQUIRE(X != 0 && (X & 15) == 0, "anc_ns_batched_bf16: X must be a 16-byte aligned device pointer");
  ANC_REQUIRE(steps >= 2 && steps <= 64 && coef != nullptr, "anc_ns_batched_bf16: steps=%d: 2..64 (the result overlays the input)",
              steps);
  ANC_REQUIRE(workspace != 0 && (workspace & 255) == 0, "anc_ns_batched_bf16: workspace must be 256-byte aligned");
  const Plan pl = make_plan(workspace, E, M, N, mode, steps);
  ANC_REQUIRE(workspace_bytes >= pl.bytes, "anc_ns_batched_bf16: workspace holds %lld bytes, %lld needed",
              (long long)workspace_bytes, (long long)pl.bytes);
  hipStream_t s = anc_stream(stream);
  const uint16_t *lo = nullptr;
  if (pl.sp.x_from == 0) {
    // pair 1 is written by the second step at the earliest: its low half serves as the zeros
    lo = pl.Xl[1];
    if (int rc = anc_fill_u32((uint64_t)lo, 0u, E * M * N / 2, stream)) return rc;
  }
  { AncProfScope prof(ANC_PROF_NS_FRO, s); hipLaunchKernelGGL((k_fro_partials<ANC_BF16, uint16_t>), dim3((unsigned)(E * pl.nchunks)),
                     dim3(kThreads), 0, s, (const uint16_t *)X, M * N, pl.nchunks, pl.partials); }
  ANC_LAUNCH_CHECK();
  NsPrologue pro{};
  add_prologue(pro, pl, X, (uint64_t)lo, (uint64_t)pl.partials, pl.nchunks, E, M * N);
  if (int rc = launch_prologue(pro, eps, s)) return rc;
  ChainProb cp{pl, (const uint16_t *)X, lo, 0, pl.recip, nullptr, (uint16_t *)X, E, M, N, nullptr};
  return run_bf16_chain(&cp, 1, steps, coef, flags, s);
}

// One weight's whole Muon step: momentum, chain, update.
extern "C" int anc_muon_resident_step(uint64_t buf, uint64_t g, int g_dtype, uint64_t p32, uint64_t p16, uint64_t u,
                                      int64_t K, int64_t N, float mom, int nesterov, float lr_scale, int steps,
                                      const float *coef, float eps, int mode, uint64_t workspace,
                                      int64_t workspace_bytes, uint64_t ctl, uint64_t stream) {
  const int64_t M = K < N ? K : N, Nn = K < N ? N : K;
  if (int rc = check_shape(1, M, Nn, mode & ~kTileFlags, "anc_muon_resident_step")) return rc;
  ANC_REQUIRE(buf && g && p32 && u && ((buf | g | p32 | u) & 15) == 0 && (p16 & 7) == 0,
              "anc_muon_resident_step: null or misaligned pointer");
  ANC_REQUIRE(g_dtype == ANC_F32 || g_dtype == ANC_BF16, "anc_muon_resident_step: bad dtype");
  ANC_REQUIRE(workspace != 0 && (workspace & 255) == 0, "anc_muon_resident_step: workspace must be 256-byte aligned");
  const Plan pl = make_plan(workspace, 1, M, Nn, mode & ~kTileFlags, steps);
  ANC_REQUIRE(workspace_bytes >= pl.bytes, "anc_muon_resident_step: workspace holds %lld bytes, %lld needed",
              (long long)workspace_bytes, (long long)pl.bytes);
  anc_muon_desc_t d{};
  d.buf = buf; d.g = g; d.p32 = p32; d.p16 = p16; d.u = u;
  d.K = (int32_t)K; d.N = (int32_t)N; d.transpose = K > N ? 1 : 0; d.g_dtype = g_dtype;
  if (int rc = anc_launch_momentum_pair_one(d, mom, nesterov, u + (uint64_t)(M * Nn * 2), pl.partials, pl.desc,
                                            (const anc_step_ctl_t *)ctl, anc_stream(stream))) return rc;
  anc_ns_problem_t prob{};
  prob.Uh = u; prob.Ul = u + (uint64_t)(M * Nn * 2); prob.fro_partials = (uint64_t)pl.partials;
  prob.workspace = workspace; prob.n_partials = M * Nn / 4096; prob.E = 1; prob.M = M; prob.N = Nn;
  prob.workspace_bytes = workspace_bytes;
  const uint64_t table = (uint64_t)pl.desc;
  NsUpdate up{};
  up.lr[0] = lr_scale;
  up.ctl = (const anc_step_ctl_t *)ctl;
  return pair_multi_impl("anc_muon_resident_step", &prob, 1, &table, &up, steps, coef, eps, mode, stream);
}

// The chain on an unnormalised bf16 pair (what anc_muon_momentum_multi_pair leaves) with the
// Frobenius partial sums already known: X0 = U / (||U|| + eps) is never materialised, the first
// step folds the scale into its epilogues.
extern "C" int anc_ns_batched_pair(uint64_t Uh, uint64_t Ul, uint64_t fro_partials, int64_t n_partials,
                                   uint64_t X32_out, int64_t E, int64_t M, int64_t N, int steps,
                                   const float *coef, float eps, int mode, uint64_t workspace,
                                   int64_t workspace_bytes, uint64_t stream) {
  const int flags = mode & kTileFlags;
  mode &= ~kTileFlags;
  if (int rc = check_shape(E, M, N, mode, "anc_ns_batched_pair")) return rc;
  ANC_REQUIRE(mode != ANC_NS_FP32, "anc_ns_batched_pair: the fp32 chain takes fp32 input (anc_ns_batched)");
  ANC_REQUIRE(Uh != 0 && Ul != 0 && ((Uh | Ul) & 15) == 0 && X32_out != 0 && (X32_out & 15) == 0,
              "anc_ns_batched_pair: pointers must be 16-byte aligned and non-null");
  ANC_REQUIRE(fro_partials != 0 && n_partials > 0 && n_partials < (1 << 30),
              "anc_ns_batched_pair: need the Frobenius partial sums (n_partials per matrix)");
  ANC_REQUIRE(steps >= 2 && steps <= 64 && coef != nullptr,
              "anc_ns_batched_pair: steps=%d: needs at least 2 steps (the fp32 result may overlay the input pair)", steps);
  ANC_REQUIRE(workspace != 0 && (workspace & 255) == 0, "anc_ns_batched_pair: workspace must be 256-byte aligned");
  const Plan pl = make_plan(workspace, E, M, N, mode, steps);
  ANC_REQUIRE(workspace_bytes >= pl.bytes, "anc_ns_batched_pair: workspace holds %lld bytes, %lld needed",
              (long long)workspace_bytes, (long long)pl.bytes);
  hipStream_t s = anc_stream(stream);
  NsPrologue pro{};
  add_prologue(pro, pl, Uh, Ul, fro_partials, n_partials, E, M * N);
  if (int rc = launch_prologue(pro, eps, s)) return rc;
  ChainProb cp{pl, (const uint16_t *)Uh, (const uint16_t *)Ul, 0, pl.recip, (float *)X32_out, nullptr, E, M, N, nullptr};
  return run_bf16_chain(&cp, 1, steps, coef, flags, s);
}

// n_probs <= 8 independent batches (the shape groups of one optimizer step) through the chain
// side by side: each product of each step is one launch over all of them, which keeps the
// CUs busy where per-batch launches would each end in a partly filled last wave. Same
// results, bit for bit, as anc_ns_batched_pair on each batch. All dims multiples of 128.
static int pair_multi_impl(const char *who, const anc_ns_problem_t *probs, int32_t n_probs,
                           const uint64_t *desc_tables, const NsUpdate *upd, int steps, const float *coef,
                           float eps, int mode, uint64_t stream) {
  ANC_REQUIRE(probs != nullptr && n_probs >= 1 && n_probs <= kMaxGroups, "%s: 1..%d problems", who, kMaxGroups);
  ANC_REQUIRE((mode & ~kTileFlags) != ANC_NS_FP32, "%s: bf16 modes only", who);
  ANC_REQUIRE(steps >= 2 && steps <= 64 && coef != nullptr, "%s: steps=%d: 2..64", who, steps);
  const int flags = mode & kTileFlags;
  mode &= ~kTileFlags;
  hipStream_t s = anc_stream(stream);
  ChainProb cp[kMaxGroups];
  int order[kMaxGroups];
  for (int q = 0; q < n_probs; ++q) {
    const anc_ns_problem_t &b = probs[q];
    if (int rc = check_shape(b.E, b.M, b.N, mode, who)) return rc;
    ANC_REQUIRE(b.Uh != 0 && b.Ul != 0 && ((b.Uh | b.Ul | b.X32_out) & 15) == 0,
                "%s: pointers must be 16-byte aligned and non-null", who);
    if (desc_tables == nullptr) ANC_REQUIRE(b.X32_out != 0, "%s: null X32_out", who);
    else ANC_REQUIRE(desc_tables[q] != 0 && (desc_tables[q] & 7) == 0, "%s: null or misaligned descriptor table", who);
    ANC_REQUIRE(b.fro_partials != 0 && b.n_partials > 0 && b.n_partials < (1 << 30),
                "%s: need the Frobenius partial sums", who);
    ANC_REQUIRE(b.workspace != 0 && (b.workspace & 255) == 0, "%s: workspace must be 256-byte aligned", who);
    order[q] = q;
  }
  // longest tiles first: by N (the Gram product's K), then by M
  for (int a = 0; a < n_probs; ++a)
    for (int c = a + 1; c < n_probs; ++c) {
      const anc_ns_problem_t &x = probs[order[a]], &y = probs[order[c]];
      if (y.N > x.N || (y.N == x.N && y.M > x.M)) { const int t = order[a]; order[a] = order[c]; order[c] = t; }
    }
  NsPrologue pro{};
  for (int q = 0; q < n_probs; ++q) {
    const anc_ns_problem_t &b = probs[order[q]];
    const Plan pl = make_plan(b.workspace, b.E, b.M, b.N, mode, steps);
    ANC_REQUIRE(b.workspace_bytes >= pl.bytes, "%s: workspace holds %lld bytes, %lld needed", who,
                (long long)b.workspace_bytes, (long long)pl.bytes);
    add_prologue(pro, pl, b.Uh, b.Ul, b.fro_partials, b.n_partials, b.E, b.M * b.N);
    cp[q] = ChainProb{pl, (const uint16_t *)b.Uh, (const uint16_t *)b.Ul, 0, pl.recip, (float *)b.X32_out, nullptr, b.E, b.M, b.N,
                      desc_tables ? (const anc_muon_desc_t *)desc_tables[order[q]] : nullptr};
  }
  if (int rc = launch_prologue(pro, eps, s)) return rc;
  return run_bf16_chain(cp, n_probs, steps, coef, flags, s, upd);
}

extern "C" int anc_ns_batched_pair_multi(const anc_ns_problem_t *probs, int32_t n_probs, int steps,
                                         const float *coef, float eps, int mode, uint64_t stream) {
  return pair_multi_impl("anc_ns_batched_pair_multi", probs, n_probs, nullptr, nullptr, steps, coef, eps, mode, stream);
}

// The same chain with the Muon weight update applied by the last step's epilogue: problem q's
// matrix e is the orthogonalised update of the weight desc_tables[q][e] (p32, p16, K, N,
// transpose, scale_idx and seed are read; p16t with ANC_MUON_P16T). Same bits in p32 and p16 as the chain
// followed by anc_muon_update_multi, without the fp32 hand-off in between.
extern "C" int anc_muon_ns_update_multi(const anc_ns_problem_t *probs, int32_t n_probs,
                                        const uint64_t *desc_tables, int steps, const float *coef, float eps,
                                        int mode, const float *lr_scales, int sr, uint32_t seed_base,
                                        uint64_t ctl, uint64_t stream) {
  ANC_REQUIRE(desc_tables != nullptr && lr_scales != nullptr, "anc_muon_ns_update_multi: null descriptor tables or lr_scales");
  NsUpdate u{};
  for (int k = 0; k < ANC_MUON_MAX_SCALES; ++k) u.lr[k] = lr_scales[k];
  const int sr_only = sr & ~ANC_MUON_P16T;
  ANC_REQUIRE(sr_only == 0 || sr_only == ANC_SR_ON || sr_only == (ANC_SR_ON | ANC_SR_STEP_SEED),
              "anc_muon_ns_update_multi: sr must be 0, ANC_SR_ON or ANC_SR_ON | ANC_SR_STEP_SEED, with or without ANC_MUON_P16T");
  ANC_REQUIRE(!(sr & ANC_SR_STEP_SEED) || ctl != 0, "anc_muon_ns_update_multi: ANC_SR_STEP_SEED needs the control block");
  u.sr = sr;
  u.seed_base = seed_base;
  u.ctl = (const anc_step_ctl_t *)ctl;
  return pair_multi_impl("anc_muon_ns_update_multi", probs, n_probs, desc_tables, &u, steps, coef, eps, mode, stream);
}
