// Input-embedding weight gradient by deterministic sorted scatter, for gfx950.
// Replaces `_embed_dw_scatter` (ancora/kernels/fused.py:387-408; host side `build_id_groups`,
// :411-424; launched from ancora/model/resident_moe_model.py:333-334):
//     out[gid[g]] += sum over r < cnt[g] of f32(bf16 dy[srt[start[g] + r]])
// The host stable-sorts the token ids into groups (one per distinct id, rows in their original
// order). One workgroup owns one (group, 256-column chunk): a single writer per output element,
// no atomics, and the rows of a group are added one after the other in sorted order starting from
// zero, then added onto `out`: the association order of the reference's loop, so the result is
// bit-identical to a sequential fp32 evaluation and the same on every run. The indices of 64 rows come in
// by one load per lane, rows are fetched 32, 8, 2 and 1 at a time while that many are left; the additions stay in
// order. (The largest group bounds the launch: with 8 rows in flight behind their own index loads, a frequent id
// of 150 rows among 8192 took 33 us. Most groups are one row and want a short path: guarding each of 32
// loads instead took 77 us.)
#include <algorithm>
#include <new>
#include <type_traits>
#include <vector>

#include "common.h"

namespace {

constexpr int kChunk = 256;     // columns per wavefront: 64 lanes x 4; up to 4 wavefronts (1024 columns) per workgroup

__global__ void __launch_bounds__(256)
k_embed_dw_scatter(const int32_t *__restrict__ cnt, const int32_t *__restrict__ start,
                   const int32_t *__restrict__ gid, const int32_t *__restrict__ srt,
                   const uint16_t *__restrict__ dy, float *__restrict__ out, float *__restrict__ compact,
                   int H, int64_t M, int64_t V) {
  const int g = (int)blockIdx.x;
  const int n = cnt[g];
  if (n <= 0) return;                                   // padding group
  const int st = start[g];
  const int64_t row = gid[g];
  if (st < 0 || (int64_t)st + n > M || row < 0 || (compact == nullptr && row >= V)) return;   // malformed group: no write
  // (every lane stays: its index load serves the others)
  const int lane = (int)(threadIdx.x & 63);
  const int col = (int)(blockIdx.y * blockDim.x + threadIdx.x) * 4;
  const bool live = col < H;
  const int c0 = live ? col : 0;
  float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  bool bad = false;                                     // an index outside dy: the group writes nothing
  for (int r0 = 0; r0 < n; r0 += 64) {
    const int i = r0 + lane;
    int idx = i < n ? srt[st + i] : 0;
    if (idx < 0 || (int64_t)idx >= M) { idx = 0; bad = true; }       // malformed index: stay inside dy
    const int left = n - r0 < 64 ? n - r0 : 64;
    int q = 0;
    auto take = [&](auto deep) {
      constexpr int D = decltype(deep)::value;
      for (; q + D <= left; q += D) {
        anc_u32x2 v[D];
#pragma unroll
        for (int j = 0; j < D; ++j) v[j] = *(const anc_u32x2 *)(dy + (int64_t)__builtin_amdgcn_readlane(idx, q + j) * H + c0);
#pragma unroll
        for (int j = 0; j < D; ++j) {
          acc[0] = acc[0] + __uint_as_float(v[j].x << 16);
          acc[1] = acc[1] + __uint_as_float(v[j].x & 0xFFFF0000u);
          acc[2] = acc[2] + __uint_as_float(v[j].y << 16);
          acc[3] = acc[3] + __uint_as_float(v[j].y & 0xFFFF0000u);
        }
      }
    };
    take(std::integral_constant<int, 32>{});
    take(std::integral_constant<int, 8>{});
    take(std::integral_constant<int, 2>{});
    take(std::integral_constant<int, 1>{});
  }
  bad = __any((int)bad) != 0;
  if (bad || !live) return;
  if (compact != nullptr) {
    const anc_f32x4 o = {acc[0], acc[1], acc[2], acc[3]};
    *(anc_f32x4 *)(compact + (int64_t)g * H + c0) = o;
  } else {
    float *p = out + row * H + c0;
    const anc_f32x4 b = *(const anc_f32x4 *)p;
    const anc_f32x4 o = {b.x + acc[0], b.y + acc[1], b.z + acc[2], b.w + acc[3]};
    *(anc_f32x4 *)p = o;
  }
}

}  // namespace

extern "C" int anc_embed_dw_scatter(uint64_t cnt, uint64_t start, uint64_t gid, uint64_t srt, uint64_t dy,
                                    uint64_t out, uint64_t compact, int64_t M, int64_t V, int64_t H,
                                    uint64_t stream) {
  ANC_REQUIRE(cnt && start && gid && srt && dy && (out != 0) != (compact != 0),
              "anc_embed_dw_scatter: null pointer, or both / neither of out and compact given");
  ANC_REQUIRE(M > 0 && M < (1ll << 31) && H > 0 && H % 64 == 0 && H <= 65536 * (int64_t)kChunk && (out == 0 || V > 0),
              "anc_embed_dw_scatter: M=%lld, V=%lld, H=%lld (H must be a multiple of 64)", (long long)M,
              (long long)V, (long long)H);
  ANC_REQUIRE(((cnt | start | gid | srt) & 3) == 0 && (dy & 7) == 0 && ((out | compact) & 15) == 0,
              "anc_embed_dw_scatter: misaligned pointers");
  AncProfScope prof(ANC_PROF_MISC, anc_stream(stream));
  const int64_t waves = (H + kChunk - 1) / kChunk, wide = waves < 4 ? waves : 4;
  hipLaunchKernelGGL(k_embed_dw_scatter, dim3((unsigned)M, (unsigned)((waves + wide - 1) / wide)), dim3((unsigned)(64 * wide)), 0,
                     anc_stream(stream), (const int32_t *)cnt, (const int32_t *)start, (const int32_t *)gid,
                     (const int32_t *)srt, (const uint16_t *)dy, (float *)out, (float *)compact, (int)H, M, V);
  ANC_LAUNCH_CHECK();
  return ANC_OK;
}

// ---- token ids -> groups, on the host ------------------------------------------------------------
// Distinct ids in ascending order and, for each, its positions in their original order. Ids of a batch lie in a range
// not much larger than a vocabulary, so the order comes from a bitmap over the range: a word's prefix count plus
// the bits below an id is the id's rank, and one counting pass by rank sorts stably (8192 ids of 152 K: 25 us;
// comparison sorts took 200 us for this and again for the distinct ids). A range beyond 64 ids per
// token is sorted.
namespace {

// (the rank wants the popcount instruction, which the baseline instruction set does not have)
#if defined(__x86_64__) && !defined(__HIP_DEVICE_COMPILE__)
#define ANC_POPCNT __attribute__((target("popcnt")))
#else
#define ANC_POPCNT
#endif

struct IdRank {
  std::vector<uint64_t> bits;
  std::vector<int32_t> below;        // distinct ids before each word
  int64_t lo = 0, distinct = 0;
  bool ok = false;                   // false: the range is too wide for a bitmap
};
__attribute__((always_inline)) inline void rank_fill(IdRank &r, const int32_t *ids, int64_t n) {
  int32_t mn = ids[0], mx = ids[0];
  for (int64_t i = 1; i < n; ++i) { mn = ids[i] < mn ? ids[i] : mn; mx = ids[i] > mx ? ids[i] : mx; }
  r.lo = mn;
  const int64_t range = (int64_t)mx - mn + 1;
  if (range > 64 * n + 65536) return;
  r.bits.assign((size_t)((range + 63) / 64), 0);
  uint64_t *bits = r.bits.data();
  for (int64_t i = 0; i < n; ++i) { const uint64_t d = (uint64_t)(ids[i] - r.lo); bits[d >> 6] |= 1ull << (d & 63); }
  r.below.resize(r.bits.size());
  int32_t at = 0;
  for (size_t w = 0; w < r.bits.size(); ++w) { r.below[w] = at; at += __builtin_popcountll(bits[w]); }
  r.distinct = at;
  r.ok = true;
}
__attribute__((always_inline)) inline void rank_groups(const IdRank &r, const int32_t *ids, int64_t n, int32_t *srt, int32_t *start,
                                                       int32_t *cnt) {
  std::vector<int32_t> rank((size_t)n), at((size_t)r.distinct);
  const uint64_t *bits = r.bits.data();
  const int32_t *below = r.below.data();
  for (int64_t i = 0; i < n; ++i) {
    const uint64_t d = (uint64_t)(ids[i] - r.lo), w = d >> 6;
    const int32_t g = below[w] + __builtin_popcountll(bits[w] & ((1ull << (d & 63)) - 1));
    rank[(size_t)i] = g;
    ++cnt[g];
  }
  int32_t sum = 0;
  for (int64_t g = 0; g < r.distinct; ++g) { start[g] = at[(size_t)g] = sum; sum += cnt[g]; }
  for (int64_t i = 0; i < n; ++i) srt[at[(size_t)rank[(size_t)i]]++] = (int32_t)i;
}
void rank_emit(const IdRank &r, int32_t *out) {
  for (size_t w = 0; w < r.bits.size(); ++w)
    for (uint64_t m = r.bits[w]; m != 0; m &= m - 1) *out++ = (int32_t)(r.lo + (int64_t)w * 64 + __builtin_ctzll(m));
}
ANC_POPCNT void rank_fill_hw(IdRank &r, const int32_t *ids, int64_t n) { rank_fill(r, ids, n); }
ANC_POPCNT void rank_groups_hw(const IdRank &r, const int32_t *ids, int64_t n, int32_t *srt, int32_t *start, int32_t *cnt) {
  rank_groups(r, ids, n, srt, start, cnt);
}
bool hw_popcnt() {
#if defined(__x86_64__) && !defined(__HIP_DEVICE_COMPILE__)
  return __builtin_cpu_supports("popcnt");
#else
  return false;
#endif
}
IdRank make_rank(const int32_t *ids, int64_t n) {
  IdRank r;
  if (hw_popcnt()) rank_fill_hw(r, ids, n); else rank_fill(r, ids, n);
  return r;
}
int no_memory(const char *who, int64_t n) {
  anc_set_error("%s: no memory to group %lld ids", who, (long long)n);
  return ANC_ERR_ARG;
}

}  // namespace

extern "C" int anc_unique_ids(const int32_t *ids, int64_t n, int32_t *out, int64_t *n_out) try {
  ANC_REQUIRE(ids != nullptr && out != nullptr && n_out != nullptr && n >= 0 && n < (1ll << 31), "anc_unique_ids: bad arguments");
  *n_out = 0;
  if (n == 0) return ANC_OK;
  const IdRank r = make_rank(ids, n);
  if (r.ok) {
    rank_emit(r, out);
    *n_out = r.distinct;
    return ANC_OK;
  }
  std::vector<int32_t> v(ids, ids + n);
  std::sort(v.begin(), v.end());
  *n_out = (int64_t)(std::unique_copy(v.begin(), v.end(), out) - out);
  return ANC_OK;
} catch (const std::bad_alloc &) {
  return no_memory("anc_unique_ids", n);
}

extern "C" int anc_id_groups(const int32_t *ids, int64_t n, int32_t *srt, int32_t *start, int32_t *cnt, int32_t *gid,
                             int64_t *n_groups) try {
  ANC_REQUIRE(ids != nullptr && srt != nullptr && start != nullptr && cnt != nullptr && gid != nullptr && n_groups != nullptr &&
                  n >= 0 && n < (1ll << 31),
              "anc_id_groups: bad arguments");
  *n_groups = 0;
  if (n == 0) return ANC_OK;
  std::fill(start, start + n, 0);
  std::fill(cnt, cnt + n, 0);
  std::fill(gid, gid + n, 0);
  const IdRank r = make_rank(ids, n);
  if (r.ok) {
    if (hw_popcnt()) rank_groups_hw(r, ids, n, srt, start, cnt); else rank_groups(r, ids, n, srt, start, cnt);
    rank_emit(r, gid);
    *n_groups = r.distinct;
    return ANC_OK;
  }
  for (int64_t i = 0; i < n; ++i) srt[i] = (int32_t)i;
  std::stable_sort(srt, srt + n, [ids](int32_t a, int32_t b) { return ids[a] < ids[b]; });
  int64_t g = -1;
  for (int64_t i = 0; i < n; ++i) {
    if (i == 0 || ids[srt[i]] != gid[g]) { ++g; gid[g] = ids[srt[i]]; start[g] = (int32_t)i; }
    ++cnt[g];
  }
  *n_groups = g + 1;
  return ANC_OK;
} catch (const std::bad_alloc &) {
  return no_memory("anc_id_groups", n);
}
