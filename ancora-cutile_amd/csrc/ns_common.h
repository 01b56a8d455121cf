// Shared declarations of the Newton-Schulz GEMM kernels: the argument block, the
// epilogue kinds, the XCD-aware tile remap.
#pragma once
#include "common.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));

// B-operand fragment of v_mfma_f32_32x32x16_bf16 from a (k, n) row-major LDS tile: two
// ds_read_b64_tr_b16. Within each group of 16 lanes, lane i receives the i%4-th 16-bit element
// of the 8 bytes addressed by lanes i/4, i/4+4, i/4+8, i/4+12 of the group. With lane s of a
// group pointing at row k0 + s/4, columns n0 + 4*(s%4) .. +3, lane i therefore receives
// column n0 + i of rows k0 .. k0+3. `p0` addresses rows k0.., `p1` rows k0+4..; the result
// holds 8 consecutive k of one column, the layout the matrix instruction wants.
__device__ __forceinline__ bf16x8 anc_lds_tr_frag(const void *p0, const void *p1) {
  const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4 *)p0);
  const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4 *)p1);
  const s16x8 v = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  return __builtin_bit_cast(bf16x8, v);
}

// Two fp32 -> one dword of two bf16 (round to nearest even, v_cvt_pk_bf16_f32): a in the low half.
typedef __bf16 anc_bf16x2 __attribute__((ext_vector_type(2)));
typedef float anc_f32x2v __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t anc_pk_bf16(float a, float b) {
  const anc_f32x2v v = {a, b};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, anc_bf16x2));
}
// The bf16 pair of two values: hi = bf16(x), lo = bf16(x - hi), each packed as above.
__device__ __forceinline__ void anc_pk_pair(float a, float b, uint32_t &hi, uint32_t &lo) {
  hi = anc_pk_bf16(a, b);
  lo = anc_pk_bf16(a - __uint_as_float(hi << 16), b - __uint_as_float(hi & 0xFFFF0000u));
}

constexpr int kCondParts = 64;           // partial sums per matrix of the conditioning proxy
constexpr int kXcds = 8;

enum { EPI_GRAM = 0, EPI_BMAT = 1, EPI_BX = 2 };
enum { VAR_NONE = 0, VAR_UPDATE = 1, VAR_PLAIN = 2, VAR_UPDATE_T = 3, VAR_STREAM = 4, VAR_STATS = 5 };   // variants of the epilogue (1 .. 3: of EPI_BX)
enum { kStream128 = 1, kStream256 = 2 };                                                  // NsGemm::stream_out

// Workgroup id -> logical tile id such that logical ids [start(x), start(x+1)) run on XCD x
// (hardware deals consecutive workgroup ids round-robin over the 8 XCDs).
__device__ __forceinline__ int xcd_remap(int bid, int grid) {
  const int x = bid % kXcds, q = bid / kXcds;
  const int base = grid / kXcds, rem = grid % kXcds;
  return x * base + (x < rem ? x : rem) + q;
}

struct NsGemm {
  const uint16_t *A[2];      // high and low half of the operand whose rows are the output's rows
  const uint16_t *B[2];      // the same for the output's columns. GRAM, BMAT: one row per column, ld = K
                             // ("NT" product); BX: the iterate itself, (K, N) row-major, ld = N
  // 1: A[0] B[0]; 2: + A[0] B[1]; 3: + A[1] B[0]. With more than one term the terms advance together, 32 k at a
  // time: hh of k 0..15, hh of k 16..31, hl and lh of 16..31, hl and lh of 0..15. The halves of both operands are
  // then fetched once per K tile (4 fetches for 3 products instead of 6), and every kernel adds in this order.
  int nterms;
  int K;
  int ldA;                   // elements between consecutive rows of A; 0 means K (only the plain
                             // product sets it: its A is a K-range of a longer row)
  int64_t strideA, strideB;  // elements between consecutive matrices
  int tiles_m, tiles_n;
  int lower;                 // symmetric output: 64x64 blocks on and below the diagonal only, mirrored: 1 = by the workgroup that
                             // multiplied them, 2 (64-wide tiles) = by another that multiplies the same block again
  int plain_sum;             // plain product: 1 = write X32 = (A32, if not null, else 0) + A B and, if Yh is
                             // not null, its bf16 copy (RNE) to Yh; 0 = write X32 = A B
  int fits256;               // the chain's dims are multiples of 256 (and no flag says otherwise): 256-wide tiles may run
  int blk_r, blk_c;          // plain product and X = a X + B X: the tile sequence of a matrix runs block by block, blocks of
                             // blk_r x blk_c tiles (rows x columns): (tiles_m, 1) = column panel by column
                             // panel, (1, tiles_n) or 0 = row by row
  int M, N;                  // matrix dims of the chain (A, B are MxM; X is MxN)
  float ca, cb, cc;
  float *A32;                // (E,M,M) fp32 A            GRAM out, BMAT in
  // With a32_gated set the fp32 copy of A exists only for the matrices that a32_flag marks (a null
  // a32_flag marks none): GRAM writes A32 for those alone and BMAT takes the off-diagonal entries
  // of A from Fh (bf16) for every other matrix.
  int a32_gated;
  const int32_t *a32_flag;   // (E)
  uint16_t *Fh;              // (E,M,M) bf16 off-diag A   GRAM out
  uint16_t *Fl, *Bl;         // bf16 residuals of F and Boff; null unless this step splits them
  float *dA;                 // (E,M)   diag A            GRAM out, BMAT in
  uint16_t *Bh;              // (E,M,M) bf16 off-diag B   BMAT out
  float *dB;                 // (E,M)   diag B            BMAT out, BX in
  const uint16_t *Xh, *Xl;   // (E,M,N) current iterate as a bf16 pair, X = Xh + Xl   BX in
  int lo_zero;               // the input has no low half (a bf16 matrix): Xl is one zeroed 16-byte piece that every
                             // read of a low half goes to
  int stream_out;            // past the caches: on tiles of 256 (kStream256) what the launch writes, on tiles of 128 (kStream128) the
                             // iterate that BX writes and the A32 that BMAT reads
                             // (VAR_STREAM; rules of ns.hip, one answer per launch)
  uint16_t *Yh, *Yl;         // (E,M,N) next iterate as a bf16 pair   BX out, null on the last step
  float *X32;                // (E,M,N) fp32 result                   BX out on the last step, else null
  uint16_t *X16;             // (E,M,N) the result rounded to bf16, instead of X32
  const anc_muon_desc_t *upd;  // BX, last step only: if set, matrix e is the Newton-Schulz result of the
                             // weight upd[e] and the epilogue applies W -= lr*O to it (p32, p16) instead
                             // of writing X32
  const double *cond;        // null, or (E) the conditioning proxy's sum (see
                             // k_ns_cond): a matrix whose sum exceeds cond_thresh multiplies
                             // nterms_hard terms instead of nterms (its list is a prefix of the hard one)
  double cond_thresh;
  int nterms_hard;
  const int32_t *order;      // (E) or null (as they come): the matrix in each place of the launch's sequence of matrices
  // Second gate: a matrix flagged from its statistics (a spectrum spread over decades, many
  // moderately large columns, a low-rank signal over weak noise) multiplies nterms_wide terms;
  // wide_flag null or nterms_wide 0 = no such gate. It takes precedence over the gate above. With
  // lo_gated set, the residual outputs Fl / Bl are written for such matrices only (else for every
  // matrix when non-null).
  const int32_t *wide_flag;  // (E)
  int nterms_wide;
  int lo_gated;
  const float *scale;        // (E) or null. The operands are an unnormalised iterate U and the step
                             // acts on X = scale*U: GRAM multiplies its accumulator by scale^2, BX
                             // multiplies the accumulator and the epilogue's X by scale.
  // Panel layout of a bf16 matrix with R rows: element (r, c) at ((c / 32) * R + r) * 32 + c % 32,
  // i.e. 32-column panels, each (R, 32) row-major. The K tile of a product is one or two panels, so the
  // rows a tile fetches are one contiguous block instead of 64-byte pieces of rows that lie a
  // whole row pitch apart. R = M for every matrix of the chain. Everything the chain writes for itself (F, B, every
  // iterate after the input) is in this layout.
  int x_panel;               // the input iterate (operands X of GRAM and BX, Xh/Xl of the BX epilogue) is too
  // 8-bit low halves. Where the low half of a matrix's
  // iterate is never a matrix-core operand it is kept as one byte per element (anc_low8_encode), in the first M*N bytes of the matrix's Xl (Yl) region, panels of
  // (M, 32) bytes: the epilogue then reads and writes 3 instead of 4 bytes per element. A matrix
  // takes the format on the input side if l8_in > 0, it is not flagged in l8_wide and its proxy
  // sum (l8_cond, the units of cond_thresh) does not exceed l8_in; l8_out likewise for the output.
  // The launches that read an iterate must be given the threshold it was written with.
  const double *l8_cond;     // (E) or null (no matrix takes the format)
  const int32_t *l8_wide;    // (E) or null
  double l8_in, l8_out;
};


// Per-matrix statistics and flags were written by earlier kernels and are the same for every lane:
// read through the constant address space they come in by scalar loads, which neither occupy the
// vector memory counter nor wait behind the kernel's own vector traffic.
template <typename T> __device__ __forceinline__ T anc_ld_const(const T *p) {
  return *(const __attribute__((address_space(4))) T *)(p);
}

// Did the classification flag matrix e for the second gate?
__device__ __forceinline__ bool anc_ns_wide(const NsGemm &p, int e) {
  return p.wide_flag != nullptr && anc_ld_const(p.wide_flag + e) != 0;
}
// Does matrix e keep the fp32 copy of A (GRAM writes it, BMAT reads it)?
__device__ __forceinline__ bool anc_ns_has_a32(const NsGemm &p, int e) {
  if (p.A32 == nullptr) return false;
  return p.a32_gated == 0 || (p.a32_flag != nullptr && anc_ld_const(p.a32_flag + e) != 0);
}
// Is the low half of matrix e's iterate one byte per element (thresh = p.l8_in or p.l8_out)?
__device__ __forceinline__ bool anc_ns_low8(const NsGemm &p, int e, double thresh) {
  if (!(thresh > 0.0) || p.l8_cond == nullptr) return false;
  if (p.l8_wide != nullptr && anc_ld_const(p.l8_wide + e) != 0) return false;
  return !(anc_ld_const(p.l8_cond + e) > thresh);
}
// The 8-bit low half of y next to its high half h = bf16(y), in the integer space of the fp32 bit
// patterns, where rounding to bf16 is rounding to a multiple of 0x10000: d = bits(y) - (h << 16) lies
// in -0x8000 .. 0x8000, and q = (d + 0x80) >> 8 (capped at 127) is d rounded to 8 bits. The pair reads
// back as the float whose bits are (h << 16) + (q << 8): y to 24 bits, exponent carries and borrows
// included, no special cases. `htop` is h in the upper half of a dword (lower half zero).
__device__ __forceinline__ uint32_t anc_low8_encode(float y, uint32_t htop) {
  int d = (int)(__float_as_uint(y) - htop) + 0x80;
  d = d < 0x7FFF ? d : 0x7FFF;
  return ((uint32_t)d >> 8) & 0xFFu;
}
// x = Xh + Xl from htop and the byte q, sign-extended
__device__ __forceinline__ float anc_low8_decode(uint32_t htop, int q) {
  return __uint_as_float(htop + ((uint32_t)q << 8));
}
// The matrix in place e of a launch's sequence
__device__ __forceinline__ int anc_ns_matrix(const NsGemm &p, int e) { return p.order == nullptr ? e : anc_ld_const(p.order + e); }
// Number of accumulation terms of matrix e: p.nterms, or more for a matrix that a gate marks.
__device__ __forceinline__ int anc_ns_terms(const NsGemm &p, int e) {
  if (p.nterms_wide > 0 && anc_ns_wide(p, e)) return p.nterms_wide;
  if (p.cond == nullptr) return p.nterms;
  return anc_ld_const(p.cond + e) > p.cond_thresh ? p.nterms_hard : p.nterms;
}

// Up to 8 independent problems of the same kind (the same product of different shape groups)
// in one launch: tiles[k] workgroups belong to problem k. One launch over all groups keeps the
// CUs busy where separate launches would each end in a partly filled last wave.
#ifndef ANC_MAX_GROUPS
#define ANC_MAX_GROUPS 8
#endif
constexpr int kMaxGroups = ANC_MAX_GROUPS;
// G: problems there is room for. A launch's arguments travel to the device with it, 3.5 KB for eight problems (a chain of
// one (128,128) matrix, which the host's launches bound: 76.7 -> 73.4 us with room for one).
template <int G> struct NsGemmArgs {
  int n;
  int seq;                   // plain product: 1 = anc_seq_tile dealing, 0 = anc_group_tile
  int tiles[G];     // 0 past n
  NsGemm g[G];
  // fused weight update (problems with `upd` set): lr*shape_scale by descriptor scale index,
  // stochastic-rounding switch and seed, the step's control block (skip flag) or null
  float lr[ANC_MUON_MAX_SCALES];
  int sr;
  uint32_t seed_base;
  const anc_step_ctl_t *ctl;
};
using NsGemmMulti = NsGemmArgs<kMaxGroups>;
struct NsUpdate {
  float lr[ANC_MUON_MAX_SCALES];
  int sr;
  uint32_t seed_base;
  const anc_step_ctl_t *ctl;
};

// Workgroup id -> (problem, tile index inside the problem). Every XCD gets an eighth of every problem's tiles, a run
// of consecutive ones, problems in the order given (longest tiles first), so that all have the same mix and a
// problem's consecutive tiles -- the tiles of one matrix -- stay on one XCD. What a problem's count leaves over 8
// goes to the XCDs after those that the problems before it gave one more tile to, which is how the hardware deals the
// launch's workgroup ids: an XCD's counts add up to the workgroups it runs. (About ten scalar instructions per problem;
// a tile of the 256-wide symmetric kernel has a CU to itself and waits for them.)
template <int G>
__device__ __forceinline__ void anc_group_tile(const NsGemmArgs<G> &pm, int bid, int &g, int &L) {
  const int x = bid % kXcds;
  int q = bid / kXcds, off = 0;
#pragma unroll
  for (g = 0; g < G; ++g) {
    const int base = pm.tiles[g] / kXcds, rem = pm.tiles[g] % kXcds, xr = (x - off) & (kXcds - 1);
    const int c = base + (xr < rem ? 1 : 0);
    if (q < c || g + 1 >= pm.n) {
      L = xr * base + (xr < rem ? xr : rem) + q;
      return;
    }
    q -= c;
    off += rem;
  }
}

// The other dealing: the problems' tile sequences one after the other, cut into 8 contiguous runs,
// one per XCD. An XCD then works on one or two problems only and fetches their operands into its
// L2 once, where the dealing above makes every XCD fetch a part of every problem's operands. For
// launches whose tiles all cost the same (the plain product: one K length).
__device__ __forceinline__ void anc_seq_tile(const NsGemmMulti &pm, int bid, int grid, int &g, int &L) {
  int pos = xcd_remap(bid, grid);
  g = 0;
  while (g + 1 < pm.n && pos >= pm.tiles[g]) { pos -= pm.tiles[g]; ++g; }
  L = pos;
}

// One product of the chain for n <= kMaxGroups problems (ps[k] with batch size Es[k]) on the tiles that suit
// the launch (ns.hip: the rule), or on tiles of `force` (64, 128, 256; 0: the rule). Every choice gives the
// same bits. `upd` carries the scalars of the fused weight update for problems whose `upd` is set.
int anc_ns_gemm_multi(int epi, const NsGemm *ps, const int64_t *Es, int n, int force, hipStream_t s,
                      const NsUpdate *upd = nullptr);
// The kernels behind it. 256x256 tiles for the symmetric products, 128x256 for X = a X + B X
// (ns_gemm_big.hip; M and N multiples of 256); `by_rows`: X = a X + B X reads its B by rows k.
int anc_ns_gemm_big_multi(int epi, const NsGemm *ps, const int64_t *Es, int n, hipStream_t s, bool by_rows,
                          const NsUpdate *upd);
// Tiles of 64x64 (`tile` 64), 128x64 (kTile128x64) or 128x128 (128) outputs (ns_gemm_tile.hip; M and N multiples of 128);
// `plain`: the bare product.
constexpr int kTile128x64 = 12864;
int anc_ns_gemm_tile_multi(int epi, const NsGemm *ps, const int64_t *Es, int n, hipStream_t s, int tile, bool by_rows,
                           const NsUpdate *upd, bool plain, const struct NsStatOne *stat = nullptr);
// Bare fp32 products C[e] = A[e] B[e] on the same K loops; a_transposed: A is
// given as (K, M) row-major with row pitch ldA (and strideA between matrices), C = A^T B. The tiles are chosen
// by a rule of their own (pick_tile_plain); the bits are the same on all.
int anc_ns_gemm_plain(const NsGemm *ps, const int64_t *Es, int n, hipStream_t s, bool a_transposed);
int anc_ns_gemm_big_plain(const NsGemm *ps, const int64_t *Es, int n, hipStream_t s, bool a_transposed = false);
// Momentum of one weight as a bf16 pair (muon_elem.hip): high halves to d.u, low halves to `lo`, a sum of u*u per 4096
// elements to `fro`; leaves `d` in device memory at `desc_out` for the chain's last product.
int anc_launch_momentum_pair_one(const anc_muon_desc_t &d, float mom, int nesterov, uint64_t lo, double *fro,
                                 anc_muon_desc_t *desc_out, const anc_step_ctl_t *ctl, hipStream_t s);
