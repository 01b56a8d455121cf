// The products of the Newton-Schulz chain (A = X X^T, B = b A + c A A, X = a X + B X with their
// epilogues; see ns.hip for the arithmetic) on 64x64 and 128x128 tiles, and the bare product of the
// weight-gradient GEMM on the same tiles and on 128x64 ones: for launches that the 256-wide tiles of ns_gemm_big.hip
// would leave most of the chip idle, and for dims that are multiples of 128 only.
//
// What bounds it. Operand bytes come into LDS at some 20 .. 25 B per clock and CU with the L2 hits these launches have (50 .. 58
// where all hit, 12 where none does), and a wavefront has its instructions to issue, so a product lasts as long as the
// CU with the most tiles needs: a single 1024x1024 output is 10 tiles of 256x256 (10 CUs at work, 512 K-bytes each
// step) or 136 of 64x64 (136 CUs, 128), a quarter of the time although the operands are fetched four times as
// often. Which tile a launch takes is a rule of ns.hip (pick_tile, pick_tile_plain).
//
// Layout. NW = 4 or 8 wavefronts as 2 x NW/2, each WM x WN blocks of v_mfma_f32_32x32x16_bf16 (tile 64 WM x 16 NW WN). 128x128 tiles run on
// eight, four per SIMD with two workgroups on a CU: with half as many the matrix pipe was busy for 40 % of X = a X + B X of
// the projections of six 640-wide layers, and a wavefront waiting for its fragments or storing its outputs for the rest (that step
// 1230 -> 1201 us; chains of 24 x (512,512) on such tiles 354 -> 332, 42 x (640,640) 961 -> 913, 24 x (1152,1152) 1442 -> 1411).
// A stage is KP = 2 (64x64) or 1 panels of 32 k of both operands, 16 KiB (12 KiB of a 128x64 tile). Operands arrive in pieces of 16
// rows x 64 bytes, one LDS-DMA instruction each. Stages form a ring of four, two workgroups per CU (three of 128x64
// tiles); 64x64 tiles that outnumber the CUs run on a ring of three, three workgroups per CU, whose
// K loops and epilogues overlap (chains of five steps: 16 x (512,512) 358 -> 331 us, 4 x (1024,3072) 625 ->
// 570 us; a single (512,1536), one workgroup per CU, loses 3 % to the shorter ring).
// An operand whose rows are tile rows ("NT") lies in LDS as [panel][row][64 bytes] with the 16-byte chunk index
// XORed with bits 2..3 of the row; an operand whose rows are k (the iterate in X = a X + B X, its symmetric B
// from M = 1024 on, activations and output gradients) lies as [32-column block][k][64 bytes] without a swizzle:
// a transposing read touches 4 rows x 64 contiguous bytes, all banks once.
// In panel layout both are contiguous in memory as well.
//
// Epilogue: block by block through a 32x36 fp32 buffer of the wavefront, so that a lane holds 16
// consecutive columns of a row (or, for mirrored halves, transposed weights and their transposed copies, 16
// consecutive rows of a column): a 32x32 block in panel layout is 2 KiB contiguous.
//
// Same bits as the 256-wide tiles: one accumulator, k ascending, the terms of a step together, and a symmetric product is
// computed directly inside the 64x64 blocks on the diagonal and mirrored from below, where residual terms make element
// (i, j) and element (j, i) differ in the last bit. (Blocks of 256 before: 24 x (256,512) 150 -> 131 us per chain, 12 x
// (512,1536) 424 -> 354 us with the order of the several terms' reads below.)
#include <type_traits>

#include "lds_dma.h"
#include "ns_common.h"
#include "ns_stats.h"

namespace {

constexpr int kSgPitch = 36;                              // floats per row of the epilogue buffer

// BYTES (4, 8 or 16) between memory and registers, one instruction.
template <int BYTES>
__device__ __forceinline__ void ld_run(const void *p, uint32_t *w) {
  if constexpr (BYTES == 16) { const anc_u32x4 t = *(const anc_u32x4 *)p; w[0] = t.x; w[1] = t.y; w[2] = t.z; w[3] = t.w; }
  else if constexpr (BYTES == 8) { const anc_u32x2 t = *(const anc_u32x2 *)p; w[0] = t.x; w[1] = t.y; }
  else w[0] = *(const uint32_t *)p;
}
// (STREAM: past the caches)
template <int BYTES, bool STREAM = false>
__device__ __forceinline__ void st_run(void *p, const uint32_t *w) {
  auto st = [](auto *q, auto v) {
    if constexpr (STREAM) anc_st_stream(q, v);
    else *q = v;
  };
  if constexpr (BYTES == 16) st((anc_u32x4 *)p, anc_u32x4{w[0], w[1], w[2], w[3]});
  else if constexpr (BYTES == 8) st((anc_u32x2 *)p, anc_u32x2{w[0], w[1]});
  else st((uint32_t *)p, w[0]);
}

// What the weight update reads and writes once: past the caches where a launch has many tiles (WIDE: the 128-wide ones), so
// that the operands stay in them. The full step of a model of 4 layers, hidden size 512: 602 -> 576 us.
template <bool WIDE, typename T> __device__ __forceinline__ T ld_once(const T *p) {
  if constexpr (WIDE) return anc_ld_stream(p);
  else return *p;
}
template <bool WIDE, typename T> __device__ __forceinline__ void st_once(T *p, T v) {
  if constexpr (WIDE) anc_st_stream(p, v);
  else *p = v;
}

// Workgroups a CU takes: what its 160 KiB of LDS hold, but not more than two rings of four 16 KiB stages. (wm, wn: 64-row and
// 64-column blocks of a tile)
constexpr int tile_per_cu(int wm, int wn, int ring) { return (wm == 1 ? ring == 3 : wn == 1) ? 3 : 2; }

// Tiles on and below the diagonal in the first `rows` rows of square tiles
__host__ __device__ constexpr int anc_sym_tiles(int rows) { return rows * (rows + 1) / 2; }

// SOLO: the launch has one problem, its arguments lie at fixed places.
// VAR_STATS (B = b A + c A A of one matrix): the workgroups behind the tiles make the gates' statistics.
// (by specialisation: an expression in the kernel's signature enters its name, and an unnamed enum has other names there on the host)
template <int VAR, bool SOLO> struct TileArgs { using type = NsGemmArgs<SOLO ? 1 : kMaxGroups>; };
template <> struct TileArgs<VAR_STATS, true> { using type = NsStatArgs; };
template <int EPI, int WM, int WN, int NW, bool AT, int VAR, int kRing, bool SOLO>
__global__ void __launch_bounds__(64 * NW, tile_per_cu(WM, WN * NW / 4, kRing) * NW / 4) k_ns_gemm_tile(typename TileArgs<VAR, SOLO>::type pm) {
  constexpr int WC = NW / 2, TM = 64 * WM, TN = 32 * WN * WC, KP = WM == 1 ? 2 : 1, TK = 32 * KP;
  constexpr bool BT = EPI == EPI_BX, PLAINV = VAR == VAR_PLAIN;
  constexpr int kHalf = TM * TK * 2, kStageBytes = kHalf + TN * TK * 2;      // A's part of a stage, a stage
  constexpr int PA = TM * KP / (16 * NW), PB = TN * KP / (16 * NW), kIps = PA + PB;        // DMA instructions per wavefront and stage
  static_assert(!AT || BT, "A by rows k: X = a X + B X and the plain product only");
  __shared__ __attribute__((aligned(1024))) unsigned char lds[kRing * kStageBytes];

  int gsel = 0, L;
  if constexpr (VAR == VAR_STATS) {
    static_assert(SOLO && NW == 4 && sizeof(lds) >= sizeof(ColLds), "a statistic's workgroup");
    if ((int)blockIdx.x >= pm.tiles_only) {
      stat_block(pm.stat, (int)blockIdx.x - pm.tiles_only, lds);
      return;
    }
    L = xcd_remap((int)blockIdx.x, pm.tiles_only);
  } else if constexpr (SOLO) L = xcd_remap((int)blockIdx.x, (int)gridDim.x);
  else if (PLAINV && pm.seq) anc_seq_tile(pm, (int)blockIdx.x, (int)gridDim.x, gsel, L);
  else anc_group_tile(pm, (int)blockIdx.x, gsel, L);
  const NsGemm &p = pm.g[gsel];
  int e = 0, tm, tn;
  constexpr bool kImages = EPI != EPI_BX && WM == 1 && kRing == 4;      // (see NsGemm::lower)
  bool image = false;
  // (the blocks' edges are powers of two; a division of two variables is 40 instructions, and a launch that this
  // kernel is made for has little else to do)
  const int sr = __builtin_ctz(p.blk_r), sc_ = __builtin_ctz(p.blk_c);
  if (EPI != EPI_BX) {
    // Tiles on and below the diagonal, in rows of blocks of blk_r x blk_c tiles, blk_r = blk_c: the whole blocks of a row, then the
    // tiles of its block on the diagonal. (Written with blk_r alone, 24 x (512,512) 323.0 -> 325.2 us per chain.)
    static_assert(EPI == EPI_BX || TM == TN, "symmetric products: square tiles");
    const int tri = anc_sym_tiles(p.tiles_m), per = kImages && p.lower == 2 ? p.tiles_m * p.tiles_m : tri;
    if (L >= per) { e = L / per; L -= e * per; }
    const int on_diag = anc_sym_tiles(p.blk_r);
    int bm = 0, row = on_diag;
    image = kImages && L >= tri;
    while (!image && L >= row) { L -= row; row += p.blk_r * p.blk_c; ++bm; }
    const int whole = row - on_diag;
    if (image) {
      tn = L - tri;
      for (tm = 1; tn >= tm; ++tm) tn -= tm;
    } else if (L < whole) {
      const int i = L & (p.blk_r * p.blk_c - 1);
      tm = (bm << sr) + (i >> sc_);
      tn = ((L >> (sr + sc_)) << sc_) + (i & (p.blk_c - 1));
    } else {
      int i = L - whole, r = 0;
      while (i >= r + 1) { i -= r + 1; ++r; }
      tm = (bm << sr) + r;
      tn = (bm << sc_) + i;
    }
  } else {
    const int per = p.tiles_m * p.tiles_n, across = p.tiles_n >> sc_;
    if (L >= per) { e = L / per; L -= e * per; }
    const int b = L >> (sr + sc_), i = L & (p.blk_r * p.blk_c - 1);
    const int br = b / across, bc = b - br * across;
    tm = (br << sr) + (i >> sc_);
    tn = (bc << sc_) + (i & (p.blk_c - 1));
  }
  if constexpr (!PLAINV) e = anc_ns_matrix(p, e);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WC, wn = wave % WC;
  const int K = p.K, nk = (K + TK - 1) / TK;
  const int nterms = anc_ns_terms(p, e);
  // plain product only: K % 32 == 0, so with two panels per step the last step may hold one
  const bool half_tail = PLAINV && KP == 2 && (K & 63) != 0;

  // ---- DMA addressing. Bytes between rows and between 32-element panels of an operand.
  const int M = p.M, N = p.N;
  const bool a_pan = !PLAINV && (EPI != EPI_GRAM || p.x_panel != 0);
  const bool b_pan = !PLAINV && (EPI == EPI_BMAT || p.x_panel != 0);
  const int64_t panel = (int64_t)M * 64;
  const int64_t rpA = a_pan ? 64 : (int64_t)(p.ldA > 0 ? p.ldA : K) * 2, rpB = b_pan ? 64 : (int64_t)(BT ? N : K) * 2;
  const int64_t psA = a_pan ? panel : 64, psB = b_pan ? panel : 64;
  const int dr = lane >> 2, dc = lane & 3;
  const uint32_t voA = (uint32_t)(dr * rpA) + (AT ? dc : dc ^ (dr >> 2)) * 16;
  const uint32_t voB = (uint32_t)(dr * rpB) + (BT ? dc : dc ^ (dr >> 2)) * 16;
  int64_t offA[PA], offB[PB], lA[PA], lB[PB], cutA[PA], cutB[PB];     // this wavefront's pieces; cut: see half_tail
#pragma unroll
  for (int j = 0; j < PA; ++j) {
    const int q = wave * PA + j, pa = AT ? q / (TK / 16) : q / (TM / 16), ra = AT ? q % (TK / 16) : q % (TM / 16);
    offA[j] = pa * psA + ra * 16 * rpA;
    lA[j] = offA[j] + voA;
    cutA[j] = AT ? (ra >= 2 ? 32 * rpA : 0) : (pa >= 1 ? psA : 0);
  }
#pragma unroll
  for (int j = 0; j < PB; ++j) {
    const int q = wave * PB + j, pb = BT ? q / (TK / 16) : q / (TN / 16), rb = BT ? q % (TK / 16) : q % (TN / 16);
    offB[j] = pb * psB + rb * 16 * rpB;
    lB[j] = offB[j] + voB;
    cutB[j] = BT ? (rb >= 2 ? 32 * rpB : 0) : (pb >= 1 ? psB : 0);
  }
  const int64_t baseA = (int64_t)e * p.strideA * 2 + (AT ? (int64_t)(tm * (TM / 32)) * psA : (int64_t)tm * TM * rpA);
  const int64_t baseB = (int64_t)e * p.strideB * 2 + (BT ? (int64_t)(tn * (TN / 32)) * psB : (int64_t)tn * TN * rpB);
  const int64_t advA = AT ? TK * rpA : KP * psA, advB = BT ? TK * rpB : KP * psB;
  const char *curA = (const char *)p.A[0] + baseA, *curB = (const char *)p.B[0] + baseB;
  int is_kt = 0;
  // Adding up addresses in scalar registers leaves the vector pipe to the matrix instructions; a wavefront that has its
  // SIMD to itself is quicker without the longer chain of scalar instructions (the step of one (1024,3072) weight: 1.4 % slower with it).
  // (`lane_at`: at + off)
  auto dma = [&](const char *g, int64_t at, int64_t lane_at, uint32_t off, uint32_t lds_base) {
    if (WM == 1 && kRing == 4) dma16(g + lane_at, lds_base);
    else                       dma16(g + at, off, lds_base);
  };
  auto piece = [&](int i, unsigned char *st, bool whole = false) {      // DMA instruction i of a stage: PA of A, PB of B
    const bool cut = !whole && half_tail && is_kt + 1 == nk;            // (the missing panel's pieces fetch the one that is there)
    if (i < PA) {
      dma(curA - (cut ? cutA[i] : 0), offA[i], lA[i], voA, lds_addr(st + (wave * PA + i) * 1024));
    } else {
      const int j = i - PA;
      dma(curB - (cut ? cutB[j] : 0), offB[j], lB[j], voB, lds_addr(st + kHalf + (wave * PB + j) * 1024));
    }
  };
  auto advance = [&]() { curA += advA; curB += advB; ++is_kt; };
  // A 128-wide tile on the diagonal of a symmetric product: its two operands are the same rows, so A's alone are fetched
  // and B's fragments come from A's part of a stage (42 x (640,640) 978 -> 968 us per chain). 64-wide tiles lose by
  // the second K loop: 16 x (768,768) 593 -> 611.
  constexpr bool kDiag = EPI != EPI_BX && WM > 1;
  const bool on_diag = kDiag && tm == tn;

  // ---- fragment addressing: tr = [block][k][64 B] by transposing reads, else [panel][row][64 B]
  const int l31 = lane & 31, hh = lane >> 5, g16 = lane >> 4, s16 = lane & 15;
  const int tr_lane = (8 * (g16 >> 1) + (s16 >> 2)) * 64 + 32 * (g16 & 1) + 8 * (s16 & 3);
  // (rows_k: k rows of a block in the stage; rows: the operand's rows per panel)
  auto frag = [&](auto tr, const unsigned char *half, int blk, int kk, int rows_k, int rows) -> bf16x8 {
    if constexpr (decltype(tr)::value) {
      const unsigned char *q = half + blk * (rows_k * 64) + kk * 16 * 64 + tr_lane;
      return anc_lds_tr_frag(q, q + 4 * 64);
    } else {
      return *(const bf16x8 *)(half + (kk >> 1) * (rows * 64) + (blk * 32 + l31) * 64 + ((((kk & 1) * 2 + hh) ^ ((l31 >> 2) & 3)) * 16));
    }
  };
  using TrA = std::bool_constant<AT>;
  using TrB = std::bool_constant<BT>;

  // ---- what the epilogue of X = a X + B X reads at the output position is requested before the K loop, so that it has
  // arrived when the loop ends (one (256,512) matrix 124.8 -> 121.5 us per chain against fetching it behind the loop; B = b A +
  // c A A reads half as much, and only launches of one workgroup per CU gain by it, kEarlyA). The loads are older than
  // every DMA below, so the waits of the ring hold. Eight wavefronts have no
  // registers for it (16 .. 32 would spill, 42 x (640,640) 913 -> 970) and request it behind the loop, all blocks at once.
  const int64_t mm = (int64_t)e * M * M, mn = (int64_t)e * M * N, mv = (int64_t)e * M;
  float *sg = (float *)lds + wave * 32 * kSgPitch;
  float sc = 1.0f;
  if (EPI != EPI_BMAT && !PLAINV && p.scale != nullptr) sc = anc_ld_const(p.scale + e);
  const float acc_scale = (EPI == EPI_GRAM) ? sc * sc : sc;
  const bool write_lo = (EPI == EPI_GRAM ? p.Fl != nullptr : EPI == EPI_BMAT ? p.Bl != nullptr : false) &&
                        (p.lo_gated == 0 || anc_ns_wide(p, e));
  const bool has_a32 = EPI != EPI_BX && anc_ns_has_a32(p, e);
  const bool in8 = EPI == EPI_BX && !PLAINV && anc_ns_low8(p, e, p.l8_in);
  const bool out8 = EPI == EPI_BX && !PLAINV && anc_ns_low8(p, e, p.l8_out);
  // This lane's 16 elements of a 32x32 block: NR runs of RUN consecutive columns (reading the block transposed, rows),
  // run r in row lrow + RS r from column c0. 32/RUN neighbouring lanes share a row, so that one instruction covers
  // whole lines.
  constexpr int RUN = (PLAINV || VAR == VAR_UPDATE) ? 4 : 8, NR = 16 / RUN, LPR = 32 / RUN, RS = 64 / LPR;
  const int lrow = lane / LPR, c0 = (lane % LPR) * RUN;
  const int gi_w = tm * TM + wm * (32 * WM), gj_w = tn * TN + wn * (32 * WN);
  // symmetric output: this wavefront's block lies above the 64x64 blocks of the diagonal (nobody needs it), or below
  const bool idle = EPI != EPI_BX && WM > 1 && (gi_w >> 6) < (gj_w >> 6), mirror = EPI != EPI_BX && (gi_w >> 6) > (gj_w >> 6) && (!kImages || p.lower != 2 || image);
  // run 0 of block b in a matrix of M rows in panel layout (run r: RS * 32 r further)
  auto pan_of = [&](int b) { return ((int64_t)((gj_w + (b % WN) * 32) / 32) * M + gi_w + (b / WN) * 32 + lrow) * 32 + c0; };
  constexpr int NB = WM * WN;
  uint32_t pre_h[NB][8], pre_l[NB][8];                  // 16 bf16, or (pre_l, 8-bit low halves) 16 bytes in the first 4
  float drow[WM][NR];
  // With several terms the K loop brings both halves of all rows of the tile's columns of X through LDS, those at the output position
  // among them: they are kept in registers as they pass, and X is not read again behind the loop (a launch over the
  // projections of six 640-wide layers reads 295 MB instead of 368, 109 -> 106 us, the last one with the weight update 140 -> 134; chains of
  // 24 x (640,1792) 1016 -> 1010, 24 x (512,512) 309 -> 304, 40 x (256,768) 248 -> 240; the full step of a model of 4 layers, hidden size 512,
  // 526 -> 524, within what its runs differ by). One workgroup per CU (the ring of four) has them earlier by a request before the loop. Eight wavefronts make room by
  // sharing the registers of a step's low fragments (kShare); four have it, and lose by the sharing (4 x (512,1536) 180 -> 184 us per chain).
  constexpr bool kKeep = EPI == EPI_BX && !PLAINV && (NW == 8 || kRing == 3), kShare = EPI == EPI_BX && NW == 8;
  if constexpr (EPI == EPI_BX && !PLAINV && NW == 4) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      if (kKeep && nterms > 1) break;
      const int64_t xo = mn + (p.x_panel ? pan_of(b) : (int64_t)(gi_w + (b / WN) * 32 + lrow) * N + gj_w + (b % WN) * 32 + c0);
      const int64_t xr = p.x_panel ? RS * 32 : (int64_t)RS * N;
#pragma unroll
      for (int r = 0; r < NR; ++r) ld_run<RUN * 2>(p.Xh + xo + r * xr, &pre_h[b][r * (RUN / 2)]);
      if (in8) {
#pragma unroll
        for (int r = 0; r < NR; ++r)
          ld_run<RUN>((const char *)p.Xl + mn * 2 + pan_of(b) + r * RS * 32, &pre_l[b][r * (RUN / 4)]);
      } else if (!p.lo_zero) {
#pragma unroll
        for (int r = 0; r < NR; ++r) ld_run<RUN * 2>(p.Xl + xo + r * xr, &pre_l[b][r * (RUN / 2)]);
      }
    }
#pragma unroll
    for (int bi = 0; bi < WM; ++bi)
#pragma unroll
      for (int r = 0; r < NR; ++r) drow[bi][r] = p.dB[mv + gi_w + bi * 32 + lrow + RS * r];
  }
  // (the master's block, or what the plain product adds to, too where registers allow: one block per wavefront)
  const bool plain_add = PLAINV && p.plain_sum && p.A32 != nullptr;
  anc_f32x4 wpre[4];
  if constexpr (VAR == VAR_UPDATE && NB == 1) {
    const anc_muon_desc_t &d = p.upd[e];
    const bool wtr = d.transpose != 0;
    const int64_t we = (int64_t)((wtr ? gj_w : gi_w) + lrow) * d.N + (wtr ? gi_w : gj_w) + c0;
#pragma unroll
    for (int r = 0; r < 4; ++r) wpre[r] = *(const anc_f32x4 *)((const float *)d.p32 + we + (int64_t)r * RS * d.N);
  }
  if constexpr (PLAINV && NB == 1) {
    if (plain_add) {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        wpre[r] = *(const anc_f32x4 *)(p.A32 + mn + (int64_t)(gi_w + lrow + RS * r) * N + gj_w + c0);
    }
  }

  // A at the output position, with at most one workgroup per CU
  constexpr bool kEarlyA = EPI == EPI_BMAT && NB == 1 && kRing == 4;
  anc_f32x4 a32[4];
  float pre_di[NR], pre_dj[RUN];
  if constexpr (kEarlyA) {
    if (has_a32) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        a32[i] = *(const anc_f32x4 *)(p.A32 + mm + (int64_t)(gi_w + lrow + RS * (4 * i / RUN)) * M + gj_w + c0 + 4 * i % RUN);
    } else {
#pragma unroll
      for (int r = 0; r < NR; ++r) ld_run<RUN * 2>(p.Fh + mm + pan_of(0) + r * RS * 32, &pre_h[0][r * (RUN / 2)]);
    }
#pragma unroll
    for (int r = 0; r < NR; ++r) pre_di[r] = p.dA[mv + gi_w + lrow + RS * r];
#pragma unroll
    for (int c = 0; c < RUN; c += 4) {
      const anc_f32x4 w = *(const anc_f32x4 *)(p.dA + mv + gj_w + c0 + c);
      pre_dj[c] = w.x; pre_dj[c + 1] = w.y; pre_dj[c + 2] = w.z; pre_dj[c + 3] = w.w;
    }
  }

  f32x16 acc[WM][WN];
#pragma unroll
  for (int bi = 0; bi < WM; ++bi)
#pragma unroll
    for (int bj = 0; bj < WN; ++bj)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[bi][bj][r] = 0.0f;

  auto mma = [&](const bf16x8 (&a)[WM], const bf16x8 (&b)[WN]) {
#pragma unroll
    for (int bi = 0; bi < WM; ++bi)
#pragma unroll
      for (int bj = 0; bj < WN; ++bj)      // operands exchanged: a lane ends with runs of 4 columns of one row
        acc[bi][bj] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b[bj], a[bi], acc[bi][bj], 0, 0, 0);
  };

  auto frags = [&](const unsigned char *st, int kk, bf16x8 (&fa)[WM], bf16x8 (&fb)[WN]) {
#pragma unroll
    for (int i = 0; i < WM; ++i) fa[i] = frag(TrA{}, st, wm * WM + i, kk, TK, TM);
#pragma unroll
    for (int i = 0; i < WN; ++i) fb[i] = frag(TrB{}, st + (on_diag ? 0 : kHalf), wn * WN + i, kk, TK, TN);
  };
  // ---- one term. Step k lives in stage k % kRing.
  auto single = [&](auto one_operand) {
    constexpr int kI = decltype(one_operand)::value ? PA : kIps;      // DMA instructions per wavefront and stage
    auto issue = [&](unsigned char *st, bool whole = false) {
#pragma unroll
      for (int i = 0; i < kI; ++i) piece(i, st, whole);
      advance();
    };
    if constexpr (WM == 1) {
      // At the top of step k a wavefront waits for its own DMA of the step (the younger ones stay in flight), the
      // workgroup meets, and the DMA of step k + kRing - 1 goes out into the stage everybody has just left.
#pragma unroll
      for (int s0 = 0; s0 < kRing - 1; ++s0)
        if (s0 < nk) issue(lds + s0 * kStageBytes);
      auto body = [&](auto steady, int step, int s0) {
        constexpr bool kSteady = decltype(steady)::value;
        if (kSteady || step + kRing - 1 <= nk) wait_vm<(kRing - 2) * kI>(); else wait_vm<0>();
        lds_barrier();
        if (kSteady || step + kRing - 1 < nk) issue(lds + ((s0 + kRing - 1) % kRing) * kStageBytes, kSteady);
        const unsigned char *st = lds + s0 * kStageBytes;
        const bool cut = !kSteady && half_tail && step + 1 == nk;
#pragma unroll
        for (int kk = 0; kk < TK / 16; ++kk) {
          if (PLAINV && kk >= 2 && cut) break;
          bf16x8 a[WM], b[WN];
          frags(st, kk, a, b);
          mma(a, b);
        }
      };
      int step = 0;
      // Rounds in which even the last step's refill is a whole stage that is there, without a branch (one (1024,3072) matrix
      // 203 -> 194 us per chain, (1024,1024) 147 -> 142. Three workgroups per CU hide the branches, and lose 1 % by the
      // code: 4 x (1024,1024) 293 -> 297. Fragments a step ahead give nothing here either.)
      for (; kRing == 4 && step + 2 * kRing - 1 < nk; step += kRing) {
#pragma unroll
        for (int s0 = 0; s0 < kRing; ++s0) body(std::true_type{}, step + s0, s0);
      }
      for (; step < nk; step += kRing) {
#pragma unroll
        for (int s0 = 0; s0 < kRing; ++s0)
          if (step + s0 < nk) body(std::false_type{}, step + s0, s0);
      }
    } else {
      // Fragments are read into registers one step ahead. At the top of step k a wavefront waits for its own DMA of step
      // k + 1 and the workgroup meets: everybody has the fragments of step k, so its stage takes the DMA of step
      // k + kRing, which goes out between the matrix instructions together with the reads of step k + 1. (Weight
      // gradients of 896 tiles of 64 at 8192 tokens 88 -> 74 us. On 64x64 tiles, whose DMA is the bound, the
      // longer way to the first product costs 0.7 us and gives nothing.)
      constexpr int KK = TK / 16, U = kRing;
      static_assert(kRing == 4, "rounds of four");
      bf16x8 a[2][KK][WM], b[2][KK][WN];
#pragma unroll
      for (int s0 = 0; s0 < kRing; ++s0)
        if (s0 < nk) issue(lds + s0 * kStageBytes);
      if (kRing <= nk) wait_vm<(kRing - 1) * kI>(); else wait_vm<0>();
      lds_barrier();
      if (idle) {                        // (its share of the DMA, and the meetings)
        for (int step = 0, at = 0; step < nk; ++step) {
          if (step + kRing <= nk) wait_vm<(kRing - 2) * kI>(); else wait_vm<0>();
          lds_barrier();
          if (step + kRing < nk) issue(lds + at);
          at = at + kStageBytes == kRing * kStageBytes ? 0 : at + kStageBytes;
        }
      } else {
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) frags(lds, kk, a[0][kk], b[0][kk]);
        auto body = [&](auto steady, int step, auto s0v) {
          constexpr bool kSteady = decltype(steady)::value;
          constexpr int s0 = decltype(s0v)::value % kRing, x = decltype(s0v)::value % 2;
          const bool more = kSteady || step + 1 < nk, refill = kSteady || step + kRing < nk;
          if (kSteady || step + kRing <= nk) wait_vm<(kRing - 2) * kI>(); else wait_vm<0>();
          lds_barrier();
#pragma unroll
          for (int kk = 0; kk < KK; ++kk) {
            mma(a[x][kk], b[x][kk]);
            __builtin_amdgcn_sched_barrier(0);
            if (refill) {
#pragma unroll
              for (int i = kk * kI / KK; i < (kk + 1) * kI / KK; ++i) piece(i, lds + s0 * kStageBytes);
            }
            if (more) frags(lds + (s0 + 1) % kRing * kStageBytes, kk, a[1 - x][kk], b[1 - x][kk]);
            __builtin_amdgcn_sched_barrier(0);
          }
          if (refill) advance();
        };
        auto round = [&](auto steady, int step) {
          auto one = [&](auto s0) {
            if (decltype(steady)::value || step + decltype(s0)::value < nk) body(steady, step + decltype(s0)::value, s0);
          };
          one(std::integral_constant<int, 0>{});
          one(std::integral_constant<int, 1>{});
          one(std::integral_constant<int, 2>{});
          one(std::integral_constant<int, 3>{});
        };
        int step = 0;
        for (; step + U - 1 + kRing < nk; step += U) round(std::true_type{}, step);
        for (; step < nk; step += U) round(std::false_type{}, step);
      }
    }
  };
  // ---- K loop
  if (PLAINV || nterms == 1) {
    if constexpr (kDiag) {
      if (on_diag) single(std::true_type{});
      else single(std::false_type{});
    } else {
      single(std::false_type{});
    }
  } else {
    // ---- several terms: a step is one panel of 32 k of both halves of both operands, high stage then low stage.
    constexpr int kPanA = TM * 64, kPanB = TN * 64, kLow = kPanA + kPanB, kPair = 2 * kLow, kPairs = kRing * kStageBytes / kPair;
    constexpr int QA = TM / (16 * NW), QB = TN / (16 * NW);         // pieces per wavefront of a panel of A and of B
    int64_t oA[QA], oB[QB], vA[QA], vB[QB];
#pragma unroll
    for (int j = 0; j < QA; ++j) {
      const int q = wave * QA + j;
      oA[j] = (AT ? (q >> 1) * psA + (q & 1) * 16 * rpA : q * 16 * rpA);
      vA[j] = oA[j] + voA;
    }
#pragma unroll
    for (int j = 0; j < QB; ++j) {
      const int q = wave * QB + j;
      oB[j] = (BT ? (q >> 1) * psB + (q & 1) * 16 * rpB : q * 16 * rpB);
      vB[j] = oB[j] + voB;
    }
    const char *pAl = (const char *)p.A[1] + baseA, *pBl = (const char *)p.B[1] + baseB;
    const int64_t adA = AT ? 32 * rpA : psA, adB = BT ? 32 * rpB : psB;
    const int at_b = on_diag ? 0 : kPanA;
    auto terms = [&](auto nt, auto one_operand) {
      constexpr bool ONE = decltype(one_operand)::value;
      constexpr int NT = decltype(nt)::value, kIpp = ONE ? 2 * QA : NT == 3 ? 2 * (QA + QB) : QA + 2 * QB;   // DMA instructions per wavefront and step
      auto issue_pair = [&](unsigned char *st) {
#pragma unroll
        for (int j = 0; j < QA; ++j) {
          dma(curA, oA[j], vA[j], voA, lds_addr(st + (wave * QA + j) * 1024));
          if (NT == 3) dma(pAl, oA[j], vA[j], voA, lds_addr(st + kLow + (wave * QA + j) * 1024));
        }
#pragma unroll
        for (int j = 0; j < (ONE ? 0 : QB); ++j) {
          dma(curB, oB[j], vB[j], voB, lds_addr(st + kPanA + (wave * QB + j) * 1024));
          dma(pBl, oB[j], vB[j], voB, lds_addr(st + kLow + kPanA + (wave * QB + j) * 1024));
        }
        curA += adA; curB += adB; pAl += adA; pBl += adB;
      };
      const int np = K / 32;
      // The first fragments of step k are in registers when it begins, the others are read under its matrix
      // instructions (kShare: the low ones of k 0..15 take the place of those of 16..31, which leaves eight wavefronts the
      // registers for kKeep). Before its last product a wavefront waits for its own DMA of step k + 1 and the workgroup meets:
      // everybody has read stage k, which takes the DMA of step k + kPairs, and the next step's first fragments are read
      // under that product. B's fragments of k 0..15 and 16..31 change places from step to step.
#pragma unroll
      for (int s0 = 0; s0 < kPairs; ++s0)
        if (s0 < np) issue_pair(lds + s0 * kPair);
      if (kPairs <= np) wait_vm<(kPairs - 1) * kIpp>(); else wait_vm<0>();
      lds_barrier();
      if (idle) {
        for (int step = 0, at = 0; step < np; ++step) {
          if (step + kPairs <= np) wait_vm<(kPairs - 2) * kIpp>(); else wait_vm<0>();
          lds_barrier();
          if (step + kPairs < np) issue_pair(lds + at);
          at = at + kPair == kPairs * kPair ? 0 : at + kPair;
        }
        return;
      }
      bf16x8 ah[2][WM], bh[2][WN], al[kShare ? 1 : 2][WM], bl[kShare ? 1 : 2][WN];
      auto rd_a = [&](const unsigned char *half, int kk, bf16x8 (&f)[WM]) {
#pragma unroll
        for (int i = 0; i < WM; ++i) f[i] = frag(TrA{}, half, wm * WM + i, kk, 32, TM);
      };
      auto rd_b = [&](const unsigned char *half, int kk, bf16x8 (&f)[WN]) {
#pragma unroll
        for (int i = 0; i < WN; ++i) f[i] = frag(TrB{}, half, wn * WN + i, kk, 32, TN);
      };
      auto fence = []() { __builtin_amdgcn_sched_barrier(0); };
      rd_a(lds, 0, ah[0]);
      rd_b(lds + at_b, 0, bh[0]);
      // (see kKeep: the step's rows of X are those of block row bi of this wavefront's outputs)
      auto keep = [&](const unsigned char *st, int step) {
#pragma unroll
        for (int bi = 0; bi < WM; ++bi)
          if (step == (gi_w >> 5) + bi) {
#pragma unroll
            for (int bj = 0; bj < WN; ++bj) {
              const unsigned char *q = st + kPanA + (wn * WN + bj) * 2048 + lrow * 64 + c0 * 2;
#pragma unroll
              for (int r = 0; r < NR; ++r) {
                ld_run<RUN * 2>(q + r * RS * 64, &pre_h[bi * WN + bj][r * (RUN / 2)]);
                ld_run<RUN * 2>(q + kLow + r * RS * 64, &pre_l[bi * WN + bj][r * (RUN / 2)]);
              }
            }
          }
      };
      auto body = [&](auto steady, int step, auto s0v) {
        constexpr int s0 = decltype(s0v)::value % kPairs, x = decltype(s0v)::value % 2, y = 1 - x;
        const unsigned char *st = lds + s0 * kPair, *nx = lds + (s0 + 1) % kPairs * kPair;
        const bool more = decltype(steady)::value || step + 1 < np, refill = decltype(steady)::value || step + kPairs < np;
        rd_a(st, 1, ah[1]);
        rd_b(st + at_b, 1, bh[y]);
        if constexpr (kKeep) keep(st, step);
        fence();
        mma(ah[0], bh[x]);                                    // hh 0..15
        fence();
        if constexpr (kShare) {
          rd_b(st + kLow + at_b, 1, bl[0]);
          if (NT == 3) rd_a(st + kLow, 1, al[0]);
          fence();
          mma(ah[1], bh[y]);                                  // hh 16..31
          mma(ah[1], bl[0]);                                  // hl 16..31
          fence();
          rd_b(st + kLow + at_b, 0, bl[0]);
          fence();
          if (NT == 3) {
            mma(al[0], bh[y]);                                // lh 16..31
            fence();
            rd_a(st + kLow, 0, al[0]);
            fence();
            mma(ah[0], bl[0]);                                // hl 0..15
          }
        } else {
          rd_b(st + kLow + at_b, 1, bl[1]);
          if (NT == 3) rd_a(st + kLow, 1, al[1]);
          fence();
          mma(ah[1], bh[y]);
          fence();
          rd_b(st + kLow + at_b, 0, bl[0]);
          if (NT == 3) rd_a(st + kLow, 0, al[0]);
          fence();
          mma(ah[1], bl[1]);
          if (NT == 3) {
            mma(al[1], bh[y]);
            mma(ah[0], bl[0]);
          }
        }
        fence();
        if (decltype(steady)::value || step + kPairs <= np) wait_vm<(kPairs - 2) * kIpp>(); else wait_vm<0>();
        lds_barrier();
        if (refill) issue_pair(lds + s0 * kPair);
        if (NT == 3 && more) rd_a(nx, 0, ah[0]);
        if (more) rd_b(nx + at_b, 0, bh[y]);
        fence();
        if (NT == 3) mma(al[0], bh[x]);                       // lh 0..15
        else         mma(ah[0], bl[0]);                       // (of two terms: hl 0..15)
        fence();
        if (NT != 3 && more) rd_a(nx, 0, ah[0]);
      };
      constexpr int U = kPairs % 2 == 0 ? kPairs : 2 * kPairs;
      static_assert(U == 2 || U == 4 || U == 6, "rounds");
      auto round = [&](auto steady, int step) {
        auto one = [&](auto s0) {
          if (decltype(steady)::value || step + decltype(s0)::value < np) body(steady, step + decltype(s0)::value, s0);
        };
        one(std::integral_constant<int, 0>{});
        one(std::integral_constant<int, 1>{});
        if constexpr (U > 2) {
          one(std::integral_constant<int, 2>{});
          one(std::integral_constant<int, 3>{});
        }
        if constexpr (U > 4) {
          one(std::integral_constant<int, 4>{});
          one(std::integral_constant<int, 5>{});
        }
      };
      int step = 0;
      for (; step + U - 1 + kPairs < np; step += U) round(std::true_type{}, step);
      for (; step < np; step += U) round(std::false_type{}, step);
    };
    if (EPI == EPI_BX && nterms == 2) {
      terms(std::integral_constant<int, 2>{}, std::false_type{});
    } else if constexpr (kDiag) {
      if (on_diag) terms(std::integral_constant<int, 3>{}, std::true_type{});
      else terms(std::integral_constant<int, 3>{}, std::false_type{});
    } else {
      terms(std::integral_constant<int, 3>{}, std::false_type{});
    }
  }
  // (the requests from above once more: as one lambda they cost the 64-wide kernels 40 instructions, 1 % of the chain of
  // one (512,512) matrix)
  if constexpr (EPI == EPI_BX && !PLAINV && NW > 4) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      if (kKeep && nterms > 1) break;
      const int64_t xo = mn + (p.x_panel ? pan_of(b) : (int64_t)(gi_w + (b / WN) * 32 + lrow) * N + gj_w + (b % WN) * 32 + c0);
      const int64_t xr = p.x_panel ? RS * 32 : (int64_t)RS * N;
#pragma unroll
      for (int r = 0; r < NR; ++r) ld_run<RUN * 2>(p.Xh + xo + r * xr, &pre_h[b][r * (RUN / 2)]);
      if (in8) {
#pragma unroll
        for (int r = 0; r < NR; ++r)
          ld_run<RUN>((const char *)p.Xl + mn * 2 + pan_of(b) + r * RS * 32, &pre_l[b][r * (RUN / 4)]);
      } else if (!p.lo_zero) {
#pragma unroll
        for (int r = 0; r < NR; ++r) ld_run<RUN * 2>(p.Xl + xo + r * xr, &pre_l[b][r * (RUN / 2)]);
      }
    }
#pragma unroll
    for (int bi = 0; bi < WM; ++bi)
#pragma unroll
      for (int r = 0; r < NR; ++r) drow[bi][r] = p.dB[mv + gi_w + bi * 32 + lrow + RS * r];
  }
  __syncthreads();

  // ---- epilogue
  if (VAR == VAR_UPDATE && pm.ctl != nullptr && pm.ctl->skip != 0u) return;   // skipped step
  if (idle) return;
  float v[16];
  auto put_rows = [&]() {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const anc_f32x4 w = {v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]};
      *(anc_f32x4 *)(sg + (lrow + RS * (4 * i / RUN)) * kSgPitch + c0 + 4 * i % RUN) = w;
    }
    lds_wave_sync();
  };
  auto get_cols = [&]() {
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = sg[(c0 + i % RUN) * kSgPitch + lrow + RS * (i / RUN)];
  };
  auto unpack = [&](const uint32_t (&u)[8], float (&x)[16]) {
#pragma unroll
    for (int i = 0; i < 8; ++i) { x[2 * i] = __uint_as_float(u[i] << 16); x[2 * i + 1] = __uint_as_float(u[i] & 0xFFFF0000u); }
  };
  constexpr bool kStreamX = EPI == EPI_BX && VAR == VAR_STREAM;
  // 16 floats -> bf16 runs at out + r * step, and the residuals at lo likewise if not null
  auto put_bf16 = [&](uint16_t *out, uint16_t *lo, int64_t step) {
    uint32_t h[8], l[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if (lo != nullptr) anc_pk_pair(v[2 * i], v[2 * i + 1], h[i], l[i]);
      else h[i] = anc_pk_bf16(v[2 * i], v[2 * i + 1]);
    }
#pragma unroll
    for (int r = 0; r < NR; ++r) st_run<RUN * 2, kStreamX>(out + r * step, h + r * (RUN / 2));
    if (lo != nullptr) {
#pragma unroll
      for (int r = 0; r < NR; ++r) st_run<RUN * 2, kStreamX>(lo + r * step, l + r * (RUN / 2));
    }
  };
#pragma unroll
  for (int bi = 0; bi < WM; ++bi) {
#pragma unroll
    for (int bj = 0; bj < WN; ++bj) {
      const int gi0 = gi_w + bi * 32, gj0 = gj_w + bj * 32;
      const int gi = gi0 + lrow, gj = gj0 + c0;
      const int64_t pan = pan_of(bi * WN + bj), pst = RS * 32;
      // four consecutive columns from column gj + 4 i % RUN of row gi + RS (4 i / RUN), in a matrix with `pitch` columns
      auto quad = [&](int i, int64_t pitch) { return (int64_t)(gi + RS * (4 * i / RUN)) * pitch + gj + 4 * i % RUN; };
      if constexpr (PLAINV && NB > 1) {
        if (plain_add) {
#pragma unroll
          for (int i = 0; i < 4; ++i) wpre[i] = *(const anc_f32x4 *)(p.A32 + mn + quad(i, N));
        }
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const anc_f32x4 w = {acc[bi][bj][4 * q], acc[bi][bj][4 * q + 1], acc[bi][bj][4 * q + 2], acc[bi][bj][4 * q + 3]};
        *(anc_f32x4 *)(sg + l31 * kSgPitch + 8 * q + 4 * hh) = w;
      }
      lds_wave_sync();
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const anc_f32x4 w = *(const anc_f32x4 *)(sg + (lrow + RS * (4 * i / RUN)) * kSgPitch + c0 + 4 * i % RUN);
        v[4 * i] = w.x; v[4 * i + 1] = w.y; v[4 * i + 2] = w.z; v[4 * i + 3] = w.w;
      }
      lds_wave_sync();                       // the buffer is free again
      if constexpr (EPI != EPI_BX) {
        // A block on the diagonal: one of the lane's elements, at most, has its row for a column. Picked by selects,
        // not branches: these blocks are in the launch's longest workgroups.
        const bool diag = gi0 == gj0;
        auto on_diag = [&](int k) { return diag && lrow + RS * (k / RUN) == c0 + k % RUN; };
        float dv = 0.0f;
        int dc = -1;                         // its value and column
        if (EPI == EPI_GRAM) {
#pragma unroll
          for (int k = 0; k < 16; ++k) v[k] = v[k] * acc_scale;
          if (has_a32 && !image) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
              *(anc_f32x4 *)(p.A32 + mm + quad(i, M)) = anc_f32x4{v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]};
          }
          if (diag) {
#pragma unroll
            for (int k = 0; k < 16; ++k) {
              const bool on = on_diag(k);
              dv = on ? v[k] : dv;
              dc = on ? k % RUN : dc;
              v[k] = on ? 0.0f : v[k];
            }
            if (dc >= 0) p.dA[mv + gj + dc] = dv;
          }
        } else {
          float a[16];
          if (has_a32) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const anc_f32x4 w = kEarlyA ? a32[i] : ld_once<VAR == VAR_STREAM>((const anc_f32x4 *)(p.A32 + mm + quad(i, M)));
              a[4 * i] = w.x; a[4 * i + 1] = w.y; a[4 * i + 2] = w.z; a[4 * i + 3] = w.w;
            }
          } else {
            if constexpr (!kEarlyA) {
#pragma unroll
              for (int r = 0; r < NR; ++r) ld_run<RUN * 2>(p.Fh + mm + pan + r * pst, &pre_h[0][r * (RUN / 2)]);
            }
            unpack(pre_h[0], a);
          }
          if constexpr (!kEarlyA) {
#pragma unroll
            for (int i = 0; i < RUN; i += 4) {
              const anc_f32x4 w = *(const anc_f32x4 *)(p.dA + mv + gj + i);
              pre_dj[i] = w.x; pre_dj[i + 1] = w.y; pre_dj[i + 2] = w.z; pre_dj[i + 3] = w.w;
            }
#pragma unroll
            for (int r = 0; r < NR; ++r) pre_di[r] = p.dA[mv + gi + RS * r];
          }
#pragma unroll
          for (int r = 0; r < NR; ++r) {
            const float di = pre_di[r];
#pragma unroll
            for (int c = 0; c < RUN; ++c) {
              const int k = r * RUN + c;
              const bool on = on_diag(k);
              const float dd = di * di, da = di * a[k] + a[k] * pre_dj[c];         // symmetric in (i,j)
              const float a2 = v[k] + (on ? dd : da);
              v[k] = p.cb * (on ? di : a[k]) + p.cc * a2;
              dv = on ? v[k] : dv;
              dc = on ? c : dc;
              v[k] = on ? 0.0f : v[k];
            }
          }
          if (dc >= 0) p.dB[mv + gj + dc] = dv;
        }
        uint16_t *oh = EPI == EPI_GRAM ? p.Fh : p.Bh, *ol = EPI == EPI_GRAM ? p.Fl : p.Bl;
        if (!image) put_bf16(oh + mm + pan, write_lo ? ol + mm + pan : nullptr, pst);
        if (mirror) {                        // mirror image: rows gj0 .., 32-column panel gi0/32
          put_rows();
          get_cols();
          const int64_t pt = ((int64_t)(gi0 / 32) * M + gj0 + lrow) * 32 + c0;
          put_bf16(oh + mm + pt, write_lo ? ol + mm + pt : nullptr, pst);
          lds_wave_sync();
        }
      } else if constexpr (PLAINV) {
        if (p.plain_sum) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const anc_f32x4 w = plain_add ? wpre[i] : anc_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            v[4 * i] = w.x + v[4 * i]; v[4 * i + 1] = w.y + v[4 * i + 1];
            v[4 * i + 2] = w.z + v[4 * i + 2]; v[4 * i + 3] = w.w + v[4 * i + 3];
          }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const anc_f32x4 w = {v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]};
          __builtin_nontemporal_store(w, (anc_f32x4 *)(p.X32 + mn + quad(i, N)));
        }
        if (p.plain_sum && p.Yh != nullptr) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const anc_u32x2 h = {(anc_bf16_rne_bits(v[4 * i]) & 0xFFFFu) | (anc_bf16_rne_bits(v[4 * i + 1]) << 16),
                                 (anc_bf16_rne_bits(v[4 * i + 2]) & 0xFFFFu) | (anc_bf16_rne_bits(v[4 * i + 3]) << 16)};
            __builtin_nontemporal_store(h, (anc_u32x2 *)(p.Yh + mn + quad(i, N)));
          }
        }
      } else {
        // y = (a + dB) x + B X. Only the first iteration carries the input's scale.
        float x[16];
        unpack(pre_h[bi * WN + bj], x);
        if (in8) {
#pragma unroll
          for (int k = 0; k < 16; ++k)
            x[k] = anc_low8_decode(__float_as_uint(x[k]), (int)(pre_l[bi * WN + bj][k >> 2] << (24 - 8 * (k & 3))) >> 24);
        } else if (!p.lo_zero) {
          float xl[16];
          unpack(pre_l[bi * WN + bj], xl);
#pragma unroll
          for (int k = 0; k < 16; ++k) x[k] = x[k] + xl[k];
        }
        if (p.scale != nullptr) {
#pragma unroll
          for (int k = 0; k < 16; ++k) v[k] = (p.ca + drow[bi][k / RUN]) * (x[k] * sc) + v[k] * acc_scale;
        } else {
#pragma unroll
          for (int k = 0; k < 16; ++k) v[k] = (p.ca + drow[bi][k / RUN]) * x[k] + v[k];
        }
        if constexpr (VAR == VAR_UPDATE) {
          // W -= lr O on the block's 32x32 elements of the weight (transposed where the chain ran on W^T)
          const anc_muon_desc_t &d = p.upd[e];
          float *W32 = (float *)d.p32;
          uint16_t *W16 = (uint16_t *)d.p16, *W16t = (uint16_t *)d.p16t;
          const bool wtr = d.transpose != 0;
          const float wlr = pm.lr[d.scale_idx & (ANC_MUON_MAX_SCALES - 1)];
          const uint32_t wseed = pm.seed_base + d.seed + ((pm.sr & ANC_SR_STEP_SEED) ? ANC_SR_SEED_STRIDE * pm.ctl->t : 0u);
          const int wr0 = wtr ? gj0 : gi0, wc0 = wtr ? gi0 : gj0;
          const int64_t we = (int64_t)(wr0 + lrow) * d.N + wc0 + c0, wst = (int64_t)RS * d.N;
          anc_f32x4 pv[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) pv[r] = NB == 1 ? wpre[r] : ld_once<(WM > 1)>((const anc_f32x4 *)(W32 + we + r * wst));
          if (wtr) {
            put_rows();
            get_cols();
            lds_wave_sync();
          }
          uint32_t hw[8];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            float pp[4] = {pv[r].x, pv[r].y, pv[r].z, pv[r].w};
            uint32_t hb[4];
#pragma unroll
            for (int k4 = 0; k4 < 4; ++k4) {
              pp[k4] = pp[k4] - wlr * v[4 * r + k4];
              const uint64_t el = (uint64_t)(we + r * wst + k4);
              hb[k4] = ((pm.sr & ANC_SR_ON) ? anc_bf16_sr_bits(pp[k4], (uint32_t)(el >> 6), (uint32_t)(el & 63u), wseed)
                                            : anc_bf16_rne_bits(pp[k4])) & 0xFFFFu;
            }
            st_once<(WM > 1)>((anc_f32x4 *)(W32 + we + r * wst), anc_f32x4{pp[0], pp[1], pp[2], pp[3]});
            hw[2 * r] = hb[0] | (hb[1] << 16);
            hw[2 * r + 1] = hb[2] | (hb[3] << 16);
          }
          if (W16 != nullptr) {
#pragma unroll
            for (int r = 0; r < 4; ++r) st_once<(WM > 1)>((anc_u32x2 *)(W16 + we + r * wst), anc_u32x2{hw[2 * r], hw[2 * r + 1]});
          }
          if (W16t != nullptr) {             // the (N, K) bf16 copy: the block's columns as rows
            uint16_t *sh = (uint16_t *)sg;   // [32][40]
#pragma unroll
            for (int r = 0; r < 4; ++r) st_run<8>(sh + (lrow + RS * r) * 40 + c0, hw + 2 * r);
            lds_wave_sync();
#pragma unroll
            for (int i = 0; i < 8; ++i) {
              const uint16_t *q = sh + (c0 + (2 * i) % RUN) * 40 + lrow + RS * (2 * i / RUN);
              hw[i] = (uint32_t)q[0] | ((uint32_t)q[40] << 16);
            }
            lds_wave_sync();
#pragma unroll
            for (int r = 0; r < 4; ++r)
              st_once<(WM > 1)>((anc_u32x2 *)(W16t + (int64_t)(wc0 + lrow + RS * r) * d.K + wr0 + c0), anc_u32x2{hw[2 * r], hw[2 * r + 1]});
          }
        } else if (p.X32 != nullptr) {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            *(anc_f32x4 *)(p.X32 + mn + quad(i, N)) = anc_f32x4{v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]};
        } else if (p.X16 != nullptr) {
          put_bf16(p.X16 + mn + (int64_t)gi * N + gj, nullptr, (int64_t)RS * N);
        } else if (out8) {
          uint32_t h[8], q[4] = {0u, 0u, 0u, 0u};
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            h[i] = anc_pk_bf16(v[2 * i], v[2 * i + 1]);
            q[i >> 1] |= (anc_low8_encode(v[2 * i], h[i] << 16) | (anc_low8_encode(v[2 * i + 1], h[i] & 0xFFFF0000u) << 8)) << (16 * (i & 1));
          }
#pragma unroll
          for (int r = 0; r < NR; ++r) {
            st_run<RUN * 2, kStreamX>(p.Yh + mn + pan + r * pst, h + r * (RUN / 2));
            st_run<RUN, kStreamX>((char *)p.Yl + mn * 2 + pan + r * pst, q + r * (RUN / 4));
          }
        } else {
          put_bf16(p.Yh + mn + pan, p.Yl + mn + pan, pst);
        }
      }
    }
  }
}

// Weight gradients on 128x128 tiles, us at 288 / 432 / 768 / 1344 tiles of 64 (written), four / eight wavefronts: 768 tokens
// 10.4 / 9.5, 10.7 / 9.4, 11.4 / 10.6, 17.4 / 17.5; 2048 tokens 17.8 / 16.4, 18.7 / 16.6, 19.2 / 18.5, 34.9 / 35.8; 8192 tokens
// 54 / 52, 55 / 51, 61 / 57, 119 / 122, and 1024 tiles at 4096 tokens 36.8 / 39.7. Added up in two workgroups per CU, level up to
// 640 tokens (1536 tiles 15.6 / 15.7 at 384, 18.7 / 19.0 at 640), but with eight some of the cards took 16 .. 21 there.
constexpr int kLongPlain = 2048;

template <int EPI, bool AT, int VAR>
void launch_tile(int tile, unsigned grid, hipStream_t s, const NsGemmMulti &pm, const NsStatOne *stat = nullptr) {
  if constexpr (VAR == VAR_PLAIN) {
    if (tile == kTile128x64) {
      hipLaunchKernelGGL((k_ns_gemm_tile<EPI, 2, 1, 4, AT, VAR, 4, false>), dim3(grid), dim3(256), 0, s, pm);
      return;
    }
    // (see kLongPlain)
    const bool adds = pm.g[0].plain_sum != 0 && pm.g[0].A32 != nullptr;
    if (tile == 128 && (pm.g[0].K > kLongPlain || (adds && grid > 256 && grid <= 512))) {
      hipLaunchKernelGGL((k_ns_gemm_tile<EPI, 2, 2, 4, AT, VAR, 4, false>), dim3(grid), dim3(256), 0, s, pm);
      return;
    }
  }
  if constexpr (VAR == VAR_NONE && EPI != EPI_GRAM) {
    if (tile == 128 && (pm.g[0].stream_out & kStream128)) {
      hipLaunchKernelGGL((k_ns_gemm_tile<EPI, 2, 1, 8, AT, VAR_STREAM, 4, false>), dim3(grid), dim3(512), 0, s, pm);
      return;
    }
  }
  if (tile == 128)      hipLaunchKernelGGL((k_ns_gemm_tile<EPI, 2, 1, 8, AT, VAR, 4, false>), dim3(grid), dim3(512), 0, s, pm);
  else if (grid > 256)  hipLaunchKernelGGL((k_ns_gemm_tile<EPI, 1, 1, 4, AT, VAR, 3, false>), dim3(grid), dim3(256), 0, s, pm);
  else if (pm.n > 1)    hipLaunchKernelGGL((k_ns_gemm_tile<EPI, 1, 1, 4, AT, VAR, 4, false>), dim3(grid), dim3(256), 0, s, pm);
  else {
    NsStatArgs one;
    one.n = 1;
    one.seq = pm.seq;
    one.g[0] = pm.g[0];
    for (int k = 0; k < ANC_MUON_MAX_SCALES; ++k) one.lr[k] = pm.lr[k];
    one.sr = pm.sr;
    one.seed_base = pm.seed_base;
    one.ctl = pm.ctl;
    if constexpr (EPI == EPI_BMAT && VAR == VAR_NONE) {
      if (stat != nullptr) {
        one.tiles_only = (int)grid;
        one.stat = *stat;
        hipLaunchKernelGGL((k_ns_gemm_tile<EPI, 1, 1, 4, AT, VAR_STATS, 4, true>), dim3(grid + kCondParts + stat->parts), dim3(256), 0, s, one);
        return;
      }
    }
    hipLaunchKernelGGL((k_ns_gemm_tile<EPI, 1, 1, 4, AT, VAR, 4, true>), dim3(grid), dim3(256), 0, s, (const NsGemmArgs<1> &)one);
  }
}

}  // namespace

// n <= kMaxGroups problems of the same product in one launch on tiles of 64, 128 or 128x64 (kTile128x64). EPI_BX:
// `by_rows` as for the 256-wide tiles; `plain`: the bare product, A transposed (by_rows) or not.
int anc_ns_gemm_tile_multi(int epi, const NsGemm *ps, const int64_t *Es, int n, hipStream_t s, int tile, bool by_rows,
                           const NsUpdate *upd, bool plain, const NsStatOne *stat) {
  const int TM = tile == 64 ? 64 : 128, TN = tile == 128 ? 128 : 64;
  ANC_REQUIRE(plain || TM == TN, "anc_ns_gemm_tile: tiles of 128x64 are the plain product's");
  NsGemmMulti pm{};
  pm.n = n;
  int64_t grid = 0, full = 0, longest = 0;
  for (int k = 0; k < n; ++k) {
    full += Es[k] * (ps[k].M / 64) * (ps[k].M / 64);
    longest = ps[k].K > longest ? ps[k].K : longest;
  }
  // Where CUs are left over, a symmetric product's tile above the diagonal is a workgroup of its own, instead of a second, transposed
  // store behind the one below: the launch lasts as long as its longest workgroup, and a short K has nothing to hide the store
  // behind. The tiles fetched twice cost more the more workgroups share what they fetch and the longer K is. Measured, us per
  // chain, one workgroup per pair of tiles / one per tile in A = X X^T (K = N) and B / in B alone (tiles in all, tiles * K of A in Ki):
  //   up to 128 tiles  1 x (128,128) 78.7 / 75.1 (4, 1), 4 x (128,4096) 208.4 / 201.8 / 206.1 (16, 64), 1 x (256,256) 90.5 / 85.8 (16, 4), 8 x (256,512)
  //               100.7 / 98.1 / 99.2 (128, 64), 2 x (512,1536) 155.6 / 153.3 / 155.4 (128, 192), 16 x (128,3072) 216.4 / 214.1 / 214.5 (64, 192),
  //               32 x (128,1536) 191.7 / 190.3 / 189.9 (128, 192), 1 x (640,2048) 172.4 / 171.3 / 172.1 (100, 200), 3 x (384,2048) 176.6 /
  //               175.4 / 176.8 (108, 216); 1 x (640,2560) 190.8 / 192.0 / 191.0 (100, 250), 2 x (512,2048) 176.1 / 174.9 / 175.9 (128, 256), 8 x
  //               (256,2048) 173.9 / 173.3 / 172.7 (128, 256), 1 x (640,3072) 211.7 / 215.4 / 211.7 (100, 300), 8 x (256,3072) 218.4 / 221.6 / 217.6
  //               (128, 384), 2 x (512,4096) 256.1 / 261.7 / 255.7 (128, 512)
  //   more        64 x (128,128) 95.9 / 93.4 (256), 64 x (128,256) 110.8 / 108.4 / 108.7 (256), 16 x (256,256) 99.4 / 97.2 (256); 16 x (256,512) 120.4 /
  //               125.8 / 118.2 (256), 3 x (512,512) 121.4 / 120.8 (192), 7 x (384,384) 114.5 / 116.2 (252), 2 x (640,1024) 153.6 / 157.5 / 155.8
  //               (200), 4 x (512,512) 126.5 / 172.3 (256)
  const bool images = epi != EPI_BX && tile == 64 && (full <= 128 ? full * longest <= 225 << 10 : full <= 256 && longest <= 256);
  for (int k = 0; k < n; ++k) {
    NsGemm &g = pm.g[k];
    g = ps[k];
    ANC_REQUIRE(g.M % 128 == 0 && g.N % 128 == 0 && g.K % (plain ? 32 : 128) == 0 && g.K > 0,
                "anc_ns_gemm_tile: dims must be multiples of 128");
    g.tiles_m = g.M / TM;
    g.tiles_n = (epi == EPI_BX ? g.N : g.M) / TN;
    g.lower = epi == EPI_BX ? 0 : images ? 2 : 1;
    // walked in blocks of 256 x 256 (see launch_bx of the 256-wide kernel: what an XCD fetches)
    const int cols = epi == EPI_BX ? g.N : g.M;
    g.blk_r = (g.M % 256 == 0 ? 256 : 128) / TM;
    g.blk_c = (cols % 256 == 0 ? 256 : 128) / TN;
    const int64_t per = !g.lower || images ? (int64_t)g.tiles_m * g.tiles_n : anc_sym_tiles(g.tiles_m);
    ANC_REQUIRE(per > 0 && Es[k] * per < (1ll << 30), "anc_ns_gemm_tile: grid out of range");
    pm.tiles[k] = (int)(Es[k] * per);
    grid += pm.tiles[k];
  }
  ANC_REQUIRE(grid < (1ll << 31), "anc_ns_gemm_tile: grid out of range");
  ANC_REQUIRE(stat == nullptr || (n == 1 && epi == EPI_BMAT && tile == 64 && grid <= kStatTiles),
              "anc_ns_gemm_tile: statistics go with one matrix's B on tiles of 64");
  const unsigned gr = (unsigned)grid;
  if (plain) {
    if (by_rows) launch_tile<EPI_BX, true, VAR_PLAIN>(tile, gr, s, pm);
    else         launch_tile<EPI_BX, false, VAR_PLAIN>(tile, gr, s, pm);
  } else if (epi == EPI_GRAM) {
    launch_tile<EPI_GRAM, false, VAR_NONE>(tile, gr, s, pm);
  } else if (epi == EPI_BMAT) {
    launch_tile<EPI_BMAT, false, VAR_NONE>(tile, gr, s, pm, stat);
  } else if (upd != nullptr) {
    for (int k = 0; k < ANC_MUON_MAX_SCALES; ++k) pm.lr[k] = upd->lr[k];
    pm.sr = upd->sr;
    pm.seed_base = upd->seed_base;
    pm.ctl = upd->ctl;
    if (by_rows) launch_tile<EPI_BX, true, VAR_UPDATE>(tile, gr, s, pm);
    else         launch_tile<EPI_BX, false, VAR_UPDATE>(tile, gr, s, pm);
  } else {
    if (by_rows) launch_tile<EPI_BX, true, VAR_NONE>(tile, gr, s, pm);
    else         launch_tile<EPI_BX, false, VAR_NONE>(tile, gr, s, pm);
  }
  ANC_LAUNCH_CHECK();
  return ANC_OK;
}
