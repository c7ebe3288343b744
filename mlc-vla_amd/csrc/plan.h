// Host-side launch planners: how the attention, the skinny GEMM and the prefill tile GEMM
// split their work, and the workspace each plan needs.  Plain C++ (no HIP types), so that
// the plans and their invariants are checked by a CPU build under the sanitizers
// (tests/plan_check.cpp).
#pragma once

#include <algorithm>
#include <cstddef>

namespace mlcv {

// ---- joint attention (attn_impl.h) ------------------------------------------------------
constexpr int ATTN_ROWS = 64;  // query rows per workgroup
constexpr int ATTN_KCH = 32;   // keys per chunk

// Key splits of `rows` query rows against Sp prefix keys (+ one split for Ts > 0 suffix keys):
// about target_blocks workgroups, prefix splits of whole chunks, at most 31 of them, none
// empty.  *kps: prefix keys per split.
inline void attn_plan(int rows, int Sp, int Ts, int target_blocks, int* nsplit, int* kps) {
  const int rb = (rows + ATTN_ROWS - 1) / ATTN_ROWS;
  const int chunks = (Sp + ATTN_KCH - 1) / ATTN_KCH;
  int ns = (target_blocks + rb - 1) / rb - (Ts > 0 ? 1 : 0);
  ns = std::min(ns, 31);
  ns = std::min(ns, chunks);
  ns = std::max(ns, 1);
  const int cps = chunks > 0 ? (chunks + ns - 1) / ns : 1;
  *kps = cps * ATTN_KCH;
  *nsplit = (chunks > 0 ? (chunks + cps - 1) / cps : 0) + (Ts > 0 ? 1 : 0);
}

// Split partials of a plan: fp16 O [KV][nsplit][rpad][hd] in the first KV*nsplit*rpad*hd
// floats (half of them used), then fp32 (m, l) [KV][nsplit][rpad][2].  None for one split.
inline size_t attn_ws_floats(int KV, int rows, int hd, int nsplit) {
  const int rpad = ((rows + ATTN_ROWS - 1) / ATTN_ROWS) * ATTN_ROWS;
  return nsplit > 1 ? (size_t)KV * nsplit * rpad * (hd + 2) : 0;
}

// ---- float32 attention (attn_f32.hip) ------------------------------------------------------
constexpr int F32_ATTN_TARGET = 512;  // workgroups: two per CU
// Key splits of `rows` query rows per kv head against nk keys: about two workgroups per CU, at least
// two chunks per split (a split costs its partials and the combine launch), none empty.
// *cps: chunks per split.
inline void f32_attn_plan(int rows, int KV, int nk, int* nsplit, int* cps) {
  const int rb = (rows + ATTN_ROWS - 1) / ATTN_ROWS * KV, chunks = (nk + ATTN_KCH - 1) / ATTN_KCH;
  const int ns = std::max(1, std::min({F32_ATTN_TARGET / std::max(rb, 1), (chunks + 1) / 2, 64}));
  *cps = std::max(1, (chunks + ns - 1) / ns);
  *nsplit = std::max(1, (chunks + *cps - 1) / *cps);
}
// fp32 partials O [KV][nsplit][rpad][hd], then (m, l) [KV][nsplit][rpad][2]; none for one split
inline size_t f32_attn_ws_floats(int KV, int rows, int hd, int nsplit) {
  const size_t rpad = (size_t)((rows + ATTN_ROWS - 1) / ATTN_ROWS) * ATTN_ROWS;
  return nsplit > 1 ? (size_t)KV * nsplit * rpad * (hd + 2) : 0;
}

// ---- float32 linears (gemm_f32.hip) ---------------------------------------------------------
// Tile edge of the many-row kernel, or 0 for the few-row kernel's 16-row slabs: tiles where they fill the
// CUs (128 x 128 twice over: half the LDS traffic per flop).  Equally shaped linears over the same rows (a
// table: the modulations of up to 64 steps) are slabs at any size, the kernel that takes them all in one
// launch.
inline int f32_tile(int M, int N, bool table, int cus) {
  const long t128 = (long)((M + 127) / 128) * ((N + 127) / 128), t64 = (long)((M + 63) / 64) * ((N + 63) / 64);
  if (table) return 0;
  return M > 64 && t128 >= 2L * cus ? 128 : M > 32 && t64 >= cus ? 64 : 0;
}

// ---- skinny GEMM (gemm_skinny.hip) ------------------------------------------------------
constexpr int SK_KC = 128;        // k per chunk
constexpr int SK_MAX_SPLIT = 8;   // K slices at most

struct SkPlan {
  int splitk, kper;  // K slices, k per slice (whole chunks)
};

// splits > 0: that many K slices (at most one per chunk); otherwise enough slices for about
// one workgroup per CU of a 256-CU part, at most SK_MAX_SPLIT.  No slice is empty.
inline SkPlan sk_plan(int ntiles, int K, int mblocks, int splits) {
  const int chunks = (K + SK_KC - 1) / SK_KC;
  int want = splits;
  if (want <= 0) {
    const int blocks = std::max(ntiles * mblocks, 1);
    want = (256 + blocks - 1) / blocks;
  }
  want = std::min(want, SK_MAX_SPLIT);
  want = std::min(want, chunks);
  want = std::max(want, 1);
  const int cps = (chunks + want - 1) / want;
  SkPlan p;
  p.kper = cps * SK_KC;
  p.splitk = (chunks + cps - 1) / cps;
  return p;
}

// fp32 partials of a split plan: [ntiles][mblocks][splitk][tr x 64]
inline size_t sk_ws_floats(int ntiles, int mblocks, const SkPlan& p, int tr) {
  return p.splitk > 1 ? (size_t)ntiles * mblocks * p.splitk * tr * 64 : 0;
}

// fp32 partials of the modulation pieces on 64-row tiles (T >= 64 or more than 16 steps): layer
// 0's two norms, then the other NM - 2, of 3 W1 rows each.  The smaller piece takes more K slices,
// so either can need the larger workspace (at W1 = 1024: 96 tiles in 3 slices against none).
inline size_t sk_mod_ws_floats(int NM, int W1, int mblocks) {
  const int per = (3 * W1 + 63) / 64;
  size_t n = 0;
  for (int segs : {2, NM - 2}) {
    if (segs <= 0) continue;
    n = std::max(n, sk_ws_floats(segs * per, mblocks, sk_plan(segs * per, W1, mblocks, 0), 64));
  }
  return n;
}

// ---- prefill tile GEMM, 256-row tiles (gemm_tile.hip) -------------------------------------
constexpr int TG_BM = 256, TG_BK = 64, TG_NXCD = 8;

// ---- linears over a few hundred rows (gemm_mid.hip) ---------------------------------------
enum MidTile : int { MID_64x96 = 0, MID_64x64 = 1, MID_32x64 = 2, MID_32x32 = 3 };
// The tile with the least operand rows per CU, rounds of workgroups x (BM + BN): a CU takes its
// tiles' rows out of the L2 at a fixed rate.  n tile j runs on XCD j % 8 with all its m tiles.  Ties go
// to the larger tile.  *rows: that figure.  *rounds: tiles of the busiest CU.
inline int mid_plan(int M, int N, int cus, long* rows = nullptr, long* rounds = nullptr) {
  constexpr int BMS[4] = {64, 64, 32, 32}, BNS[4] = {96, 64, 64, 32};
  int best = 0;
  long least = 0;
  for (int i = 0; i < 4; ++i) {
    const long mt = (M + BMS[i] - 1) / BMS[i], nt = (N + BNS[i] - 1) / BNS[i];
    const long xcd = (nt + TG_NXCD - 1) / TG_NXCD * mt, per = std::max(cus / TG_NXCD, 1);  // tiles, CUs per XCD
    const long r = (xcd + per - 1) / per * (BMS[i] + BNS[i]);
    if (i == 0 || r < least) {
      best = i;
      least = r;
    }
  }
  if (rows) *rows = least;
  if (rounds) *rounds = least / (BMS[best] + BNS[best]);
  return best;
}

// Linears of the image tower that run on this kernel, not on the long-M tile GEMM (256 rows of 128 or 256
// outputs, K split) and an epilogue pass.  This kernel's tiles read more operand rows per product and K is not
// split, so it is the slower one past 1024 rows, in many rounds and at long K.  Towers, us, the tile GEMM and
// pass / this kernel for all linears: 4 layers of width 1152 of 256 patches 444 / 268, 1024 patches 654 / 646,
// 1369 patches 894 / 1060.  3 layers, and with this rule: width 1152 of 1024 patches 602 / 457 / 461, 2048 (MLP
// 8192) of 784 832 / 793 / 746, 3072 (8192) of 784 1064 / 1141 / 1014, 4096 (16384) of 256 889 / 947 / 802 and of
// 1024 2008 / 2707 / 1975.
inline bool mid_vs_tile(int M, int N, int K, int cus) {
  long rows = 0, rounds = 0;
  mid_plan(M, N, cus, &rows, &rounds);
  return M <= 1024 && rounds <= 3 && rows * K <= 1400000;
}

// fp16 linears (mlcv_linear) that run on this kernel, not on the skinny one: the shapes of more than 64
// rows and K > 256 where it is the faster of the two.  Kernel times over 2800 shapes of 65 to 16384 rows on
// 256 CUs, skinny / this, us; inside it is 0.95 to 4 times as fast.
// - One round of tiles: 100 x 2048 x 2048 9.7 / 6.1, 457 x 2048 x 2560 30.4 / 14.3, 256 x 512 x 4096 7.6 / 6.4.
//   Few outputs are a few n tiles, whose m tiles share an XCD each, while the skinny kernel splits K: past
//   1024 rows 1100 x 8192 x 64 19.8 / 24.3, 1226 x 14112 x 256 49.1 / 57.1.  Rows that straddle 128-byte lines
//   (K % 64 = 32) cost a wave two lines a row and stage; with few outputs that loses at K just below 8192
//   and near 16384: 285 x 7968 x 64 14.5 / 16.4, 126 x 16160 x 28 21.4 / 25.3, but 227 x 9888 x 8 20.5 / 13.6.
//   Just below 4096 the two are about even: 956 x 4064 x 56 12.5 / 12.8.
// - More rounds: up to K = 512 968 x 512 x 4096 17.6 / 20.4, 457 x 288 x 16384 26.0 / 35.8; past it 968 x
//   768 x 16384 106.8 / 78.1, 671 x 608 x 2680 16.1 / 15.1.  More than 900 straddling rows: 942 x 672 x 2128 14.4 /
//   15.9, from K = 800 on faster.  Past 2048 rows or below 1024 outputs: 3846 x 800 x 2324 55.8 / 65.0, 16384 x
//   512 x 256 19.5 / 42.2.
inline bool mid_linear(int M, int K, int N, int cus) {
  if (M <= 64 || K <= 256 || K % 32 != 0) return false;
  const bool straddle = K % 64 != 0;
  long rounds = 0;
  mid_plan(M, N, cus, nullptr, &rounds);
  if (rounds == 1) {
    const bool even = (K > 7168 && K <= 8192) || K > 13312;
    return N >= (M <= 1024 ? 256 : 512) || (M <= 1024 && !(straddle && even));
  }
  return M <= 2048 && N >= 1024 && K > (straddle && M > 900 ? 799 : 512);
}

// ---- the prefill tile GEMM's plan
struct TilePlanIn {
  int M, N, K;
  int F;           // GeGLU: outputs (the gate rows, then F up rows)
  int n1, n2;      // weight segment boundaries in N
  int lda, ldb, ldc;
  bool geglu, small_tiles;
  bool split_ws;   // a split-K workspace and meeting counters are given
  size_t ws_floats;
  int sync_tiles;  // tiles with meeting counters
  int cus;         // compute units of the device
  bool m128 = true;  // 128 x 128 tiles allowed (tuning switch)
  bool n64m128 = true;  // 128 x 64 tiles where 128 x 128 ones fill at most half the CUs (tuning switch)
};

struct TilePlan {
  int bm, bn, splitk, kt_per;  // m tile, n tile, K slices, k tiles (of TG_BK) per slice
  int mtiles, ntiles;          // ntiles: n tiles of bn (GeGLU: of bn / 2 outputs)
};

// fp32 partials of one split of a tile: [4 waves][bn / 64 blocks][4][4][64] f4
inline size_t tile_part_floats(int bn) { return (size_t)4 * (bn / 64) * 4 * 4 * 64 * 4; }

// Launch slots of a tile grid: tiles dealt round-robin to the XCDs, rounded to whole rounds.
inline int tile_slots(int tiles) { return ((tiles + TG_NXCD - 1) / TG_NXCD) * TG_NXCD; }

// false: the shape needs the 128 x 128 kernel.  A split-K plan keeps every workgroup of the
// grid resident at once (slots x splits <= CUs, one workgroup per CU), because the splits of
// a tile meet through a bounded wait, and its partials within the workspace.
inline bool tile_plan(const TilePlanIn& a, TilePlan& p) {
  if (a.small_tiles || a.K % 8 != 0 || a.M < 1 || a.lda % 8 != 0 || a.ldb % 8 != 0 || a.ldc % 4 != 0) return false;
  p.bm = TG_BM;
  if (a.geglu) {
    if (a.F % 128 != 0) return false;
    p.bn = 256;
    p.ntiles = a.F / 128;
  } else {
    if (a.N % 4 != 0) return false;
    if ((a.n1 % 8 != 0 && a.n1 != a.N) || (a.n2 % 8 != 0 && a.n2 != a.N)) return false;
    // long K (down_proj): 256 x 256 tiles over up to 8 K slices load a third less through
    // L2 than 256 x 128 tiles over 4.  Shorter K, over the whole K, when the tiles give at
    // least half a workgroup per CU: 128 x 128 (the prefill's q/k/v at P = 968), or 128 x 64
    // where 128 x 128 would leave half the CUs idle (o_proj: 256 tiles instead of 128); else
    // 256 x 64; else 256 x 128.
    const int mt = (a.M + TG_BM - 1) / TG_BM, mt2 = (a.M + 127) / 128;
    // (the 256 x 256 kernel stores every tile's product as a split partial and meets on the
    // tile's counter, also over one slice: only where the workspace and counters hold its tiles)
    const long t256 = (long)mt * (a.N / 256);
    if (a.K >= 8192 && a.N % 256 == 0 && (a.n1 % 16 == 0 || a.n1 == a.N) && (a.n2 % 16 == 0 || a.n2 == a.N) &&
        a.split_ws && t256 <= a.sync_tiles && (size_t)t256 * tile_part_floats(256) <= a.ws_floats) {
      p.bn = 256;
    } else if (a.K < 8192 && a.m128 && 2 * mt2 * ((a.N + 127) / 128) >= a.cus && a.cus > 0) {
      p.bm = 128;
      p.bn = a.n64m128 && mt2 * ((a.N + 127) / 128) <= a.cus / 2 ? 64 : 128;
    } else if (a.K < 8192 && 2 * mt * ((a.N + 63) / 64) >= a.cus && a.cus > 0) {
      p.bn = 64;
    } else {
      p.bn = 128;
    }
    p.ntiles = (a.N + p.bn - 1) / p.bn;
  }
  p.mtiles = (a.M + p.bm - 1) / p.bm;
  const int tiles = p.mtiles * p.ntiles, kts = (a.K + TG_BK - 1) / TG_BK;
  const int slots = tile_slots(tiles);
  int S = 1;
  if (!a.geglu && p.bn != 64 && p.bm == TG_BM && a.split_ws && tiles <= a.sync_tiles && a.cus > 0) {
    // at least 4 k tiles per slice
    S = std::min({8, a.cus / slots, kts / 4});
    const size_t part = tile_part_floats(p.bn);
    while (S > 1 && (size_t)tiles * S * part > a.ws_floats) --S;
    S = std::max(S, 1);
  }
  p.kt_per = (kts + S - 1) / S;
  p.splitk = (kts + p.kt_per - 1) / p.kt_per;
  return true;
}

}  // namespace mlcv
