// CPU check of the launch planners (mlc-vla_amd/csrc/plan.h) over sweeps of shapes, built with
// the address and undefined-behaviour sanitizers by tests/test_planners.py.  Every plan must
// cover its whole K (or key) range with no empty slice, stay within its workspace, and -- for
// the split-K tile GEMM, whose splits meet through a bounded wait -- keep the whole grid
// resident (one workgroup per CU).  Prints the number of plans checked; exits 1 on a failure.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "../mlc-vla_amd/csrc/plan.h"

using namespace mlcv;

static long checked = 0;
static int failures = 0;

#define CHECK(cond, ...)                             \
  do {                                               \
    if (!(cond)) {                                   \
      if (failures++ < 20) {                         \
        std::fprintf(stderr, "FAIL %s: ", #cond);    \
        std::fprintf(stderr, __VA_ARGS__);           \
        std::fprintf(stderr, "\n");                  \
      }                                              \
    }                                                \
  } while (0)

static void check_attn() {
  for (int rows : {1, 8, 16, 50, 63, 64, 65, 400, 800, 7744, 8192})
    for (int Sp : {0, 1, 31, 32, 33, 256, 800, 968, 1018, 4096})
      for (int Ts : {0, 1, 8, 50, 64})
        for (int target : {1, 7, 64, 100, 128, 224, 256, 1000}) {
          if (Sp == 0 && Ts == 0) continue;
          int ns = -1, kps = -1;
          attn_plan(rows, Sp, Ts, target, &ns, &kps);
          ++checked;
          const int nsp = ns - (Ts > 0 ? 1 : 0);
          CHECK(ns >= 1 && ns <= 32, "rows %d Sp %d Ts %d target %d: nsplit %d", rows, Sp, Ts, target, ns);
          CHECK(kps >= ATTN_KCH && kps % ATTN_KCH == 0, "kps %d", kps);
          if (Sp > 0) {
            CHECK(nsp >= 1 && (long)nsp * kps >= Sp, "Sp %d nsp %d kps %d: keys not covered", Sp, nsp, kps);
            CHECK((long)(nsp - 1) * kps < Sp, "Sp %d nsp %d kps %d: an empty prefix split", Sp, nsp, kps);
          } else {
            CHECK(nsp == 0, "no prefix keys but %d prefix splits", nsp);
          }
          // every partial the kernels write lies inside the workspace
          for (int KV : {1, 2, 8}) {
            const int hd = 256;
            const size_t ws = attn_ws_floats(KV, rows, hd, ns);
            if (ns == 1) {
              CHECK(ws == 0, "one split needs no workspace");
              continue;
            }
            const size_t rpad = (size_t)((rows + ATTN_ROWS - 1) / ATTN_ROWS) * ATTN_ROWS;
            const size_t last_row = ((size_t)(KV - 1) * ns + (ns - 1)) * rpad + (rows - 1);
            const size_t o_end_halfs = (last_row + 1) * hd;           // fp16 O
            const size_t ml_off = (size_t)KV * ns * rpad * hd;        // floats, after O
            const size_t ml_end = ml_off + (last_row + 1) * 2;
            CHECK(o_end_halfs <= 2 * ml_off, "O partials overlap (m, l)");
            CHECK(ml_end <= ws, "rows %d ns %d KV %d: (m, l) end %zu > workspace %zu", rows, ns, KV, ml_end, ws);
          }
        }
}

static void check_f32_attn() {
  for (int rows : {1, 16, 63, 64, 65, 400, 7744})
    for (int KV : {1, 2, 8})
      for (int nk : {1, 31, 32, 33, 64, 65, 100, 968, 1018, 16000}) {
        int ns = -1, cps = -1;
        f32_attn_plan(rows, KV, nk, &ns, &cps);
        ++checked;
        const int chunks = (nk + ATTN_KCH - 1) / ATTN_KCH;
        CHECK(ns >= 1 && ns <= 64 && cps >= 1, "rows %d KV %d nk %d: %d x %d", rows, KV, nk, ns, cps);
        CHECK((long)ns * cps >= chunks && (long)(ns - 1) * cps < chunks, "rows %d nk %d: %d x %d chunks of %d", rows, nk, ns, cps, chunks);
        const size_t rpad = (size_t)((rows + ATTN_ROWS - 1) / ATTN_ROWS) * ATTN_ROWS, hd = 256;
        const size_t end = (size_t)KV * ns * rpad * hd + 2 * ((((size_t)KV - 1) * ns + ns - 1) * rpad + rows);
        CHECK(ns == 1 || end <= f32_attn_ws_floats(KV, rows, (int)hd, ns), "partials past the workspace");
      }
}

// A float32 table launch (the modulations of up to 64 steps) takes the few-row kernel at any width and
// device size; a plain one takes tiles where they fill the CUs
static void check_f32_tile() {
  for (int cus : {8, 32, 64, 256, 304})
    for (int M : {1, 16, 32, 33, 64, 65, 968})
      for (int N : {8, 192, 3072, 16368, 65536}) {
        ++checked;
        CHECK(f32_tile(M, N, true, cus) == 0, "table M %d N %d cus %d on tiles", M, N, cus);
        const int bm = f32_tile(M, N, false, cus);
        CHECK(bm == 0 || (M > bm / 2 && (long)((M + bm - 1) / bm) * ((N + bm - 1) / bm) >= (bm == 128 ? 2L : 1L) * cus),
              "M %d N %d cus %d: tile %d", M, N, cus, bm);
      }
  // what test_gpu_f32.py's shapes are there for, on 256 CUs
  CHECK(f32_tile(100, 8192, false, 256) == 64 && f32_tile(150, 32768, false, 256) == 128, "gate_up tiles");
  CHECK(f32_tile(520, 2112, false, 256) == 64 && f32_tile(520, 2056, false, 256) == 64, "q/k/v, o_proj and down tiles");
  CHECK(f32_tile(1000, 8448, false, 256) == 128 && f32_tile(1000, 8200, false, 256) == 128, "the same of 128");
}

static void check_skinny() {
  for (int ntiles : {1, 2, 3, 8, 16, 40, 64, 160, 256, 512, 1024})
    for (int K : {32, 96, 128, 129, 512, 1024, 2048, 4096, 16384})
      for (int mblocks : {1, 2, 4, 16})
        for (int splits : {-1, 0, 1, 2, 3, 4, 8, 9, 100}) {
          const SkPlan p = sk_plan(ntiles, K, mblocks, splits);
          ++checked;
          CHECK(p.splitk >= 1 && p.splitk <= SK_MAX_SPLIT, "splitk %d", p.splitk);
          CHECK(p.kper >= SK_KC && p.kper % SK_KC == 0, "kper %d", p.kper);
          CHECK((long)p.kper * p.splitk >= K, "K %d: %d x %d does not cover it", K, p.splitk, p.kper);
          CHECK((long)(p.splitk - 1) * p.kper < K, "K %d: %d x %d leaves an empty slice", K, p.splitk, p.kper);
          if (splits > 0) CHECK(p.splitk <= splits, "asked %d splits, got %d", splits, p.splitk);
          const size_t ws = sk_ws_floats(ntiles, mblocks, p, 4);
          CHECK((ws == 0) == (p.splitk == 1), "workspace %zu for %d splits", ws, p.splitk);
          if (p.splitk > 1)
            CHECK(ws == (size_t)ntiles * mblocks * p.splitk * 4 * 64, "workspace %zu", ws);
        }
}

// The mid-size linears' tile: no other tile gives the busiest CU fewer operand rows, and ties go to the
// larger one
static void check_mid() {
  const int bm[4] = {64, 64, 32, 32}, bn[4] = {96, 64, 64, 32};
  for (int cus : {8, 64, 256, 304})
    for (int M : {1, 32, 33, 64, 65, 100, 256, 457, 968, 1024})
      for (int N : {4, 32, 36, 1024, 1152, 2048, 2560, 4304, 16384}) {
        long rows = 0;
        const int t = mid_plan(M, N, cus, &rows);
        ++checked;
        CHECK(t >= 0 && t < 4, "tile %d", t);
        for (int i = 0; i < 4; ++i) {
          // the busiest XCD's tiles, counted one by one
          long most = 0;
          for (int x = 0; x < 8; ++x) {
            long n = 0;
            for (int j = x; j * bn[i] < N; j += 8) n += (M + bm[i] - 1) / bm[i];
            most = std::max(most, n);
          }
          const long per = std::max(cus / 8, 1), r = (most + per - 1) / per * (bm[i] + bn[i]);
          CHECK(i == t ? r == rows : i < t ? r > rows : r >= rows, "M %d N %d: tile %d has %ld rows, %d has %ld", M, N,
                t, rows, i, r);
        }
      }
}

// fp16 linears on the mid-size kernel: never below its row count and depth, or where the kernel times
// (us, skinny / mid) say that it is the slower one
static void check_mid_linear() {
  struct Shape {
    int M, K, N;
    bool in;
  };
  const Shape shapes[] = {
      {457, 2048, 2560, true},   // 30.4 / 14.3
      {256, 512, 4096, true},    // 7.6 / 6.4: one round
      {968, 512, 4096, false},   // 17.6 / 20.4: two
      {457, 288, 16384, false},  // 26.0 / 35.8
      {83, 416, 15748, false},   // 9.5 / 11.2
      {968, 768, 16384, true},   // 106.8 / 78.1
      {942, 672, 2128, false},   // 14.4 / 15.9: rows across lines
      {671, 608, 2680, true},    // 16.1 / 15.1
      {582, 928, 2908, true},    // 17.6 / 14.1
      {640, 8192, 64, true},     // 16.3 / 14.0
      {1100, 8192, 64, false},   // 19.8 / 24.3: an XCD or two
      {1226, 14112, 256, false}, // 49.1 / 57.1
      {285, 7968, 64, false},    // 14.5 / 16.4: rows across lines
      {126, 16160, 28, false},   // 21.4 / 25.3
      {227, 9888, 8, true},      // 20.5 / 13.6
      {801, 3328, 32, true},     // 11.2 / 8.1
      {3846, 800, 2324, false},  // 55.8 / 65.0
      {16384, 512, 256, false},  // 19.5 / 42.2
      {64, 2048, 2048, false},   // the skinny kernel's rows
      {200, 256, 4096, false},
  };
  for (const Shape& s : shapes) {
    ++checked;
    CHECK(mid_linear(s.M, s.K, s.N, 256) == s.in, "linear %d x %d x %d", s.M, s.K, s.N);
  }
}

// The image tower's linears on the mid-size kernel, or (many rows, many rounds, long K) on the tile GEMM
static void check_mid_vs_tile() {
  for (int M : {4, 64, 196, 256, 576, 1024})
    for (int N : {1152, 3456, 4304, 2048}) {
      ++checked;
      CHECK(mid_vs_tile(M, N, N == 1152 ? 4304 : 1152, 256), "So400m linear %d x %d", M, N);
    }
  CHECK(!mid_vs_tile(1025, 1152, 1152, 256), "rows");
  CHECK(mid_vs_tile(784, 6144, 1152, 256) == false && mid_vs_tile(289, 16384, 64, 256) == false, "rounds");
  CHECK(!mid_vs_tile(256, 4096, 16384, 256) && !mid_vs_tile(784, 4096, 4096, 256), "long K");
}

// The modulation pieces of mlcv_bind_params on 64-row tiles (layer 0's two norms, then the other
// NM - 2, 3 W1 rows each): the workspace mlcv_create allocates holds the partials of each piece.
static void check_modulations() {
  for (int D : {1, 2, 3, 4, 11, 18})
    for (int W1 : {64, 128, 256, 1024, 2048})
      for (int mblocks : {1, 2}) {
        const int NM = 2 * D + 1, per = (3 * W1 + 63) / 64;
        const size_t ws = sk_mod_ws_floats(NM, W1, mblocks);
        for (int segs : {2, NM - 2}) {
          ++checked;
          const SkPlan p = sk_plan(segs * per, W1, mblocks, 0);
          const size_t end = p.splitk > 1 ? (size_t)segs * per * mblocks * p.splitk * 64 * 64 : 0;
          CHECK(end <= ws, "D %d W1 %d: a piece of %d norms needs %zu floats of %zu", D, W1, segs, end, ws);
        }
      }
}

static void check_tile() {
  for (int cus : {8, 80, 256, 304})
    for (int M : {1, 32, 255, 256, 257, 968, 4096})
      for (int N : {4, 256, 1024, 2048, 2560, 8192, 16384})
        for (int K : {8, 64, 200, 512, 1024, 2048, 4096, 16384})
          for (int geglu : {0, 1})
            for (int ws_given : {0, 1}) {
              TilePlanIn in{};
              in.M = M;
              in.N = N;
              in.K = K;
              in.F = N;
              in.n1 = in.n2 = geglu ? 2 * N : N;
              in.lda = K;
              in.ldb = K;
              in.ldc = N;
              in.geglu = geglu != 0;
              in.small_tiles = false;
              in.split_ws = ws_given != 0;
              in.ws_floats = (size_t)cus * TG_BM * 256;  // one 256 x 256 partial per CU
              in.sync_tiles = cus;
              in.cus = cus;
              TilePlan p{};
              if (!tile_plan(in, p)) {
                ++checked;
                CHECK(geglu ? N % 128 != 0 : (N % 4 != 0 || K % 8 != 0), "M %d N %d K %d: no 256-row plan", M, N, K);
                continue;
              }
              ++checked;
              const int tiles = p.mtiles * p.ntiles, kts = (K + TG_BK - 1) / TG_BK;
              CHECK(p.bm == TG_BM || (p.bm == 128 && (p.bn == 128 || p.bn == 64) && p.splitk == 1 && !geglu), "m tile %d", p.bm);
              CHECK((long)p.mtiles * p.bm >= M && (long)(p.mtiles - 1) * p.bm < M, "m tiles %d for M %d", p.mtiles, M);
              const long ncover = geglu ? (long)p.ntiles * (p.bn / 2) : (long)p.ntiles * p.bn;
              CHECK(ncover >= N, "n tiles %d x %d for N %d", p.ntiles, p.bn, N);
              CHECK(p.splitk >= 1 && p.kt_per >= 1, "splitk %d kt_per %d", p.splitk, p.kt_per);
              CHECK((long)p.kt_per * p.splitk >= kts && (long)(p.splitk - 1) * p.kt_per < kts,
                    "K %d: %d slices of %d k tiles", K, p.splitk, p.kt_per);
              CHECK(p.bn == 64 || p.bn == 128 || p.bn == 256, "n tile %d", p.bn);
              if (p.bn == 64) CHECK(p.splitk == 1 && 2 * tiles >= cus, "256 x 64 tiles: %d tiles, %d splits", tiles, p.splitk);
              // the 256 x 256 kernel (not GeGLU) stores split partials and meets even over one slice
              if (p.bn == 256 && !geglu) {
                CHECK(ws_given && tiles <= in.sync_tiles, "256 x 256: %d tiles, workspace %d", tiles, ws_given);
                CHECK((size_t)tiles * p.splitk * tile_part_floats(p.bn) <= in.ws_floats, "256 x 256 partials overflow");
              }
              if (p.splitk > 1) {
                CHECK(!geglu && ws_given, "split-K without a workspace or with the GeGLU epilogue");
                CHECK(tiles <= in.sync_tiles, "%d tiles, %d meeting counters", tiles, in.sync_tiles);
                CHECK((long)tile_slots(tiles) * p.splitk <= cus,
                      "M %d N %d K %d cus %d: %d slots x %d splits not resident at once", M, N, K, cus,
                      tile_slots(tiles), p.splitk);
                CHECK((size_t)tiles * p.splitk * tile_part_floats(p.bn) <= in.ws_floats, "partials overflow");
                CHECK(p.kt_per >= 4, "slices of %d k tiles", p.kt_per);
              }
            }
}

int main() {
  check_attn();
  check_f32_attn();
  check_f32_tile();
  check_skinny();
  check_modulations();
  check_mid();
  check_mid_linear();
  check_mid_vs_tile();
  check_tile();
  std::printf("plans checked: %ld, failures: %d\n", checked, failures);
  return failures ? 1 : 0;
}
