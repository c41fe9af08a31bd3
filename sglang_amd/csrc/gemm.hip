// Host side of the FP8 GEMM entry points: argument checks mirrored from the reference ops, kernel
// choice, launch.  No allocation, no synchronisation.
#include <algorithm>
#include <atomic>
#include <mutex>

#include "gemm_bmm.h"
#include "gemm_direct.h"
#include "gemm_direct_quant.h"
#include "gemm_skinny.h"
#include "gemm_tile128.h"
#include "gemm_tile64.h"

#include "../../include/fp8k_tune.h"

namespace fp8k {

struct Plan {
  int kind;    // 0 = generic, 1 = tile256, 2 = weight-streaming through LDS (33..128 rows), 3 = direct (<= 32 rows),
               // 4 = tiles of 128 weight rows, 5 = direct with K cut across the waves of a workgroup (<= 16 rows, N below 16 K),
               // 7 = skinny strips over all of K (<= 64 rows, N up to 16 K), 8 = tiles of 64 weight rows
  int splits;  // >1: split-K through the float workspace
  int kb_per_split;
  int tm;      // rows per block of the streaming kernels, activation rows of a tile (kind 4)
  int tail_first;   // tile256: first tile that is cut along K or into halves (== number of tiles when none is)
  int halves;       // tile256: the tiles from tail_first on are computed as two 128-row halves; kinds 5, 7: waves along n
  int64_t ws_bytes; // float workspace the plan needs
};

// tuning aid: force the kernel family (and the K split of the uniform-split families) of later calls made by the
// calling thread; other threads keep the automatic choice
static thread_local int g_force_kind = -1, g_force_splits = 0;
static thread_local int g_tail_halves = 1;  // tuning aid: 0 keeps the last round of 256x256 tiles whole

static Plan plan_tile128(int64_t M, int64_t N, int kb, int splits, int tm) {
  Plan pl{4, 1, 0, 0, 0, 0};
  pl.tm = tm;
  if (splits > kb) splits = kb;
  if (splits < 1) splits = 1;
  pl.kb_per_split = (kb + splits - 1) / splits;
  pl.splits = (kb + pl.kb_per_split - 1) / pl.kb_per_split;
  pl.ws_bytes = pl.splits > 1 ? (int64_t)pl.splits * M * N * 4 : 0;
  return pl;
}

static Plan plan_tile64(int64_t M, int64_t N, int kb, int splits) {
  Plan pl = plan_tile128(M, N, kb, splits, kT64);
  pl.kind = 8;
  return pl;
}

// decode-sized, up to 32 rows: weights go HBM -> registers -> matrix core.  K is cut into about 512 workgroups (two per CU, one
// round, up to 16 rows; above, the LDS of the activations leaves one per CU and they run in two) of at least 8 K blocks each, while
// the float partials stay a small fraction of the weight bytes
static Plan plan_direct(int64_t M, int64_t N, int64_t K) {
  Plan pl{3, 1, 0, 0, 0, 0};
  const int kb = (int)(K / kTileK);
  pl.tm = M <= 16 ? 16 : 32;
  const int64_t tiles_n = (N + kDirTileN - 1) / kDirTileN;
  int64_t splits = std::max<int64_t>(1, 512 / tiles_n);
  splits = std::min<int64_t>(splits, std::max<int64_t>(1, kb / kDirDepth));
  splits = std::min<int64_t>(splits, std::max<int64_t>(1, K / (64 * M)));
  // 128 and more n tiles keep half the CUs streaming on their own: no K cut and no reduction launch (18432 x 7168:
  // 26.6 us against 28.6 us with three cuts; two cuts, 288 workgroups, leave the CUs unevenly loaded: 33 us)
  if (tiles_n >= 128) splits = 1;
  // a share of 9 or 10 K blocks is one full prefetch round of 8 and a round for the one or two left over: one more cut
  // gives every workgroup a single shorter round (7168 x 2304, 18 K blocks: 10.2 -> 8.5 us at M = 1 with three cuts)
  while (splits > 1 && splits < kb) {
    const int64_t per = (kb + splits - 1) / splits;
    if (per > kDirDepth && per % kDirDepth >= 1 && per % kDirDepth <= 2 && (kb + splits) / (splits + 1) >= 4) ++splits;
    else break;
  }
  if (g_force_kind == 3 && g_force_splits > 0) splits = std::min<int64_t>(g_force_splits, kb);  // tuning aid
  const int kbps = (int)((kb + splits - 1) / splits);
  pl.kb_per_split = kbps;
  pl.splits = (kb + kbps - 1) / kbps;
  pl.ws_bytes = pl.splits > 1 ? (int64_t)pl.splits * M * N * 4 : 0;
  return pl;
}

// decode-sized with fewer than 128 tiles of 128 weight rows: a workgroup owns 16 (or 32) weight rows and its waves cut
// K between them, so that every CU streams without float partials in memory or a reduction launch.  `splits` stays 1
// (nothing goes through the workspace); kb_per_split is the K range of one wave, tm reuses the row-count slot, and
// the number of waves along n travels in `halves`.
constexpr int64_t kWaveKMaxN = 16384;
static Plan plan_wavek(int64_t M, int64_t N, int64_t K, int cu) {
  Plan pl{5, 1, 0, 0, 0, 0};
  const int kb = (int)(K / kTileK);
  pl.tm = 16;
  // waves along n: the choice that leaves the busiest CU the fewest weight rows (workgroups go two to a CU at most);
  // among equals the widest workgroup whose waves still get at most 16 K blocks each (measured: wider workgroups
  // re-read less of the activations, longer per-wave K ranges start to serialise)
  int nw = 1;
  int64_t best_rows = -1;
  for (int cand = 1; cand <= 4; cand *= 2) {
    const int64_t wgs = (N + 16 * cand - 1) / (16 * cand);
    if (wgs > 2 * (int64_t)cu && cand < 4) continue;
    const int64_t rows = (wgs + cu - 1) / cu * 16 * cand;
    const int per_wave = (kb + 8 / cand - 1) / (8 / cand);
    if (best_rows < 0 || rows < best_rows || (rows == best_rows && per_wave <= 16)) { best_rows = rows; nw = cand; }
  }
  if (g_force_kind == 5 && (g_force_splits == 1 || g_force_splits == 2 || g_force_splits == 4 || g_force_splits == 8))
    nw = g_force_splits;  // tuning aid
  pl.halves = nw;
  pl.kb_per_split = (kb + 8 / nw - 1) / (8 / nw);
  return pl;
}
// Up to 64 rows: the strips of weight rows that one workgroup each runs over all of K are as narrow as leaves every CU one.
constexpr int64_t kSkinnyMaxN = 16384;
static Plan plan_skinny(int64_t M, int64_t N, int64_t K, int cu) {
  Plan pl{7, 1, 0, 0, 0, 0};
  pl.tm = M <= 16 ? 16 : M <= 32 ? 32 : 64;
  pl.halves = N <= 16 * cu ? 1 : N <= 32 * cu ? 2 : 4;
  if (g_force_kind == 7 && (g_force_splits == 1 || g_force_splits == 2 || g_force_splits == 4)) pl.halves = g_force_splits;  // tuning aid
  return pl;
}
// Where it is ahead (M = 4 .. 64 x 16 widths up to 20480 x 9 depths up to 18432, timed against the other decode kernels and the
// 64-row tiles under every K cut):
//  * more than 64 weight rows per CU's strip cost more activation traffic than a K cut costs partials, from 9 rows on;
//  * 17 .. 32 rows in 64-row strips that leave a quarter of the CUs idle: up to K = 6144;
//  * 33 .. 64 rows: that traffic grows with rows x K, so up to a K where the 64-row tiles are level (370 shapes, weights out of HBM;
//    time over the tiles': up to 4096 weight rows 0.63 at K = 1536 .. 3072, 0.75 at 5120, 0.92 at 7168, 1.04 at 10240; up to 8192
//    0.71, 0.89, 0.94 at 6144, 1.05 at 8192), and in 64-row strips from K = 1664 (0.82 - 0.95; level below) to 4608, or 10240
//    where the strips fill the chip.
static bool prefers_skinny(int64_t M, int64_t N, int64_t K, int cu) {
  if (M > kSkinnyMaxM || N > kSkinnyMaxN) return false;
  const bool wide = N > 32 * cu, fills = N >= 48 * cu;
  if (M <= 8) return K <= 9216;  // above: the wave-cut kernel, whose waves keep all of their K range in flight
  if (M <= 16) return true;
  if (M <= 32) return !wide || fills || K <= 6144;
  if (wide) return K > 1536 && K <= (fills ? 10240 : 4608);
  return K <= (N <= 16 * cu ? 7168 : 6144);
}
// Activations few enough for every workgroup to quantise them for itself (gemm_wavek_quant_kernel): up to 16 rows of at most
// kQuantFuseMax elements together.  The share of the quantisation grows with M * K while the launch it saves does not (the gain
// falls from 1.5 .. 1.85 times at 4096 elements to 1.2 .. 1.3 at 32768; twice as many would take another 32 registers per lane
// and with them the second workgroup of a CU).  The GEMM of these sizes is the wave-cut kernel's also where the activations come
// quantised, so that a linear's result does not depend on the way it took.
static bool few_activations(int64_t M, int64_t N, int64_t K) {
  return M <= 16 && M * K <= kQuantFuseMax && N < kWaveKMaxN && (M <= 8 || N * K <= (24LL << 20));
}

// up to 128 rows: stream the weights once, every CU takes a K slice of one 256-row weight tile
static Plan plan_stream(int64_t M, int64_t N, int64_t K) {
  Plan pl{2, 1, 0, 0, 0, 0};
  const int kb = (int)(K / kTileK);
  pl.tm = M <= 64 ? 64 : 128;
  const int64_t tiles_n = (N + kTileN - 1) / kTileN;
  int splits = (int)(256 / tiles_n);
  if (splits > kb / 4) splits = kb / 4;
  if (splits < 1) splits = 1;
  pl.kb_per_split = (kb + splits - 1) / splits;
  pl.splits = (kb + pl.kb_per_split - 1) / pl.kb_per_split;
  pl.ws_bytes = pl.splits > 1 ? (int64_t)pl.splits * M * N * 4 : 0;
  return pl;
}

// One workgroup (one CU) per 256x256 tile.  The tiles of the last, partial round over the CUs are cut along K
// so that the round keeps every CU busy for 1/splits of a tile time (>= 4 K blocks per piece).
static Plan plan_tile256(int64_t M, int64_t N, int64_t K, int cu) {
  Plan pl{1, 1, 0, 0, 0, 0};
  const int kb = (int)(K / kTileK);
  const int64_t tiles = ((M + kTileM - 1) / kTileM) * ((N + kTileN - 1) / kTileN);
  const int64_t rest = tiles % cu;
  int splits = rest ? (int)(cu / rest) : 1;
  if (splits > kb / 4) splits = kb / 4;
  if (splits < 1) splits = 1;
  // With at least one full round before it, the cut only pays when the tile time it saves (about 2 us per K block)
  // outweighs writing and re-reading the float partials (256 KB per piece): measured break-even.
  if (tiles > cu && kb * (splits - 1) * 8 <= rest * splits * splits) splits = 1;
  pl.kb_per_split = (kb + splits - 1) / splits;
  pl.splits = (kb + pl.kb_per_split - 1) / pl.kb_per_split;
  pl.tail_first = (int)(pl.splits > 1 ? tiles - rest : tiles);
  pl.ws_bytes = pl.splits > 1 ? rest * pl.splits * (int64_t)(kTileM * kTileN) * 4 : 0;
  // A last round that fills at most half the CUs and is not worth a K cut: its tiles run as two 128-row halves, one
  // workgroup each (half the matrix-core time per K block, nothing to reduce).
  if (pl.splits == 1 && tiles > cu && rest > 0 && rest <= cu / 2 && M > kTileM / 2 && g_tail_halves) {
    pl.halves = 1;
    pl.tail_first = (int)(tiles - rest);
  }
  return pl;
}

// the plan without the 128-row tiles: skinny / direct / streaming / 256x256 tiles by the number of rows
static Plan plan_base(int64_t M, int64_t N, int64_t K, int cu) {
  const bool fits32 = M * K < (1LL << 31);
  if (g_force_kind == 3 && M <= 32 && fits32) return plan_direct(M, N, K);
  if (g_force_kind == 5 && M <= 16 && fits32) return plan_wavek(M, N, K, cu);
  if (g_force_kind == 7 && M <= kSkinnyMaxM && fits32) return plan_skinny(M, N, K, cu);
  if (g_force_kind == 2 && M <= 128 && fits32) return plan_stream(M, N, K);
  if (g_force_kind == 1) return plan_tile256(M, N, K, cu);
  if (fits32 && few_activations(M, N, K)) return plan_wavek(M, N, K, cu);
  if (fits32 && prefers_skinny(M, N, K, cu)) return plan_skinny(M, N, K, cu);
  if (fits32 && M <= 8 && N < kWaveKMaxN) return plan_wavek(M, N, K, cu);
  if (M <= 32 && fits32) return plan_direct(M, N, K);
  if (M <= 128 && fits32) return plan_stream(M, N, K);
  return plan_tile256(M, N, K, cu);
}

// Device-time models in microseconds of the two tile kernels, fitted to 2500 shapes (M = 33 .. 2400, N = 512 .. 24576, K = 512 .. 18432,
// block scales, weights out of HBM, every K cut; rms error 6 and 5 %).  Over those with more than 128 rows the choice they make
// is 0.4 % behind the best of all plans on average, 14 % at worst.
//  * tiles of 128 weight rows and TM = 128 or 64 activation rows: 0.43 (0.34) per K block - the serial chain of a trip more than its
//    work - and a little more when the weights are new to the chip and the chip is full; 3 us of first loads and write-out per
//    round of tiles, at most two rounds; a K cut adds the reduction launch and the float partials.  A cut counts as 12 us at least:
//    where the product without one takes that little, it is not cut, and among cuts below 12 us the fewest runs are taken.  Both
//    sides, whole linears of 150 such shapes (N up to some 2500, 4 % of all), us, replayed from a graph / launched one by one: without
//    a cut 11.8 / 12.5, with the six runs the model would choose 12.4 / 13.7 (152 x 832 x 2304; 166 x 1216 x 2432 12.4 / 13.0 and
//    12.8 / 14.4, but 218 x 640 x 2560 14.7 / 14.7 and 12.7 / 14.1); four runs 13.3 / 14.6, eight 12.2 / 13.7 (99 x 512 x 4736; 82 x
//    2304 x 3328, four and seven: 13.2 / 14.2 and 13.7 / 14.6).  On average the model without that floor is 3 % ahead in a graph and 2 %
//    outside of one.
//  * 256x256 tiles: 1.5 per K block on a full chip (0.7 for a workgroup alone), 4.4 per tile, 15 us + partials for a cut last round.
static double est_tile128(int64_t M, int64_t N, int kb, int cu, int* best_splits, int* best_tm) {
  double best = 1e30;
  const int64_t tn = (N + kT128 - 1) / kT128;
  for (int rows = 64; rows <= (M > 64 ? 128 : 64); rows += 64) {
    const int64_t tm = (M + rows - 1) / rows;
    for (int s = 1; s <= 8; ++s) {
      const int64_t wgs = tm * tn * s, rounds = (wgs + cu - 1) / cu;
      if (rounds > 2 || (s > 1 && (rounds > 1 || s > kb / 3))) break;  // a K cut stays within one round of workgroups
      const double fill = std::min(1.0, (double)wgs / cu), cold = 1.0 / (double)tm;
      const double tb = rows == 64 ? 0.342 + 0.048 * cold + fill * (0.159 * cold + 0.008) : 0.433 + 0.018 * cold + fill * (0.056 * cold + 0.065);
      double t = 1.4 + (double)rounds * ((kb + s - 1) / s * tb + (rows == 64 ? 2.8 : 3.4));
      if (rounds == 2) t *= 0.985;
      if (s > 1) t += 3.1 + (double)s * M * N * 8.0 / 4.15e6;
      t = std::max(t, s > 1 ? 12.0 : 8.0);
      if (t < best) { best = t; *best_splits = s; *best_tm = rows; }
    }
  }
  return best;
}

// The same for tiles of 64 x 64, as many as the chip has CUs at most (one round), more than 64 rows and more than eight K blocks (up
// to eight they are level with the larger tiles, 0.95 - 1.05): a wave runs 0.9 us per K block of its own, every fourth of the range, and
// more where the weights come out of HBM for this tile alone and the chip is full.  Fitted to 137 pairs of shape and K cut (65 .. 1150
// rows, N = 512 .. 9856, K = 896 .. 17664; rms error 6 %).  On 105 other such shapes, even over the logarithm of 65 .. 1300 rows, N up
// to 12000 and K up to 18000, the GEMM takes 0.92 (0.73 - 1.00) of the time that the larger tiles and the strips took there with
// weights out of HBM, 0.88 (0.73 - 1.04) out of the last-level cache; whole linears, us, replayed from a graph, HBM / cache: 238 x 3456 x
// 3072 18.2 -> 14.5 / 13.1 -> 10.8, 159 x 4288 x 4224 20.8 -> 16.4 / 15.8 -> 12.4, 73 x 576 x 2688 13.9 -> 11.6 / 13.3 -> 10.2, 411 x 1024 x
// 3200 15.6 -> 13.3 / 14.7 -> 12.5, 128 x 4096 x 4096 18.1 -> 16.4 / 15.7 -> 11.2.
static double est_tile64(int64_t M, int64_t N, int kb, int cu, int* best_splits) {
  double best = 1e30;
  const int64_t tm = (M + kT64 - 1) / kT64, tiles = tm * ((N + kT64 - 1) / kT64);
  if (M <= kT64 || kb <= 8) return best;
  for (int s = 1; s <= 8 && tiles * s <= cu && (s == 1 || s <= kb / 8); ++s) {
    const double cold = 1.0 / (double)tm, fill = (double)(tiles * s) / cu;
    double t = 4.75 + (((kb + s - 1) / s + 3) / 4) * (0.91 + cold * (0.64 * fill - 0.26));
    if (s > 1) t += 2.7 + (double)s * M * N * 8.0 / 6.9e6;
    if (t < best) { best = t; *best_splits = s; }
  }
  return best;
}

static double est_tile256(const Plan& pl, int64_t M, int64_t N, int kb, int cu) {
  const int64_t tiles = ((M + kTileM - 1) / kTileM) * ((N + kTileN - 1) / kTileN), rest = tiles % cu;
  auto per_kb = [&](int64_t wgs) { return 0.68 + 0.87 * std::min(1.0, (double)wgs / cu); };
  if (pl.splits == 1) {
    const double rounds = pl.halves ? (double)(tiles / cu) + 0.6 : (double)((tiles + cu - 1) / cu);
    return 4.7 + rounds * (kb * per_kb(tiles) + 4.4);
  }
  return 4.7 + (double)(tiles / cu) * (kb * per_kb(cu) + 4.4) + pl.kb_per_split * per_kb(rest * pl.splits) + 15.4 +
         (double)rest * pl.splits * 0.0205;
}

static Plan make_plan(int64_t M, int64_t N, int64_t K) {
  Plan pl{0, 1, 0, 0, 0, 0};
  if (K % kTileK != 0 || N % 4 != 0) return pl;
  const int kb = (int)(K / kTileK), cu = num_cu();  // once: asking the runtime for the device costs more than all of the arithmetic
  // tuning aid: the K cut in the low byte, 256 for tiles of 64 activation rows
  if (g_force_kind == 4 && N % 8 == 0) return plan_tile128(M, N, kb, g_force_splits & 255, g_force_splits & 256 ? 64 : 128);
  if (g_force_kind == 8 && N % 8 == 0) return plan_tile64(M, N, kb, g_force_splits);
  pl = plan_base(M, N, K, cu);
  if (g_force_kind >= 0 || N % 8 != 0 || M <= 16) return pl;
  int splits = 1, rows = 0, splits64 = 1;
  // The streaming kernel keeps 256-row tiles x 2 - 3 K ranges where 128-row tiles are a little more than half a chip and a K cut
  // would be a second round: 97 x 18240 x 15104 70 us against 79, 97 x 17152 x 8192 41 against 45; 122 x 20288 x 6400 42 against 39,
  // 106 x 23040 x 5760 41 against 35.  Everywhere else the tiles are ahead, up to twice (108 x 15616 x 1024 8.2 against 19.3).
  if (pl.kind == 1 || (pl.kind == 2 && !(N > 64 * cu && N <= 80 * cu && K >= 8192))) {
    const double t128 = est_tile128(M, N, kb, cu, &splits, &rows), t64 = est_tile64(M, N, kb, cu, &splits64);
    if (pl.kind == 2 || std::min(t128, t64) < est_tile256(pl, M, N, kb, cu)) {
      if (t64 < t128) return plan_tile64(M, N, kb, splits64);
      if (rows) return plan_tile128(M, N, kb, splits, rows);
    }
  } else if (pl.kind == 3 && N > 32 * cu && N < 48 * cu && K > 6144) {
    // 17 .. 32 rows of weights too wide for one 32-row strip per CU and too narrow for 64-row strips: 64-row tiles with a K cut
    // (us, against the direct kernel: 26 x 8768 x 6400 17.3 / 23.7, 18 x 8640 x 9984 21.6 / 25.8, 23 x 10688 x 14208 31.9 / 36.4)
    est_tile128(M, N, kb, cu, &splits, &rows);
    return plan_tile128(M, N, kb, splits, rows);
  }
  return pl;
}

static int64_t workspace_bytes(int64_t M, int64_t N, int64_t K) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  return make_plan(M, N, K).ws_bytes;
}

// Row-major activation scales ([M, K/128], the layout of the reference's Triton path) make every lane of a tile
// kernel's scale load touch a cache line of its own: 32 lines per load instead of one, which costs the 256x256
// kernel 17 % and the streaming kernel 20 %.  When the caller's workspace has room, the block GEMM first copies
// them into column-major order behind the float partials (a few microseconds for at most M*K/128 floats) and
// runs on the copy; fp8k_block_gemm_workspace_bytes counts that area for every call that could need it.
static int64_t align256(int64_t v) { return (v + 255) & ~(int64_t)255; }
// The skinny kernel's waves fetch 16 scales per load instead of 32: there the copy (2 - 3 us) is level at 16 rows x 128 K blocks
// and ahead above (without it 32 x 128 takes 34.8 us against 27.4 with column-major scales, 64 x 64 32.4 against 21.1).
static bool wants_scale_copy(const Plan& pl, int64_t M, int64_t K) {
  return pl.kind == 7 ? M * (K / kTileK) >= 2048 : M > 32 && (pl.kind == 1 || pl.kind == 2 || pl.kind == 4 || pl.kind == 8);
}
static int64_t block_gemm_workspace_bytes(int64_t M, int64_t N, int64_t K) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  const Plan pl = make_plan(M, N, K);
  return wants_scale_copy(pl, M, K) ? align256(pl.ws_bytes) + M * ((K + kTileK - 1) / kTileK) * 4 : pl.ws_bytes;
}
__global__ __launch_bounds__(256) void scale_to_column_major_kernel(const float* __restrict__ src, float* __restrict__ dst,
                                                                    int M, int kb, int64_t stride_m) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;  // m fastest: the writes are contiguous
  if (i >= (int64_t)M * kb) return;
  const int k = (int)(i / M), m = (int)(i - (int64_t)k * M);
  dst[i] = src[(int64_t)m * stride_m + k];
}

// the tile kernels (plan kinds 1, 4 and 8); `a` carries the operands, the plan the tiling
template <int MODE, int OUT_DT, int BIAS_DT>
static int launch_tiles(const GemmArgs& a0, const Plan& pl, hipStream_t st) {
  GemmArgs a = a0;
  a.tiles_m = (a.M + kTileM - 1) / kTileM;
  a.tiles_n = (a.N + kTileN - 1) / kTileN;
  a.splits = pl.splits;
  a.kb_per_split = pl.kb_per_split;
  if (pl.kind == 4) {
    a.tiles_m = (a.M + pl.tm - 1) / pl.tm;
    a.tiles_n = (a.N + kT128 - 1) / kT128;
    const unsigned nwg = (unsigned)(((int64_t)a.tiles_m * a.tiles_n * pl.splits + 7) / 8 * 8);
#define FP8K_T128(SPLIT, TM) hipLaunchKernelGGL((gemm_tile128_kernel<MODE, OUT_DT, BIAS_DT, SPLIT, TM>), dim3(nwg), dim3(512), 0, st, a)
    if (pl.splits == 1) {
      if (pl.tm == 64) FP8K_T128(false, 64);
      else FP8K_T128(false, 128);
    } else {
      if (pl.tm == 64) FP8K_T128(true, 64);
      else FP8K_T128(true, 128);
    }
#undef FP8K_T128
    int rc = check_launch("gemm_tile128");
    if (rc || pl.splits == 1) return rc;
    const int64_t quads = (int64_t)a.M * (a.N / 4);
    hipLaunchKernelGGL((splitk_reduce_kernel<MODE, OUT_DT, BIAS_DT>), dim3((unsigned)((quads + 255) / 256)), dim3(256),
                       0, st, a);
    return check_launch("splitk_reduce");
  }
  if (pl.kind == 8) {
    a.tiles_m = (a.M + kT64 - 1) / kT64;
    a.tiles_n = (a.N + kT64 - 1) / kT64;
    const unsigned nwg = (unsigned)(((int64_t)a.tiles_m * a.tiles_n * pl.splits + 7) / 8 * 8);
    if (pl.splits == 1) hipLaunchKernelGGL((gemm_tile64_kernel<MODE, OUT_DT, BIAS_DT, false>), dim3(nwg), dim3(256), 0, st, a);
    else hipLaunchKernelGGL((gemm_tile64_kernel<MODE, OUT_DT, BIAS_DT, true>), dim3(nwg), dim3(256), 0, st, a);
    int rc = check_launch("gemm_tile64");
    if (rc || pl.splits == 1) return rc;
    const int64_t quads = (int64_t)a.M * (a.N / 4);
    hipLaunchKernelGGL((splitk_reduce_kernel<MODE, OUT_DT, BIAS_DT>), dim3((unsigned)((quads + 255) / 256)), dim3(256), 0, st, a);
    return check_launch("splitk_reduce");
  }
  const int ntiles = a.tiles_m * a.tiles_n;
  a.tail_first = pl.tail_first;
  a.tail_halves = pl.halves;
  const int ncu8 = std::max(8, num_cu() / 8 * 8);
  const int tail_units = (ntiles - pl.tail_first) * (pl.halves ? 2 : pl.splits);
  unsigned nwg;
  if (pl.tail_first >= ncu8) {
    // at least as many whole tiles as CUs: one walking workgroup per CU, which also takes a unit of the tail at the end
    a.walkers = ncu8;
    a.tail_shared = 1;
    nwg = (unsigned)std::max(ncu8, tail_units);
  } else {
    a.walkers = (pl.tail_first + 7) / 8 * 8;
    a.tail_shared = 0;
    nwg = (unsigned)(a.walkers + tail_units);
  }
  hipLaunchKernelGGL((gemm_tile256_kernel<MODE, OUT_DT, BIAS_DT>), dim3(nwg), dim3(512), 0, st, a);
  int rc = check_launch("gemm_tile256");
  if (rc || pl.tail_first == ntiles || pl.halves) return rc;
  hipLaunchKernelGGL((tile_reduce_kernel<MODE, OUT_DT, BIAS_DT>), dim3((unsigned)((ntiles - pl.tail_first) * 64)), dim3(256),
                     0, st, a);
  return check_launch("tile_reduce");
}

template <int MODE, int OUT_DT, int BIAS_DT>
static int launch(const GemmArgs& a0, const Plan& pl, hipStream_t st) {
  GemmArgs a = a0;
  if (pl.kind == 0) {
    dim3 grid((unsigned)((a.N + 63) / 64), (unsigned)((a.M + 3) / 4));
    hipLaunchKernelGGL((gemm_generic_kernel<MODE, OUT_DT, BIAS_DT>), grid, dim3(256), 0, st, a);
    return check_launch("gemm_generic");
  }
  a.tiles_m = (a.M + kTileM - 1) / kTileM;
  a.tiles_n = (a.N + kTileN - 1) / kTileN;
  a.splits = pl.splits;
  a.kb_per_split = pl.kb_per_split;
  if (pl.kind == 3) {
    a.m_blocks = 1;
    a.tiles_n = (a.N + kDirTileN - 1) / kDirTileN;
    const unsigned nwg = (unsigned)(a.tiles_n * pl.splits);
#define FP8K_DIRECT(TM)                                                                                             \
  do {                                                                                                              \
    if (pl.splits == 1)                                                                                             \
      hipLaunchKernelGGL((gemm_direct_kernel<TM, MODE, OUT_DT, BIAS_DT, false, false>), dim3(nwg), dim3(512), 0, st, a); \
    else                                                                                                            \
      hipLaunchKernelGGL((gemm_direct_kernel<TM, MODE, OUT_DT, BIAS_DT, true, false>), dim3(nwg), dim3(512), 0, st, a);  \
  } while (0)
    if (pl.tm == 16) FP8K_DIRECT(16);
    else FP8K_DIRECT(32);
#undef FP8K_DIRECT
    int rc = check_launch("gemm_direct");
    if (rc || pl.splits == 1) return rc;
    const int64_t quads = (int64_t)a.M * (a.N / 4);
    hipLaunchKernelGGL((splitk_reduce_kernel<MODE, OUT_DT, BIAS_DT>), dim3((unsigned)((quads + 255) / 256)), dim3(256),
                       0, st, a);
    return check_launch("splitk_reduce");
  }
  if (pl.kind == 5) {
    a.wk_nw = pl.halves;
    const unsigned nwg = (unsigned)((a.N + 16 * a.wk_nw - 1) / (16 * a.wk_nw));
    hipLaunchKernelGGL((gemm_wavek_kernel<MODE, OUT_DT, BIAS_DT>), dim3(nwg), dim3(512), 0, st, a);
    return check_launch("gemm_wavek");
  }
  if (pl.kind == 7) {
    a.wk_nw = pl.halves;
    a.tiles_n = (a.N + 16 * a.wk_nw - 1) / (16 * a.wk_nw);
    const dim3 grid((unsigned)((a.tiles_n + 7) / 8 * 8));
#define FP8K_SKINNY(TM, NW) hipLaunchKernelGGL((gemm_skinny_kernel<TM, NW, MODE, OUT_DT, BIAS_DT>), grid, dim3(TM <= 32 ? 640 : 768), 0, st, a)
#define FP8K_SKINNY_NW(TM)                    \
  do {                                        \
    if (pl.halves == 1) FP8K_SKINNY(TM, 1);   \
    else if (pl.halves == 2) FP8K_SKINNY(TM, 2); \
    else FP8K_SKINNY(TM, 4);                  \
  } while (0)
    if (pl.tm == 16) FP8K_SKINNY_NW(16);
    else if (pl.tm == 32) FP8K_SKINNY_NW(32);
    else FP8K_SKINNY_NW(64);
#undef FP8K_SKINNY_NW
#undef FP8K_SKINNY
    return check_launch("gemm_skinny");
  }
  if (pl.kind == 2) {
    a.m_blocks = 1;
    const unsigned nwg = (unsigned)(((a.tiles_n + 7) / 8) * 8 * pl.splits);
#define FP8K_STREAM(TM, NST, NW)                                                                                      \
  do {                                                                                                                \
    if (pl.splits == 1)                                                                                               \
      hipLaunchKernelGGL((gemm_stream_kernel<TM, NST, NW, MODE, OUT_DT, BIAS_DT, false, false>), dim3(nwg),           \
                         dim3(NW * 64), 0, st, a);                                                                    \
    else                                                                                                              \
      hipLaunchKernelGGL((gemm_stream_kernel<TM, NST, NW, MODE, OUT_DT, BIAS_DT, true, false>), dim3(nwg),            \
                         dim3(NW * 64), 0, st, a);                                                                    \
  } while (0)
    if (pl.tm == 64) FP8K_STREAM(64, 3, 8);
    else FP8K_STREAM(128, 3, 8);
#undef FP8K_STREAM
    int rc = check_launch("gemm_stream");
    if (rc || pl.splits == 1) return rc;
    const int64_t quads = (int64_t)a.M * (a.N / 4);
    hipLaunchKernelGGL((splitk_reduce_kernel<MODE, OUT_DT, BIAS_DT>), dim3((unsigned)((quads + 255) / 256)), dim3(256),
                       0, st, a);
    return check_launch("splitk_reduce");
  }
  return launch_tiles<MODE, OUT_DT, BIAS_DT>(a, pl, st);
}

static int common_checks(const char* op, const void* A, const void* B, void* C, int64_t M, int64_t N, int64_t K,
                         int64_t lda, int64_t ldb, int64_t ldc, int out_dtype) {
  FP8K_REQUIRE(M >= 0 && N >= 0 && K >= 0, "%s: negative shape", op);
  FP8K_REQUIRE(M <= 0x7fffffffLL && N <= 0x7fffffffLL && K <= 0x7fffffffLL, "%s: shape too large", op);
  FP8K_REQUIRE(out_dtype == FP8K_F16 || out_dtype == FP8K_BF16, "%s: out_dtype must be Half or BFloat16", op);
  FP8K_REQUIRE(K % 16 == 0, "%s: mat_a must be multiple of 16 bytes for memory alignment", op);
  FP8K_REQUIRE((N * 2) % 16 == 0, "%s: out must be multiple of 16 bytes for memory alignment", op);
  FP8K_REQUIRE(lda >= K && ldb >= K && ldc >= N, "%s: leading dimension smaller than the row length", op);
  FP8K_REQUIRE(lda % 16 == 0 && ldb % 16 == 0 && (ldc * 2) % 8 == 0, "%s: rows must be 16-byte aligned", op);
  FP8K_REQUIRE(lda < (1LL << 23) && ldb < (1LL << 23) && K < (1LL << 23), "%s: rows longer than 8 MiB are not supported", op);
  if (M == 0 || N == 0) return FP8K_OK;
  FP8K_REQUIRE(A && B && C, "%s: null pointer", op);
  FP8K_REQUIRE(aligned(A, 16) && aligned(B, 16) && aligned(C, 8), "%s: operands must be 16-byte aligned", op);
  return FP8K_OK;
}

}  // namespace fp8k

using namespace fp8k;

extern "C" void fp8k_tune_force_gemm_plan(int kind, int splits) {
  g_tail_halves = kind != -2;  // -2: automatic choice with the last round of 256x256 tiles kept whole
  g_force_kind = kind == -2 ? -1 : kind;
  g_force_splits = splits;
}

extern "C" int64_t fp8k_block_gemm_workspace_bytes(int64_t M, int64_t N, int64_t K) { return block_gemm_workspace_bytes(M, N, K); }
extern "C" int64_t fp8k_scaled_mm_workspace_bytes(int64_t M, int64_t N, int64_t K) { return workspace_bytes(M, N, K); }

static int block_gemm_impl(const void* A, const void* B, const float* As, const float* Bs, void* C, int64_t M, int64_t N,
                           int64_t K, int64_t lda, int64_t ldb, int64_t as_stride_m, int64_t as_stride_k,
                           int64_t bs_stride_n, int64_t bs_stride_k, int64_t ldc, int out_dtype, void* workspace,
                           int64_t workspace_bytes_given, void* stream) {
  int rc = common_checks("fp8_blockwise_scaled_mm", A, B, C, M, N, K, lda, ldb, ldc, out_dtype);
  if (rc) return rc;
  if (M == 0 || N == 0) return FP8K_OK;
  FP8K_REQUIRE(K > 0, "fp8_blockwise_scaled_mm: K must be positive");
  FP8K_REQUIRE(As && Bs, "fp8_blockwise_scaled_mm: null scale pointer");
  FP8K_REQUIRE(as_stride_m >= 0 && as_stride_k >= 0 && bs_stride_n >= 0 && bs_stride_k >= 0,
               "fp8_blockwise_scaled_mm: negative scale stride");
  FP8K_REQUIRE((M - 1) * as_stride_m + ((K + kTileK - 1) / kTileK - 1) * as_stride_k < 0x38000000LL,
               "fp8_blockwise_scaled_mm: scales_a spans more than 3.5 GiB");
  const Plan pl = make_plan(M, N, K);
  const int64_t kb = (K + kTileK - 1) / kTileK;
  const int64_t need = wants_scale_copy(pl, M, K) ? align256(pl.ws_bytes) + M * kb * 4 : pl.ws_bytes;
  if (need > 0 && (!workspace || workspace_bytes_given < need))
    return fail(FP8K_ERR_WORKSPACE, "fp8_blockwise_scaled_mm: workspace of %lld bytes required, %lld given",
                (long long)need, (long long)(workspace ? workspace_bytes_given : 0));
  GemmArgs a{};
  a.X = (const uint8_t*)A; a.W = (const uint8_t*)B; a.sx = As; a.sw = Bs; a.bias = nullptr; a.C = C;
  a.partial = (float*)workspace;
  a.M = (int)M; a.N = (int)N; a.K = (int)K; a.ldx = lda; a.ldw = ldb; a.ldc = ldc;
  a.sx_m = as_stride_m; a.sx_k = as_stride_k; a.sw_n = bs_stride_n; a.sw_k = bs_stride_k;
  hipStream_t st = (hipStream_t)stream;
  if (wants_scale_copy(pl, M, K) && as_stride_k == 1 && as_stride_m > 1 && kb > 1) {
    float* cm = reinterpret_cast<float*>(static_cast<char*>(workspace) + align256(pl.ws_bytes));
    hipLaunchKernelGGL(scale_to_column_major_kernel, dim3((unsigned)((M * kb + 255) / 256)), dim3(256), 0, st, As, cm, (int)M,
                       (int)kb, as_stride_m);
    rc = check_launch("scale_to_column_major");
    if (rc) return rc;
    a.sx = cm; a.sx_m = 1; a.sx_k = M;
  }
  return out_dtype == FP8K_BF16 ? launch<kModeBlock, FP8K_BF16, FP8K_BF16>(a, pl, st)
                                : launch<kModeBlock, FP8K_F16, FP8K_F16>(a, pl, st);
}

extern "C" int fp8k_block_gemm(const void* A, const void* B, const float* As, const float* Bs, void* C, int64_t M,
                               int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t as_stride_m, int64_t as_stride_k,
                               int64_t bs_stride_n, int64_t bs_stride_k, int64_t ldc, int out_dtype, void* workspace,
                               int64_t workspace_bytes_given, void* stream) {
  clear_error();
  return block_gemm_impl(A, B, As, Bs, C, M, N, K, lda, ldb, as_stride_m, as_stride_k, bs_stride_n, bs_stride_k, ldc,
                         out_dtype, workspace, workspace_bytes_given, stream);
}

// ---- the same GEMM for callers that cannot allocate: its scratch is a fixed array in device memory, one copy per GPU
// that loads this library, held until the process ends.  In host code the array's name is only a handle for
// hipGetSymbolAddress; kernels and every other use take the device address that call returns, kept per device.
constexpr int64_t kStaticScratchBytes = 80ll << 20;  // 64 MiB of float partials (one 256x256 tile per CU) + 16 MiB of copied scales
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

static int static_scratch(void** out, hipStream_t stream) {
  constexpr int kMaxDev = 64;
  static std::mutex mu;
  static void* ptrs[kMaxDev];  // device address of `scratch` on each device, resolved on the first call there
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return fail(FP8K_ERR_LAUNCH, "fp8k_block_gemm_noalloc: hipGetDevice: %s", hipGetErrorString(e));
  if (dev < 0 || dev >= kMaxDev) return fail(FP8K_ERR_UNSUPPORTED, "fp8k_block_gemm_noalloc: device index %d not supported", dev);
  // every GPU holds its own copy of the array: the copy used must be the one of the GPU the launches go to
  if (stream) {
    int sdev = -1;
    e = hipStreamGetDevice(stream, &sdev);
    if (e != hipSuccess) return fail(FP8K_ERR_LAUNCH, "fp8k_block_gemm_noalloc: hipStreamGetDevice: %s", hipGetErrorString(e));
    if (sdev != dev)
      return fail(FP8K_ERR_INVALID, "fp8k_block_gemm_noalloc: the stream belongs to device %d but device %d is current; make the "
                  "stream's device current before the call", sdev, dev);
  }
  std::lock_guard<std::mutex> lock(mu);
  if (!ptrs[dev]) {
    // the look-up is not a stream operation; under a capture it would break the capture, so it is refused there
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if (stream && hipStreamIsCapturing(stream, &cs) == hipSuccess && cs != hipStreamCaptureStatusNone)
      return fail(FP8K_ERR_UNSUPPORTED, "fp8k_block_gemm_noalloc: the first call on a device resolves the scratch address and "
                  "cannot run while the stream is capturing; make one call outside the capture first");
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return fail(FP8K_ERR_LAUNCH, "fp8k_block_gemm_noalloc: hipGetSymbolAddress: %s", hipGetErrorString(e));
    ptrs[dev] = p;
  }
  *out = ptrs[dev];
  return FP8K_OK;
}

extern "C" int fp8k_block_gemm_noalloc(const void* A, const void* B, const float* As, const float* Bs, void* C, int64_t M,
                                       int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t as_stride_m,
                                       int64_t as_stride_k, int64_t bs_stride_n, int64_t bs_stride_k, int64_t ldc,
                                       int out_dtype, void* stream) {
  clear_error();
  const int64_t need = block_gemm_workspace_bytes(M, N, K);
  if (need > kStaticScratchBytes)
    return fail(FP8K_ERR_WORKSPACE, "fp8k_block_gemm_noalloc: M=%lld N=%lld K=%lld needs %lld bytes of scratch, the built-in "
                "buffer holds %lld; use fp8k_block_gemm with a caller-owned workspace", (long long)M, (long long)N,
                (long long)K, (long long)need, (long long)kStaticScratchBytes);
  void* ws = nullptr;
  if (need > 0) {
    const int rc = static_scratch(&ws, (hipStream_t)stream);
    if (rc) return rc;
  }
  // nothing in the buffer has to start at zero: every float partial and every copied scale that a launch reads was
  // written by the same call
  return block_gemm_impl(A, B, As, Bs, C, M, N, K, lda, ldb, as_stride_m, as_stride_k, bs_stride_n, bs_stride_k, ldc,
                         out_dtype, ws, need > 0 ? kStaticScratchBytes : 0, stream);
}

extern "C" int fp8k_block_gemm_ue8m0(const void* A, const void* B, const int32_t* As_packed, const float* Bs, void* C,
                                     int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t as_stride_m,
                                     int64_t as_stride_w, int64_t bs_stride_n, int64_t bs_stride_k, int64_t ldc,
                                     int out_dtype, void* workspace, int64_t workspace_bytes_given, void* stream) {
  clear_error();
  const char* op = "block_gemm_ue8m0";
  int rc = common_checks(op, A, B, C, M, N, K, lda, ldb, ldc, out_dtype);
  if (rc) return rc;
  if (M == 0 || N == 0) return FP8K_OK;
  FP8K_REQUIRE(K > 0, "%s: K must be positive", op);
  FP8K_REQUIRE(As_packed && Bs, "%s: null scale pointer", op);
  FP8K_REQUIRE(as_stride_m >= 0 && as_stride_w >= 0 && bs_stride_n >= 0 && bs_stride_k >= 0, "%s: negative scale stride", op);
  FP8K_REQUIRE((M - 1) * as_stride_m + ((K + kTileK - 1) / kTileK / 4) * as_stride_w < (1LL << 31), "%s: scales span more than 2^31 elements", op);
  // the matrix core applies the scales only in the tile kernels, and every plan for more than 128 rows and whole K blocks is one of
  // them; smaller problems take the float-scale entry point with the exponents expanded to floats
  const Plan pl = make_plan(M, N, K);
  FP8K_REQUIRE(M > 128 && (pl.kind == 1 || pl.kind == 4 || pl.kind == 8), "%s: built for M > 128 with K a multiple of 128 (got M=%lld, K=%lld); expand the "
               "scales and call fp8k_block_gemm", op, (long long)M, (long long)K);
  const int64_t need = pl.ws_bytes;
  if (need > 0 && (!workspace || workspace_bytes_given < need))
    return fail(FP8K_ERR_WORKSPACE, "%s: workspace of %lld bytes required, %lld given", op, (long long)need,
                (long long)(workspace ? workspace_bytes_given : 0));
  GemmArgs a{};
  a.X = (const uint8_t*)A; a.W = (const uint8_t*)B; a.sx = reinterpret_cast<const float*>(As_packed); a.sw = Bs;
  a.bias = nullptr; a.C = C; a.partial = (float*)workspace;
  a.M = (int)M; a.N = (int)N; a.K = (int)K; a.ldx = lda; a.ldw = ldb; a.ldc = ldc;
  a.sx_m = as_stride_m; a.sx_k = as_stride_w; a.sw_n = bs_stride_n; a.sw_k = bs_stride_k;
  hipStream_t st = (hipStream_t)stream;
  return out_dtype == FP8K_BF16 ? launch_tiles<kModeScaled, FP8K_BF16, FP8K_F32>(a, pl, st)
                                : launch_tiles<kModeScaled, FP8K_F16, FP8K_F32>(a, pl, st);
}

extern "C" int fp8k_scaled_mm(const void* A, const void* B, const float* sa, const float* sb, const void* bias, void* C,
                              int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t ldc, int out_dtype,
                              int bias_dtype, void* workspace, int64_t workspace_bytes_given, void* stream) {
  clear_error();
  int rc = common_checks("fp8_scaled_mm", A, B, C, M, N, K, lda, ldb, ldc, out_dtype);
  if (rc) return rc;
  if (M == 0 || N == 0) return FP8K_OK;
  FP8K_REQUIRE(K > 0, "fp8_scaled_mm: K must be positive");
  FP8K_REQUIRE(sa && sb, "fp8_scaled_mm: null scale pointer");
  FP8K_REQUIRE(aligned(sb, 16), "fp8_scaled_mm: scales_b must be 16-byte aligned");
  if (bias)
    FP8K_REQUIRE(bias_dtype == FP8K_F32 || bias_dtype == FP8K_F16 || bias_dtype == FP8K_BF16,
                 "fp8_scaled_mm: bias dtype must be float32, float16 or bfloat16");
  const Plan pl = make_plan(M, N, K);
  const int64_t need = pl.ws_bytes;
  if (need > 0 && (!workspace || workspace_bytes_given < need))
    return fail(FP8K_ERR_WORKSPACE, "fp8_scaled_mm: workspace of %lld bytes required, %lld given", (long long)need,
                (long long)(workspace ? workspace_bytes_given : 0));
  GemmArgs a{};
  a.X = (const uint8_t*)A; a.W = (const uint8_t*)B; a.sx = sa; a.sw = sb; a.bias = bias; a.C = C;
  a.partial = (float*)workspace;
  a.M = (int)M; a.N = (int)N; a.K = (int)K; a.ldx = lda; a.ldw = ldb; a.ldc = ldc;
  a.sx_m = a.sw_n = 1;
  hipStream_t st = (hipStream_t)stream;
  const int bd = bias ? bias_dtype : FP8K_F32;
#define FP8K_SMM(O, B) launch<kModeRow, O, B>(a, pl, st)
  if (out_dtype == FP8K_BF16) {
    if (bd == FP8K_F32) return FP8K_SMM(FP8K_BF16, FP8K_F32);
    if (bd == FP8K_BF16) return FP8K_SMM(FP8K_BF16, FP8K_BF16);
    return FP8K_SMM(FP8K_BF16, FP8K_F16);
  }
  if (bd == FP8K_F32) return FP8K_SMM(FP8K_F16, FP8K_F32);
  if (bd == FP8K_BF16) return FP8K_SMM(FP8K_F16, FP8K_BF16);
  return FP8K_SMM(FP8K_F16, FP8K_F16);
#undef FP8K_SMM
}

// ---- whole linears, quantisation included.  Of a few rows: one launch (gemm_wavek_quant_kernel).
static bool fuses_quant(int64_t M, int64_t N, int64_t K) {
  if (M < 1 || N < 1 || N % 8 != 0 || K < kTileK || K % kTileK != 0) return false;
  return g_force_kind < 0 && few_activations(M, N, K);
}

template <int MODE, int OUT_DT, int BIAS_DT>
static int launch_quant_linear(const GemmArgs& a, hipStream_t st) {
  const dim3 grid((unsigned)((a.N + 16 * a.wk_nw - 1) / (16 * a.wk_nw))), block(512);
  const unsigned lds = (unsigned)(a.M * wq_row_bytes(a.K));
  const int64_t pieces = (int64_t)a.M * a.K / 8;
  if (pieces <= 2 * 512) hipLaunchKernelGGL((gemm_wavek_quant_kernel<2, 8, MODE, OUT_DT, BIAS_DT>), grid, block, lds, st, a);
  else if (pieces <= 4 * 512) hipLaunchKernelGGL((gemm_wavek_quant_kernel<4, 8, MODE, OUT_DT, BIAS_DT>), grid, block, lds, st, a);
  else hipLaunchKernelGGL((gemm_wavek_quant_kernel<8, 4, MODE, OUT_DT, BIAS_DT>), grid, block, lds, st, a);
  return check_launch("gemm_wavek_quant");
}

// Workspace of a linear: the quantised activations, their scales, what the GEMM's plan needs.
struct LinearLayout {
  Plan pl{};
  int64_t s = 0, work = 0, bytes = 0;  // offsets behind the quantised activations at 0
};
static LinearLayout linear_layout(int64_t M, int64_t N, int64_t K, bool block_mode) {
  LinearLayout l;
  l.pl = make_plan(M, N, K);
  l.s = align256(M * K);
  l.work = l.s + align256(M * (block_mode ? K / kTileK : 1) * 4);
  l.bytes = l.work + l.pl.ws_bytes;
  return l;
}

static int quant_linear(const char* op, bool block_mode, const void* x, const void* B, const float* Bs, int64_t bs_n, int64_t bs_k,
                        const void* bias, int bias_dtype, void* C, int64_t M, int64_t N, int64_t K, int64_t ldb, int64_t ldc, float eps,
                        int dtype, void* workspace, int64_t workspace_bytes_given, void* stream) {
  clear_error();
  int rc = common_checks(op, x, B, C, M, N, K, K, ldb, ldc, dtype);
  if (rc) return rc;
  if (M == 0 || N == 0) return FP8K_OK;
  FP8K_REQUIRE(K > 0 && (!block_mode || K % kTileK == 0), "%s: K must be a positive multiple of %d (got %lld)", op, block_mode ? kTileK : 16,
               (long long)K);
  FP8K_REQUIRE(Bs, "%s: null scale pointer", op);
  FP8K_REQUIRE(bs_n >= 0 && bs_k >= 0, "%s: negative scale stride", op);
  FP8K_REQUIRE(block_mode || ((bs_n == 0 || bs_n == 1) && (bs_n == 0 || aligned(Bs, 16))),
               "%s: channel scales must be contiguous and 16-byte aligned", op);
  FP8K_REQUIRE(!block_mode || M * (K / kTileK) < 0x38000000LL, "%s: activation scales span more than 3.5 GiB", op);
  FP8K_REQUIRE(!bias || bias_dtype == FP8K_F32 || bias_dtype == FP8K_F16 || bias_dtype == FP8K_BF16,
               "%s: bias dtype must be float32, float16 or bfloat16", op);
  const int bd = bias ? bias_dtype : FP8K_F32;
  GemmArgs a{};
  a.X = (const uint8_t*)x; a.W = (const uint8_t*)B; a.sw = Bs; a.bias = bias; a.C = C;
  a.M = (int)M; a.N = (int)N; a.K = (int)K; a.ldx = K; a.ldw = ldb; a.ldc = ldc;
  a.sw_n = bs_n; a.sw_k = bs_k;
  hipStream_t st = (hipStream_t)stream;
#define FP8K_QL(FN, O, ...) (bd == FP8K_F32    ? FN<kModeRow, O, FP8K_F32>(__VA_ARGS__) \
                             : bd == FP8K_BF16 ? FN<kModeRow, O, FP8K_BF16>(__VA_ARGS__) \
                                               : FN<kModeRow, O, FP8K_F16>(__VA_ARGS__))
#define FP8K_LINEAR(FN, ...)                                                                                                      \
  (block_mode ? (dtype == FP8K_BF16 ? FN<kModeBlock, FP8K_BF16, FP8K_BF16>(__VA_ARGS__) : FN<kModeBlock, FP8K_F16, FP8K_F16>(__VA_ARGS__)) \
   : dtype == FP8K_BF16 ? FP8K_QL(FN, FP8K_BF16, __VA_ARGS__)                                                                     \
                        : FP8K_QL(FN, FP8K_F16, __VA_ARGS__))
  if (fuses_quant(M, N, K)) {
    const Plan pl = plan_wavek(M, N, K, num_cu());
    a.q_eps = quant_eps(eps, dtype);
    a.wk_nw = pl.halves; a.kb_per_split = pl.kb_per_split;
    return FP8K_LINEAR(launch_quant_linear, a, st);
  }
  const LinearLayout l = linear_layout(M, N, K, block_mode);
  if (!workspace || workspace_bytes_given < l.bytes)
    return fail(FP8K_ERR_WORKSPACE, "%s: workspace of %lld bytes required, %lld given", op, (long long)l.bytes,
                (long long)(workspace ? workspace_bytes_given : 0));
  FP8K_REQUIRE(aligned(workspace, 256), "%s: the workspace must be 256-byte aligned", op);
  char* const ws = static_cast<char*>(workspace);
  float* const s = reinterpret_cast<float*>(ws + l.s);
  rc = quant_for_linear(block_mode, x, ws, s, M, K, eps, dtype, st);
  if (rc) return rc;
  a.X = reinterpret_cast<const uint8_t*>(ws);
  a.sx = s; a.sx_m = 1; a.sx_k = block_mode ? M : 0;
  a.partial = reinterpret_cast<float*>(ws + l.work);
  return FP8K_LINEAR(launch, a, l.pl, st);
#undef FP8K_LINEAR
#undef FP8K_QL
}

extern "C" int fp8k_linear_fuses_quant(int64_t M, int64_t N, int64_t K) { return fuses_quant(M, N, K) ? 1 : 0; }

extern "C" int64_t fp8k_linear_workspace_bytes(int64_t M, int64_t N, int64_t K, int block_mode) {
  if (M <= 0 || N <= 0 || K <= 0 || fuses_quant(M, N, K)) return 0;
  return linear_layout(M, N, K, block_mode != 0).bytes;
}

extern "C" int fp8k_block_linear(const void* x, const void* B, const float* Bs, const void* bias, void* C, int64_t M, int64_t N, int64_t K,
                                 int64_t ldb, int64_t bs_stride_n, int64_t bs_stride_k, int64_t ldc, float eps, int dtype, void* workspace,
                                 int64_t workspace_bytes_given, void* stream) {
  return quant_linear("block_linear", true, x, B, Bs, bs_stride_n, bs_stride_k, bias, dtype, C, M, N, K, ldb, ldc, eps, dtype, workspace,
                      workspace_bytes_given, stream);
}

extern "C" int fp8k_token_linear(const void* x, const void* B, const float* sb, int64_t sb_stride, const void* bias, int bias_dtype,
                                 void* C, int64_t M, int64_t N, int64_t K, int64_t ldb, int64_t ldc, int dtype, void* workspace,
                                 int64_t workspace_bytes_given, void* stream) {
  return quant_linear("token_linear", false, x, B, sb, sb_stride, 0, bias, bias_dtype, C, M, N, K, ldb, ldc, 0.f, dtype, workspace,
                      workspace_bytes_given, stream);
}

// ---- batched per-tensor-scaled FP8 GEMM (the MLA absorbed products): every batch entry is a row-mode GEMM on the short-K
// kernel or, for long K, on the 128x128 tile kernel (grid y = entry), whose per-row / per-column scale vectors are shared by all entries.
// Up to eight K blocks the short-K kernel is ahead at every row count (1 .. 4096 rows, 16 and 128 entries: 1.03 - 3.7 times;
// 128 entries of 64 x 512 x 128: 14.7 -> 6.2 us).  At 16 blocks the tile kernel's ring and larger tile are ahead with 4096 rows (16
// entries 98 against 107 us, 128 entries 773 against 816) and at 32 blocks with 16 entries of up to 64 rows (17.1 against 19.1); in
// between the short-K kernel still is, most with many entries of few rows (128 entries of 64 rows, K = 1536 / 2048 / 4096: 24.7 /
// 31.6 / 54.1 against 47.7 / 56.1 / 93.1).  The line is where it is right for every count.
constexpr int64_t kBmmShortK = 1024;
static int bmm_impl(const void* A, const void* B, const float* sa, const float* sb, int64_t scale_stride, void* C, int64_t batch,
                    int64_t M, int64_t N, int64_t K, int64_t a_stride_b, int64_t lda, int64_t b_stride_b, int64_t ldb,
                    int64_t c_stride_b, int64_t ldc, int out_dtype, void* stream) {
  clear_error();
  const char* op = "bmm_fp8";
  int rc = common_checks(op, A, B, C, M, N, K, lda, ldb, ldc, out_dtype);
  if (rc) return rc;
  FP8K_REQUIRE(batch >= 0 && batch <= 65535, "%s: batch must be in [0, 65535] (got %lld)", op, (long long)batch);
  if (batch == 0 || M == 0 || N == 0) return FP8K_OK;
  FP8K_REQUIRE(K > 0 && K % kTileK == 0, "%s: K must be a positive multiple of 128 (got %lld)", op, (long long)K);
  FP8K_REQUIRE(N % 8 == 0, "%s: N must be a multiple of 8 (got %lld)", op, (long long)N);
  FP8K_REQUIRE(sa && sb, "%s: null scale pointer", op);
  FP8K_REQUIRE(scale_stride == 0 || aligned(sb, 16), "%s: the column scale vector must be 16-byte aligned", op);
  FP8K_REQUIRE(a_stride_b % 16 == 0 && b_stride_b % 16 == 0 && (c_stride_b * 2) % 16 == 0 && a_stride_b >= 0 && b_stride_b >= 0 &&
               c_stride_b >= 0, "%s: batch strides must be non-negative multiples of 16 bytes", op);
  GemmArgs a{};
  a.X = (const uint8_t*)A; a.W = (const uint8_t*)B; a.sx = sa; a.sw = sb; a.bias = nullptr; a.C = C; a.partial = nullptr;
  a.M = (int)M; a.N = (int)N; a.K = (int)K; a.ldx = lda; a.ldw = ldb; a.ldc = ldc;
  a.sx_m = a.sw_n = scale_stride;
  a.batch_x = a_stride_b; a.batch_w = b_stride_b; a.batch_c = c_stride_b;
  hipStream_t st = (hipStream_t)stream;
  a.batch = (int)batch;
  if ((g_force_kind == 6 || (g_force_kind < 0 && K <= kBmmShortK)) && M * lda < (1LL << 31) && N * ldb < (1LL << 31)) {
    a.tiles_m = (int)((M + kBmmTileM - 1) / kBmmTileM);
    a.tiles_n = (int)((N + kBmmTileN - 1) / kBmmTileN);
    const int64_t blocks = (int64_t)a.tiles_m * a.tiles_n * ((batch + 7) / 8 * 8);
    FP8K_REQUIRE(blocks <= 0x7fffffffLL, "%s: too many tiles for one launch", op);
    if (out_dtype == FP8K_BF16) hipLaunchKernelGGL(gemm_bmm_short_kernel<FP8K_BF16>, dim3((unsigned)blocks), dim3(256), 0, st, a);
    else hipLaunchKernelGGL(gemm_bmm_short_kernel<FP8K_F16>, dim3((unsigned)blocks), dim3(256), 0, st, a);
    return check_launch(op);
  }
  a.tiles_m = (int)((M + kT128 - 1) / kT128);
  a.tiles_n = (int)((N + kT128 - 1) / kT128);
  a.splits = 1;
  a.kb_per_split = (int)(K / kTileK);
  const unsigned nwg = (unsigned)(((int64_t)a.tiles_m * a.tiles_n + 7) / 8 * 8);
  if (out_dtype == FP8K_BF16)
    hipLaunchKernelGGL((gemm_tile128_kernel<kModeRow, FP8K_BF16, FP8K_F32, false, 128>), dim3(nwg, (unsigned)batch), dim3(512), 0, st, a);
  else
    hipLaunchKernelGGL((gemm_tile128_kernel<kModeRow, FP8K_F16, FP8K_F32, false, 128>), dim3(nwg, (unsigned)batch), dim3(512), 0, st, a);
  return check_launch(op);
}

extern "C" int fp8k_bmm_fp8(const void* A, const void* B, const float* sa, const float* sb, void* C, int64_t batch, int64_t M,
                            int64_t N, int64_t K, int64_t a_stride_b, int64_t lda, int64_t b_stride_b, int64_t ldb,
                            int64_t c_stride_b, int64_t ldc, int out_dtype, void* stream) {
  return bmm_impl(A, B, sa, sb, 1, C, batch, M, N, K, a_stride_b, lda, b_stride_b, ldb, c_stride_b, ldc, out_dtype, stream);
}

extern "C" int fp8k_bmm_fp8_tensor_scales(const void* A, const void* B, const float* sa, const float* sb, void* C, int64_t batch,
                                          int64_t M, int64_t N, int64_t K, int64_t a_stride_b, int64_t lda, int64_t b_stride_b,
                                          int64_t ldb, int64_t c_stride_b, int64_t ldc, int out_dtype, void* stream) {
  return bmm_impl(A, B, sa, sb, 0, C, batch, M, N, K, a_stride_b, lda, b_stride_b, ldb, c_stride_b, ldc, out_dtype, stream);
}
