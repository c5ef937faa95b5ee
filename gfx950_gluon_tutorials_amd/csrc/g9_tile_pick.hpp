// Choice of the output tile of a data-parallel GEMM: one of the small tiles
// (g9_tile.hpp) or the 256x256 kernels' tile.  Host code only.
#pragma once

#include <climits>

namespace g9 {

struct GemmParams;
typedef void (*TileKernelFn)(GemmParams);
struct TileLaunch {
  TileKernelFn fn;
  int tm, tn, threads;
};
// Small-tile kernel `shape` (an index of kTileShapes) of operand type `dtype`,
// dense or grouped.
bool tile_kernel(int dtype, bool moe, int shape, TileLaunch& out);

// The small tiles, and last the 256x256 kernels' tile.
constexpr int kNumTiles = 8;
constexpr int kTileShapes[kNumTiles + 1][2] = {{16, 16},  {16, 32},   {32, 32},   {64, 32},  {64, 64},
                                               {128, 64}, {128, 128}, {256, 128}, {256, 256}};

// Whether a small tile can address its A rows (lda bytes apart) and row-major
// A scales (ldsa): its buffer ranges stay below 2^31 bytes, so that dead
// offsets are out of range.  Row strides go up to 2^24 bytes, which 128 rows
// allow; the 256-row tile takes them below 2^23.
inline bool tile_addresses(int tm, long long lda, long long ldsa) {
  return tm <= 128 || (lda < (1 << 23) && ldsa < (1 << 23));
}

// Cost of one tile in microseconds, fixed + per K stage (128 bytes of a row),
// by operand size (16-bit, BF8, MXFP4): the least-squares fit (in the
// logarithm) of predict() to the kernels' times on 43 shapes from 1 x 1024 to
// 8192 x 512 and 5000 x 4096, K 512-14336, one MI355X (256 CUs), operands in
// the 256 MB memory-side cache.  Over those shapes and the three types the tile
// picked takes 0.2% longer than the fastest one on average, 10% at most; they
// are the shapes of the fit.  Stages that straddle two 128-byte lines (by the
// rows' distance, their base or a K tail) take the small tiles up to twice as
// long as predicted, but of 470 drawn data-parallel calls with such stages (up
// to 600 256x256 tiles) none took more than 3% longer than on 256x256 tiles.
struct TileCost {
  float fixed, stage;
};
constexpr TileCost kTileCost[3][kNumTiles + 1] = {
    {{0.8f, 0.059f}, {0.9f, 0.071f}, {0.8f, 0.087f}, {0.4f, 0.135f}, {0.4f, 0.184f}, {1.7f, 0.28f}, {2.4f, 0.39f},
     {4.8f, 0.60f}, {6.5f, 0.95f}},
    {{1.0f, 0.050f}, {1.1f, 0.057f}, {0.9f, 0.080f}, {1.0f, 0.117f}, {0.9f, 0.160f}, {2.7f, 0.23f}, {3.7f, 0.32f},
     {5.9f, 0.51f}, {7.0f, 0.89f}},
    {{0.9f, 0.070f}, {1.1f, 0.074f}, {0.9f, 0.101f}, {1.1f, 0.140f}, {1.1f, 0.194f}, {2.7f, 0.30f}, {3.6f, 0.44f},
     {5.6f, 0.75f}, {6.9f, 1.00f}}};

// Predicted time (us) of `tiles` tiles of shape index `shape` over `ns` K
// stages on `cus` CUs, `bytes` the operands and outputs: whole rounds of one
// tile per CU (their time times `slow`), against reading the operands at
// 5.2 TB/s; a quarter of the smaller of the two does not overlap.
inline double tile_time(int family, int shape, double tiles, int ns, double bytes, int cus, double slow = 1.0) {
  const TileCost& c = kTileCost[family][shape];
  const double rounds = (double)(long long)((tiles + cus - 1) / cus);
  const double x = slow * (c.fixed + ns * (double)c.stage) * (rounds < 1 ? 1 : rounds), y = 1.0 + bytes * (1.0 / 5.2e6);
  return 2.5 + (x > y ? x + 0.25 * y : y + 0.25 * x);
}

// What the choice depends on: an M x N output of operand size `family`, `ns` K
// stages, `bytes` of operands and output, A rows (and row-major A scales) lda
// (ldsa) bytes apart, on `cus` CUs.
struct TileProblem {
  int family;
  long long M, N;
  int ns;
  double bytes;
  long long lda, ldsa;
  int cus;
};

inline double tile_count(long long M, long long N, int shape) {
  return (double)((M + kTileShapes[shape][0] - 1) / kTileShapes[shape][0]) *
         (double)((N + kTileShapes[shape][1] - 1) / kTileShapes[shape][1]);
}

// Shape index with the smallest predicted time among the tiles that can
// address the operands.  The 256x256 tile (kNumTiles) is preferred within 7%:
// its many-round times, where the chip is power-limited, are the model's least
// accurate ones.
inline int pick_tile(const TileProblem& p) {
  int best = kNumTiles;
  double best_t = 0;
  for (int i = kNumTiles; i >= 0; --i) {
    const double tiles = tile_count(p.M, p.N, i);
    if (i < kNumTiles && (tiles > INT_MAX || !tile_addresses(kTileShapes[i][0], p.lda, p.ldsa))) continue;
    const double t = tile_time(p.family, i, tiles, p.ns, p.bytes, p.cus) * (i == kNumTiles ? 0.93 : 1.0);
    if (i == kNumTiles || t < best_t) {
      best = i;
      best_t = t;
    }
  }
  return best;
}

// Predicted time (us) of split-K with S segments for each of `tiles` 256x256
// tiles: launches and a tile's fixed cost, a segment's stages (`ragged`: stages
// of a row straddle two 128-byte lines), and a share per 256 KiB partial of the
// reduction.  Least-squares fit to the split's times on 231
// drawn shapes near the rule below (rms error 7%).
constexpr float kSplitStage[3] = {1.16f, 1.12f, 1.35f};
inline double splitk_time(int family, int ns, long long tiles, int S, bool ragged) {
  return 13.1 + kSplitStage[family] * (ragged ? 1.12 : 1.0) * ((ns + S - 1) / S) + 0.0515 * (double)(tiles * S);
}

// Whether a split-K call runs data-parallel on small tile `shape` instead.
// The tiles' times depend on where the operands are: as predicted in the
// memory-side cache, 1.2 to 1.5 times that from HBM, where the split's, on
// tiles that read each operand less often, grow by 1 to 5%.  A launch cannot
// know, so the factors take the smallest geometric mean of both over the 231
// shapes (0.3% above the better of the two on average): FP16/BF16 tiles, whose
// predictions are up to 15% high, within 1.05 of the split, BF8 and MXFP4
// below 0.88, and stages off 128-byte lines, which cost the tiles up to twice
// their prediction, below 0.7.  Operands of more than 140 MB do not stay in
// the cache from one call to the next.  None of the 231 then loses to the
// split with its operands in the cache; with 1.0, 1.0 and 0.65 in their place
// 13 did, by up to 1.5 times (BF8 7972 x 896 x 22272: 159 against 122 us).
inline bool tile_beats_split(const TileProblem& p, int shape, long long tiles, int S, bool ragged) {
  if (shape >= kNumTiles) return false;
  const double slow = p.bytes > 140e6 ? 1.3 : 1.0;
  const double t = tile_time(p.family, shape, tile_count(p.M, p.N, shape), p.ns, p.bytes, p.cus, slow);
  return t < (ragged ? 0.7 : p.family == 0 ? 1.05 : 0.88) * splitk_time(p.family, p.ns, tiles, S, ragged);
}

// The choice for a grouped GEMM of p.M rows over E experts.  The rows per
// expert are on the device: an expert is taken to have the average of the
// experts that can have rows, and half an m-tile more than its rows fill.
inline int pick_moe_tile(const TileProblem& p, long long E) {
  const long long rows_e = E < p.M ? E : p.M;
  const double experts = (double)rows_e, rows = p.M / experts;
  int best = kNumTiles;
  double best_t = 0;
  for (int i = kNumTiles; i >= 0; --i) {
    const int tm = kTileShapes[i][0];
    const long long tn = (p.N + kTileShapes[i][1] - 1) / kTileShapes[i][1];
    // The grid's bound (launch_moe) has to be a 32-bit number.
    if (i < kNumTiles && ((double)((p.M + rows_e * (tm - 1)) / tm) * tn > INT_MAX || !tile_addresses(tm, p.lda, p.ldsa)))
      continue;
    const double per = rows / tm + 0.5;
    const double tiles = experts * (per < 1 ? 1 : per) * (double)tn;
    const double t = tile_time(p.family, i, tiles, p.ns, p.bytes, p.cus) * (i == kNumTiles ? 0.93 : 1.0);
    if (i == kNumTiles || t < best_t) {
      best = i;
      best_t = t;
    }
  }
  return best;
}

}  // namespace g9
