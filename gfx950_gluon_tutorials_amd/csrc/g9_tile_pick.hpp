// Choice of the output tile of a data-parallel GEMM: one of the small tiles
// (g9_tile.hpp) or the 256x256 kernels' tile.  Host code only.
#pragma once

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
// 8192 x 512 and 5000 x 4096, K 512-14336, one MI355X (256 CUs).  Over those
// shapes and the three types the tile picked takes 0.2% longer than the
// fastest one on average, 10% at most.
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
// tile per CU, against reading the operands at 5.2 TB/s; a quarter of the
// smaller of the two does not overlap.
inline double tile_time(int family, int shape, double tiles, int ns, double bytes, int cus) {
  const TileCost& c = kTileCost[family][shape];
  const double rounds = (double)(long long)((tiles + cus - 1) / cus);
  const double x = (c.fixed + ns * (double)c.stage) * (rounds < 1 ? 1 : rounds), y = 1.0 + bytes * (1.0 / 5.2e6);
  return 2.5 + (x > y ? x + 0.25 * y : y + 0.25 * x);
}

// Shape index with the smallest predicted time for an M x N output.  The
// 256x256 tile (kNumTiles) is preferred within 7%: its many-round times, where
// the chip is power-limited, are the model's least accurate ones.
inline int pick_tile(int family, long long M, long long N, int ns, double bytes, int cus, double* time = nullptr) {
  int best = kNumTiles;
  double best_t = 0;
  for (int i = kNumTiles; i >= 0; --i) {
    const double tiles = (double)((M + kTileShapes[i][0] - 1) / kTileShapes[i][0]) *
                         (double)((N + kTileShapes[i][1] - 1) / kTileShapes[i][1]);
    const double t = tile_time(family, i, tiles, ns, bytes, cus) * (i == kNumTiles ? 0.93 : 1.0);
    if (i == kNumTiles || t < best_t) {
      best = i;
      best_t = t;
    }
  }
  if (time) *time = best_t;
  return best;
}

// The same for a grouped GEMM of T rows over E experts.  The rows per expert
// are on the device: an expert is taken to have the average of the experts
// that can have rows, and half an m-tile more than its rows fill.
inline int pick_moe_tile(int family, long long T, long long E, long long N, int ns, double row_bytes, int cus) {
  const double experts = (double)(E < T ? E : T), rows = T / experts;
  const double bytes = (T + experts * N) * row_bytes + 2.0 * T * N;
  int best = kNumTiles;
  double best_t = 0;
  for (int i = kNumTiles; i >= 0; --i) {
    const double per = rows / kTileShapes[i][0] + 0.5;
    const double tiles = experts * (per < 1 ? 1 : per) * (double)((N + kTileShapes[i][1] - 1) / kTileShapes[i][1]);
    const double t = tile_time(family, i, tiles, ns, bytes, cus) * (i == kNumTiles ? 0.93 : 1.0);
    if (i == kNumTiles || t < best_t) {
      best = i;
      best_t = t;
    }
  }
  return best;
}

}  // namespace g9
