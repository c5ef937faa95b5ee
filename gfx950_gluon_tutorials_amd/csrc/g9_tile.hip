// Small-tile kernels (g9_tile.hpp), dense and grouped, and the rule that
// chooses between them and the 256x256 kernels.
#include "g9_tile_pick.hpp"

#include "../../include/gfx950_gemm.h"
#include "g9_tile.hpp"

using namespace g9;

// Tile TM x TN of operand type OP: NW waves, WM x WN of them computing, and as
// many ring slots as leave two workgroups to a CU (tiles up to 64x64, whose
// barriers and latencies then overlap) or fill its LDS (larger tiles).  MXFP4
// gives up slots for its scale ring.
#define G9_TILE_SHAPES(X, NAME, OP, S)      \
  X(NAME, OP, 16, 16, 4, 1, 1, S ? 16 : 20)  \
  X(NAME, OP, 16, 32, 2, 1, 2, S ? 12 : 13)  \
  X(NAME, OP, 32, 32, 4, 2, 2, S ? 8 : 10)   \
  X(NAME, OP, 64, 32, 4, 2, 2, 6)            \
  X(NAME, OP, 64, 64, 4, 2, 2, S ? 4 : 5)    \
  X(NAME, OP, 128, 64, 4, 2, 2, S ? 4 : 6)   \
  X(NAME, OP, 128, 128, 4, 2, 2, S ? 4 : 5)  \
  X(NAME, OP, 256, 128, 4, 2, 2, 3)

#define G9_TILE_KERNEL(NAME, OP, TM, TN, NW, WM, WN, NS)                                                \
  using NAME##_t##TM##x##TN = Tile<OP, TM, TN, NW, WM, WN, NS>;                                         \
  extern "C" __global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(                  \
      NAME##_t##TM##x##TN::kWavesPerSimd, NAME##_t##TM##x##TN::kWavesPerSimd))) void                    \
  NAME##_dp_t##TM##x##TN(GemmParams p) {                                                                \
    __shared__ __attribute__((aligned(1024))) char smem[NAME##_t##TM##x##TN::kLds];                     \
    int tm, tn;                                                                                         \
    tile_coords(blockIdx.x, p.tiles_m * p.tiles_n, p.tiles_m, p.tiles_n, p.num_xcds, p.group_m, tm, tn); \
    tile_gemm<NAME##_t##TM##x##TN>(p, smem, tm, tn, p.out, epilogue_scale<OP>(p));                      \
  }

// Grouped (MoE): the tile of the expert that owns it.
#define G9_TILE_MOE_KERNEL(NAME, OP, TM, TN, NW, WM, WN, NS)                                            \
  extern "C" __global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(                  \
      NAME##_t##TM##x##TN::kWavesPerSimd, NAME##_t##TM##x##TN::kWavesPerSimd))) void                    \
  NAME##_moe_t##TM##x##TN(GemmParams p) {                                                               \
    __shared__ __attribute__((aligned(1024))) char smem[NAME##_t##TM##x##TN::kLds];                     \
    int expert, tm, tn, row0, rows;                                                                     \
    if (!moe_find<TM>(p, blockIdx.x, expert, tm, tn, row0, rows)) return;                               \
    const GemmParams q = moe_params<OP>(p, expert, row0, rows);                                         \
    tile_gemm<NAME##_t##TM##x##TN>(q, smem, tm, tn, p.out, epilogue_scale<OP>(q));                      \
  }

G9_TILE_SHAPES(G9_TILE_KERNEL, g9_a16w16_f16, Op::F16, false)
G9_TILE_SHAPES(G9_TILE_KERNEL, g9_a16w16_bf16, Op::BF16, false)
G9_TILE_SHAPES(G9_TILE_KERNEL, g9_a8w8, Op::BF8, false)
G9_TILE_SHAPES(G9_TILE_KERNEL, g9_a4w4, Op::FP4, true)
G9_TILE_SHAPES(G9_TILE_KERNEL, g9_a4w4km, Op::FP4K, true)
G9_TILE_SHAPES(G9_TILE_KERNEL, g9_a4w4ps, Op::FP4P, true)

G9_TILE_SHAPES(G9_TILE_MOE_KERNEL, g9_a16w16_f16, Op::F16, false)
G9_TILE_SHAPES(G9_TILE_MOE_KERNEL, g9_a16w16_bf16, Op::BF16, false)
G9_TILE_SHAPES(G9_TILE_MOE_KERNEL, g9_a8w8, Op::BF8, false)
G9_TILE_SHAPES(G9_TILE_MOE_KERNEL, g9_a4w4, Op::FP4, true)

namespace {

struct TileEntry {
  int dtype, moe, tm, tn, threads;
  TileKernelFn fn;
};
#define G9_TILE_ENTRY(DT, NAME, TM, TN, NW) {DT, 0, TM, TN, 64 * NW, NAME##_dp_t##TM##x##TN},
#define G9_MOE_ENTRY(DT, NAME, TM, TN, NW) {DT, 1, TM, TN, 64 * NW, NAME##_moe_t##TM##x##TN},
#define G9_TILE_ENTRIES(G9_TILE_ENTRY, DT, NAME)                                                                       \
  G9_TILE_ENTRY(DT, NAME, 16, 16, 4) G9_TILE_ENTRY(DT, NAME, 16, 32, 2) G9_TILE_ENTRY(DT, NAME, 32, 32, 4) \
  G9_TILE_ENTRY(DT, NAME, 64, 32, 4) G9_TILE_ENTRY(DT, NAME, 64, 64, 4) G9_TILE_ENTRY(DT, NAME, 128, 64, 4) \
  G9_TILE_ENTRY(DT, NAME, 128, 128, 4) G9_TILE_ENTRY(DT, NAME, 256, 128, 4)

const TileEntry kTiles[] = {
    G9_TILE_ENTRIES(G9_TILE_ENTRY, G9_F16, g9_a16w16_f16) G9_TILE_ENTRIES(G9_TILE_ENTRY, G9_BF16, g9_a16w16_bf16) G9_TILE_ENTRIES(G9_TILE_ENTRY, G9_BF8, g9_a8w8)
    G9_TILE_ENTRIES(G9_TILE_ENTRY, G9_FP4, g9_a4w4) G9_TILE_ENTRIES(G9_TILE_ENTRY, G9_FP4K, g9_a4w4km) G9_TILE_ENTRIES(G9_TILE_ENTRY, G9_FP4P, g9_a4w4ps)
    G9_TILE_ENTRIES(G9_MOE_ENTRY, G9_F16, g9_a16w16_f16) G9_TILE_ENTRIES(G9_MOE_ENTRY, G9_BF16, g9_a16w16_bf16)
    G9_TILE_ENTRIES(G9_MOE_ENTRY, G9_BF8, g9_a8w8) G9_TILE_ENTRIES(G9_MOE_ENTRY, G9_FP4, g9_a4w4)};

}  // namespace

namespace g9 {

bool tile_kernel(int dtype, bool moe, int shape, TileLaunch& out) {
  int n = 0;
  for (const TileEntry& t : kTiles)
    if (t.dtype == dtype && t.moe == (int)moe && n++ == shape) {
      out = TileLaunch{t.fn, t.tm, t.tn, t.threads};
      return true;
    }
  return false;
}

}  // namespace g9
