// tile_rows.hip -- tile_gemm.h's kernel in its "rows" output form.
#define CRANE_TILE_KERNEL
#include "tile_gemm.h"

namespace crane {
bool launch_tile_rows(const TileCfg& c, const TileArgs& a, hipStream_t st) { return launch_tile_form<kTileRows>(c, a, st); }
}  // namespace crane
