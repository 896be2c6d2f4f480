// tile_gated.hip -- tile_gemm.h's kernel in its "gated" output form.
#define CRANE_TILE_KERNEL
#include "tile_gemm.h"

namespace crane {
bool launch_tile_gated(const TileCfg& c, const TileArgs& a, hipStream_t st) { return launch_tile_form<kTileGated>(c, a, st); }
}  // namespace crane
