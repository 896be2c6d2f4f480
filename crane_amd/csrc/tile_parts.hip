// tile_parts.hip -- tile_gemm.h's kernel in its "parts" output form.
#define CRANE_TILE_KERNEL
#include "tile_gemm.h"

namespace crane {
bool launch_tile_parts(const TileCfg& c, const TileArgs& a, hipStream_t st) { return launch_tile_form<kTileParts>(c, a, st); }
}  // namespace crane
