#include "gemm_tiles.h"

namespace mfh {
MFH_TILES_SMALL(MFH_TILE_DEFINE)
}  // namespace mfh
