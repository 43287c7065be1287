#include "gemm_tiles.h"

namespace mfh {
MFH_TILES_MID(MFH_TILE_DEFINE)
}  // namespace mfh
