#include "gemm_tiles.h"

namespace mfh {
MFH_TILES_SINGLE_MID(MFH_TILE_DEFINE)
}  // namespace mfh
