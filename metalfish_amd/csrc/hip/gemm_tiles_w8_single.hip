#include "gemm_tiles.h"

namespace mfh {
MFH_TILES_W8_SINGLE(MFH_TILE_DEFINE)
}  // namespace mfh
