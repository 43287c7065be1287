#include "gemm_tiles.h"

namespace mfh {
MFH_TILES_W8_A(MFH_TILE_DEFINE)
}  // namespace mfh
