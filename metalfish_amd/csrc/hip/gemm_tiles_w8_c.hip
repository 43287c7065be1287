#include "gemm_tiles.h"

namespace mfh {
MFH_TILES_W8_C(MFH_TILE_DEFINE)
}  // namespace mfh
