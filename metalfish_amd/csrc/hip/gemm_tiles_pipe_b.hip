#include "gemm_tiles.h"

namespace mfh {
MFH_TILES_PIPE_B(MFH_TILE_DEFINE)
}  // namespace mfh
