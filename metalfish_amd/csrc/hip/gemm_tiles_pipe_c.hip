#include "gemm_tiles.h"

namespace mfh {
MFH_TILES_PIPE_C(MFH_TILE_DEFINE)
}  // namespace mfh
