// PackInputPlanesRaw (reference src/nn/input_plane_packing.h:30-83) on the
// host: planes[batch * 112 * 64] -> masks[batch * 112], values[batch * 112].
#pragma once

#include <cstdint>

namespace mfh {

void PackPlanes(const float *planes, int batch, std::uint64_t *masks, float *values);

}  // namespace mfh
