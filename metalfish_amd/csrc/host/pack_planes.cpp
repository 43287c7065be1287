// Packing a batch of float planes: 28 KiB read per position, a mask and a
// value written per plane.  What bounds it is reading the planes, so a
// plane's 64 compares run four to an instruction (SSE2, part of every x86-64)
// and the mask is put together from their sign bits; the element loop before
// it took a branch per square.  256 positions (7.3 MB) on one core:
// 0.69 -> 0.10 ms.
#include "pack_planes.h"

#if defined(__SSE2__)
#include <emmintrin.h>
#endif

namespace mfh {
namespace {

constexpr int kPlanes = 112, kSquares = 64;

// Bit sq set where plane[sq] != 0 (NaN counts, -0 does not).
std::uint64_t NonZeroMask(const float *plane) {
  std::uint64_t mask = 0;
#if defined(__SSE2__)
  const __m128 zero = _mm_setzero_ps();
  for (int i = 0; i < kSquares / 16; ++i) {
    const float *p = plane + 16 * i;
    const __m128i a = _mm_castps_si128(_mm_cmpneq_ps(_mm_loadu_ps(p), zero));
    const __m128i b = _mm_castps_si128(_mm_cmpneq_ps(_mm_loadu_ps(p + 4), zero));
    const __m128i c = _mm_castps_si128(_mm_cmpneq_ps(_mm_loadu_ps(p + 8), zero));
    const __m128i d = _mm_castps_si128(_mm_cmpneq_ps(_mm_loadu_ps(p + 12), zero));
    const __m128i bytes = _mm_packs_epi16(_mm_packs_epi32(a, b), _mm_packs_epi32(c, d));
    mask |= static_cast<std::uint64_t>(static_cast<std::uint16_t>(_mm_movemask_epi8(bytes)))
            << (16 * i);
  }
#else
  for (int sq = 0; sq < kSquares; ++sq)
    mask |= static_cast<std::uint64_t>(plane[sq] != 0.0f) << sq;
#endif
  return mask;
}

}  // namespace

void PackPlanes(const float *planes, int batch, std::uint64_t *masks, float *values) {
  for (int b = 0; b < batch; ++b)
    for (int p = 0; p < kPlanes; ++p, planes += kSquares, ++masks, ++values) {
      const bool uniform = (p < 104 && p % 13 == 12) || p == 106 || p == 107 || p >= 109;
      if (uniform) {
        *values = planes[0];
        *masks = planes[0] != 0.0f ? ~0ULL : 0ULL;
        continue;
      }
      *masks = NonZeroMask(planes);
      *values = *masks ? planes[__builtin_ctzll(*masks)] : 0.0f;
    }
}

}  // namespace mfh
