// The GEMM tiles that exist (LaunchW's template arguments: BM, BN, BK, ring
// stages, waves along M and N, split activations, fp8 weights, fp8
// activations, pipelined loop, fp8 lo correction), in the lists that one
// translation unit each (gemm_tiles_*.hip) compiles: device code generation
// for one tile's epilogues takes tens of seconds, so the lists build in
// parallel.
#pragma once

#include "gemm_kernel.h"

#define MFH_TILES_PIPE_A(X)                                 \
  X(256, 256, 32, 2, 4, 2, true, false, false, true, false) \
  X(256, 256, 32, 3, 4, 2, true, false, false, true, false)
#define MFH_TILES_PIPE_B(X) \
  X(256, 256, 32, 4, 4, 2, false, false, false, true, true)
#define MFH_TILES_PIPE_C(X)                                 \
  X(128, 256, 32, 3, 2, 4, true, false, false, true, false) \
  X(128, 256, 32, 2, 2, 2, true, false, false, true, false)
#define MFH_TILES_MID(X)                                    \
  X(128, 128, 64, 3, 2, 4, true, false, false, true, false) \
  X(64, 128, 64, 4, 2, 4, true, false, false, true, false)
#define MFH_TILES_SINGLE(X)                                   \
  X(256, 256, 32, 4, 4, 2, false, false, false, true, false)  \
  X(256, 128, 32, 3, 4, 2, false, false, false, true, false)  \
  X(256, 128, 64, 3, 4, 2, false, false, false, true, false)  \
  X(256, 256, 64, 2, 4, 2, false, false, true, false, false)  \
  X(128, 128, 64, 2, 2, 4, false, false, true, false, false)
#define MFH_TILES_SINGLE_MID(X)                              \
  X(128, 128, 64, 4, 2, 4, false, false, false, true, false) \
  X(128, 128, 64, 2, 2, 4, false, false, false, true, false) \
  X(64, 128, 64, 3, 2, 2, false, false, false, true, false)
#define MFH_TILES_SMALL(X)                                  \
  X(64, 64, 32, 2, 2, 2, true, false, false, false, false)  \
  X(64, 64, 32, 2, 2, 2, false, false, false, false, false) \
  X(64, 64, 64, 2, 2, 2, true, false, false, true, false)   \
  X(64, 64, 64, 2, 2, 2, false, false, false, true, false)  \
  X(64, 64, 64, 3, 2, 2, true, false, false, true, false)   \
  X(64, 64, 64, 3, 2, 2, false, false, false, true, false)
#define MFH_TILES_W8_A(X)                                  \
  X(256, 256, 32, 2, 4, 2, true, true, false, true, false) \
  X(256, 256, 32, 3, 4, 2, true, true, false, true, false)
#define MFH_TILES_W8_B(X)                                  \
  X(128, 256, 32, 3, 2, 4, true, true, false, true, false) \
  X(128, 256, 32, 2, 2, 2, true, true, false, true, false)
#define MFH_TILES_W8_C(X)                                  \
  X(128, 128, 64, 3, 2, 4, true, true, false, true, false) \
  X(64, 128, 64, 4, 2, 4, true, true, false, true, false)
#define MFH_TILES_W8_SINGLE(X)                              \
  X(256, 256, 32, 4, 4, 2, false, true, false, true, false) \
  X(256, 128, 64, 3, 4, 2, false, true, false, true, false) \
  X(128, 128, 64, 4, 2, 4, false, true, false, true, false) \
  X(128, 128, 64, 2, 2, 4, false, true, false, true, false) \
  X(64, 128, 64, 3, 2, 2, false, true, false, true, false)
#define MFH_TILES_W8_SMALL(X)                               \
  X(64, 64, 32, 2, 2, 2, true, true, false, false, false)  \
  X(64, 64, 32, 2, 2, 2, false, true, false, false, false) \
  X(64, 64, 64, 2, 2, 2, true, true, false, true, false)   \
  X(64, 64, 64, 2, 2, 2, false, true, false, true, false)  \
  X(64, 64, 64, 3, 2, 2, true, true, false, true, false)   \
  X(64, 64, 64, 3, 2, 2, false, true, false, true, false)

#define MFH_TILES(X)                                                               \
  MFH_TILES_PIPE_A(X) MFH_TILES_PIPE_B(X) MFH_TILES_PIPE_C(X) MFH_TILES_MID(X)     \
  MFH_TILES_SINGLE(X) MFH_TILES_SINGLE_MID(X) MFH_TILES_SMALL(X) MFH_TILES_W8_A(X) \
  MFH_TILES_W8_B(X) MFH_TILES_W8_C(X) MFH_TILES_W8_SINGLE(X) MFH_TILES_W8_SMALL(X)

#define MFH_TILE_DECLARE(...) \
  extern template hipError_t LaunchW<__VA_ARGS__>(const GemmParams &, hipStream_t);
#define MFH_TILE_DEFINE(...) \
  template hipError_t LaunchW<__VA_ARGS__>(const GemmParams &, hipStream_t);
