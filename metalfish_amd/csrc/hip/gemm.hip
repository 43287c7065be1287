// Tile choice and launch of the MFMA GEMM (gemm_kernel.h), and the split-K
// reduce kernel.
#include "gemm_kernel.h"
#include "gemm_tiles.h"

#include <algorithm>

namespace mfh {
MFH_TILES(MFH_TILE_DECLARE)

namespace {

// Sums the k_splits fp32 partial tiles of a split-K launch in slice order
// and applies the epilogue: one thread per four consecutive outputs.  With
// LN, the GEMM read folded rows (x o gamma) and the epilogue applies their
// LayerNorm (p.fold_c, p.ln_stats) before the bias.
template <int MODE, int ACT, bool LN = false>
__global__ __launch_bounds__(256) void ReduceEpilogueKernel(GemmParams p, const float *part,
                                                            int splits) {
  const int groups = (p.N + 3) / 4;
  const int idx = blockIdx.x * 256 + threadIdx.x;
  const int row = idx / groups;
  if (row >= p.M)
    return;
  const int col = (idx % groups) * 4;
  const size_t plane = static_cast<size_t>(p.M) * p.N;
  const float *src = part + static_cast<size_t>(row) * p.N + col;
  f32x4 a = f32x4{0.f, 0.f, 0.f, 0.f};
  if (p.vec && col + 3 < p.N) {
    a = sum_parts4(src, plane, splits);
  } else {
    for (int s = 0; s < splits; ++s)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (col + r < p.N)
          a[r] += src[s * plane + r];
  }
  float b[4];
#pragma unroll
  for (int r = 0; r < 4; ++r)
    b[r] = (p.bias && col + r < p.N) ? p.bias[col + r] : 0.f;
  Epilogue4<MODE, ACT, LN>(p, row, col, a, b);
}

template <int MODE, int ACT, bool LN = false>
hipError_t LaunchReduce(const GemmParams &p, const float *part, int splits,
                        hipStream_t stream) {
  const long threads = static_cast<long>(p.M) * ((p.N + 3) / 4);
  hipLaunchKernelGGL((ReduceEpilogueKernel<MODE, ACT, LN>), dim3((threads + 255) / 256),
                     dim3(256), 0, stream, p, part, splits);
  return hipGetLastError();
}

hipError_t Reduce(const GemmParams &p, const float *part, int splits, hipStream_t stream) {
  if (p.fold_c) {
    // A folded LayerNorm's consumer (bf16 output only).
    if (p.out_mode != GEMM_OUT_BF16 || !p.ln_stats)
      return hipErrorInvalidValue;
    return p.act == ACT_NONE
               ? LaunchReduce<GEMM_OUT_BF16, ACT_NONE, true>(p, part, splits, stream)
               : LaunchReduce<GEMM_OUT_BF16, ACT_RUNTIME, true>(p, part, splits, stream);
  }
  if (p.out_mode == GEMM_OUT_RESID_F32)
    return LaunchReduce<GEMM_OUT_RESID_F32, ACT_NONE>(p, part, splits, stream);
  if (p.out_mode == GEMM_OUT_F32)
    return p.act == ACT_NONE ? LaunchReduce<GEMM_OUT_F32, ACT_NONE>(p, part, splits, stream)
                             : LaunchReduce<GEMM_OUT_F32, ACT_RUNTIME>(p, part, splits, stream);
  if (p.act == ACT_NONE)
    return LaunchReduce<GEMM_OUT_BF16, ACT_NONE>(p, part, splits, stream);
  if (p.act == ACT_MISH)
    return LaunchReduce<GEMM_OUT_BF16, ACT_MISH>(p, part, splits, stream);
  return LaunchReduce<GEMM_OUT_BF16, ACT_RUNTIME>(p, part, splits, stream);
}

// Narrow outputs (the smolgen compression: 32 columns, K = 1024) at many
// rows.  There is no reuse to stage for: a workgroup takes 32 rows x 32
// columns, its eight waves an eighth of K each, straight from memory into
// registers with every load of 128 K elements in flight at once, and the
// partial tiles are summed in wave order through LDS before the epilogue.
// What bounds it: the rows' bytes at large batches, the launch and one
// latency at small ones; the ring of 64 x 64 tiles that it replaces had 16 to
// 32 latencies in a row on too few workgroups, or a split over K with a
// second launch to sum it.
constexpr int kNarrowWaves = 8, kNarrowTile = 32;
template <bool SPLIT, bool W8, bool LN>
__global__ __launch_bounds__(kNarrowWaves * 64, 2) void NarrowKernel(GemmParams p) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int P = SPLIT ? 2 : 1, PITCH = kNarrowTile + 4;
  __shared__ float red[kNarrowWaves][kNarrowTile][PITCH];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int fr = lane & 15, fc = lane >> 4;
  const int m0 = blockIdx.x * kNarrowTile, n0 = blockIdx.y * kNarrowTile;
  const int ks = p.K / kNarrowWaves, first = wave * ks;
  const std::uint16_t *ar[P][2];
  size_t wr[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    // (Rows and columns past the edge repeat the last one.)
    const size_t row = min(m0 + i * 16 + fr, p.M - 1), col = min(n0 + i * 16 + fr, p.N - 1);
    ar[0][i] = p.A + row * p.lda + first + fc * 8;
    if constexpr (SPLIT)
      ar[1][i] = p.A_lo + row * p.lda + first + fc * 8;
    wr[i] = col * p.ldw + first + fc * 8;
  }
  // The epilogue's operands, asked for with the first rows: a thread of the
  // first four waves ends up with four outputs of row r.
  const int r = threadIdx.x / 8, c = threadIdx.x % 8 * 4;
  const bool out = r < kNarrowTile && m0 + r < p.M && n0 + c < p.N;
  float b[4] = {}, mu = 0.f, rs = 1.f, fold[4] = {}, scale[4] = {1.f, 1.f, 1.f, 1.f};
  using WRaw = std::conditional_t<W8, u32x2, bf16x8>;
  f32x4 acc[2][2] = {};
  for (int k = 0; k < ks; k += 128) {
    bf16x8 a[4][P][2];
    WRaw w[4][2];
#pragma unroll
    for (int t = 0; t < 4; ++t)
      if (k + 32 * t < ks)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
#pragma unroll
          for (int q = 0; q < P; ++q)
            a[t][q][i] = *reinterpret_cast<const bf16x8 *>(ar[q][i] + k + 32 * t);
          if constexpr (W8)
            w[t][i] = *reinterpret_cast<const WRaw *>(p.W8 + wr[i] + k + 32 * t);
          else
            w[t][i] = *reinterpret_cast<const WRaw *>(p.W + wr[i] + k + 32 * t);
        }
    if (k == 0 && out) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int col = n0 + c + e;  // (N is a multiple of 4)
        b[e] = p.bias ? p.bias[col] : 0.f;
        scale[e] = p.wscale ? p.wscale[col] : 1.f;
        if constexpr (LN)
          fold[e] = p.fold_c[col];
      }
      if constexpr (LN)
        RowLnStats(p.ln_stats, p.ln_width, p.ln_eps, m0 + r, mu, rs);
    }
#pragma unroll
    for (int t = 0; t < 4; ++t)
      if (k + 32 * t < ks) {
        bf16x8 wb[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          if constexpr (W8)
            wb[j] = Fp8x8ToBf16(w[t][j]);
          else
            wb[j] = w[t][j];
        }
#pragma unroll
        for (int q = 0; q < P; ++q)
#pragma unroll
          for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
              acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wb[j], a[t][q][i], acc[i][j],
                                                                  0, 0, 0);
      }
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
      *reinterpret_cast<f32x4 *>(&red[wave][i * 16 + fr][j * 16 + fc * 4]) = acc[i][j];
  __syncthreads();
  if (!out)
    return;
  f32x4 sum = *reinterpret_cast<const f32x4 *>(&red[0][r][c]);
#pragma unroll
  for (int v = 1; v < kNarrowWaves; ++v)
    sum += *reinterpret_cast<const f32x4 *>(&red[v][r][c]);
#pragma unroll
  for (int e = 0; e < 4; ++e)
    sum[e] = rs * (sum[e] * scale[e] - mu * fold[e]);
  GemmParams q = p;
  q.wscale = nullptr;
  Epilogue4<GEMM_OUT_BF16, ACT_NONE, false>(q, m0 + r, n0 + c, sum, b);
#endif
}

template <bool SPLIT, bool W8, bool LN>
hipError_t LaunchNarrowW(const GemmParams &p, hipStream_t stream) {
  const dim3 grid((p.M + kNarrowTile - 1) / kNarrowTile, (p.N + kNarrowTile - 1) / kNarrowTile);
  hipLaunchKernelGGL((NarrowKernel<SPLIT, W8, LN>), grid, dim3(kNarrowWaves * 64), 0, stream, p);
  return hipGetLastError();
}

// From 17 positions, where the compression is a launch of its own, to 47: the
// forward at batch 17 2002 -> 1971 us, 24 2038 -> 1996, 32 2192 -> 2166, 45
// 2701 -> 2680, bf16 at 32 2001 -> 1953.  Past that its waves and the loads
// of the same weights by every 32 rows hold up Q|K|V beside it: 48 2 %
// slower, 128 2.4 %, 300 2 %.
constexpr int kNarrowRows = 1088, kNarrowRowsEnd = 3072;
bool NarrowOk(const GemmParams &p) {
  return p.M >= kNarrowRows && p.M < kNarrowRowsEnd && p.N < 128 && p.N % 4 == 0 &&
         p.K % (32 * kNarrowWaves) == 0 && p.k_splits == 1 && p.out_mode == GEMM_OUT_BF16 &&
         p.act == ACT_NONE && !p.A8 && !p.A_lo8 && !p.C_lo8 && p.split_n >= p.N &&
         (!p.fold_c || (p.A_lo && !p.W8));
}

hipError_t LaunchNarrow(const GemmParams &p, hipStream_t stream) {
  if (p.fold_c)
    return LaunchNarrowW<true, false, true>(p, stream);
  if (p.A_lo)
    return p.W8 ? LaunchNarrowW<true, true, false>(p, stream)
                : LaunchNarrowW<true, false, false>(p, stream);
  return p.W8 ? LaunchNarrowW<false, true, false>(p, stream)
              : LaunchNarrowW<false, false, false>(p, stream);
}

// A tile with bf16 or fp8 weights on the pipelined loops.
template <int BM, int BN, int BK, int ST, int WM, int WN, bool SPLIT>
hipError_t LaunchPipe(const GemmParams &p, hipStream_t stream) {
  return p.W8 ? LaunchW<BM, BN, BK, ST, WM, WN, SPLIT, true, false, true>(p, stream)
              : LaunchW<BM, BN, BK, ST, WM, WN, SPLIT, false, false, true>(p, stream);
}

// 64 x 64 over BK = 32, lock-step (K a multiple of 32, or little LDS).
template <bool SPLIT> hipError_t LaunchStep32(const GemmParams &p, hipStream_t stream) {
  return p.W8 ? LaunchW<64, 64, 32, 2, 2, 2, SPLIT, true>(p, stream)
              : LaunchW<64, 64, 32, 2, 2, 2, SPLIT, false>(p, stream);
}

bool Aligned(const void *ptr, std::uintptr_t bytes) {
  return (reinterpret_cast<std::uintptr_t>(ptr) & (bytes - 1)) == 0;
}

}  // namespace

// Rows from which the tile rules for large problems apply (below them,
// 64 x 64 tiles over the whole K or split-K).
constexpr int kLargeRows = 1536;
// Rows from which the time model below is fitted for a long K (LaunchGemm).
// With bf16 weights up to 16 positions: at 17 to 23, beside the smolgen chain,
// it moved the forward by -0.4 to +0.7 %; with e4m3 weights 20 gained 1.8 %.
constexpr int kModelRows = 256, kModelRowsEnd = 1088;

// 256 x 256 tiles where they fill whole rounds of 256 workgroups (bf16
// activations, one K slice, from the large-problem rows).
bool GemmWholeRoundTiles(const GemmParams &p) {
  const long big_tiles = static_cast<long>((p.M + 255) / 256) * ((p.N + 255) / 256);
  return p.M >= kLargeRows && p.N >= 128 && p.k_splits == 1 && big_tiles % 256 == 0 && !p.A8;
}

// (Split precision: two 128 x 256 tiles per CU.)
bool GemmFillsCus(const GemmParams &p) {
  const long wide = static_cast<long>((p.M + 127) / 128) * ((p.N + 255) / 256);
  return GemmWholeRoundTiles(p) || (p.A_lo && p.M >= kLargeRows && wide >= 512);
}

namespace {

// The tiles of the GEMMs from kLargeRows rows on (LDS sizes with bf16
// weights).  Those of split precision compile a folded LayerNorm's epilogue.
enum class Tile {
  kNone,
  kLo8,      // 256 x 256, BF16X2_FP8LO
  k256,      // 256 x 256, three stages of 48 KiB (one workgroup per CU)
  k256Two,   // 256 x 256, two stages (beside the smolgen chain)
  k128x256,  // 128 x 256, eight waves, three stages of 32 KiB
  kWide,     // 128 x 256, four waves, two stages of 32 KiB (beside the chain)
  k128,      // 128 x 128 over BK = 64, three stages of 48 KiB
  k64x128,   // 64 x 128 over BK = 64, four stages of 32 KiB
  k64Three,  // 64 x 64 over BK = 64, three stages of 24 KiB (two per CU)
  k64,       // 64 x 64 over BK = 64, two stages of 24 KiB (three per CU)
  kNarrow,   // 64 x 64 over BK = 32, two stages (narrow N, beside the chain)
  kSplitK,   // split over K, the reduce kernel applying the LayerNorm
  // Single bf16.
  kOne256,      // 256 x 256, four stages of 32 KiB
  kOneSlim,     // 256 x 128, three stages of 24 KiB (beside the chain)
  kOne256x128,  // 256 x 128 over BK = 64, three stages of 48 KiB
  kOne128,      // 128 x 128 over BK = 64, four stages of 32 KiB
  kOne128Two,   // 128 x 128 over BK = 64, two stages (two per CU)
  kOne64x128,   // 64 x 128 over BK = 64, three stages of 24 KiB (two per CU)
  kOne64,       // 64 x 64 over BK = 64, three stages of 16 KiB (three per CU)
};

// Time of a launch, in microseconds as measured on MI355X: 3 for the launch,
// and per round of `slots` workgroups start + (per_k + fill_k * f) * K / 1024
// with f the share of the slots the round fills (fewer busy CUs clock higher
// and share less bandwidth); a residual epilogue adds resid, an activation
// act (nothing where a CU's other workgroups run meanwhile).  Fitted to
// isolated launches at the BT4 widths and 1536 to 19200 rows; the model is
// within 10 % of most of them and orders the tiles as measured, e.g. (split)
// 2048 rows out-projection 12.6 us on 64 x 128, 16.5 on 128 x 128, 27.9 on
// 128 x 256; 4096 rows 19.1 on 128 x 128, 21.0 on 64 x 128; 16384 rows 67.6
// on 256 x 256, 80.7 on 128 x 128; FFN1 there 108.6 on 128 x 256 against
// 119.6 on 256 x 256 (1.5 rounds).  Single bf16, out-projection at 4096 rows:
// 14.7 on 128 x 128 (20.0-23.5 on the tiles it took before).
struct TileTime {
  Tile tile;
  int bm, bn, slots;
  float start, resid, act, per_k, fill_k;
};
constexpr TileTime kOneTimes[] = {
    {Tile::kOne256, 256, 256, 256, 6.f, 7.f, 5.f, 18.f, 10.f},
    {Tile::kOneSlim, 256, 128, 256, 6.5f, 3.f, 0.f, 10.5f, 4.5f},
    {Tile::kOne256x128, 256, 128, 256, 5.f, 2.f, 2.5f, 9.6f, 5.4f},
    {Tile::kOne128, 128, 128, 256, 2.f, 0.5f, 1.f, 6.f, 3.f},
    {Tile::kOne128Two, 128, 128, 512, 2.f, 0.5f, 0.f, 10.5f, 11.f},
    {Tile::kOne64x128, 64, 128, 512, 1.5f, 0.5f, 0.f, 4.f, 7.f},
    {Tile::kOne64, 64, 64, 768, 1.5f, 0.5f, 0.f, 2.1f, 6.4f},
};
constexpr TileTime kTileTimes[] = {
    {Tile::k256, 256, 256, 256, 6.f, 9.f, 5.f, 29.f, 20.f},
    {Tile::k128x256, 128, 256, 256, 3.f, 3.f, 2.f, 19.f, 8.5f},
    {Tile::k128, 128, 128, 256, 2.5f, 1.5f, 1.f, 9.5f, 5.f},
    {Tile::k64x128, 64, 128, 256, 1.5f, 1.f, 0.5f, 5.8f, 2.5f},
    {Tile::k64, 64, 64, 768, 2.f, 1.f, 0.f, 6.f, 6.5f},
    {Tile::k64Three, 64, 64, 256, 0.5f, 1.f, 0.f, 3.3f, 1.9f},
};

float LaunchTime(const TileTime &t, int M, const GemmParams &p) {
  const long tiles = static_cast<long>((M + t.bm - 1) / t.bm) * ((p.N + t.bn - 1) / t.bn);
  const float k = p.K / 1024.f;
  const float start = t.start + (p.out_mode == GEMM_OUT_RESID_F32 ? t.resid : 0.f) +
                      (p.act != ACT_NONE ? t.act : 0.f);
  const long full = tiles / t.slots, rem = tiles % t.slots;
  float us = 3.f + full * (start + (t.per_k + t.fill_k) * k);
  if (rem)
    us += start + (t.per_k + t.fill_k * rem / t.slots) * k;
  return us;
}

// The fastest tile by that model for M rows of p; a folded LayerNorm takes
// whole tiles, on the residual side of kLnStatCols columns at least.
Tile BestTile(const GemmParams &p, int M, float *us) {
  const bool ln_res = p.out_gamma || p.res_stats;
  Tile best = Tile::kNone;
  *us = 0.f;
  const auto consider = [&](const TileTime &t) {
    if (((p.fold_c || ln_res) && p.N % t.bn) || (ln_res && t.bn < kLnStatCols))
      return;
    if (p.W8 && t.tile == Tile::kOneSlim)  // (its e4m3 stage is no whole wave-loads)
      return;
    const float c = LaunchTime(t, M, p);
    if (best == Tile::kNone || c < *us) {
      best = t.tile;
      *us = c;
    }
  };
  if (p.A_lo)
    for (const TileTime &t : kTileTimes)
      consider(t);
  else
    for (const TileTime &t : kOneTimes)
      consider(t);
  return best;
}

// A short K under a wide output (the smolgen global projection): the time
// goes into the stores, which two workgroups per CU overlap with each
// other's loads.  N = 4096, K = 256, split with fp32 output: 8192 rows 47.6
// us (256 x 256 tiles 53.1), 9600 59.1 (71.7), 16384 106 (112), but 2048
// 17.8 (128 x 256 with eight waves 17.2); single bf16 8192 rows 30.2 (256 x 256 34.3),
// 9600 35.7 (256 x 128 39.7), 16384 56.3 (60.7), 32768 131 (122.9).  Past 16384
// rows the 256 x 256 tiles' rounds are long enough (batch 1024 0.6 % slower).
bool StoreBound(const GemmParams &p) {
  return p.K <= 256 && p.M > 2048 && p.M <= 16384 && p.N >= 2048 && p.N % 256 == 0 &&
         p.act == ACT_NONE && !p.beside_chain && p.out_mode != GEMM_OUT_RESID_F32 && !p.fold_c;
}

// Rows of p to run on whole rounds of 256 x 256 tiles, the rest following as
// a launch of its own on smaller ones (0: one launch).  A last round that is
// nearly empty costs as much as a full one: out-projection at 19200 rows
// (300 tiles of 256 x 256) 129 us on them, 100 on 128 x 128, 67 + 20 split.
int RowsFirst(const GemmParams &p) {
  if (p.N % 256 || p.K % 64 || p.beside_chain || p.M < kLargeRows || StoreBound(p))
    return 0;
  const TileTime &whole = p.A_lo ? kTileTimes[0] : kOneTimes[0];
  const int nbn = p.N / 256, nbm = p.M / 256;
  const long rounds = static_cast<long>(nbm) * nbn / 256;
  if (rounds < 1)
    return 0;
  const int rows = static_cast<int>(rounds * 256 / nbn) * 256;
  if (rows >= p.M)
    return 0;
  float one, rest;
  BestTile(p, p.M, &one);
  BestTile(p, p.M - rows, &rest);
  return LaunchTime(whole, rows, p) + rest < 0.97f * one ? rows : 0;
}

// The tile of a large GEMM, or of one with a folded LayerNorm (kNone: none
// of these).
Tile LargeTile(const GemmParams &p) {
  const bool res = p.out_mode == GEMM_OUT_RESID_F32;
  const bool ln = p.fold_c || p.out_gamma || p.res_stats;
  if (p.A8 || p.k_splits != 1 || (ln && p.W8))
    return Tile::kNone;
  if (p.K % 64) {
    // The tiles over BK = 32, on whole rounds.  Isolated, single bf16, against
    // the lock-step 64 x 64 ones: 16384 x 1024 over K = 1056 104 -> 52 us,
    // 65536 x 256 over 224 42 -> 27, 16384 x 1024 over 96 28 -> 24.
    if (ln || p.A_lo8 || !GemmWholeRoundTiles(p))
      return Tile::kNone;
    return !p.A_lo ? Tile::kOne256 : p.beside_chain ? Tile::k256Two : Tile::k256;
  }
  if (p.A_lo8)
    return !ln || p.N % 256 == 0 ? Tile::kLo8 : Tile::kNone;
  if (!p.A_lo) {
    if (ln || p.M < kLargeRows || p.N < 128)
      return Tile::kNone;
    if (StoreBound(p))
      return Tile::kOne128Two;
    if (p.beside_chain)
      return GemmWholeRoundTiles(p) ? Tile::kOne256 : p.W8 ? Tile::kOne128Two : Tile::kOneSlim;
    float us;
    return BestTile(p, p.M, &us);
  }
  if (p.N < 128) {
    // Narrow consumers (the smolgen compression): split over K where the
    // launcher splits them (the split GEMM sums x o gamma and the reduce
    // kernel applies the LayerNorm before the bias).
    if (!ln || res)
      return Tile::kNone;
    return !p.small_lds && GemmAutoSplits(p) > 1 ? Tile::kSplitK : Tile::kNarrow;
  }
  if (p.M < kLargeRows)
    return Tile::kNone;
  if (p.beside_chain && !res) {
    // Q|K|V beside the smolgen chain: two-stage tiles, so that the chain's
    // run on the same CUs.  Forward with 128 x 256 four-wave tiles against
    // 256 x 128 ones: batch 24 and 32 equal, 64 3155 -> 3038 us, 128 5586 ->
    // 5464, 200 8594 -> 8357; on 128 x 128 tiles (144 KiB) 32 was 4 % slower,
    // 64 4 %, 200 4 %.
    if (GemmWholeRoundTiles(p) && p.N % 256 == 0)
      return Tile::k256Two;
    return !ln || p.N % 256 == 0 ? Tile::kWide : Tile::kNone;
  }
  if (StoreBound(p))
    return Tile::kWide;
  float us;
  return BestTile(p, p.M, &us);
}

// Rows first .. first + rows - 1 of p.
GemmParams RowRange(const GemmParams &p, int first, int rows) {
  GemmParams q = p;
  const size_t r = first;
  const auto bf16 = [](const std::uint16_t *x, size_t off) { return x ? x + off : nullptr; };
  const bool f32 = p.out_mode != GEMM_OUT_BF16 && !p.out_gamma;
  const auto out = [&](void *c, int ld) -> void * {
    return c ? static_cast<char *>(c) + r * ld * (f32 ? 4 : 2) : nullptr;
  };
  q.M = rows;
  q.A = bf16(p.A, r * p.lda);
  q.A_lo = bf16(p.A_lo, r * p.lda);
  q.C = out(p.C, p.ldc);
  q.C_lo = out(p.C_lo, p.ldc);
  q.C2 = out(p.C2, p.ldc2);
  q.C2_lo = out(p.C2_lo, p.ldc2);
  q.resid = p.resid ? p.resid + r * p.ldr : nullptr;
  q.resid16 = bf16(p.resid16, r * p.ldr);
  q.resid16_lo = bf16(p.resid16_lo, r * p.ldr);
  q.C_lo8 = p.C_lo8 ? p.C_lo8 + r * p.ldc8 : nullptr;
  q.A_lo8 = p.A_lo8 ? p.A_lo8 + r * p.lda8 : nullptr;
  const size_t stats = p.ln_width ? r * (p.ln_width / kLnStatCols) * 2 : 0;
  q.ln_stats = p.ln_stats ? p.ln_stats + stats : nullptr;
  q.res_stats = p.res_stats ? p.res_stats + stats : nullptr;
  q.out_stats = p.out_stats ? p.out_stats + stats : nullptr;
  return q;
}

// The pipelined tiles address an operand with 32-bit byte offsets from its
// first element, below 2^31 (past that a buffer load reads zeros).  Rows of p
// within reach: all of them, or how many to take at a time, in equal ranges of
// whole 256-row tiles (0: the weights, or 256 rows, are past it).
constexpr long kReach = (1l << 31) - 1;
int RowsInReach(const GemmParams &p) {
  if (static_cast<long>(p.N) * p.ldw * (p.W8 ? 1 : 2) > kReach)
    return 0;
  const long most = kReach / (2l * p.lda);
  if (p.M <= most)
    return p.M;
  if (most < 256 || p.k_splits > 1)  // (a slice's plane holds all rows)
    return 0;
  const long ranges = (p.M + most / 256 * 256 - 1) / (most / 256 * 256);
  return static_cast<int>(((p.M + ranges - 1) / ranges + 255) / 256 * 256);
}

hipError_t LaunchTile(Tile t, const GemmParams &p, hipStream_t stream) {
  switch (t) {
  case Tile::kLo8:
    return LaunchW<256, 256, 32, 4, 4, 2, false, false, false, true, true>(p, stream);
  case Tile::k256:
    return LaunchPipe<256, 256, 32, 3, 4, 2, true>(p, stream);
  case Tile::k256Two:
    return LaunchPipe<256, 256, 32, 2, 4, 2, true>(p, stream);
  case Tile::k128x256:
    return LaunchPipe<128, 256, 32, 3, 2, 4, true>(p, stream);
  case Tile::kWide:
    return LaunchPipe<128, 256, 32, 2, 2, 2, true>(p, stream);
  case Tile::k128:
    return LaunchPipe<128, 128, 64, 3, 2, 4, true>(p, stream);
  case Tile::k64x128:
    return LaunchPipe<64, 128, 64, 4, 2, 4, true>(p, stream);
  case Tile::k64:
    return LaunchPipe<64, 64, 64, 2, 2, 2, true>(p, stream);
  case Tile::k64Three:
    return LaunchPipe<64, 64, 64, 3, 2, 2, true>(p, stream);
  case Tile::kNarrow:
    return LaunchStep32<true>(p, stream);
  case Tile::kOne256:
    return LaunchPipe<256, 256, 32, 4, 4, 2, false>(p, stream);
  case Tile::kOneSlim:
    return LaunchW<256, 128, 32, 3, 4, 2, false, false, false, true>(p, stream);
  case Tile::kOne256x128:
    return LaunchPipe<256, 128, 64, 3, 4, 2, false>(p, stream);
  case Tile::kOne128:
    return LaunchPipe<128, 128, 64, 4, 2, 4, false>(p, stream);
  case Tile::kOne128Two:
    return LaunchPipe<128, 128, 64, 2, 2, 4, false>(p, stream);
  case Tile::kOne64x128:
    return LaunchPipe<64, 128, 64, 3, 2, 2, false>(p, stream);
  case Tile::kOne64:
    return LaunchPipe<64, 64, 64, 3, 2, 2, false>(p, stream);
  default:
    return hipErrorInvalidValue;
  }
}

}  // namespace

bool GemmLnFoldOk(const GemmParams &p) {
  // (The caller's parameters carry no LayerNorm yet: a consumer, or a
  // residual GEMM as producer.)
  if (p.out_mode != GEMM_OUT_BF16 && p.out_mode != GEMM_OUT_RESID_F32)
    return false;
  GemmParams q = p;
  static const float one = 1.f;
  if (q.out_mode == GEMM_OUT_RESID_F32)
    q.out_gamma = &one;
  else
    q.fold_c = &one;
  return LargeTile(q) != Tile::kNone;
}

// Split-K at few positions (64 x 64 tiles, K in 64-wide steps).  A GEMM
// kernel here costs ~5 us however short its K loop, and a separate reduce
// launch another ~4.5 us, so:
// * the slices fill at most one workgroup per CU (256): beyond that the
//   extra slices lengthen the kernel more than they shorten each loop;
// * a split whose partials need their own reduce launch (LaunchGemm) is
//   taken for long K loops only (>= 16 steps) and at least four ways: a
//   two-way split of FFN1 at 256 rows (10.1 + 4.8 us against 11.9 us whole)
//   and any split of the smolgen global projection (K = 256) lost;
// * a caller whose next kernel sums the partials anyway (the LayerNorm
//   after a residual GEMM) also takes a two-way split up to 384 workgroups.
// Measured forward (with the three-stage rings below): batch 1 1.29 ->
// 1.20 ms, 2 1.43 -> 1.26, 4 1.58 -> 1.33, 8 1.62 -> 1.48, 12 1.79 -> 1.76.
// (kSplitMaxGroups and kSplitPairMaxGroups are in mfh_kernels.h.)
constexpr int kSplitMinSteps = 16;
constexpr int kSplitMinParts = 4;

int GemmAutoSplits(const GemmParams &p, bool summed_by_consumer) {
  const bool large = p.M >= kLargeRows && p.N >= 128;
  if (large || p.k_splits != 1 || !p.partials || p.N % 4 || p.K % 64 || p.M <= 0 || p.N <= 0)
    return 1;
  const long tiles = static_cast<long>((p.M + 63) / 64) * ((p.N + 63) / 64);
  const int steps = p.K / 64;
  const auto fits = [&](int s) {
    return static_cast<size_t>(s) * p.M * p.N <= p.partials_floats;
  };
  int splits = 1;
  if (summed_by_consumer || steps >= kSplitMinSteps)
    for (int s = 2; s <= steps; ++s)
      if (steps % s == 0 && tiles * s <= kSplitMaxGroups && fits(s))
        splits = s;
  if (!summed_by_consumer && splits < kSplitMinParts)
    splits = 1;
  if (splits == 1 && summed_by_consumer && steps % 2 == 0 && tiles * 2 <= kSplitPairMaxGroups &&
      fits(2))
    splits = 2;
  return splits;
}

hipError_t LaunchGemm(const GemmParams &p_in, hipStream_t stream, std::string *err) {
  auto fail = [&](const char *why) {
    if (err)
      *err = std::string("gemm: ") + why;
    return hipErrorInvalidValue;
  };
  GemmParams p = p_in;
  const bool lo8 = p.A_lo8 != nullptr;
  if (lo8 && (!p.A || p.A_lo || !p.W || p.W8 || !p.wscale || !p.W_lo8 || p.A8 ||
              p.k_splits != 1 || p.K % 128 || p.lda8 % 128 || p.ldw8 % 128 || p.lda8 < p.K ||
              p.ldw8 < p.K || !Aligned(p.A_lo8, 16) || !Aligned(p.W_lo8, 16)))
    return fail("fp8 lo correction needs A (hi) + A_lo8 with W (bf16) + W_lo8 + wscale, "
                "one K slice, K % 128 == 0, lda8 / ldw8 % 128 == 0 and 16-byte aligned codes");
  const bool f8 = p.A8 != nullptr;
  if (f8) {
    // fp8 activations x fp8 weights: the byte operands go through the bf16
    // data path as 16-bit units (K and leading dimensions halved); the F8
    // kernels run one fp8 MFMA per 128-byte K step.
    if (p.A || p.A_lo || !p.W8 || p.W || !p.wscale || !p.ascale || p.k_splits != 1 ||
        p.K % 128 || p.lda % 16 || p.ldw % 16 || p.lda < p.K || p.ldw < p.K ||
        !Aligned(p.A8, 16) || !Aligned(p.W8, 16) || p.M < 2048)
      return fail("fp8 activations need A8 + ascale with W8 + wscale, K % 128 == 0, "
                  "lda / ldw % 16 == 0, 16-byte aligned operands and M >= 2048");
    p.A = reinterpret_cast<const std::uint16_t *>(p.A8);
    p.lda /= 2;
    p.W = reinterpret_cast<const std::uint16_t *>(p.W8);
    p.W8 = nullptr;
    p.ldw /= 2;
    p.K /= 2;
    p.partials = nullptr;
  }
  if (p.M <= 0 || p.N <= 0 || p.K <= 0)
    return fail("non-positive shape");
  if (p.K % 32)
    return fail("K must be a multiple of 32");
  if (p.k_splits < 1 || p.K % (p.k_splits * 32))
    return fail("K must split into multiples of 32");
  if (p.k_splits > 1 && (p.out_mode != GEMM_OUT_F32 || p.bias || p.act != ACT_NONE ||
                         p.split_n < p.N))
    return fail("split-K writes raw fp32 partials only (no bias, activation or split)");
  if (!p.A || (!p.W && !p.W8) || (p.W && p.W8) || !p.C)
    return fail("null operand (or both W and W8)");
  if (p.W8 && !p.wscale)
    return fail("fp8 weights need row scales");
  if (!Aligned(p.A, 16) || (p.W && !Aligned(p.W, 16)) || (p.W8 && !Aligned(p.W8, 8)) ||
      (p.A_lo && !Aligned(p.A_lo, 16)) || p.lda % 8 || p.ldw % 8 || p.lda < p.K ||
      p.ldw < p.K)
    return fail("operands must be 16-byte aligned with ld >= K, ld % 8 == 0");
  if (p.out_mode == GEMM_OUT_RESID_F32 &&
      ((!p.resid && !p.resid16) || (p.resid && p.resid16) ||
       (p.resid16 != nullptr) != (p.resid16_lo != nullptr) || p.split_n < p.N))
    return fail("residual mode needs resid (fp32) or resid16 + resid16_lo (split), and no "
                "split output");
  if (p.out_mode == GEMM_OUT_RESID_F32 && p.resid16 &&
      (!Aligned(p.resid16, 2) || !Aligned(p.resid16_lo, 2)))
    return fail("split residual planes must be 2-byte aligned");
  if (p.split_n < p.N && (!p.C2 || p.ldc2 < p.N - p.split_n || p.split_n % 4))
    return fail("split output needs C2 wide enough and split_n % 4 == 0");
  if (p.split_n < p.N && (p.C_lo != nullptr) != (p.C2_lo != nullptr))
    return fail("split output needs lo planes for both parts or neither");
  if (p.ldc < (p.split_n < p.N ? p.split_n : p.N))
    return fail("ldc too small");
  // Folded LayerNorm (see GemmParams): consumer and residual sides.
  const bool ln_res = p.out_mode == GEMM_OUT_RESID_F32 && (p.out_gamma || p.res_stats);
  constexpr int kLnCols = kLnStatCols;
  if (p.fold_c && (!p.ln_stats || p.out_mode == GEMM_OUT_RESID_F32 || p.ln_width != p.K ||
                   p.K % (2 * kLnCols) || p.K > 128 * kLnCols || !Aligned(p.fold_c, 16) ||
                   !Aligned(p.ln_stats, 16) || p.k_splits != 1))
    return fail("folded LayerNorm consumer: ln_stats, fold_c (16-byte aligned), K = ln_width a "
                "multiple of 256 up to 16384, one K slice, not the residual mode");
  if ((p.out_gamma || p.res_stats) && !ln_res)
    return fail("folded LayerNorm output / residual: residual mode only");
  if (ln_res && (!p.resid16 || p.k_splits != 1 || p.ln_width != p.N || p.N % (2 * kLnCols) ||
                 p.N > 128 * kLnCols ||
                 (p.res_stats && (!p.res_gamma || !p.res_beta || !Aligned(p.res_stats, 16) ||
                                  !Aligned(p.res_gamma, 16) || !Aligned(p.res_beta, 16))) ||
                 (p.out_gamma && (!p.out_stats || !Aligned(p.out_gamma, 16) ||
                                  !Aligned(p.out_stats, 8) || !p.C_lo))))
    return fail("folded LayerNorm residual: split residual, one K slice, N = ln_width a "
                "multiple of 256 up to 16384, gamma / beta / stats 16-byte aligned, a bf16 lo "
                "output plane with out_gamma");
  if (p.C_lo8 && !(p.out_mode == GEMM_OUT_RESID_F32 && p.out_gamma) &&
      (p.out_mode != GEMM_OUT_BF16 || p.C_lo || p.split_n < p.N || p.k_splits != 1 ||
       p.ldc8 < p.N || p.ldc8 % 8 || !Aligned(p.C_lo8, 8)))
    return fail("e4m3 lo output: bf16 mode, one output, no bf16 lo plane, ldc8 >= N, "
                "ldc8 % 8 == 0, 8-byte aligned");
  if (p.C_lo8 && p.out_gamma && (p.ldc8 < p.N || p.ldc8 % 8 || !Aligned(p.C_lo8, 8)))
    return fail("e4m3 lo output: ldc8 >= N, ldc8 % 8 == 0, 8-byte aligned");
  // Vector (4-column) stores need every output row start aligned to 4
  // elements' width; otherwise the epilogue stores element by element.
  const bool f32 = (p.out_mode != GEMM_OUT_BF16 && !p.out_gamma) || p.k_splits > 1;
  const std::uintptr_t vb = f32 ? 16 : 8;
  p.vec = Aligned(p.C, vb) && p.ldc % 4 == 0 && (!p.C_lo || Aligned(p.C_lo, vb)) &&
          (p.split_n >= p.N ||
           (Aligned(p.C2, vb) && p.ldc2 % 4 == 0 && (!p.C2_lo || Aligned(p.C2_lo, vb)))) &&
          (p.out_mode != GEMM_OUT_RESID_F32 ||
           (p.ldr % 4 == 0 && (p.resid16 ? Aligned(p.resid16, 8) && Aligned(p.resid16_lo, 8)
                                          : Aligned(p.resid, 16))));
  // Eight-column groups with 16-byte accesses (staged epilogue).
  const bool out_bf16 = p.out_mode == GEMM_OUT_BF16 || p.out_gamma;
  const int gcols = out_bf16 ? 8 : 4;  // elements per 16 bytes
  p.vec8 = p.vec && Aligned(p.C, 16) && p.ldc % gcols == 0 &&
           (!p.C_lo || Aligned(p.C_lo, 16)) &&
           (p.split_n >= p.N || (p.split_n % 8 == 0 && Aligned(p.C2, 16) &&
                                 p.ldc2 % gcols == 0 && (!p.C2_lo || Aligned(p.C2_lo, 16)))) &&
           (!p.bias || Aligned(p.bias, 16)) && (!p.wscale || Aligned(p.wscale, 16)) &&
           (p.out_mode != GEMM_OUT_RESID_F32 ||
            (p.resid16 ? Aligned(p.resid16, 16) && Aligned(p.resid16_lo, 16) && p.ldr % 8 == 0
                       : Aligned(p.resid, 16) && p.ldr % 4 == 0));
  if (NarrowOk(p))
    return LaunchNarrow(p, stream);
  const int reach = f8 ? p.M : RowsInReach(p);
  if (reach == 0) {
    // Lock-step tiles, which load through 64-bit addresses.
    if (p.fold_c || ln_res || lo8)
      return fail("folded LayerNorm or fp8 lo correction: weights below 2 GiB");
    return p.A_lo ? LaunchStep32<true>(p, stream) : LaunchStep32<false>(p, stream);
  }
  if (reach < p.M) {
    for (int first = 0; first < p.M; first += reach) {
      const GemmParams q = RowRange(p_in, first, std::min(reach, p.M - first));
      const hipError_t e = LaunchGemm(q, stream, err);
      if (e != hipSuccess)
        return e;
    }
    return hipSuccess;
  }
  // Large shapes and any folded LayerNorm: the tiles of LargeTile.  (BF16X2_FP8LO: 256 x 256 tiles
  // of eight waves, the hi pass on the four-stage single-bf16 pipelined ring,
  // 128 KiB, then the lo pass on two 64 KiB stages of code rows.)
  const Tile tile = LargeTile(p);
  if (tile == Tile::kSplitK) {
    if (!Aligned(p.partials, 16) || !p.vec || p.N % 4)
      return fail("folded LayerNorm split over K: 16-byte aligned partials, vector stores");
  } else if (tile != Tile::kNone) {
    const int rows = tile == Tile::kLo8 ? 0 : RowsFirst(p);
    if (rows == 0)
      return LaunchTile(tile, p, stream);
    float us;
    const Tile whole = p.A_lo ? Tile::k256 : Tile::kOne256;
    const hipError_t e = LaunchTile(whole, RowRange(p, 0, rows), stream);
    const GemmParams rest = RowRange(p, rows, p.M - rows);
    return e != hipSuccess ? e : LaunchTile(BestTile(rest, rest.M, &us), rest, stream);
  } else if (p.fold_c || ln_res || lo8) {
    return fail("folded LayerNorm or fp8 lo correction: split-precision activations, one K "
                "slice, K % 64 == 0 and N a multiple of the tile's width");
  }
  const bool split = p.A_lo != nullptr;
  const bool large = p.M >= kLargeRows && p.N >= 128;
  // Small problems (few positions): 64 x 64 tiles leave most CUs idle and
  // walk K serially, so the launcher splits K (GemmAutoSplits), writes fp32
  // partials to p.partials through a three-stage ring and sums them in
  // slice order in a second kernel that applies the epilogue.  The split depends on the shape
  // only: a batch size always takes the same path and gives the same bits.
  if (!large && !ln_res && p.k_splits == 1 && p.partials && Aligned(p.partials, 16) && p.vec &&
      p.N % 4 == 0) {
    const int splits = GemmAutoSplits(p);
    if (splits > 1) {
      GemmParams q = p;
      q.bias = nullptr;
      q.act = ACT_NONE;
      q.out_mode = GEMM_OUT_F32;
      q.C = p.partials;
      q.C_lo = q.C2 = q.C2_lo = nullptr;
      q.ldc = p.N;
      q.split_n = 1 << 30;
      q.resid = nullptr;
      q.fold_c = q.ln_stats = nullptr;  // plain sums of x o gamma
      q.k_splits = splits;
      q.vec = true;
      const bool small = p.small_lds && !p.W8;
      const hipError_t e = small ? (split ? LaunchStep32<true>(q, stream)
                                          : LaunchStep32<false>(q, stream))
                           : split ? LaunchPipe<64, 64, 64, 3, 2, 2, true>(q, stream)
                                   : LaunchPipe<64, 64, 64, 3, 2, 2, false>(q, stream);
      if (e != hipSuccess)
        return e;
      // The partials already carry the fp8 row scale.
      GemmParams r = p;
      r.wscale = nullptr;
      return Reduce(r, p.partials, splits, stream);
    }
  }
  if (p.fold_c)
    return fail("folded LayerNorm: no tile for this shape");
  const int kslice = p.K / p.k_splits;
  const long big_tiles = static_cast<long>((p.M + 255) / 256) * ((p.N + 255) / 256);
  if (f8)
    return big_tiles % 256 == 0 ? LaunchW<256, 256, 64, 2, 4, 2, false, false, true>(p, stream)
                                : LaunchW<128, 128, 64, 2, 2, 4, false, false, true>(p, stream);
  // Q|K|V, out-projection and FFN over the whole K at 4 to 23 positions: the
  // tile by the time model, as for the large shapes.  Measured alone against
  // the 64 x 64 tiles below, split: Q|K|V (N = 3136) at 512 rows 10.9 us on 64
  // x 128 (12.5), 768 17.5 on two-stage 64 x 64 (18.9), 1024 18.8 on 128 x 128
  // (21.8); FFN1 at 768 11.1 on 64 x 128 (12.4); single bf16 Q|K|V at 1024 12.4
  // on 128 x 128 (16.5).  (Beside the chain, from 17 positions, the 128 x 128
  // tiles' 144 KiB keep its workgroups off the CU: batch 20 4 % slower.)
  if (p.M >= kModelRows && p.M < (p.W8 ? kLargeRows : kModelRowsEnd) && p.N >= 128 &&
      p.k_splits == 1 && p.K % 64 == 0 && p.K >= 512 && !p.small_lds && !p.beside_chain) {
    float us;
    return LaunchTile(BestTile(p, p.M, &us), p, stream);
  }
  // 64 x 64 tiles over the whole K otherwise (the smolgen dense2 and other
  // short K, few rows or columns): from 256 rows up, or over K >= 1024, a
  // three-stage ring keeps two K steps in flight (batch 16 forward 2.30 ->
  // 2.05 ms, batch 8 1.75 -> 1.68, batch 256 +0.9 %, batch 3 1.51 -> 1.36;
  // Q|K|V took 16.0 us at 192 rows with two stages, 11.6 us at 256 rows
  // with three); for short K at 128 rows (smolgen dense2 at batch 128,
  // beside the Q|K|V GEMM on the other stream) it was 1.7 % slower, and four
  // stages (one workgroup per CU) were slower at every batch.
  if (p.small_lds && !p.W8)
    return split ? LaunchStep32<true>(p, stream) : LaunchStep32<false>(p, stream);
  if (kslice % 64 == 0) {
    if (p.M >= 256 || kslice >= 1024)
      return split ? LaunchPipe<64, 64, 64, 3, 2, 2, true>(p, stream)
                   : LaunchPipe<64, 64, 64, 3, 2, 2, false>(p, stream);
    return split ? LaunchPipe<64, 64, 64, 2, 2, 2, true>(p, stream)
                 : LaunchPipe<64, 64, 64, 2, 2, 2, false>(p, stream);
  }
  return split ? LaunchStep32<true>(p, stream) : LaunchStep32<false>(p, stream);
}

}  // namespace mfh
