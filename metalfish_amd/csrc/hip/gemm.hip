// Tile choice and launch of the MFMA GEMM (gemm_kernel.h), and the split-K
// reduce kernel.
#include "gemm_kernel.h"
#include "gemm_tiles.h"

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

template <int BM, int BN, int BK, int ST, int WM, int WN, bool SPLIT>
hipError_t Launch(const GemmParams &p, hipStream_t stream) {
  // fp8 weights: the ring's stages when their rows go through LDS, else two
  // (fragments from global memory).
  if (p.W8)
    return LaunchW<BM, BN, BK, W8InLds<BM, BN, BK, WM, WN, SPLIT>() ? ST : 2, WM, WN, SPLIT,
                   true>(p, stream);
  return LaunchW<BM, BN, BK, ST, WM, WN, SPLIT, false>(p, stream);
}

bool Aligned(const void *ptr, std::uintptr_t bytes) {
  return (reinterpret_cast<std::uintptr_t>(ptr) & (bytes - 1)) == 0;
}

}  // namespace

// Rows from which the tile rules for large problems apply (below them,
// 64 x 64 tiles over the whole K or split-K).  From 1536 rows (24
// positions) Q|K|V takes 256 x 128 split tiles instead of 1176-1519
// whole-K 64 x 64 ones: forward at batch 24 2.47 -> 2.41 ms, 28 2.60 ->
// 2.50, 31 2.84 -> 2.56; from 1024 rows it was slower (batch 16 2.07 ->
// 2.34).
constexpr int kLargeRows = 1536;

// 256 x 256 tiles where they fill whole rounds of 256 workgroups (bf16
// activations, one K slice, from the large-problem rows).
bool GemmWholeRoundTiles(const GemmParams &p) {
  const long big_tiles = static_cast<long>((p.M + 255) / 256) * ((p.N + 255) / 256);
  return p.M >= kLargeRows && p.N >= 128 && p.k_splits == 1 && big_tiles % 256 == 0 && !p.A8;
}

namespace {

// The instances that compile a folded LayerNorm's epilogue, and the one a
// GEMM with a folded LayerNorm runs on (the tiles the same shapes take
// without it, where those are among them): split precision (bf16 hi + lo
// activations, or the BF16X2_FP8LO codes), bf16 weights, one K slice.
enum class LnTile { kNone, kLo8, k256, k256Beside, k256x128, k64, k64x64, kSplitK };

LnTile LnFoldTile(const GemmParams &p) {
  const bool res = p.out_mode == GEMM_OUT_RESID_F32;
  if ((!p.A_lo && !p.A_lo8) || p.W8 || p.A8 || p.k_splits != 1 || p.K % 64)
    return LnTile::kNone;
  if (!res && p.out_mode != GEMM_OUT_BF16)
    return LnTile::kNone;
  // Whole rounds of 256-wide whole tiles.
  if (p.A_lo8)
    return p.N % 256 == 0 ? LnTile::kLo8 : LnTile::kNone;
  if (p.N % 256 == 0 && GemmWholeRoundTiles(p))
    return p.beside_chain && !res ? LnTile::k256Beside : LnTile::k256;
  // Fewer 128 x 128 tiles than CUs (24-62 positions at the BT4 widths): the
  // 64 x 64 tiles over the whole K that these shapes take without the fold.
  // Consumers up to 2048 wide also up to two rounds of them (FFN1 at 43-62
  // positions, 128 x 128 tiles without the fold; on 256 x 128 ones with it
  // the forward was 3.4 % slower at batch 48, 0.5 % at 56).
  const long tiles128 = static_cast<long>((p.M + 127) / 128) * ((p.N + 127) / 128);
  if (p.M >= kLargeRows && p.N >= 128 && p.N % 64 == 0 &&
      (tiles128 < 256 || (!res && p.N <= 2048 && tiles128 < 512)))
    return LnTile::k64x64;
  if (res)
    return LnTile::kNone;
  // Consumers: the small-LDS 64 x 64 tiles beside Q|K|V (any width); narrow
  // ones (the smolgen compression at 24-62 positions) split over K where
  // the launcher splits them (the split GEMM sums x o gamma and the reduce
  // kernel applies the LayerNorm before the bias), else on those 64 x 64
  // tiles; else 256 x 128 pipelined tiles.
  if (p.small_lds)
    return LnTile::k64;
  if (p.N < 128)
    return GemmAutoSplits(p) > 1 ? LnTile::kSplitK : LnTile::k64;
  return p.N % 128 == 0 ? LnTile::k256x128 : LnTile::kNone;
}

}  // namespace

bool GemmLnFoldOk(const GemmParams &p) { return LnFoldTile(p) != LnTile::kNone; }

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
  if (p.fold_c && (!p.ln_stats || p.out_mode == GEMM_OUT_RESID_F32 || p.ln_width != p.K ||
                   (p.ln_part != 64 && p.ln_part != 128) || p.K % (2 * p.ln_part) ||
                   p.K > 128 * p.ln_part ||
                   !Aligned(p.fold_c, 16) ||
                   !Aligned(p.ln_stats, 16) || p.k_splits != 1))
    return fail("folded LayerNorm consumer: ln_stats, fold_c (16-byte aligned), ln_part 64 or "
                "128, K = ln_width a multiple of 2 ln_part up to 128 ln_part, one K slice, not "
                "the residual mode");
  if ((p.out_gamma || p.res_stats) && !ln_res)
    return fail("folded LayerNorm output / residual: residual mode only");
  if (ln_res && (!p.resid16 || p.k_splits != 1 || p.ln_width != p.N ||
                 (p.ln_part != 64 && p.ln_part != 128) || p.N % (2 * p.ln_part) ||
                 p.N > 128 * p.ln_part ||
                 (p.res_stats && (!p.res_gamma || !p.res_beta || !Aligned(p.res_stats, 16) ||
                                  !Aligned(p.res_gamma, 16) || !Aligned(p.res_beta, 16))) ||
                 (p.out_gamma && (!p.out_stats || !Aligned(p.out_gamma, 16) ||
                                  !Aligned(p.out_stats, 8) || !p.C_lo))))
    return fail("folded LayerNorm residual: split residual, one K slice, ln_part 64 or 128, "
                "N = ln_width a multiple of 2 ln_part up to 128 ln_part, gamma / beta / stats "
                "16-byte aligned, a bf16 lo output plane with out_gamma");
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
  // fp8 lo correction: 256 x 256 tiles of eight waves, the hi pass on the
  // four-stage single-bf16 pipelined ring (128 KiB), then the lo pass on two
  // 64 KiB stages of code rows.
  // A folded LayerNorm: only the instances that compile its epilogue.
  if (p.fold_c || ln_res) {
    switch (LnFoldTile(p)) {
    case LnTile::kLo8:
      return LaunchW<256, 256, 32, 4, 4, 2, false, false, false, true, true>(p, stream);
    case LnTile::k256Beside:
      return LaunchW<256, 256, 32, 2, 4, 2, true, false, false, true>(p, stream);
    case LnTile::k256:
      return LaunchW<256, 256, 32, 3, 4, 2, true, false, false, true>(p, stream);
    case LnTile::k256x128:
      return LaunchW<256, 128, 32, 2, 4, 2, true, false, false, true>(p, stream);
    case LnTile::k64:
      return LaunchW<64, 64, 32, 2, 2, 2, true, false>(p, stream);
    case LnTile::k64x64:
      return LaunchW<64, 64, 64, 2, 2, 2, true, false>(p, stream);
    case LnTile::kSplitK:
      if (!Aligned(p.partials, 16) || !p.vec || p.N % 4)
        return fail("folded LayerNorm split over K: 16-byte aligned partials, vector stores");
      break;  // the split-K launch below, its reduce applying the LayerNorm
    default:
      return fail("folded LayerNorm: split-precision activations, bf16 weights, one K slice, "
                  "K % 64 == 0 and N a multiple of 256 (residual, BF16X2_FP8LO codes) or "
                  "128 (or small-LDS tiles)");
    }
  }
  if (lo8)
    return LaunchW<256, 256, 32, 4, 4, 2, false, false, false, true, true>(p, stream);
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
      const hipError_t e = small ? (split ? Launch<64, 64, 32, 2, 2, 2, true>(q, stream)
                                          : Launch<64, 64, 32, 2, 2, 2, false>(q, stream))
                           : split ? Launch<64, 64, 64, 3, 2, 2, true>(q, stream)
                                   : Launch<64, 64, 64, 3, 2, 2, false>(q, stream);
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
  // Tile choice measured on MI355X at the BT4 body shapes (M = 16384): for
  // K <= 1024, eight waves per workgroup on BK = 32 steps (split precision
  // 128 x 128 tiles as 2 x 4 waves with two 48 KiB stages, bf16 256 x 128
  // tiles as 4 x 2 waves with three 24 KiB stages); for longer K, four waves
  // on BK = 64 (split 64 x 128, bf16 128 x 128).
  // Whole rounds of 256 workgroups: 256 x 256 tiles of eight waves (4 x 2,
  // 64 x 128 per wave) and a three-stage (split) or four-stage (bf16) LDS
  // ring, 144 / 128 KiB, one workgroup per CU.  They halve the L2 traffic
  // per MFMA of the 128-wide tiles; measured faster in the forward on the
  // out-projection, FFN2 and smolgen-global shapes, slower on QKV (832 tiles,
  // a partial last round) and FFN1 (384).  bf16 weights only (the fp8 path
  // keeps two stages).
  const long big_tiles = static_cast<long>((p.M + 255) / 256) * ((p.N + 255) / 256);
  if (f8)
    return big_tiles % 256 == 0 ? LaunchW<256, 256, 64, 2, 4, 2, false, false, true>(p, stream)
                                : LaunchW<128, 128, 64, 2, 2, 4, false, false, true>(p, stream);
  if (GemmWholeRoundTiles(p)) {
    // fp8 weights too: their e4m3 rows share the ring (40 / 24 KiB stages).
    if (p.W8)
      return split ? LaunchW<256, 256, 32, 3, 4, 2, true, true>(p, stream)
                   : LaunchW<256, 256, 32, 4, 4, 2, false, true>(p, stream);
    // Beside the smolgen chain (Q|K|V at large batches): two stages, so
    // the chain's small-LDS tiles run on the same CUs instead of waiting for
    // a round of these tiles to end (batch 256 forward 23.01k -> 23.55k
    // positions/s with the chain on small-LDS tiles; two stages alone
    // 23.15k, batch 1024 unchanged).
    // bf16 weights: the software-pipelined main loop (PipelinedLoop).
    // Isolated at batch 256, split precision: Q|K|V 223 -> 209 us, the
    // out-projection 76.7 -> 70.7, FFN2 103.8 -> 93.6; single bf16 Q|K|V
    // 112 -> 104; the batch-256 forward 23.15k -> 23.64k positions/s
    // (bit-equal outputs: the MFMAs accumulate in the same order).
    if (p.beside_chain && split)
      return LaunchW<256, 256, 32, 2, 4, 2, true, false, false, true>(p, stream);
    return split ? LaunchW<256, 256, 32, 3, 4, 2, true, false, false, true>(p, stream)
                 : LaunchW<256, 256, 32, 4, 4, 2, false, false, false, true>(p, stream);
  }
  // Split precision with fewer 128 x 128 tiles than CUs (the out-projection
  // and FFN at M = 2048 .. 3072): 64 x 64 tiles, four times the workgroups
  // (out-projection at M = 2048: 13.5 instead of 25.4 us; batch 32 forward
  // 3.02 -> 2.78 ms).  64 x 128 tiles between one and three rounds were
  // faster in isolated launches but 2 % slower in the forward at batches 64
  // and 96, so those keep 128 x 128.
  const long tiles128 = static_cast<long>((p.M + 127) / 128) * ((p.N + 127) / 128);
  if (large && kslice % 64 == 0) {
    if (split && tiles128 < 256)
      return Launch<64, 64, 64, 2, 2, 2, true>(p, stream);
    if (kslice <= 1024 && split && !p.W8) {
      // 256 x 128 tiles (eight 64 x 64 waves, two 40 KiB stages, two
      // workgroups per CU) read 12 LDS fragments per 32 MFMAs, 128 x 128
      // tiles 10 per 16; a 256 x 128 tile costs ~1.8 times a 128 x 128
      // one, so it is taken when its rounds of 256 workgroups cost less and
      // it fills at least one round.  Below one round (FFN1 at batches 48
      // and 64, the out-projection at 96) it was 1-5 % slower, except for
      // Q|K|V at 2048 rows (batch 32), where its 192 tiles leave CUs to the
      // smolgen chain running beside it, the longer branch there.
      // Measured forward: batch 32 2.72 -> 2.61 ms, 96 5.32 -> 5.26, 128
      // 6.72 -> 6.66, 256 11.30 -> 11.16; 48 and 64 unchanged.
      const long t256 = static_cast<long>((p.M + 255) / 256) * ((p.N + 127) / 128);
      if ((t256 >= 256 || p.M <= 2048) &&
          9 * ((t256 + 255) / 256) < 5 * ((tiles128 + 255) / 256))
        return LaunchW<256, 128, 32, 2, 4, 2, true, false, false, true>(p, stream);
    }
    // Split precision with fp8 weights: BK = 64, whose stage holds the
    // e4m3 rows in LDS (at BK = 32 the 128 x 128 stage does not split
    // evenly over the waves).
    if (kslice <= 1024)
      return split ? (p.W8 ? LaunchW<128, 128, 64, 2, 2, 4, true, true>(p, stream)
                           : LaunchW<128, 128, 32, 2, 2, 4, true, false>(p, stream))
             : p.W8 ? LaunchW<256, 128, 32, 2, 4, 2, false, true>(p, stream)
                    : LaunchW<256, 128, 32, 3, 4, 2, false, false, false, true>(p, stream);
    return split ? Launch<64, 128, 64, 2, 2, 2, true>(p, stream)
                 : Launch<128, 128, 64, 2, 2, 2, false>(p, stream);
  }
  // 64 x 64 tiles over the whole K (Q|K|V at 4-31 positions, the
  // out-projection and FFN at 16-31, the smolgen dense2 and global
  // projection at some batches): from 256 rows up, or over K >= 1024, a
  // three-stage ring keeps two K steps in flight (batch 16 forward 2.30 ->
  // 2.05 ms, batch 8 1.75 -> 1.68, batch 256 +0.9 %, batch 3 1.51 -> 1.36;
  // Q|K|V took 16.0 us at 192 rows with two stages, 11.6 us at 256 rows
  // with three); for short K at 128 rows (smolgen dense2 at batch 128,
  // beside the Q|K|V GEMM on the other stream) it was 1.7 % slower, and four
  // stages (one workgroup per CU) were slower at every batch.
  if (p.small_lds && !p.W8)
    return split ? Launch<64, 64, 32, 2, 2, 2, true>(p, stream)
                 : Launch<64, 64, 32, 2, 2, 2, false>(p, stream);
  if (kslice % 64 == 0) {
    if (p.M >= 256 || kslice >= 1024)
      return split ? Launch<64, 64, 64, 3, 2, 2, true>(p, stream)
                   : Launch<64, 64, 64, 3, 2, 2, false>(p, stream);
    return split ? Launch<64, 64, 64, 2, 2, 2, true>(p, stream)
                 : Launch<64, 64, 64, 2, 2, 2, false>(p, stream);
  }
  return split ? Launch<64, 64, 32, 2, 2, 2, true>(p, stream)
               : Launch<64, 64, 32, 2, 2, 2, false>(p, stream);
}

}  // namespace mfh
