// The end of the smolgen chain in one launch (reference src/nn/cpu/
// cpu_network.cpp:1136-1173): the LayerNorm over a position's heads x gen
// row, then the shared global projection of each head's segment into the
// attention bias, bias[b][h][:] = LN(x_b)[h] . Wg^T.
//
// A workgroup of four waves takes the whole positions of up to 32 (position,
// head) rows.  It takes their statistics from the rows that it reads anyway,
// normalises them into LDS as bf16 (hi + lo), and each wave then holds their
// fragments in registers for the launch: K is only the gen width, so 32 rows
// over all of it are 128 registers in split precision.  The weights stream
// past them, 128 output columns at a time, through an LDS ring of 64-wide K
// stages that grows into the rows' space once they are read; a wave reads
// only weight fragments in the loop.  Each wave owns 32 of the columns, its
// weight rows permuted so that a lane ends up with eight consecutive outputs
// of a row: they go out in 16-byte stores straight from the accumulators, 128
// consecutive bytes a row in fp32, with no staging or barrier between a
// tile's stores and the next tile's MFMAs.
//
// 80 KiB of LDS and four waves, so that a workgroup fits beside one of
// Q|K|V's (64 KiB, four waves): eight waves with 64 rows, 112 to 144 KiB, had
// to wait for Q|K|V to end (batch 45, beside it: 35.7 us against 18.6).
//
// What bounds it: the launch and its chain of loads (rows, statistics,
// weights) at a few positions, then L2 reads of the weights, which every row
// group streams whole.  Measured (BT4 shape, split precision) against the
// LayerNorm and GEMM launches: 8.1 us instead of 5.1 + 4.4 and a launch at
// batch 8, 18.6 instead of 12.8 + 15.9 at 45; forward 1162 -> 1125 us at batch
// 1, 1175 -> 1141 at 2, 1373 -> 1350 at 8, 2489 -> 2443 at 36, 2697 -> 2677 at 45.  From 48
// positions on Q|K|V, on the other stream, outlasts the LayerNorm, and the
// wider tiles of the GEMM read the weights less often: 48 was 1.2 % slower on
// this kernel, 64 5 %, 256 4 %, so those keep the two launches.
#include "mfh_device.h"
#include "mfh_kernels.h"

#include <mutex>

namespace mfh {
namespace {

constexpr int kWaves = 4;
constexpr int kRows = 32;   // (position, head) rows per workgroup
constexpr int kCols = 128;  // output columns per tile
constexpr int kMaxN = 4096; // the bias of 64 x 64 squares (its row scales stay in LDS)
constexpr int kFirst = 3;   // ring stages beside the rows

// 16-byte chunk of a 128-byte LDS row (the swizzle of the GEMM tiles).
__device__ __forceinline__ int RowChunk(int row, int chunk) {
  return chunk ^ (row & 7) ^ (((row >> 3) & 1) * 5);
}

// The same for the weights, whose rows are read in the order of MFMA rows
// f = 4 (row / 8) + row % 4: lanes of a fragment meet the slots that they
// would meet over consecutive rows.
__device__ __forceinline__ int WeightRow(int row) { return ((row >> 3) & 3) * 4 + (row & 3); }

#if defined(__HIP_DEVICE_COMPILE__)
template <int N> __device__ __forceinline__ void WaitLoads() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// Waits until at most `stages` stages of LPW loads of this wave are
// outstanding (a wave-uniform count of at most MAX).
template <int LPW, int MAX> __device__ __forceinline__ void WaitStages(int stages) {
  if constexpr (MAX == 0) {
    WaitLoads<0>();
  } else {
    if (stages >= MAX)
      WaitLoads<MAX * LPW>();
    else
      WaitStages<LPW, MAX - 1>(stages);
  }
}
#endif

constexpr int StageBytes(bool w8) { return kCols * 64 * (w8 ? 1 : 2); }
constexpr int RowBytes(int kb, bool split) { return kb * (split ? 2 : 1) * kRows * 128; }
constexpr int Stages(int kb, bool split, bool w8) {
  const int more = RowBytes(kb, split) / StageBytes(w8);
  return kFirst + (more < 3 ? more : 3);
}

// KB: gen width / 64.  SPLIT: bf16 hi + lo rows and fp32 output, else bf16.
template <int KB, bool SPLIT, bool W8>
__global__ __launch_bounds__(kWaves * 64, 2) void SmolgenBiasKernel(SmolgenBiasParams p) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int P = SPLIT ? 2 : 1;
  constexpr int G = KB * 64;
  constexpr int T = kWaves * 64;
  constexpr int kWBytes = StageBytes(W8);
  constexpr int ST = Stages(KB, SPLIT, W8);
  constexpr int LPW = kWBytes / 1024 / kWaves;  // wave-loads per wave and stage
  // LDS: kFirst ring stages, then the rows; once every wave holds its
  // fragments of them, the rows' space is more ring.
  extern __shared__ __attribute__((aligned(1024))) std::uint16_t lds[];
  std::uint16_t *arows = lds + kFirst * (kWBytes / 2);
  float *scale = reinterpret_cast<float *>(arows + RowBytes(KB, SPLIT) / 2);  // W8

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fr = lane & 15, fc = lane >> 4;
  const int HG = p.heads * G;
  const int pos0 = blockIdx.x * p.positions;          // first position
  const int npos = min(p.positions, p.batch - pos0);  // of this workgroup
  const int tile0 = blockIdx.y * p.tiles;             // first column tile
  const int ntiles = min(p.tiles, p.N / kCols - tile0);
  const int total = ntiles * KB;  // stages

  // Weight loads: wave-load j of a stage covers eight 128-byte rows (16 of 64
  // bytes with W8) of the tile, lane l fetching the chunk its slot holds.
  const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<void *>(W8 ? static_cast<const void *>(p.W8) : static_cast<const void *>(p.W)),
      0, 0x7FFFFFFF, 0x00020000);
  unsigned goff[LPW];
#pragma unroll
  for (int j = 0; j < LPW; ++j) {
    const int load = wave * LPW + j;
    if constexpr (W8) {
      const int row = load * 16 + lane / 4;
      goff[j] = static_cast<unsigned>(row) * G + ((lane % 4) ^ ((WeightRow(row) >> 1) & 3)) * 16;
    } else {
      const int row = load * 8 + lane / 8;
      goff[j] = (static_cast<unsigned>(row) * G + RowChunk(WeightRow(row), lane % 8) * 8) * 2;
    }
  }
  auto fill = [&](int slot, int s) {
    const int n0 = (tile0 + s / KB) * kCols, k0 = (s % KB) * 64;
    std::uint16_t *d = lds + slot * (kWBytes / 2) + wave * LPW * 512;
#pragma unroll
    for (int j = 0; j < LPW; ++j)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, MFH_LDS_PTR(d + j * 512), 16, goff[j],
                                               (n0 * G + k0) * (W8 ? 1 : 2), 0, 0);
  };

  // The rows, four consecutive elements per thread and step: a wave's load is
  // 256 consecutive elements of one position.  Everything the prologue reads
  // is asked for at once, the first stages' weights last; past the last
  // position the loads repeat the first elements.
  constexpr int STEPS = kRows * G / (4 * T);
  const int chunks = HG / 256;  // wave loads per position
  const float *x = p.x + static_cast<size_t>(pos0) * HG;
  f32x4 v[STEPS], gm[STEPS], bt[STEPS];
  int pos[STEPS];  // position of the step's elements (wave-uniform)
#pragma unroll
  for (int i = 0; i < STEPS; ++i) {
    const int chunk = i * kWaves + wave;
    pos[i] = chunk * p.chunk_inv >> 16;  // chunk / chunks
    const bool in = pos[i] < npos;
    v[i] = *reinterpret_cast<const f32x4 *>(x + (in ? chunk * 256 : 0) + lane * 4);
    const int c = (in ? chunk - pos[i] * chunks : 0) * 256 + lane * 4;
    gm[i] = *reinterpret_cast<const f32x4 *>(p.gamma + c);
    bt[i] = *reinterpret_cast<const f32x4 *>(p.beta + c);
  }
  f32x4 ws[W8 ? kMaxN / 4 / T : 1];
  if constexpr (W8) {
#pragma unroll
    for (int i = 0; i < kMaxN / 4 / T; ++i) {
      const int c = (i * T + tid) * 4;
      ws[i] = *reinterpret_cast<const f32x4 *>(p.wscale + tile0 * kCols +
                                               (c < ntiles * kCols ? c : 0));
    }
  }
#pragma unroll
  for (int s = 0; s < kFirst; ++s)
    fill(s, min(s, total - 1));
  __builtin_amdgcn_sched_barrier(0);  // no arithmetic between the loads
  float sum[STEPS], sq[STEPS];
#pragma unroll
  for (int i = 0; i < STEPS; ++i) {
    sum[i] = v[i][0] + v[i][1] + v[i][2] + v[i][3];
    sq[i] = v[i][0] * v[i][0] + v[i][1] * v[i][1] + v[i][2] * v[i][2] + v[i][3] * v[i][3];
  }
  f32x2 *part = reinterpret_cast<f32x2 *>(arows);  // [position][wave]
  for (int q = 0; q < npos; ++q) {
    float s = 0.f, ss = 0.f;
#pragma unroll
    for (int i = 0; i < STEPS; ++i) {
      s += pos[i] == q ? sum[i] : 0.f;
      ss += pos[i] == q ? sq[i] : 0.f;
    }
    s = wave_sum(s);
    ss = wave_sum(ss);
    if (lane == 0)
      part[q * kWaves + wave] = f32x2{s, ss};
  }
  if constexpr (W8) {
#pragma unroll
    for (int i = 0; i < kMaxN / 4 / T; ++i) {
      const int c = (i * T + tid) * 4;
      if (c < ntiles * kCols)
        *reinterpret_cast<f32x4 *>(scale + c) = ws[i];
    }
  }
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  // Mean and 1 / sqrt(variance + eps) of each position, in every wave.
  float mu[STEPS], rs[STEPS];
#pragma unroll
  for (int i = 0; i < STEPS; ++i)
    mu[i] = rs[i] = 0.f;
  for (int q = 0; q < npos; ++q) {
    float s = 0.f, ss = 0.f;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      s += part[q * kWaves + w][0];
      ss += part[q * kWaves + w][1];
    }
    s /= static_cast<float>(HG);
    float var = ss / static_cast<float>(HG) - s * s;
    var = var < 0.f ? 0.f : var;
    const float inv = 1.f / sqrtf(var + p.eps);
#pragma unroll
    for (int i = 0; i < STEPS; ++i)
      if (pos[i] == q) {
        mu[i] = s;
        rs[i] = inv;
      }
  }
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
  for (int i = 0; i < STEPS; ++i) {
    const int e = ((i * kWaves + wave) * 64 + lane) * 4;
    const int row = e / G, k = e % G;
    f32x4 y;
#pragma unroll
    for (int r = 0; r < 4; ++r)
      y[r] = pos[i] < npos ? (v[i][r] - mu[i]) * rs[i] * gm[i][r] + bt[i][r] : 0.f;
    std::uint32_t h0, h1, l0 = 0, l1 = 0;
    if constexpr (SPLIT) {
      split_bf16x2(y[0], y[1], h0, l0);
      split_bf16x2(y[2], y[3], h1, l1);
    } else {
      h0 = pack_bf16x2(y[0], y[1]);
      h1 = pack_bf16x2(y[2], y[3]);
    }
    std::uint16_t *d =
        arows + ((k / 64) * P * kRows + row) * 64 + RowChunk(row, (k % 64) / 8) * 8 + (k & 4);
    *reinterpret_cast<u32x2 *>(d) = u32x2{h0, h1};
    if constexpr (SPLIT)
      *reinterpret_cast<u32x2 *>(d + kRows * 64) = u32x2{l0, l1};
  }
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  // This wave's rows for the whole launch.
  bf16x8 a[2 * KB][P][2];
#pragma unroll
  for (int kk = 0; kk < 2 * KB; ++kk)
#pragma unroll
    for (int q = 0; q < P; ++q)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int row = i * 16 + fr;
        a[kk][q][i] = *reinterpret_cast<const bf16x8 *>(
            arows + (((kk / 2) * P + q) * kRows + row) * 64 + RowChunk(row, (kk & 1) * 4 + fc) * 8);
      }

  // Weight fragments of a stage: MFMA row f of fragment j is column 8 (f / 4)
  // + f % 4 + 4 j of the wave's 32, so that a lane's eight outputs (4 fc ..
  // + 3 of both fragments) are columns 8 fc .. + 7.
  using WRaw = std::conditional_t<W8, u32x2, bf16x8>;
  struct Frags {
    WRaw w[2][2];  // [substep][fragment]
  };
  auto read = [&](Frags &f, int slot) {
    const std::uint16_t *base = lds + slot * (kWBytes / 2);
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int row = wave * 32 + 8 * (fr >> 2) + (fr & 3) + 4 * j;
        const std::uint16_t *src =
            W8 ? base + row * 32 + ((2 * kk + (fc >> 1)) ^ ((fr >> 1) & 3)) * 8 + (fc & 1) * 4
               : base + row * 64 + RowChunk(fr, kk * 4 + fc) * 8;
        f.w[kk][j] = *reinterpret_cast<const WRaw *>(src);
      }
  };
  auto conv = [](const WRaw &w) -> bf16x8 {
    if constexpr (W8)
      return Fp8x8ToBf16(w);
    else
      return w;
  };

  // Output rows of this lane.
  const int rows = npos * p.heads;
  const size_t row_base = static_cast<size_t>(pos0) * p.heads;

  // The rows are in registers and stage 0 has landed, for every wave.
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  WaitStages<LPW, kFirst - 1>(min(kFirst, total) - 1);
  asm volatile("s_barrier" ::: "memory");
#pragma unroll
  for (int s = kFirst; s < ST; ++s)
    if (s < total)
      fill(s, s);
  Frags cur, nxt;
  read(cur, 0);
  int slot = 0;  // of stage s
  f32x4 acc[2][2];
  int s = 0;
  for (int t = 0; t < ntiles; ++t) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kb = 0; kb < KB; ++kb, ++s) {
      // Stage s + 1 visible to every wave, and stage s read by all of them
      // (its fragments are in registers), so its slot takes stage s + ST.
      // Loads younger than stage s + 1's: those of the stages up to s + ST -
      // 1 that exist.  (Stores in between only make the wait stricter.)
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      WaitStages<LPW, ST - 2>(min(s + ST, total) - (s + 2));
      asm volatile("s_barrier" ::: "memory");
      if (s + ST < total)
        fill(slot, s + ST);
      slot = slot + 1 == ST ? 0 : slot + 1;
      if (s + 1 < total)
        read(nxt, slot);
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        const bf16x8 w0 = conv(cur.w[kk][0]), w1 = conv(cur.w[kk][1]);
#pragma unroll
        for (int q = 0; q < P; ++q)
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            const bf16x8 &ai = a[2 * kb + kk][q][i];
            acc[i][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w0, ai, acc[i][0], 0, 0, 0);
            acc[i][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w1, ai, acc[i][1], 0, 0, 0);
          }
      }
      cur = nxt;
    }
    const int col = (tile0 + t) * kCols + wave * 32 + 8 * fc;
    float sc[8];
    if constexpr (W8) {
      const float *src = scale + col - tile0 * kCols;
      const f32x4 s0 = *reinterpret_cast<const f32x4 *>(src);
      const f32x4 s1 = *reinterpret_cast<const f32x4 *>(src + 4);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        sc[r] = s0[r];
        sc[4 + r] = s1[r];
      }
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int row = i * 16 + fr;
      if (row >= rows)
        continue;
      const size_t off = (row_base + row) * p.N + col;
      float o[8];
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        o[r] = acc[i][r >> 2][r & 3];
        if constexpr (W8)
          o[r] *= sc[r];
      }
      if constexpr (SPLIT) {
        float *d = static_cast<float *>(p.out) + off;
        *reinterpret_cast<f32x4 *>(d) = f32x4{o[0], o[1], o[2], o[3]};
        *reinterpret_cast<f32x4 *>(d + 4) = f32x4{o[4], o[5], o[6], o[7]};
      } else {
        u32x4 h;
#pragma unroll
        for (int r = 0; r < 4; ++r)
          h[r] = pack_bf16x2(o[2 * r], o[2 * r + 1]);
        *reinterpret_cast<u32x4 *>(static_cast<std::uint16_t *>(p.out) + off) = h;
      }
    }
  }
#endif
}

template <int KB, bool SPLIT, bool W8>
hipError_t Launch(const SmolgenBiasParams &p, dim3 grid, hipStream_t stream) {
  constexpr int lds = kFirst * StageBytes(W8) + RowBytes(KB, SPLIT) + (W8 ? kMaxN * 4 : 0);
  auto kernel = SmolgenBiasKernel<KB, SPLIT, W8>;
  static std::once_flag once;
  static hipError_t attr = hipSuccess;
  std::call_once(once, [&]() {
    attr = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                               hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  });
  if (attr != hipSuccess)
    return attr;
  hipLaunchKernelGGL(kernel, grid, dim3(kWaves * 64), lds, stream, p);
  return hipGetLastError();
}

template <int KB, bool SPLIT>
hipError_t LaunchW(const SmolgenBiasParams &p, dim3 grid, hipStream_t stream) {
  return p.W8 ? Launch<KB, SPLIT, true>(p, grid, stream)
              : Launch<KB, SPLIT, false>(p, grid, stream);
}

template <int KB> hipError_t LaunchK(const SmolgenBiasParams &p, dim3 grid, hipStream_t stream) {
  return p.split ? LaunchW<KB, true>(p, grid, stream) : LaunchW<KB, false>(p, grid, stream);
}

bool Aligned16(const void *ptr) { return (reinterpret_cast<std::uintptr_t>(ptr) & 15) == 0; }

}  // namespace

bool SmolgenBiasOk(int heads, int gen, int n) {
  return heads >= 1 && heads <= kRows && (gen == 64 || gen == 128 || gen == 256) &&
         (heads * gen) % 256 == 0 && n > 0 && n <= kMaxN && n % kCols == 0;
}

hipError_t LaunchSmolgenBias(const SmolgenBiasParams &p_in, hipStream_t stream,
                             std::string *err) {
  SmolgenBiasParams p = p_in;
  auto fail = [&](const char *why) {
    if (err)
      *err = std::string("smolgen bias: ") + why;
    return hipErrorInvalidValue;
  };
  if (!SmolgenBiasOk(p.heads, p.gen, p.N) || p.batch < 1)
    return fail("up to 32 heads, gen width 64, 128 or 256, heads x gen a multiple of 256, N a "
                "multiple of 128 up to 4096");
  if (!p.x || !p.gamma || !p.beta || !p.out || (!p.W && !p.W8) || (p.W && p.W8) ||
      (p.W8 && !p.wscale))
    return fail("null operand (or both W and W8)");
  if (!Aligned16(p.x) || !Aligned16(p.gamma) || !Aligned16(p.beta) || !Aligned16(p.out) ||
      !Aligned16(p.W) || !Aligned16(p.W8) || !Aligned16(p.wscale))
    return fail("operands must be 16-byte aligned");
  // Whole positions per workgroup, and column tiles per workgroup such that
  // the rounds of 256 workgroups (one per CU) cost least: a tile takes about
  // 1 us, the rows before the first one about 3.
  p.positions = kRows / p.heads;
  const int chunks = p.heads * p.gen / 256;
  p.chunk_inv = (65536 + chunks - 1) / chunks;  // exact below 64 chunks
  const int mt = (p.batch + p.positions - 1) / p.positions, nt = p.N / kCols;
  int best = 1;
  long best_cost = -1;
  for (int ny = 1; ny <= nt; ++ny) {
    const int tiles = (nt + ny - 1) / ny;
    const int groups = (nt + tiles - 1) / tiles;
    const long cost = (static_cast<long>(mt) * groups + 255) / 256 * (tiles + 3);
    if (best_cost < 0 || cost < best_cost) {
      best_cost = cost;
      best = tiles;
    }
  }
  p.tiles = best;
  const dim3 grid(mt, (nt + best - 1) / best);
  if (p.gen == 64)
    return LaunchK<1>(p, grid, stream);
  if (p.gen == 128)
    return LaunchK<2>(p, grid, stream);
  return LaunchK<4>(p, grid, stream);
}

}  // namespace mfh
