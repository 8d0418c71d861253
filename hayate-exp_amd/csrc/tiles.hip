// Products of a prompt's rows with the model's weights: y = x W^T + residual
// (attention output and MLP down projection) and y = silu(x Wg^T) * (x Wu^T)
// (the MLP's gate and up projections in one product, so neither is written).
// Weights are (n, k) rows as torch stores them, so both operands have k
// contiguous.
//
// A workgroup of 4 waves, one wave per SIMD, owns a BM x BN tile of outputs
// (gated: BN / 2 columns, 16 rows of Wg and of Wu alternating, so a lane ends
// with gate and up of the same element). Steps of 64 k of both operands go
// straight to LDS in a ring of 2-4 stages; v_mfma_f32_32x32x16_bf16 with the weight
// rows as A, because one wave cannot issue the 16x16x32 form fast enough: on
// one wave per SIMD that form stops at 1.5 PFLOP/s even on zeros, the larger one
// reaches 2.4 (1.75 on random values, where the card's power decides).
//
// LDS rows are 128 bytes (64 k), 16-byte chunk c of row r at place c ^ (r % 8):
// a load instruction still brings whole 128-byte runs, and the 8 lanes that one
// LDS cycle serves read 8 different places.
//
// Inside a step the wave multiplies one half (32 k) while it reads the other
// half's fragments, one barrier per step. What bounds it (512 rows, gate and up,
// 256 x 160): the loads alone take 45 us, the arithmetic alone 47, both 51; below
// 200 rows the weights' way from HBM.
//
// Measured on MI355X against the library's products and the elementwise kernels
// after them (us, HIP graph, weights from HBM):
//                               64 rows    128        512        2064       8192
//   2560 -> 2 x 9728, gated     45 / 29    54 / 34    89 / 53    231 / 233  934 / 750
//   4096 -> 2560, residual      15 / 14    22 / 14    27 / 24    57 / 54    165 / 166
//   9728 -> 2560, residual      30 / 18    53 / 22    56 / 42    120 / 111  344 / 350
//   1024 -> 2 x 3072, gated     23 / 10    24 / 10    28 / 12    54 / 39    156 / 122
// A plain product without either gains nothing here and stays with the library; so
// do large products with a residual (hayate_amd/linear.py has the line and why).
#include <type_traits>

#include "hy_common.h"
#include "tile_plan.h"

namespace hy {
namespace {

constexpr int kTileThreads = 256;
constexpr int kTileWaves = 4;
constexpr int kLdsBytes = 160 * 1024;

struct TileArgs {
  const uint16_t *x;
  int64_t x_stride;
  int m, n, k;
  const uint16_t *w, *up;
  int64_t w_stride;
  const uint16_t *residual;
  int64_t r_stride;
  uint16_t *y;
  int64_t y_stride;
  float *partials;  // splits > 1: [split][column tile][row tile][accumulators]
  int row_tiles, col_tiles, splits;
  int row_group;  // row tiles that share a pass over the weights
};

// WN of the 4 waves lie along the columns; a wave's fragments are 32 x 32.
template <int BM_, int BN_, int WN_>
struct Tile {
  static constexpr int BM = BM_, BN = BN_, WN = WN_, WM = kTileWaves / WN_;
  static constexpr int FM = BM / 32 / WM, FN = BN / 32 / WN;
  static constexpr int kStage = (BM + BN) * kStepK;  // elements
  static constexpr int kFit = kLdsBytes / (2 * kStage);
  static constexpr int kStages = kFit < 4 ? kFit : 4;
  static constexpr int kLoads = (BM + BN) / 8 / kTileWaves;  // of one wave, per stage
  static_assert(FM * WM * 32 == BM && FN * WN * 32 == BN && kStages >= 2, "tile");
};

// 16 bytes per lane from a buffer straight into LDS at m0 + 16 lane. The wait
// state after writing M0 is the one the ISA asks for. In inline assembly, so the
// compiler neither waits for these loads nor orders LDS reads behind them:
// wait_barrier does both.
__device__ __forceinline__ void buffer_to_lds(uint32_t off, u32x4 rsrc, uint32_t soff,
                                              uint32_t m0) {
  __asm__ volatile("s_mov_b32 m0, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds"
                   :
                   : "v"(off), "s"(rsrc), "s"(soff), "s"(m0)
                   : "memory");
}

__device__ __forceinline__ u32x4 buffer_of(const void *p) {
  const uint64_t a = reinterpret_cast<uintptr_t>(p);
  return u32x4{static_cast<uint32_t>(a), static_cast<uint32_t>(a >> 32) & 0xffffu, 0xffffffffu,
               0x00020000u};
}

// All but the last `Newer` of this wave's loads have landed and its LDS reads are
// done, and so have every other wave's.
template <int Newer>
__device__ __forceinline__ void wait_barrier() {
  __asm__ volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(Newer) : "memory");
  __builtin_amdgcn_sched_barrier(0);
}

__device__ __forceinline__ float silu(float g) { return g / (1.0f + __expf(-g)); }

// Lane (r = l % 32, q = l / 32) of a 32 x 32 fragment holds row r, accumulator
// 4 g + e column 8 g + 4 q + e. Stores columns of g and g + 2 (lo and hi; gated:
// gate and up of column g of 32 x 16) of the fragment at row0, col0.
template <bool kGated>
__device__ __forceinline__ void store_pair(const TileArgs &a, f32x4 lo, f32x4 hi, int g, int row0,
                                           int col0, int lane) {
  const int row = row0 + (lane & 31);
  if (row >= a.m) return;
#pragma unroll
  for (int p = 0; p < (kGated ? 1 : 2); ++p) {
    const int col = col0 + 8 * (g + 2 * p) + 4 * (lane >> 5);
    if (col >= a.n) continue;  // n is a multiple of 4
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = kGated ? silu(lo[e]) * hi[e] : p ? hi[e] : lo[e];
    if (!kGated && a.residual) {
      const uint2 r = *reinterpret_cast<const uint2 *>(a.residual + row * a.r_stride + col);
      v[0] += bf16_lo(r.x);
      v[1] += bf16_hi(r.x);
      v[2] += bf16_lo(r.y);
      v[3] += bf16_hi(r.y);
    }
    *reinterpret_cast<uint2 *>(a.y + row * a.y_stride + col) =
        make_uint2(pack_bf16x2_rne(v[0], v[1]), pack_bf16x2_rne(v[2], v[3]));
  }
}

template <class T, bool kGated>
__global__ __launch_bounds__(kTileThreads, 1) void tile_kernel(const TileArgs a) {
  constexpr int FM = T::FM, FN = T::FN, kStages = T::kStages, kLoads = T::kLoads;
  constexpr int kCols = kGated ? T::BN / 2 : T::BN;
  __shared__ __attribute__((aligned(1024))) uint16_t smem[kStages * T::kStage];
  const int lane = static_cast<int>(threadIdx.x) & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

  // Workgroups go to XCDs in turn: consecutive `wg` share one.
  const int total = gridDim.x, xcd = blockIdx.x & 7;
  const int wg = xcd * (total >> 3) + min(xcd, total & 7) + static_cast<int>(blockIdx.x >> 3);
  const int group_size = a.row_group * a.col_tiles * a.splits;
  const int group = wg / group_size, in_group = wg - group * group_size;
  const int rows = min(a.row_group, a.row_tiles - group * a.row_group);
  const int rt = group * a.row_group + in_group % rows;
  const int sp = in_group / rows % a.splits, ct = in_group / rows / a.splits;
  const int m0 = rt * T::BM, n0 = ct * kCols;
  const int steps = a.k / kStepK;
  const int k0 = static_cast<int>(static_cast<int64_t>(steps) * sp / a.splits);
  const int nk = static_cast<int>(static_cast<int64_t>(steps) * (sp + 1) / a.splits) - k0;

  // Load i of a stage brings LDS rows 8 (wave + 4 i) .. + 7; rows past the operands'
  // last repeat it. The rows of one wave all belong to one of Wg and Wu.
  u32x4 rx = buffer_of(a.x + m0 * a.x_stride);
  u32x4 rw = buffer_of((kGated && (wave & 2) ? a.up : a.w) + n0 * a.w_stride);
  uint32_t off[kLoads];
  const int chunk = (lane & 7) ^ (lane >> 3);
#pragma unroll
  for (int i = 0; i < kLoads; ++i) {
    const int r = 8 * (wave + 4 * i) + (lane >> 3);
    if (32 * (i + 1) <= T::BM) {
      off[i] = static_cast<uint32_t>((min(r, a.m - 1 - m0) * a.x_stride + chunk * 8) * 2);
    } else {
      const int f = r - T::BM;
      const int c = kGated ? (f >> 5) * 16 + (f & 15) : f;
      off[i] = static_cast<uint32_t>((min(c, a.n - 1 - n0) * a.w_stride + chunk * 8) * 2);
    }
  }
  const uint32_t lds0 = static_cast<uint32_t>(
      reinterpret_cast<uintptr_t>((const __attribute__((address_space(3))) uint16_t *)smem));
  uint32_t soff = k0 * kStepK * 2;
  int left = nk;
  auto load = [&](int i, uint32_t dst) {
    buffer_to_lds(off[i], 32 * (i + 1) <= T::BM ? rx : rw, soff, dst + 1024 * (wave + 4 * i));
  };
  // After the last step the buffers have no records: loads bring nothing, and
  // the counts that wait_barrier relies on stay the same.
  auto next_step = [&] {
    soff += kStepK * 2;
    if (--left == 0) rx[2] = rw[2] = 0;
  };

  f32x16 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

  const int wm = wave % T::WM, wn = wave / T::WM;
  const int r32 = lane & 31, q = lane >> 5;
  int place[4];  // element offset of chunk 2 kk + q in this lane's rows
#pragma unroll
  for (int kk = 0; kk < 4; ++kk) place[kk] = ((2 * kk + q) ^ (lane & 7)) * 8;
  const int x_row = (wm * FM * 32 + r32) * kStepK;
  const int w_row = (T::BM + wn * FN * 32 + r32) * kStepK;
  bf16x8 xf[2][2][FM], wf[2][2][FN];  // [half][16 k][fragment]
  constexpr int kFrags = 2 * (FM + FN);
  auto read = [&](int h, int f, const uint16_t *s) {
    const int kk = f / (FM + FN), g = f % (FM + FN);
    s += place[2 * h + kk];
    if (g < FM)
      xf[h][kk][g] = *reinterpret_cast<const bf16x8 *>(s + x_row + g * 32 * kStepK);
    else
      wf[h][kk][g - FM] = *reinterpret_cast<const bf16x8 *>(s + w_row + (g - FM) * 32 * kStepK);
  };
  // Multiplies half H, and in between reads the other half's fragments from s
  // and, with kFill, loads the stage at dst. The scheduling barriers keep that
  // order: left alone, the compiler puts each read right before its use.
  constexpr int kGroups = 2 * FN;
  constexpr int kReadsPer = (kFrags + kGroups - 2) / (kGroups - 1);
  constexpr int kLoadsPer = (kLoads + kGroups - 1) / kGroups;
  auto multiply = [&](auto half, auto read_other, auto fill, const uint16_t *s, uint32_t dst) {
    constexpr int h = decltype(half)::value;
#pragma unroll
    for (int j = 0; j < kGroups; ++j) {
      if constexpr (decltype(read_other)::value) {
#pragma unroll
        for (int f = j * kReadsPer; f < (j + 1) * kReadsPer; ++f)
          if (f < kFrags) read(1 - h, f, s);
      }
      if constexpr (decltype(fill)::value) {
#pragma unroll
        for (int i = j * kLoadsPer; i < (j + 1) * kLoadsPer; ++i)
          if (i < kLoads) load(i, dst);
      }
#pragma unroll
      for (int i = 0; i < FM; ++i)
        acc[i][j % FN] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
            wf[h][j / FN][j % FN], xf[h][j / FN][i], acc[i][j % FN], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  constexpr std::integral_constant<int, 0> first{};
  constexpr std::integral_constant<int, 1> second{};
  constexpr std::true_type yes{};
  constexpr std::false_type no{};

#pragma unroll
  for (int s = 0; s < kStages; ++s) {
#pragma unroll
    for (int i = 0; i < kLoads; ++i) load(i, lds0 + 2 * s * T::kStage);
    next_step();
  }
  wait_barrier<(kStages - 1) * kLoads>();
#pragma unroll
  for (int f = 0; f < kFrags; ++f) read(0, f, smem);
  int stage = 0;
  for (int t = 0; t < nk - 1; ++t) {
    const int next = stage == kStages - 1 ? 0 : stage + 1;
    multiply(first, yes, no, smem + stage * T::kStage, 0);
    // the next step has landed, and nobody reads this one's stage any more
    wait_barrier<(kStages - 2) * kLoads>();
    multiply(second, yes, yes, smem + next * T::kStage, lds0 + 2 * stage * T::kStage);
    next_step();
    stage = next;
  }
  multiply(first, yes, no, smem + stage * T::kStage, 0);
  multiply(second, no, no, smem, 0);

#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      f32x4 v[4];
#pragma unroll
      for (int g = 0; g < 4; ++g)
        v[g] = f32x4{acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2],
                     acc[i][j][4 * g + 3]};
      if (a.splits > 1) {
        // accumulator order: a wave's stores are 1 KiB runs
        const int64_t tile = (static_cast<int64_t>(sp) * a.col_tiles + ct) * a.row_tiles + rt;
        float *p = a.partials + tile * T::BM * T::BN + ((wave * FM + i) * FN + j) * 1024 + lane * 4;
#pragma unroll
        for (int g = 0; g < 4; ++g) *reinterpret_cast<f32x4 *>(p + 256 * g) = v[g];
      } else {
#pragma unroll
        for (int g = 0; g < 2; ++g)
          store_pair<kGated>(a, v[g], v[g + 2], g, m0 + (wm * FM + i) * 32,
                             n0 + (wn * FN + j) * (kGated ? 16 : 32), lane);
      }
    }
}

// Sums the splits' partials, half a fragment per wave, and finishes as the
// unsplit kernel does. Small products have few waves here, so each has several
// splits' loads in flight.
template <class T, bool kGated>
__global__ __launch_bounds__(kTileThreads) void tile_merge_kernel(const TileArgs a) {
  constexpr int FM = T::FM, FN = T::FN;
  const int lane = static_cast<int>(threadIdx.x) & 63;
  const int half = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) + 4 * blockIdx.y;
  const int g = half & 1, frag = half >> 1;
  const int wave = frag / (FM * FN), i = frag / FN % FM, j = frag % FN;
  const int rt = blockIdx.x % a.row_tiles, ct = blockIdx.x / a.row_tiles;
  f32x4 lo = {0.0f, 0.0f, 0.0f, 0.0f}, hi = lo;
  const int64_t split_stride = static_cast<int64_t>(gridDim.x) * T::BM * T::BN;
  const float *p = a.partials + static_cast<int64_t>(blockIdx.x) * T::BM * T::BN + frag * 1024 +
                   g * 256 + lane * 4;
  constexpr int kAhead = 4;
  int sp = 0;
  for (; sp + kAhead <= a.splits; sp += kAhead, p += kAhead * split_stride) {
    f32x4 v[kAhead], w[kAhead];
#pragma unroll
    for (int s = 0; s < kAhead; ++s) {
      v[s] = *reinterpret_cast<const f32x4 *>(p + s * split_stride);
      w[s] = *reinterpret_cast<const f32x4 *>(p + s * split_stride + 512);
    }
#pragma unroll
    for (int s = 0; s < kAhead; ++s) {
      lo += v[s];
      hi += w[s];
    }
  }
  for (; sp < a.splits; ++sp, p += split_stride) {
    lo += *reinterpret_cast<const f32x4 *>(p);
    hi += *reinterpret_cast<const f32x4 *>(p + 512);
  }
  store_pair<kGated>(a, lo, hi, g, rt * T::BM + (wave % T::WM * FM + i) * 32,
                     ct * (kGated ? T::BN / 2 : T::BN) +
                         (wave / T::WM * FN + j) * (kGated ? 16 : 32),
                     lane);
}

// RMSNorm of rows, y = bf16((x * rstd) * w) with rstd = 1 / sqrt(mean(x^2) + eps)
// in fp32: one wave per row, the whole row and the weight in registers before the
// sum, so a row is one trip to memory. C chunks of 512 values.
//
// Bound by launch and latency up to 512 rows, then by the copy rate. Against the
// library's norm, rows of 2560 (us, HIP graph): 512 rows 5.3 / 4.7, 2064 9.0 / 6.3,
// 8192 22.8 / 15.0 (5.6 TB/s).
template <int C>
__global__ __launch_bounds__(kTileThreads) void row_norm_kernel(
    const uint16_t *__restrict__ x, int64_t x_stride, int m, int k,
    const uint16_t *__restrict__ w, float eps, uint16_t *__restrict__ y) {
  const int lane = static_cast<int>(threadIdx.x) & 63;
  const int row = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (row >= m) return;
  u32x4 xv[C], wv[C];
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int col = 512 * c + 8 * lane;
    xv[c] = wv[c] = u32x4{0, 0, 0, 0};
    if (col < k) {
      xv[c] = load16(x + row * x_stride + col);
      wv[c] = load16(w + col);
    }
  }
  float ss = 0.0f;
#pragma unroll
  for (int c = 0; c < C; ++c)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t v = xv[c][j];
      ss = fmaf(bf16_lo(v), bf16_lo(v), ss);
      ss = fmaf(bf16_hi(v), bf16_hi(v), ss);
    }
#pragma unroll
  for (int d = 32; d; d >>= 1) ss += __shfl_xor(ss, d);
  const float rstd = 1.0f / sqrtf(ss / static_cast<float>(k) + eps);
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int col = 512 * c + 8 * lane;
    u32x4 out;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t v = xv[c][j], u = wv[c][j];
      out[j] = pack_bf16x2_rne((bf16_lo(v) * rstd) * bf16_lo(u), (bf16_hi(v) * rstd) * bf16_hi(u));
    }
    if (col < k) store16(y + static_cast<int64_t>(row) * k + col, out);
  }
}

template <class T, bool kGated>
int launch_tiles(const TileArgs &a, hipStream_t stream) {
  const int tiles = a.row_tiles * a.col_tiles;
  hipLaunchKernelGGL((tile_kernel<T, kGated>), dim3(tiles * a.splits), dim3(kTileThreads), 0,
                     stream, a);
  if (a.splits > 1)
    hipLaunchKernelGGL((tile_merge_kernel<T, kGated>), dim3(tiles, T::BM * T::BN / 2048),
                       dim3(kTileThreads), 0, stream, a);
  return launch_status("hy_linear_tiles");
}

template <bool kGated>
int launch_shape(int shape, const TileArgs &a, hipStream_t stream) {
  switch (shape) {
    case 0: return launch_tiles<Tile<64, 128, 2>, kGated>(a, stream);
    case 1: return launch_tiles<Tile<128, 96, 1>, kGated>(a, stream);
    case 2: return launch_tiles<Tile<128, 128, 2>, kGated>(a, stream);
    case 3: return launch_tiles<Tile<128, 192, 2>, kGated>(a, stream);
    case 4: return launch_tiles<Tile<256, 128, 2>, kGated>(a, stream);
    default: return launch_tiles<Tile<256, 160, 1>, kGated>(a, stream);
  }
}

bool aligned(const void *p, int bytes) { return (reinterpret_cast<uintptr_t>(p) & (bytes - 1)) == 0; }

bool sizes_fit(int m, int n, int k) {
  // the grid's threads stay below 2^32
  return k % kStepK == 0 && n % 4 == 0 && static_cast<int64_t>(m / 64 + 1) * (n / 48 + 1) < (1 << 23);
}

}  // namespace
}  // namespace hy

extern "C" int64_t hy_linear_tiles_workspace_bytes(int32_t m, int32_t n, int32_t k, int32_t gated) {
  if (m <= 0 || n <= 0 || k <= 0 || !hy::sizes_fit(m, n, k)) return 0;
  return hy::plan_tiles(m, n, k, gated != 0).bytes;
}

extern "C" int hy_linear_tiles(const void *x, int64_t x_stride, int32_t m, int32_t k,
                               const void *weight, const void *up_weight, int64_t w_stride,
                               int32_t n, const void *residual, int64_t r_stride, void *y,
                               int64_t y_stride, void *workspace, int64_t workspace_bytes,
                               void *stream) {
  hy::clear_error();
  HY_REQUIRE(m >= 0 && n >= 0 && k > 0, "hy_linear_tiles: invalid sizes %d x %d x %d", m, n, k);
  if (m == 0 || n == 0) return HY_OK;
  HY_REQUIRE(x && weight && y, "hy_linear_tiles: null pointer argument");
  HY_REQUIRE(!(up_weight && residual), "hy_linear_tiles: a gated product takes no residual");
  HY_REQUIRE_SUPPORTED(hy::sizes_fit(m, n, k), "hy_linear_tiles: sizes %d x %d x %d unsupported", m,
                       n, k);
  HY_REQUIRE(hy::aligned(x, 16) && hy::aligned(weight, 16) && hy::aligned(up_weight, 16) &&
                 ((x_stride | w_stride) & 7) == 0,
             "hy_linear_tiles: operand rows must be 16-byte aligned");
  HY_REQUIRE(hy::aligned(y, 8) && hy::aligned(residual, 8) && ((y_stride | r_stride) & 3) == 0,
             "hy_linear_tiles: result and residual rows must be 8-byte aligned");
  // a tile's rows and the reach along k are 32-bit byte offsets
  HY_REQUIRE_SUPPORTED(x_stride >= 0 && w_stride >= 0 && x_stride < (1 << 22) &&
                           w_stride < (1 << 22) && k < (1 << 22),
                       "hy_linear_tiles: rows too long");
  const hy::TilePlan plan = hy::plan_tiles(m, n, k, up_weight != nullptr);
  HY_REQUIRE(plan.bytes == 0 || (workspace && workspace_bytes >= plan.bytes && hy::aligned(workspace, 16)),
             "hy_linear_tiles: needs %lld bytes of 16-byte aligned workspace",
             static_cast<long long>(plan.bytes));
  const hy::TileArgs a{static_cast<const uint16_t *>(x),
                       x_stride,
                       m,
                       n,
                       k,
                       static_cast<const uint16_t *>(weight),
                       static_cast<const uint16_t *>(up_weight),
                       w_stride,
                       static_cast<const uint16_t *>(residual),
                       r_stride,
                       static_cast<uint16_t *>(y),
                       y_stride,
                       static_cast<float *>(workspace),
                       plan.row_tiles,
                       plan.col_tiles,
                       plan.splits,
                       plan.row_group};
  return up_weight ? hy::launch_shape<true>(plan.shape, a, static_cast<hipStream_t>(stream))
                   : hy::launch_shape<false>(plan.shape, a, static_cast<hipStream_t>(stream));
}

extern "C" int hy_row_norm(const void *x, int64_t x_stride, int32_t m, int32_t k,
                           const void *norm_weight, float eps, void *y, void *stream) {
  hy::clear_error();
  HY_REQUIRE(m >= 0 && k > 0, "hy_row_norm: invalid sizes %d x %d", m, k);
  if (m == 0) return HY_OK;
  HY_REQUIRE(x && norm_weight && y, "hy_row_norm: null pointer argument");
  HY_REQUIRE_SUPPORTED(k % 8 == 0 && k <= 4096, "hy_row_norm: rows of %d unsupported", k);
  HY_REQUIRE(hy::aligned(x, 16) && hy::aligned(norm_weight, 16) && hy::aligned(y, 16) &&
                 (x_stride & 7) == 0,
             "hy_row_norm: rows must be 16-byte aligned");
  // one row per workgroup until every CU has several
  const int waves = m <= 4096 ? 1 : hy::kTileWaves;
#define HY_NORM(C)                                                                               \
  case C:                                                                                        \
    hipLaunchKernelGGL((hy::row_norm_kernel<C>), dim3((m + waves - 1) / waves), dim3(64 * waves), \
                       0, static_cast<hipStream_t>(stream), static_cast<const uint16_t *>(x),   \
                       x_stride, m, k, static_cast<const uint16_t *>(norm_weight), eps,         \
                       static_cast<uint16_t *>(y));                                             \
    break;
  switch ((k + 511) / 512) {
    HY_NORM(1) HY_NORM(2) HY_NORM(3) HY_NORM(4) HY_NORM(5) HY_NORM(6) HY_NORM(7) HY_NORM(8)
  }
#undef HY_NORM
  return hy::launch_status("hy_row_norm");
}
