// Products of few activation rows (decode tokens) with a large weight
// matrix, y = f(x) W^T, for M <= 32 rows: the weights are read once from HBM
// and everything around the product rides on that read.
//
//   wide_kernel    N much larger than K (the fused q/k/v projection, the MLP's
//                  gate and up projections, the vocabulary head): RMSNorm of x
//                  before the product, optionally silu(gate) * up after it.
//   tall_kernel    long K (the attention output and MLP down projections):
//                  residual added after the product.
//
// Both use v_mfma_f32_16x16x32_bf16 with 16 weight rows as A and x^T as B, so
// lane (m = l % 16, g = l / 16) ends with y[m][4 g + i] of the 16 weight rows.
//
// What bounds them is the read of the weights, and within it the order of the
// lanes. In operand order (lane l holds row l % 16) four neighbouring lanes
// touch four rows: a CU then takes 34 GB/s, measured on rows that sit in L2,
// against 105 GB/s when they share 64 bytes of a row. And a load of 64-byte
// runs asks HBM for half lines: the vocabulary head (778 MB) went from 150 to
// 122 us with 128-byte runs. So a load instruction covers 8 rows x 128 bytes;
// its registers go to LDS and come back in operand order. The LDS buffers
// belong to one wave, so no barrier is involved.
//
// The waves of a workgroup split K; their fp32 partial sums meet in LDS. Rows
// of x past M repeat row M - 1 and weight rows past the workgroup's share
// repeat its last row (addresses already in the caches); neither is stored.

#include "hy_common.h"
#include "qknorm.h"

namespace hy {
namespace {

constexpr int kSkinnyWaves = 8;             // waves per workgroup, two per SIMD
constexpr int kSkinnyThreads = 64 * kSkinnyWaves;
// LDS floats of one wave's 16 x 16 partial tile: lane (m, g) keeps its four
// sums at 80 g + 4 m (16-float gaps between the g groups spread the reads
// over all banks).
constexpr int kPartTile = 4 * 80;

// LDS place (u16) of chunk g (8 k) of row r of a tile: the xor spreads the
// 16 rows of one chunk over all banks.
constexpr int kTileElems = 16 * 32;
__device__ __forceinline__ int tile_at(int r, int g) {
  return (4 * r + (g ^ ((r >> 2) & 3))) * 8;
}

__device__ __forceinline__ f32x4 mfma16(const u32x4 &a, const u32x4 &b, const f32x4 &c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// y = norm(x) W^T or silu(norm(x) Wg^T) * (norm(x) Wu^T).
//
// Workgroup i, one per CU, owns output columns [i n / grid, (i + 1) n / grid)
// and walks them 16 weight rows at a time (gated: 8 of Wg and 8 of Wu). Wave
// w keeps its SPW steps of 32 k of all of x in registers for the whole walk,
// so a tile is SPW loads, SPW * MT MFMAs and one exchange of partial sums,
// with the next two tiles in flight. The norm's weight is folded into x (one
// bf16 rounding, as the norm's own) and its 1 / rms into the fp32 sums, so
// that no wave waits for the row sums before its products; normalising x up
// front, 1 / rms included, took 2.5 us more at 32 rows (every CU repeats it).
//
// Measured on MI355X against the library's norm, products and silu * up (us,
// HIP graph, weights from HBM; x is M x 2560):
//                       M = 1          16             32
//   N = 6144, normed    9.7 / 13.5     10.4 / 14.6    12.6 / 15.5
//   2 x 9728, gated     19.7 / 45.7    20.1 / 43.0    21.8 / 40.1
//   N = 151936, normed  120 / 252      128 / 252      136 / 177  (6.5-5.7 TB/s)
template <int MT, int SPW, bool kGated>
__global__ __launch_bounds__(kSkinnyThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
void wide_kernel(const uint16_t *__restrict__ x, int64_t ldx, int m_rows, int k_dim,
                 const uint16_t *__restrict__ norm_w, float eps, const uint16_t *__restrict__ w0,
                 const uint16_t *__restrict__ w1, int64_t ldw, int n_cols,
                 uint16_t *__restrict__ y, int64_t ldy) {
  constexpr int kTile = kGated ? 8 : 16;  // output columns per tile
  __shared__ __attribute__((aligned(16))) uint16_t tiles[kSkinnyWaves][SPW * kTileElems];
  __shared__ __attribute__((aligned(16))) float part[2][kSkinnyWaves][MT][kPartTile];
  __shared__ __attribute__((aligned(16))) uint16_t scale_w[kSkinnyWaves * SPW * 32];
  __shared__ float sums[kSkinnyWaves][16 * MT];

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int c = lane & 15;
  const int g = lane >> 4;
  const int c0 = static_cast<int>(static_cast<int64_t>(n_cols) * blockIdx.x / gridDim.x);
  const int c1 = static_cast<int>(static_cast<int64_t>(n_cols) * (blockIdx.x + 1) / gridDim.x);
  if (c0 >= c1) return;
  // This wave's SPW steps of 32 k start at s0; near the end of K the window
  // slides back into it, and B is zero for steps another wave owns (`own`).
  const int s0 = min(wave * SPW, k_dim / 32 - SPW);
  const int own = wave * SPW - s0;
  const int lr = lane >> 3;               // row and k of a row-major load
  const int lk = 32 * s0 + 8 * (lane & 7);
  uint16_t *put[2];
#pragma unroll
  for (int h = 0; h < 2; ++h)
    put[h] = tiles[wave] + ((lane >> 2) & 1) * kTileElems + tile_at(lr + 8 * h, lane & 3);
  const uint16_t *get = tiles[wave] + tile_at(c, g);

  u32x4 b[MT][SPW], nw;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const uint16_t *row =
          x + static_cast<int64_t>(min(16 * mt + 8 * h + lr, m_rows - 1)) * ldx + lk;
#pragma unroll
      for (int s = 0; s < SPW; s += 2) b[mt][s + h] = load16(row + 32 * s);
    }
  // This wave's norm weights, lane l < 4 SPW holding chunk l.
  if (norm_w != nullptr) nw = load16(norm_w + 32 * s0 + 8 * min(lane, 4 * SPW - 1));

  auto issue = [&](u32x4 (&a)[SPW], int n0) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const uint16_t *row;
      if constexpr (kGated) {
        row = (h ? w1 : w0) + static_cast<int64_t>(min(n0 + lr, c1 - 1)) * ldw + lk;
      } else {
        row = w0 + static_cast<int64_t>(min(n0 + 8 * h + lr, c1 - 1)) * ldw + lk;
      }
#pragma unroll
      for (int s = 0; s < SPW; s += 2) a[s + h] = load16_stream(row + 32 * s);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  // From load order to operand order, through this wave's buffer.
  auto turn = [&](u32x4 (&a)[SPW]) {
#pragma unroll
    for (int s = 0; s < SPW; ++s)
      *reinterpret_cast<u32x4 *>(put[s & 1] + (s & ~1) * kTileElems) = a[s];
#pragma unroll
    for (int s = 0; s < SPW; ++s) a[s] = *reinterpret_cast<const u32x4 *>(get + s * kTileElems);
  };
  u32x4 a0[SPW], a1[SPW];
  issue(a0, c0);
  issue(a1, min(c0 + kTile, c1 - 1));
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) turn(b[mt]);
  auto drop_others = [&]() {  // steps that another wave owns
    if (own == 0) return;
#pragma unroll
    for (int s = 0; s < SPW; ++s)
      if (s < own) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) b[mt][s] = u32x4{0u, 0u, 0u, 0u};
      }
  };
  drop_others();

  if (norm_w != nullptr) {
    // Row sums of squares over this wave's k: the diagonal of x x^T, whose
    // element m lies in lane (m, g = m / 4).
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      f32x4 gram = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < SPW; ++s) gram = mfma16(b[mt][s], b[mt][s], gram);
      const float ss = (c & 2) ? ((c & 1) ? gram[3] : gram[2]) : ((c & 1) ? gram[1] : gram[0]);
      if (g == c >> 2) sums[wave][16 * mt + c] = ss;
    }
    // B becomes bf16(x * weight); the row's 1 / rms multiplies the fp32 sums.
    uint16_t *sw = scale_w + wave * SPW * 32;
    if (lane < 4 * SPW) *reinterpret_cast<u32x4 *>(sw + 8 * lane) = nw;
#pragma unroll
    for (int s = 0; s < SPW; ++s) {
      float wv[8];
      unpack8(*reinterpret_cast<const u32x4 *>(sw + 32 * s + 8 * g), wv);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        float v[8];
        unpack8(b[mt][s], v);
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] *= wv[j];
        b[mt][s] = pack8_rne(v);
      }
    }
    drop_others();  // again: no 0 * inf of an infinite weight
  }

  // Output (m, n) of a tile: thread m * kTile + n, the same for every tile.
  constexpr int kOut = kTile * 16 * MT;
  static_assert(kOut <= kSkinnyThreads, "one output per thread");
  const int on = threadIdx.x % kTile;
  const int om = threadIdx.x / kTile;
  const bool out = static_cast<int>(threadIdx.x) < kOut && om < m_rows;
  float rstd = 1.0f;
  bool first = norm_w != nullptr;
  auto consume = [&](u32x4 (&a)[SPW], int buf) {
    turn(a);
    if (own > 0) {  // another wave's steps: no 0 * inf
#pragma unroll
      for (int s = 0; s < SPW; ++s)
        if (s < own) a[s] = u32x4{0u, 0u, 0u, 0u};
    }
    f32x4 acc[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < SPW; ++s)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) acc[mt] = mfma16(a[s], b[mt][s], acc[mt]);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
      *reinterpret_cast<f32x4 *>(&part[buf][wave][mt][80 * g + 4 * c]) = acc[mt];
    __builtin_amdgcn_sched_barrier(0);
  };
  auto finish = [&](int n0, int buf) {
    __syncthreads();  // the buffer of two tiles ago is free again after this one
    if (!out) return;
    if (first) {
      float ss = 0.f;
#pragma unroll
      for (int w = 0; w < kSkinnyWaves; ++w) ss += sums[w][om];
      rstd = 1.0f / sqrtf(ss / static_cast<float>(k_dim) + eps);
      first = false;
    }
    auto sum = [&](int r) {  // of weight row r of the tile
      float t = 0.f;
#pragma unroll
      for (int w = 0; w < kSkinnyWaves; ++w)
        t += part[buf][w][om >> 4][80 * (r >> 2) + 4 * (om & 15) + (r & 3)];
      return t * rstd;
    };
    float v = sum(on);
    if constexpr (kGated) {
      const float up = sum(8 + on);
      v = v / (1.0f + expf(-v)) * up;
    }
    if (n0 + on < c1) y[om * ldy + n0 + on] = static_cast<uint16_t>(f32_to_bf16_rne(v));
  };

  // Two tiles are always in flight; the steady state issues without a
  // condition, so that every wait covers only the tile it needs.
  int n0 = c0;
  for (; n0 + 3 * kTile < c1; n0 += 2 * kTile) {
    consume(a0, 0);
    issue(a0, n0 + 2 * kTile);
    finish(n0, 0);
    consume(a1, 1);
    issue(a1, n0 + 3 * kTile);
    finish(n0 + kTile, 1);
  }
  consume(a0, 0);
  if (n0 + 2 * kTile < c1) issue(a0, n0 + 2 * kTile);
  finish(n0, 0);
  if (n0 + kTile < c1) {
    consume(a1, 1);
    finish(n0 + kTile, 1);
  }
  if (n0 + 2 * kTile < c1) {
    consume(a0, 0);
    finish(n0 + 2 * kTile, 0);
  }
}

// y = x W^T (+ residual), one tile of up to 16 weight rows per workgroup (10
// for the 2,560 outputs of the default model, one workgroup per CU); the
// waves take contiguous shares of K in stages of kSteps tiles, two stages of
// weights and activations in flight. Every CU reads all of x, M / 10 times
// its share of the weights, from L2 (about 95 GB/s per CU), which is what grows
// with M. 16 waves, longer stages or a deeper ring measured the same or slower.
//
// Measured on MI355X against the library's product and addition (us):
//                     M = 1          16             20             32
//   N = 2560, K 4096  6.6 / 14.3     8.3 / 14.9     9.5 / 11.4     9.6 / 11.5
//   N = 2560, K 9728  12.9 / 20.8    15.5 / 20.1    17.8 / 21.4    19.2 / 23.0
// (at 48 and 64 rows 23.2 / 22.9 and 27.1 / 30.5 for K = 9728: not built).
template <int MT>
__global__ __launch_bounds__(kSkinnyThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
void tall_kernel(const uint16_t *__restrict__ x, int64_t ldx, int m_rows, int k_dim,
                 const uint16_t *__restrict__ w, int64_t ldw, int n_cols,
                 const uint16_t *__restrict__ res, int64_t ldr, uint16_t *__restrict__ y,
                 int64_t ldy) {
  constexpr int kSteps = 4;
  constexpr int kLoads = kSteps * (1 + MT);
  union Shared {
    uint16_t tiles[kSkinnyWaves][kLoads * kTileElems];
    float part[kSkinnyWaves][MT][kPartTile];
  };
  __shared__ __attribute__((aligned(16))) Shared sh;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int c = lane & 15;
  const int g = lane >> 4;
  const int c0 = static_cast<int>(static_cast<int64_t>(n_cols) * blockIdx.x / gridDim.x);
  const int c1 = static_cast<int>(static_cast<int64_t>(n_cols) * (blockIdx.x + 1) / gridDim.x);
  if (c0 >= c1) return;
  const int stages = k_dim / (32 * kSteps);
  const int t0 = stages * wave / kSkinnyWaves;
  const int t1 = stages * (wave + 1) / kSkinnyWaves;

  const int lr = lane >> 3;  // row and k of a row-major load
  const int lk = 8 * (lane & 7);
  const uint16_t *wr[2], *xr[MT][2];
  uint16_t *put[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    wr[h] = w + static_cast<int64_t>(min(c0 + 8 * h + lr, c1 - 1)) * ldw + lk;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
      xr[mt][h] = x + static_cast<int64_t>(min(16 * mt + 8 * h + lr, m_rows - 1)) * ldx + lk;
    put[h] = sh.tiles[wave] + ((lane >> 2) & 1) * kTileElems + tile_at(lr + 8 * h, lane & 3);
  }
  const uint16_t *get = sh.tiles[wave] + tile_at(c, g);

  f32x4 acc[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) acc[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto issue = [&](u32x4 (&r)[kLoads], int t) {
    const int k = 32 * kSteps * t;
#pragma unroll
    for (int s = 0; s < kSteps; ++s) r[s] = load16_stream(wr[s & 1] + k + 32 * (s & ~1));
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int s = 0; s < kSteps; ++s)
        r[kSteps * (1 + mt) + s] = load16(xr[mt][s & 1] + k + 32 * (s & ~1));
    __builtin_amdgcn_sched_barrier(0);
  };
  auto consume = [&](u32x4 (&r)[kLoads]) {
#pragma unroll
    for (int i = 0; i < kLoads; ++i)
      *reinterpret_cast<u32x4 *>(put[i & 1] + (i & ~1) * kTileElems) = r[i];
    auto op = [&](int i) { return *reinterpret_cast<const u32x4 *>(get + i * kTileElems); };
#pragma unroll
    for (int s = 0; s < kSteps; ++s) {
      const u32x4 a = op(s);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) acc[mt] = mfma16(a, op(kSteps * (1 + mt) + s), acc[mt]);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  if (t0 < t1) {
    u32x4 p[kLoads], q[kLoads];
    issue(p, t0);
    int t = t0;
    for (; t + 2 < t1; t += 2) {
      issue(q, t + 1);
      consume(p);
      issue(p, t + 2);
      consume(q);
    }
    if (t + 1 < t1) {
      issue(q, t + 1);
      consume(p);
      consume(q);
    } else {
      consume(p);
    }
  }
  __syncthreads();  // the partial sums reuse the tile buffers
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
    *reinterpret_cast<f32x4 *>(&sh.part[wave][mt][80 * g + 4 * c]) = acc[mt];
  __syncthreads();
  for (int o = threadIdx.x; o < 16 * 16 * MT; o += kSkinnyThreads) {
    const int n = o & 15;
    const int m = o >> 4;
    if (m >= m_rows || c0 + n >= c1) continue;
    float v = 0.f;
#pragma unroll
    for (int wv = 0; wv < kSkinnyWaves; ++wv)
      v += sh.part[wv][m >> 4][80 * (n >> 2) + 4 * (m & 15) + (n & 3)];
    if (res != nullptr) v += bf16_lo(res[m * ldr + c0 + n]);
    y[m * ldy + c0 + n] = static_cast<uint16_t>(f32_to_bf16_rne(v));
  }
}

}  // namespace
}  // namespace hy

namespace {

int num_cus() {
  static const int n = [] {
    int dev = 0, v = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || v < 1)
      v = 256;
    return v;
  }();
  return n;
}

bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// The step counts cover every K of 512 .. 4096 in multiples of 64 (rounded up,
// a wave's window slides back); two row tiles of 16 steps would not fit the
// registers, so K > 3072 takes 16 rows.
template <bool kGated>
int launch_wide(const uint16_t *x, int64_t ldx, int m, int k, const uint16_t *nw, float eps,
                const uint16_t *w0, const uint16_t *w1, int64_t ldw, int n, uint16_t *y,
                int64_t ldy, hipStream_t st) {
  const int spw = (k / 32 + hy::kSkinnyWaves - 1) / hy::kSkinnyWaves;
  const int tile = kGated ? 8 : 16;
  const int grid = min(num_cus(), (n + tile - 1) / tile);
#define HY_WIDE(MT, SPW)                                                                          \
  hipLaunchKernelGGL((hy::wide_kernel<MT, SPW, kGated>), dim3(grid), dim3(hy::kSkinnyThreads), 0, \
                     st, x, ldx, m, k, nw, eps, w0, w1, ldw, n, y, ldy)
  if (m <= 16) {
    if (spw <= 4) HY_WIDE(1, 4);
    else if (spw <= 8) HY_WIDE(1, 8);
    else if (spw <= 10) HY_WIDE(1, 10);
    else if (spw <= 12) HY_WIDE(1, 12);
    else HY_WIDE(1, 16);
  } else {
    if (spw <= 4) HY_WIDE(2, 4);
    else if (spw <= 8) HY_WIDE(2, 8);
    else if (spw <= 10) HY_WIDE(2, 10);
    else HY_WIDE(2, 12);
  }
#undef HY_WIDE
  return hy::launch_status("hy_norm_linear");
}

}  // namespace

extern "C" int hy_norm_linear(const void *x, int64_t x_stride, int32_t m, int32_t k,
                              const void *norm_weight, float eps, const void *weight,
                              const void *up_weight, int64_t w_stride, int32_t n, void *y,
                              int64_t y_stride, void *stream) {
  hy::clear_error();
  HY_REQUIRE(m >= 0 && n >= 0 && k > 0, "hy_norm_linear: invalid sizes %d x %d x %d", m, n, k);
  if (m == 0 || n == 0) return HY_OK;
  HY_REQUIRE(x && weight && y, "hy_norm_linear: null pointer argument");
  HY_REQUIRE_SUPPORTED(k % 64 == 0 && k >= 512 && k <= 4096 && m <= (k <= 3072 ? 32 : 16),
                       "hy_norm_linear: %d rows of %d unsupported", m, k);
  HY_REQUIRE(aligned16(x) && aligned16(weight) && aligned16(up_weight) && aligned16(norm_weight) &&
                 ((x_stride | w_stride) & 7) == 0,
             "hy_norm_linear: rows must be 16-byte aligned");
  const auto *xx = static_cast<const uint16_t *>(x);
  const auto *nw = static_cast<const uint16_t *>(norm_weight);
  const auto *w0 = static_cast<const uint16_t *>(weight);
  const auto *w1 = static_cast<const uint16_t *>(up_weight);
  auto *yy = static_cast<uint16_t *>(y);
  hipStream_t st = static_cast<hipStream_t>(stream);
  return w1 ? launch_wide<true>(xx, x_stride, m, k, nw, eps, w0, w1, w_stride, n, yy,
                                y_stride, st)
            : launch_wide<false>(xx, x_stride, m, k, nw, eps, w0, w1, w_stride, n, yy,
                                 y_stride, st);
}

extern "C" int hy_linear_add(const void *x, int64_t x_stride, int32_t m, int32_t k,
                             const void *weight, int64_t w_stride, int32_t n, const void *residual,
                             int64_t r_stride, void *y, int64_t y_stride, void *stream) {
  hy::clear_error();
  HY_REQUIRE(m >= 0 && n >= 0 && k > 0, "hy_linear_add: invalid sizes %d x %d x %d", m, n, k);
  if (m == 0 || n == 0) return HY_OK;
  HY_REQUIRE(x && weight && y, "hy_linear_add: null pointer argument");
  HY_REQUIRE_SUPPORTED(k % 128 == 0 && m <= 32, "hy_linear_add: %d rows of %d unsupported", m, k);
  HY_REQUIRE(aligned16(x) && aligned16(weight) && ((x_stride | w_stride) & 7) == 0,
             "hy_linear_add: rows must be 16-byte aligned");
  const int grid = max((n + 15) / 16, min(num_cus(), (n + 7) / 8));
#define HY_TALL(MT)                                                                                \
  hipLaunchKernelGGL((hy::tall_kernel<MT>), dim3(grid), dim3(hy::kSkinnyThreads), 0,             \
                     static_cast<hipStream_t>(stream), static_cast<const uint16_t *>(x), x_stride, \
                     m, k, static_cast<const uint16_t *>(weight), w_stride, n,                   \
                     static_cast<const uint16_t *>(residual), r_stride, static_cast<uint16_t *>(y), \
                     y_stride)
  if (m <= 16) HY_TALL(1);
  else HY_TALL(2);
#undef HY_TALL
  return hy::launch_status("hy_linear_add");
}
