// Batched sampling of 16-bit logits: greedy, temperature, top-k and top-p,
// without a sort.
//
// The reference sorts each row (hayate/engine/sampler.py:39-65); batched, the sort
// of 20 x 151,936 scores, the softmax and prefix sum over them and the scatter
// back took 1,040 us. What is needed of the order is only where top-k and top-p
// cut it. A 16-bit logit has 65,536 values, so a histogram of a row holds its
// whole order, and all logits of one value share one score and probability:
// counts times exp(score - max) are the cumulative masses.
//
//   cut_kernel   one workgroup per row: greedy rows end here; for the others
//                the histogram in LDS (65,536 16-bit counters; a value that
//                more than 65,535 logits share shows in the counters' sum,
//                and the row is done again with 32-bit counters, half of the
//                values at a time), the k-th value and the value in which the
//                mass passes top_p. A value that this cut splits keeps its
//                first logits by index, as a stable descending sort does.
//   draw_kernel  many workgroups per row: the largest p / q of each one's share
//                of the kept logits, q the exponential noise the caller made;
//                the draw of torch.multinomial.
//   pick_kernel  the largest of those per row.
//
// cut_kernel is bound by one CU's reads (304 KB a row of 151,936: 10 us, also
// of a greedy row), its LDS atomics (8 us), and for a top-p cut a walk over the
// counters and a second read for the ties (18 us); everything that needs an
// exponential per logit is in draw_kernel (9-11 us, 19 workgroups a row).
// Measured on MI355X, 20 rows of 151,936, noise and launches included, against
// the sort: greedy 35 -> 17 us, temperature alone 1,056 -> 38, top-k 1,060 -> 41,
// top-p 1,054 -> 62, a mix 1,020 -> 59.

#include <math.h>

#include "hy_common.h"

namespace hy {
namespace {

constexpr int kCutThreads = 1024;
constexpr int kCutWaves = kCutThreads / 64;
constexpr int kWords = 32768;                  // histogram words
constexpr int kVec = 8;                        // logits per load
constexpr int kAhead = 4;                      // loads in flight per thread
constexpr int kStep = kVec * kCutThreads;      // logits per round of the workgroup
constexpr int kMaxRounds = 512;                // rounds whose tie counts fit LDS
constexpr int kDrawThreads = 256;
constexpr int kDrawShare = kDrawThreads * kVec * kAhead;  // logits per draw workgroup
constexpr int kSampleRows = 64;                // rows of one launch
constexpr float kLog2eS = 1.4426950408889634f;

typedef short s16x2 __attribute__((ext_vector_type(2)));
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

struct SampleRow {
  float temp;     // 0: greedy
  int32_t k;      // of top-k, vocabulary size for none
  float p;        // of top-p, >= 1 for none
  int32_t noise;  // row of the noise
};
struct SampleRows {
  SampleRow r[kSampleRows];
};
// What the cut leaves of a row: keys >= low, except those == cut past index last.
struct RowCut {
  int32_t low, cut, last, ok;
  float max;  // largest score
};

// Ordered keys of two 16-bit floats: larger key, larger value.
__device__ __forceinline__ uint32_t keys_of(uint32_t w) {
  const s16x2 sign = __builtin_bit_cast(s16x2, w) >> 15;
  return w ^ ((__builtin_bit_cast(uint32_t, sign) & 0x7fff7fffu) | 0x80008000u);
}
// -0 counts as +0.
__device__ __forceinline__ uint32_t merge_zero(uint32_t key) { return key == 0x7fffu ? 0x8000u : key; }
template <bool kBf16>
constexpr uint32_t kInfBits = kBf16 ? 0x7f80u : 0x7c00u;

template <bool kBf16>
__device__ __forceinline__ float value_of(uint32_t key) {
  const uint32_t u = (key & 0x8000u) ? key & 0x7fffu : 0xffffu & ~key;
  if (kBf16) return __uint_as_float(u << 16);
  return static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(u)));
}

// v / t to within the last bit (t is in the range the entry accepts).
__device__ __forceinline__ float score_of(float v, float t, float rcp) {
  const float s = v * rcp;
  return isinf(s) ? s : __builtin_fmaf(__builtin_fmaf(-s, t, v), rcp, s);
}

// Larger value first, then smaller index.
__device__ __forceinline__ uint64_t rank_of(uint32_t value, int index) {
  return static_cast<uint64_t>(value) << 32 | (0xffffffffu - static_cast<uint32_t>(index));
}
__device__ __forceinline__ int index_of(uint64_t rank) {
  return static_cast<int>(0xffffffffu - static_cast<uint32_t>(rank));
}
__device__ __forceinline__ uint64_t wave_best(uint64_t v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const uint64_t w = __shfl_xor(static_cast<unsigned long long>(v), o);
    v = w > v ? w : v;
  }
  return v;
}

template <bool kBf16>
__global__ __launch_bounds__(kCutThreads) void cut_kernel(
    const uint16_t *__restrict__ logits, int64_t ld, int vocab, SampleRows rows,
    int64_t *__restrict__ out, RowCut *__restrict__ cuts) {
  __shared__ uint32_t hist[kWords];
  __shared__ uint64_t best[kCutWaves];
  __shared__ uint32_t wave_cnt[kCutWaves];
  __shared__ float wave_mass[kCutWaves];
  __shared__ uint32_t tie_cnt[kMaxRounds];
  __shared__ struct {
    int kth;  // key of the k-th largest logit, -1 while unknown
    int cut;  // key that the top-p cut lies in, -1 while unknown
    uint32_t cut_keep, cut_count;  // its logits kept, and all of them
    int last;  // index of the last kept logit of the cut's value
  } sh;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const SampleRow row = rows.r[blockIdx.x];
  const uint16_t *x = logits + blockIdx.x * ld;
  const bool greedy = row.temp == 0.f;
  const bool use_k = !greedy && row.k < vocab;
  const bool use_p = !greedy && row.p < 1.f;
  const float temp = greedy ? 1.f : row.temp;
  const float rcp = 1.0f / temp;

  // Calls f(keys, index of the first, how many) for this thread's logits, up to
  // kVec at a time (two keys a word), in index order.
  const int n_vec = vocab / kVec;
  auto each = [&](auto f) __attribute__((always_inline)) {
#pragma unroll 1
    for (int v = tid; v < n_vec; v += kAhead * kCutThreads) {
      u32x4 w[kAhead];
#pragma unroll
      for (int a = 0; a < kAhead; ++a)  // rows may start at any logit
        __builtin_memcpy(&w[a], x + kVec * min(v + a * kCutThreads, n_vec - 1), sizeof(w[a]));
#pragma unroll
      for (int a = 0; a < kAhead; ++a) {
        const int va = v + a * kCutThreads;
        if (va >= n_vec) break;
#pragma unroll
        for (int j = 0; j < kVec / 2; ++j) w[a][j] = keys_of(w[a][j]);
        f(w[a], kVec * va, kVec);
      }
    }
    if (vocab % kVec && tid == n_vec % kCutThreads) {
      u32x4 w = {0u, 0u, 0u, 0u};
#pragma unroll
      for (int j = 0; j < kVec; ++j)
        w[j >> 1] |= static_cast<uint32_t>(x[min(kVec * n_vec + j, vocab - 1)]) << (16 * (j & 1));
#pragma unroll
      for (int j = 0; j < kVec / 2; ++j) w[j] = keys_of(w[j]);
      f(w, kVec * n_vec, vocab % kVec);
    }
  };
  auto key_at = [](const u32x4 &w, int j) { return (w[j >> 1] >> (16 * (j & 1))) & 0xffffu; };
  auto block_best = [&](uint64_t v) __attribute__((always_inline)) {
    v = wave_best(v);
    __syncthreads();  // earlier readers of best are done
    if (lane == 0) best[wave] = v;
    __syncthreads();
    v = best[0];
#pragma unroll
    for (int w = 1; w < kCutWaves; ++w) v = best[w] > v ? best[w] : v;
    return v;
  };

  const bool filter = use_k || use_p;
  if (filter)
    for (int i = tid; i < kWords; i += kCutThreads) hist[i] = 0;
  if (tid == 0) {
    sh.kth = use_k ? -1 : 0;
    sh.cut = use_p ? -1 : 0;
    sh.cut_keep = sh.cut_count = 0;
    sh.last = vocab;
  }
  __syncthreads();

  // One read: the largest key and this thread's first load that holds it,
  // whether there is a NaN (a magnitude above infinity), and the histogram.
  // Past the end of the row a tail repeats its last logit, which changes
  // none of these.
  u16x2 mag2 = {0, 0};
  uint32_t my_key = 0;
  int my_load = 0;
  each([&](const u32x4 &w, int i0, int n) __attribute__((always_inline)) {
    u16x2 top2 = {0, 0};
#pragma unroll
    for (int j = 0; j < kVec / 2; ++j) {
      const uint32_t word = w[j];  // a bit cast of w[j] itself reads w[0]
      const u16x2 k2 = __builtin_bit_cast(u16x2, word);
      top2 = __builtin_elementwise_max(top2, k2);
      // a key or its complement is 0x8000 + the magnitude
      const u16x2 neg = __builtin_bit_cast(u16x2, ~word);
      mag2 = __builtin_elementwise_max(mag2, __builtin_elementwise_max(k2, neg));
    }
    const uint32_t top = max(top2[0], top2[1]);
    if (top > my_key) {
      my_key = top;
      my_load = i0;
    }
    if (filter) {
#pragma unroll
      for (int j = 0; j < kVec; ++j) {
        const uint32_t key = key_at(w, j);
        if (j < n) atomicAdd(&hist[key >> 1], 1u << (16 * (key & 1)));
      }
    }
  });
  const uint32_t mag = max(mag2[0], mag2[1]) & 0x7fffu;
  const uint64_t top = block_best(rank_of(my_key, my_load));
  const uint32_t top_key = merge_zero(static_cast<uint32_t>(top >> 32));
  const bool nan = __syncthreads_or(mag > kInfBits<kBf16>);

  if (greedy) {
    // the first logit of the largest value; a NaN counts as the largest
    int first = vocab;
    if (nan || top_key == 0x8000u) {  // several keys count as the largest
      each([&](const u32x4 &w, int i0, int n) __attribute__((always_inline)) {
#pragma unroll
        for (int j = kVec - 1; j >= 0; --j) {
          const uint32_t key = key_at(w, j);
          const bool is_nan = key > (0x8000u | kInfBits<kBf16>) || key < 0x7fffu - kInfBits<kBf16>;
          if (j < n && (nan ? is_nan : merge_zero(key) == top_key)) first = min(first, i0 + j);
        }
      });
    } else if (tid < kVec) {
      const int i = index_of(top) + tid;
      if (i < vocab && (keys_of(x[i]) & 0xffffu) == top_key) first = i;
    }
    const uint64_t b = block_best(rank_of(1, first));
    if (tid == 0) {
      out[blockIdx.x] = index_of(b);
      cuts[blockIdx.x].ok = -1;
    }
    return;
  }
  const float mx = score_of(value_of<kBf16>(top_key), temp, rcp);
  // softmax of such a row has no probabilities
  if (nan || isinf(mx)) {
    if (tid == 0) {
      out[blockIdx.x] = 0;
      cuts[blockIdx.x].ok = 0;
    }
    return;
  }
  auto finish = [&]() __attribute__((always_inline)) {
    if (tid == 0)
      cuts[blockIdx.x] = {max(sh.kth, sh.cut), sh.cut, sh.last, 1, mx};
  };
  if (!filter) {
    finish();
    return;
  }
  // exp(score - max), in the exp2 domain. The logits are subtracted before they
  // are scaled: of score * log2(e) and max * log2(e) the roundings alone are
  // hundreds apart at a temperature of 1e-8, and one fma of the two would leave
  // infinite or no mass.
  const float slope = rcp * kLog2eS, top_value = value_of<kBf16>(top_key);
  auto mass_of = [&](uint32_t key) __attribute__((always_inline)) {
    return __builtin_amdgcn_exp2f((value_of<kBf16>(key) - top_value) * slope);
  };

  // `wide`: 32-bit counters of the keys of one half (bit 15 `held`) at a time.
  bool wide = false;
  int held = 1;
  auto build = [&](int half) __attribute__((always_inline)) {
    held = half;
    __syncthreads();
    for (int i = tid; i < kWords; i += kCutThreads) hist[i] = 0;
    __syncthreads();
    each([&](const u32x4 &w, int, int n) __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < kVec; ++j) {
        const uint32_t key = merge_zero(key_at(w, j));
        if (j < n && static_cast<int>(key >> 15) == half) atomicAdd(&hist[key & 0x7fff], 1u);
      }
    });
    __syncthreads();
  };
  // This thread's words, in an order that spreads a wave over the banks.
  constexpr int kSpan = kWords / kCutThreads;
  const int top_word = kWords - 1 - kSpan * tid;
  auto my_word = [&](int i) { return top_word - ((i + tid) & (kSpan - 1)); };
  // Keys and counts of a word: two in 16 bits, or one.
  auto key_of_word = [&](int w) { return wide ? held << 15 | w : 2 * w; };
  auto wave_scan = [&](auto v) __attribute__((always_inline)) {
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const auto u = __shfl_up(v, o);
      if (lane >= o) v += u;
    }
    return v;
  };
  // Counts above this thread's keys, and of all held keys after cnt0.
  uint32_t cnt, above;
  auto scan_counts = [&](uint32_t cnt0) __attribute__((always_inline)) {
    cnt = 0;
#pragma unroll 4
    for (int i = 0; i < kSpan; ++i) {
      const uint32_t c = hist[my_word(i)];
      cnt += wide ? c : (c >> 16) + (c & 0xffffu);
    }
    const uint32_t ci = wave_scan(cnt);
    __syncthreads();
    if (lane == 63) wave_cnt[wave] = ci;
    __syncthreads();
    uint32_t all = cnt0;
    above = cnt0 + ci - cnt;
    for (int w = 0; w < kCutWaves; ++w) {
      if (w < wave) above += wave_cnt[w];
      all += wave_cnt[w];
    }
    return all;
  };
  // The keys of lane `owner`'s words in descending order, one per lane of its
  // wave, with their counts.
  auto spread = [&](int owner, int &key, uint32_t &n) __attribute__((always_inline)) {
    const int w = __shfl(top_word, owner) - (wide ? lane & (kSpan - 1) : lane >> 1);
    const uint32_t c = hist[w];
    key = wide ? key_of_word(w) : 2 * w + 1 - (lane & 1);
    n = wide ? (lane < kSpan ? c : 0) : (key & 1 ? c >> 16 : c & 0xffffu);
  };
  auto find_kth = [&]() __attribute__((always_inline)) {
    const uint32_t k = static_cast<uint32_t>(row.k);
    const uint64_t owners = __ballot(above < k && k <= above + cnt);
    if (owners) {
      const int owner = __ffsll(static_cast<long long>(owners)) - 1;
      int key;
      uint32_t n;
      spread(owner, key, n);
      const uint32_t with = __shfl(above, owner) + wave_scan(n);
      if (with - n < k && k <= with) sh.kth = key;
    }
    __syncthreads();
  };
  // Masses of the kept keys above this thread's (and with them), after mass0.
  float mass_above, mass_with;
  auto scan_masses = [&](float mass0) __attribute__((always_inline)) {
    float s = 0.f;
    const int kth = sh.kth;
    if ((key_of_word(top_word) | 1) >= kth) {
#pragma unroll 1
      for (int i = 0; i < kSpan; ++i) {
        const int w = my_word(i);
        const uint32_t c = hist[w];
        const int key = key_of_word(w);
        if (wide) {
          if (c && key >= kth) s += c * mass_of(key);
        } else {
          if (c >> 16 && key + 1 >= kth) s += (c >> 16) * mass_of(key + 1);
          if ((c & 0xffffu) && key >= kth) s += (c & 0xffffu) * mass_of(key);
        }
      }
    }
    const float si = wave_scan(s);
    float se = __shfl_up(si, 1);  // the neighbour's own sum
    if (lane == 0) se = 0.f;
    __syncthreads();
    if (lane == 63) wave_mass[wave] = si;
    __syncthreads();
    float base = mass0, all = mass0;
    for (int w = 0; w < kCutWaves; ++w) {
      if (w < wave) base += wave_mass[w];
      all += wave_mass[w];
    }
    mass_above = base + se;
    mass_with = base + si;
    return all;
  };
  // A thread's range starts with the very sum its neighbour's ends with, so
  // some thread's straddles a target below the total; of several (the sums of
  // a scan need not grow) the first one is taken, and so for its keys.
  // Rounding can leave the keys' own sums short of the target: then it keeps
  // all of them.
  auto find_cut = [&](float target) __attribute__((always_inline)) {
    int my_cut = -1;
    uint32_t my_keep = 0, my_count = 0;
    const uint64_t owners = __ballot(mass_above <= target && target < mass_with);
    if (owners) {
      const int owner = __ffsll(static_cast<long long>(owners)) - 1;
      int key;
      uint32_t n;
      spread(owner, key, n);
      if (key < sh.kth) n = 0;
      const float e = n ? mass_of(key) : 0.f;
      const float base = __shfl(mass_above, owner);
      const float with = base + wave_scan(n * e);
      float before = __shfl_up(with, 1);
      if (lane == 0) before = base;
      const uint64_t at = __ballot(n && before <= target && target < with);
      const uint64_t some = __ballot(n != 0);
      const int pick = at ? __ffsll(static_cast<long long>(at)) - 1
                          : (some ? 63 - __clzll(static_cast<long long>(some)) : 0);
      if (lane == pick) {
        // logit j of the value stays if the mass before it is within the target
        const float over = (target - before) / e;
        my_cut = some ? key : key + 1;
        my_count = n;
        my_keep = at && over < static_cast<float>(n) ? min(n, static_cast<uint32_t>(over) + 1u) : n;
        atomicMax(&sh.cut, my_cut);
      }
    }
    __syncthreads();
    if (my_cut >= 0 && my_cut == sh.cut) {
      sh.cut_keep = my_keep;
      sh.cut_count = my_count;
    }
    __syncthreads();
  };

  // The two zeros become one value; then, did every counter hold its count?
  const uint32_t zeros = (hist[0x7fff >> 1] >> 16) + (hist[0x4000] & 0xffffu);
  __syncthreads();
  if (tid == 0 && zeros <= 0xffffu) {
    hist[0x4000] += hist[0x7fff >> 1] >> 16;
    hist[0x7fff >> 1] &= 0xffffu;
  }
  __syncthreads();
  uint32_t up_cnt = scan_counts(0);
  if (up_cnt != static_cast<uint32_t>(vocab) || zeros > 0xffffu) {
    wide = true;
    build(1);
    up_cnt = scan_counts(0);
  }
  if (use_k) {
    find_kth();
    if (wide && sh.kth < 0) {
      build(0);
      scan_counts(up_cnt);
      find_kth();
    }
  }
  if (use_p) {
    if (wide && !held) build(1);
    const float up_mass = scan_masses(0.f);
    float z = up_mass;
    if (wide && sh.kth < 0x8000) {
      build(0);
      z = scan_masses(up_mass);
    }
    const float target = row.p * z;
    if (wide && !held && target < up_mass) {
      build(1);
      scan_masses(0.f);
    }
    find_cut(target);
    if (sh.cut < 0) {  // the target is not reached: everything stays
      __syncthreads();
      if (tid == 0) sh.cut = 0;
      __syncthreads();
    }
  }
  // A value that the cut splits keeps its first logits by index: count it by
  // rounds, then find the last kept one in its round.
  if (sh.cut_keep < sh.cut_count) {
    const uint32_t cut = sh.cut;
    for (int i = tid; i < kMaxRounds; i += kCutThreads) tie_cnt[i] = 0;
    __syncthreads();
    each([&](const u32x4 &w, int i0, int n) __attribute__((always_inline)) {
      // a word with the cut's key in either half (or, rarely, beside it)
      uint32_t any = 0;
#pragma unroll
      for (int j = 0; j < kVec / 2; ++j) {
        const uint32_t d = w[j] ^ (cut * 0x10001u);
        any |= (d - 0x10001u) & ~d & 0x80008000u;
      }
      if (!any && cut != 0x8000u) return;
      uint32_t c = 0;
#pragma unroll
      for (int j = 0; j < kVec; ++j) c += j < n && merge_zero(key_at(w, j)) == cut;
      if (c) atomicAdd(&tie_cnt[i0 / kStep], c);
    });
    __syncthreads();
    uint32_t before = 0;
    int round = 0;
    while (before + tie_cnt[round] < sh.cut_keep) before += tie_cnt[round++];
    const uint32_t want = sh.cut_keep - before;  // the want-th of this round, from 1
    const int i0 = round * kStep + kVec * tid;
    auto is_cut = [&](int i) { return i < vocab && merge_zero(keys_of(x[i]) & 0xffffu) == cut; };
    uint32_t c = 0;
#pragma unroll 1
    for (int j = 0; j < kVec; ++j) c += is_cut(i0 + j);
    uint32_t ci = c;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t cu = __shfl_up(ci, o);
      if (lane >= o) ci += cu;
    }
    if (lane == 63) wave_cnt[wave] = ci;
    __syncthreads();
    for (int w = 0; w < wave; ++w) ci += wave_cnt[w];
    if (ci - c < want && want <= ci) {
      uint32_t at = ci - c;
#pragma unroll 1
      for (int j = 0; j < kVec; ++j)
        if (is_cut(i0 + j) && ++at == want) sh.last = i0 + j;
    }
    __syncthreads();
  }
  finish();
}

// Grid (shares of a row, rows): the best p / q of kDrawShare logits.
template <bool kBf16>
__global__ __launch_bounds__(kDrawThreads) void draw_kernel(
    const uint16_t *__restrict__ logits, int64_t ld, int vocab, SampleRows rows,
    const float *__restrict__ noise, const RowCut *__restrict__ cuts, uint64_t *__restrict__ bests) {
  __shared__ uint64_t best[kDrawThreads / 64];
  const SampleRow row = rows.r[blockIdx.y];
  if (row.temp == 0.f) return;
  const RowCut cut = cuts[blockIdx.y];
  if (cut.ok != 1) return;
  const uint16_t *x = logits + blockIdx.y * ld;
  const float *q = noise + static_cast<int64_t>(row.noise) * vocab;
  const float rcp = 1.0f / row.temp;
  const int i0 = blockIdx.x * kDrawShare + kVec * threadIdx.x;
  constexpr int kRound = kDrawThreads * kVec;

  u32x4 w[kAhead];
#pragma unroll
  for (int a = 0; a < kAhead; ++a) {
    const int i = i0 + a * kRound;
    if (i + kVec <= vocab) {
      __builtin_memcpy(&w[a], x + i, sizeof(w[a]));
    } else {
      w[a] = u32x4{0u, 0u, 0u, 0u};
#pragma unroll
      for (int j = 0; j < kVec; ++j)
        w[a][j >> 1] |= static_cast<uint32_t>(x[min(i + j, vocab - 1)]) << (16 * (j & 1));
    }
  }
  float r_best = -1.f;
  int i_best = vocab;
#pragma unroll
  for (int a = 0; a < kAhead; ++a) {
    const int i = i0 + a * kRound;
    uint32_t key[kVec];
    bool keep[kVec], any = false;
#pragma unroll
    for (int j = 0; j < kVec; ++j) {
      key[j] = merge_zero((keys_of(w[a][j >> 1]) >> (16 * (j & 1))) & 0xffffu);
      keep[j] = i + j < vocab && static_cast<int>(key[j]) >= cut.low &&
                !(static_cast<int>(key[j]) == cut.cut && i + j > cut.last);
      any = any || keep[j];
    }
    if (!any) continue;  // no noise is read for these
    float qv[kVec];
    if (i + kVec <= vocab) {
      __builtin_memcpy(qv, q + i, sizeof(qv));
    } else {
#pragma unroll
      for (int j = 0; j < kVec; ++j) qv[j] = q[min(i + j, vocab - 1)];
    }
#pragma unroll
    for (int j = 0; j < kVec; ++j) {
      const float s = score_of(value_of<kBf16>(key[j]), row.temp, rcp);
      const float p = exp2f((s - cut.max) * kLog2eS);  // up to the row's common factor
      const float r = p / qv[j];
      if (keep[j] && r > r_best) {
        r_best = r;
        i_best = i + j;
      }
    }
  }
  // r >= 0 orders as its bits; 0 marks "nothing kept"
  uint64_t b = wave_best(i_best < vocab ? rank_of(__float_as_uint(r_best) + 1u, i_best) : 0);
  if ((threadIdx.x & 63) == 0) best[threadIdx.x >> 6] = b;
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int v = 1; v < kDrawThreads / 64; ++v) b = best[v] > b ? best[v] : b;
    bests[blockIdx.y * gridDim.x + blockIdx.x] = b;
  }
}

// One wave per row; `valid` collects whether every row had a distribution
// (the first launch of a call sets it, the following ones only clear it).
__global__ __launch_bounds__(1024) void pick_kernel(int rows, int shares, bool first_rows,
                                                    const RowCut *__restrict__ cuts,
                                                    const uint64_t *__restrict__ bests,
                                                    int64_t *__restrict__ out,
                                                    uint8_t *__restrict__ valid) {
  const int lane = threadIdx.x & 63;
  bool bad = false;
  for (int r = threadIdx.x >> 6; r < rows; r += 16) {
    const int ok = cuts[r].ok;
    bad = bad || ok == 0;
    if (ok != 1) continue;
    uint64_t b = 0;
    for (int s = lane; s < shares; s += 64) {
      const uint64_t v = bests[r * shares + s];
      b = v > b ? v : b;
    }
    b = wave_best(b);
    if (lane == 0) out[r] = index_of(b);
  }
  const bool any_bad = __syncthreads_or(bad);
  if (threadIdx.x == 0 && valid != nullptr && (first_rows || any_bad)) *valid = !any_bad;
}

int64_t cut_bytes(int rows) { return (static_cast<int64_t>(rows) * sizeof(RowCut) + 255) / 256 * 256; }

}  // namespace
}  // namespace hy

extern "C" int64_t hy_sample_workspace_bytes(int32_t n_rows, int32_t vocab) {
  if (n_rows <= 0 || vocab <= 0) return 0;
  const int rows = n_rows < hy::kSampleRows ? n_rows : hy::kSampleRows;
  const int64_t shares = (static_cast<int64_t>(vocab) + hy::kDrawShare - 1) / hy::kDrawShare;
  return hy::cut_bytes(rows) + rows * shares * static_cast<int64_t>(sizeof(uint64_t));
}

extern "C" int hy_sample(const void *logits, int64_t row_stride, int32_t dtype, int32_t n_rows,
                         int32_t vocab, const float *temperature, const int32_t *top_k,
                         const float *top_p, const float *noise, int64_t *out, uint8_t *valid,
                         void *workspace, int64_t workspace_bytes, void *stream) {
  hy::clear_error();
  HY_REQUIRE(n_rows >= 0 && vocab >= 1, "hy_sample: invalid sizes %d x %d", n_rows, vocab);
  HY_REQUIRE(dtype == 0 || dtype == 1, "hy_sample: dtype %d (0: bf16, 1: fp16)", dtype);
  HY_REQUIRE_SUPPORTED(vocab <= hy::kStep * hy::kMaxRounds, "hy_sample: vocabulary %d too large",
                       vocab);
  if (n_rows == 0) return HY_OK;
  HY_REQUIRE(logits && temperature && top_k && top_p && out && workspace,
             "hy_sample: null pointer argument");
  if (workspace_bytes < hy_sample_workspace_bytes(n_rows, vocab)) {
    hy::set_error("hy_sample: workspace too small: need %lld bytes, got %lld",
                  static_cast<long long>(hy_sample_workspace_bytes(n_rows, vocab)),
                  static_cast<long long>(workspace_bytes));
    return HY_ENOSPACE;
  }
  int sampled = 0;
  for (int r = 0; r < n_rows; ++r) {
    const float t = temperature[r];
    if (t == 0.f) continue;
    HY_REQUIRE_SUPPORTED(t >= 1e-30f && t <= 1e30f, "hy_sample: temperature %g", t);
    HY_REQUIRE(top_k[r] >= 1 && top_p[r] > 0.f, "hy_sample: row %d has top_k %d, top_p %g", r,
               top_k[r], top_p[r]);
    ++sampled;
  }
  HY_REQUIRE(sampled == 0 || (noise && valid), "hy_sample: null pointer argument");
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int shares = (vocab + hy::kDrawShare - 1) / hy::kDrawShare;
  int noise_row = 0;
  for (int r0 = 0; r0 < n_rows; r0 += hy::kSampleRows) {
    const int n = n_rows - r0 < hy::kSampleRows ? n_rows - r0 : hy::kSampleRows;
    hy::SampleRows rows{};
    for (int i = 0; i < n; ++i) {
      const float t = temperature[r0 + i];
      rows.r[i] = {t, top_k[r0 + i] < vocab ? top_k[r0 + i] : vocab, top_p[r0 + i],
                   t == 0.f ? 0 : noise_row++};
    }
    const uint16_t *x = static_cast<const uint16_t *>(logits) + r0 * row_stride;
    auto *cuts = static_cast<hy::RowCut *>(workspace);
    auto *bests = reinterpret_cast<uint64_t *>(static_cast<char *>(workspace) + hy::cut_bytes(n));
    auto cut = dtype == 0 ? hy::cut_kernel<true> : hy::cut_kernel<false>;
    auto draw = dtype == 0 ? hy::draw_kernel<true> : hy::draw_kernel<false>;
    hipLaunchKernelGGL(cut, dim3(n), dim3(hy::kCutThreads), 0, st, x, row_stride, vocab, rows,
                       out + r0, cuts);
    if (sampled == 0) continue;
    hipLaunchKernelGGL(draw, dim3(shares, n), dim3(hy::kDrawThreads), 0, st, x, row_stride, vocab,
                       rows, noise, cuts, bests);
    hipLaunchKernelGGL(hy::pick_kernel, dim3(1), dim3(1024), 0, st, n, shares, r0 == 0, cuts,
                       bests, out + r0, valid);
  }
  return hy::launch_status("hy_sample");
}
