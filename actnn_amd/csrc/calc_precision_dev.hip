// Per-sample sensitivities and the greedy per-sample bit allocation on the device, for the case the
// layers use at every step: all items start at the same width and have unit weight (replaces the host
// round trip around calc_precision.cc:9-50 in QScheme.compute_quantization_bits,
// actnn/actnn/qscheme.py:80-94).
//
// The reference pops, K = N * initial - target times, the largest (delta, index) pair of a
// priority queue and pushes the popped item's next step.  The steps of one item get strictly more
// expensive (delta more negative) as its width shrinks - or stay equal when C is 0 - so the popped
// set is exactly the K largest of all N * (initial - 1) candidate steps under the order
// (delta, index, earlier step first).  One block finds the delta of the K-th of them by radix selection
// - 11, 11 and 10 bits of the deltas' ordered bit patterns, a histogram in LDS each - gives every item
// the steps above it, hands the steps equal to it to the items of the largest index, and scans the
// widths for the offsets of the packed stream while it holds them.
//
// What bounds it: not memory but the chain of block barriers (about twenty) and, from some thousand
// items on, the LDS atomics of the histograms.  The candidates are walked so that the lanes of a wave
// hold different steps of neighbouring items: the exponents of an item's steps lie two apart, so few
// lanes of an atomic meet in one bin.
#include "bn_finalize.h"
#include "device_utils.h"

namespace actnn {
namespace {

constexpr int kThreads = 256;
constexpr int kMaxCand = 8192;                       // actnn_calc_precision_device's limit
constexpr int64_t kMaxAllocated = int64_t(1) << 20;  // candidates actnn_allocate_bits_device takes

// ---------------------------------------------------------------------------- sensitivities
// factor * mult * sum_g (mx[n,g] - mn[n,g])^2 (the difference rounded to T, as the tensor subtraction
// of qscheme.py:80 rounds it).  The order of the fp32 additions is fixed whatever the kernel: 256
// running sums, sum t over the groups t, t + 256, ..., folded in halves.  mult: nothing, one device
// scalar or one value per sample.
template <typename T> ACTNN_DEV float range_term(const T* mn, const T* mx, int64_t i) {
  return Conv<T>::round(Conv<T>::load(mx, i) - Conv<T>::load(mn, i));
}
ACTNN_DEV float finish_sensitivity(float sum, float factor, const float* mult, int mult_stride, int64_t n) {
  const float v = sum * factor;
  return mult ? v * mult[n * mult_stride] : v;
}

// One block per sample: few samples of many groups.  The running sums are chains of additions, but their terms
// are loaded kAhead at a time: with one load per turn the pass was the latency of G / 256 loads in a row
// (2 samples of 158080 groups in fp16: 171 us, 23.6 now; 3 of 21576 in bf16: 24.5 and 6.2 us).
template <typename T>
ACTNN_DEV void range_sqr_of_block(const T* __restrict__ mn, const T* __restrict__ mx, float* __restrict__ out, int64_t n, int64_t G,
                                  float factor, const float* __restrict__ mult, int mult_stride) {
  __shared__ float s_part[kThreads];
  float acc = 0.0f;
  constexpr int kAhead = 16;
  for (int64_t g0 = threadIdx.x; g0 < G; g0 += kThreads * kAhead) {
    float d[kAhead];
#pragma unroll
    for (int j = 0; j < kAhead; ++j) {
      const int64_t g = g0 + j * kThreads < G ? g0 + j * kThreads : g0;      // (a valid address; dropped below)
      d[j] = range_term(mn, mx, n * G + g);
    }
#pragma unroll
    for (int j = 0; j < kAhead; ++j)
      if (g0 + j * kThreads < G) acc = fmaf(d[j], d[j], acc);
  }
  s_part[threadIdx.x] = acc;
  __syncthreads();
  for (int w = kThreads / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) s_part[threadIdx.x] += s_part[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[n] = finish_sensitivity(s_part[0], factor, mult, mult_stride, n);
}
template <typename T>
__global__ __launch_bounds__(kThreads) void range_sqr_kernel(const T* __restrict__ mn,
                                                             const T* __restrict__ mx,
                                                             float* __restrict__ out, int64_t G,
                                                             float factor, const float* __restrict__ mult,
                                                             int mult_stride) {
  range_sqr_of_block(mn, mx, out, (int64_t)blockIdx.x, G, factor, mult, mult_stride);
}

// The same sum by one wave, lane l holding the running sums l, l + 64, l + 128 and l + 192: valid in lane 0.
template <typename T> ACTNN_DEV float range_sqr_of_wave(const T* __restrict__ mn, const T* __restrict__ mx, int64_t first, int64_t G) {
  const int lane = threadIdx.x & 63;
  float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int64_t g0 = lane; g0 < G; g0 += 256) {
    float d[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) d[j] = g0 + 64 * j < G ? range_term(mn, mx, first + g0 + 64 * j) : 0.0f;
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[j] = fmaf(d[j], d[j], acc[j]);
  }
  float v = (acc[0] + acc[2]) + (acc[1] + acc[3]);
#pragma unroll
  for (int w = 32; w > 0; w >>= 1) v += __shfl_down(v, w);
  return v;
}

// One wave per sample: many samples of few groups (8192 samples of 16: 7.6 us with a block each).
constexpr int64_t kWaveGroups = 512;
template <typename T>
__global__ __launch_bounds__(kThreads) void range_sqr_wave_kernel(const T* __restrict__ mn,
                                                                  const T* __restrict__ mx,
                                                                  float* __restrict__ out, int64_t N, int64_t G,
                                                                  float factor, const float* __restrict__ mult,
                                                                  int mult_stride) {
  const int64_t n = (int64_t)blockIdx.x * (kThreads / 64) + (threadIdx.x >> 6);
  if (n >= N) return;
  const float v = range_sqr_of_wave(mn, mx, n * G, G);
  if ((threadIdx.x & 63) == 0) out[n] = finish_sensitivity(v, factor, mult, mult_stride, n);
}

// Either kernel in the first sample_blocks blocks; the others fold batch norm's partial sums, a wave per channel.  The two do not
// wait for each other, and each is a few microseconds of latency: bf16 [256, 512, 28, 28] 6.2 + 4.7 us one after the other,
// 7.3 side by side (the widths could come from the same launch, made by the block that is the last to arrive: 14.6 us for the three,
// and 9.0 for the two of bf16 [32, 64, 56, 56], where two launches take 6.6).
template <typename T, bool WAVES>
__global__ __launch_bounds__(kThreads) void range_sqr_and_fold_kernel(const T* __restrict__ mn, const T* __restrict__ mx,
                                                                      float* __restrict__ out, int64_t N, int64_t G, float factor,
                                                                      const float* __restrict__ mult, int mult_stride,
                                                                      unsigned sample_blocks, BnFinalize fold) {
  const int wave = threadIdx.x >> 6;
  if (blockIdx.x >= sample_blocks) {
    const int64_t c = (int64_t)(blockIdx.x - sample_blocks) * (kThreads / 64) + wave;
    if (c < fold.C) bn_finalize_channel(fold, c);
  } else if constexpr (WAVES) {
    const int64_t n = (int64_t)blockIdx.x * (kThreads / 64) + wave;
    if (n >= N) return;
    const float v = range_sqr_of_wave(mn, mx, n * G, G);
    if ((threadIdx.x & 63) == 0) out[n] = finish_sensitivity(v, factor, mult, mult_stride, n);
  } else {
    range_sqr_of_block(mn, mx, out, (int64_t)blockIdx.x, G, factor, mult, mult_stride);
  }
}

template <typename T>
int launch_range_sqr_and_fold(const void* mn, const void* mx, float* out, int64_t N, int64_t G, float factor, const float* mult,
                              int stride, const BnFinalize& fold, hipStream_t s) {
  const T* lo = static_cast<const T*>(mn);
  const T* hi = static_cast<const T*>(mx);
  const bool waves = G <= kWaveGroups;
  const int64_t blocks = waves ? (N + 3) / 4 : N, folds = (fold.C + kThreads / 64 - 1) / (kThreads / 64);
  if (blocks + folds > 0x7fffffffLL) return ACTNN_EINVAL;
  const dim3 grid((unsigned)(blocks + folds)), blk(kThreads);
  if (waves) range_sqr_and_fold_kernel<T, true><<<grid, blk, 0, s>>>(lo, hi, out, N, G, factor, mult, stride, (unsigned)blocks, fold);
  else range_sqr_and_fold_kernel<T, false><<<grid, blk, 0, s>>>(lo, hi, out, N, G, factor, mult, stride, (unsigned)blocks, fold);
  ACTNN_RETURN_LAUNCH_STATUS();
}

template <typename T>
int launch_range_sqr(const void* mn, const void* mx, float* out, int64_t N, int64_t G, float factor, const float* mult,
                     int stride, hipStream_t s) {
  const T* lo = static_cast<const T*>(mn);
  const T* hi = static_cast<const T*>(mx);
  if (G <= kWaveGroups)
    range_sqr_wave_kernel<T><<<dim3((unsigned)((N + 3) / 4)), dim3(kThreads), 0, s>>>(lo, hi, out, N, G, factor, mult, stride);
  else
    range_sqr_kernel<T><<<dim3((unsigned)N), dim3(kThreads), 0, s>>>(lo, hi, out, G, factor, mult, stride);
  ACTNN_RETURN_LAUNCH_STATUS();
}

// ---------------------------------------------------------------------------- allocation
constexpr int kBins = 2048;
constexpr int kLdsItems = 16384;                     // sensitivities kept in LDS (64 KiB)

// 1/(2^b - 1)^2 - 1/(2^(b-1) - 1)^2: what the step from b to b - 1 bits multiplies the sensitivity with
constexpr double step_factor(int b) {
  const double full = (double)((1 << b) - 1), less = (double)((1 << (b - 1)) - 1);
  return 1.0 / (full * full) - 1.0 / (less * less);
}
__constant__ const double kStepFactor[9] = {0.0, 0.0, step_factor(2), step_factor(3), step_factor(4),
                                            step_factor(5), step_factor(6), step_factor(7), step_factor(8)};

// Order-preserving bit pattern of the cost of a step: larger = popped earlier.
ACTNN_DEV uint32_t step_order(float C, double factor) {
  float d = (float)((double)C * factor);               // calc_precision.cc:24-28, weight 1
  if (d == 0.0f) d = -0.0f;                            // one representation for "no cost"
  const uint32_t u = as_uint(d);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);   // monotone in the float order
}

// Inclusive sum over the lanes of the wave, the lane exchange inside the additions (row shifts, then
// the last lane of each row of 16 into the rows behind it).
ACTNN_DEV uint32_t wave_scan(uint32_t v) {
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false);     // row_shr:1
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, false);     // row_shr:2
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, false);     // row_shr:4
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, false);     // row_shr:8
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false);     // row_bcast:15 into rows 1, 3
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false);     // row_bcast:31 into rows 2, 3
  return v;
}

// Inclusive sum of v over the threads of the block; `total` receives the sum of all.  s_wave: a word
// of LDS per wave, free again after the caller's next barrier.
template <int THREADS> ACTNN_DEV uint32_t block_scan(uint32_t v, uint32_t* s_wave, uint32_t& total) {
  const int wave = threadIdx.x >> 6;
  v = wave_scan(v);
  if ((threadIdx.x & 63) == 63) s_wave[wave] = v;
  __syncthreads();
  uint32_t before = 0, sum = 0;
#pragma unroll
  for (int w = 0; w < THREADS / 64; ++w) {
    const uint32_t t = s_wave[w];
    before += w < wave ? t : 0u;
    sum += t;
  }
  total = sum;
  return before + v;
}

// KEYS > 0: the patterns of a thread's candidates (at most KEYS) stay in registers over the passes; 0:
// evaluated anew in each.
template <int THREADS, int KEYS>
__global__ __launch_bounds__(THREADS) void allocate_kernel(const float* __restrict__ sens, int32_t* __restrict__ bits,
                                                           int32_t* __restrict__ prefix, int N, int initial,
                                                           int64_t K) {
  constexpr int kPer = kBins / THREADS;                // bins a thread scans
  constexpr int kItems = KEYS > 0 ? THREADS * KEYS : kLdsItems;
  __shared__ double factors[8];
  __shared__ float C_s[kItems];
  __shared__ uint32_t hist[kBins];
  __shared__ uint32_t s_wave[THREADS / 64];
  __shared__ uint32_t s_digit, s_above, s_inside;
  const int L = initial - 1;
  const int total = N * L;
  const bool in_lds = N <= kItems;
  const bool select = K > 0 && K < total;              // otherwise nothing or everything is taken
  if (in_lds && select)
    for (int n = threadIdx.x; n < N; n += THREADS) C_s[n] = sens[n];
  if ((int)threadIdx.x < L) factors[threadIdx.x] = kStepFactor[initial - (int)threadIdx.x];
  // taken are the steps above `cut`, and the first `left` of those equal to it
  uint32_t cut = 0, left = 0;
  if (select) {
    left = (uint32_t)K;
    const int i0 = (int)threadIdx.x / L, l0 = (int)threadIdx.x - i0 * L;
    const int di = THREADS / L, dl = THREADS - di * L;
    uint32_t key[KEYS > 0 ? KEYS : 1];
#pragma unroll 1
    for (int pass = 0; pass < 3; ++pass) {
      const int shift = pass == 0 ? 21 : pass == 1 ? 10 : 0, width = pass == 2 ? 10 : 11;
      const uint32_t last = (1u << width) - 1u;
#pragma unroll
      for (int k = 0; k < kPer; ++k) hist[k * THREADS + threadIdx.x] = 0;
      __syncthreads();
      // (the dearest steps in the last bin; a shift by 32 is what pass 0 would ask for)
      auto count = [&](uint32_t o) {
        if (pass == 0 || (o >> (shift + width)) == cut) atomicAdd(&hist[last - ((o >> shift) & last)], 1u);
      };
      if (KEYS > 0) {
        if (pass == 0) {
          int i = i0, l = l0;
#pragma unroll
          for (int k = 0; k < KEYS; ++k) {
            if ((int)threadIdx.x + k * THREADS < total) key[k] = step_order(C_s[i], factors[l]);
            i += di;
            l += dl;
            if (l >= L) { l -= L; ++i; }
          }
        }
#pragma unroll
        for (int k = 0; k < KEYS; ++k)
          if ((int)threadIdx.x + k * THREADS < total) count(key[k]);
      } else {
        int i = i0, l = l0;
        for (int c = threadIdx.x; c < total; c += THREADS) {
          count(step_order(in_lds ? C_s[i] : sens[i], factors[l]));
          i += di;
          l += dl;
          if (l >= L) { l -= L; ++i; }
        }
      }
      __syncthreads();
      uint32_t h[kPer], mine = 0;
#pragma unroll
      for (int k = 0; k < kPer; ++k) {
        h[k] = hist[threadIdx.x * kPer + k];
        mine += h[k];
      }
      uint32_t all;
      uint32_t before = block_scan<THREADS>(mine, s_wave, all) - mine;
      if (before < left && left <= before + mine) {    // one thread: the step sought lies in one of its bins
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
          if (before < left && left <= before + h[k]) {
            s_digit = last - (threadIdx.x * kPer + k);
            s_above = before;
            s_inside = h[k];
            before = left;                             // found: it only grows from here, so no later bin compares
          } else {
            before += h[k];
          }
        }
      }
      __syncthreads();
      cut = (cut << width) | s_digit;
      left -= s_above;
      if (left == s_inside) {                          // the whole bin is taken: its lower end is the cut
        cut = (cut << shift) - 1u;                     // (no step has the pattern 0: that is a NaN's)
        left = 0;
        break;
      }
    }
  }
  __syncthreads();
  // A thread owns a run of items.  Steps of exactly the cost `cut` of which not all are taken go to
  // the items of the largest index.
  const int per = (N + THREADS - 1) / THREADS;
  const int lo = (int)threadIdx.x * per < N ? (int)threadIdx.x * per : N;
  const int hi = lo + per < N ? lo + per : N;
  if (left > 0) {                                      // (the same for all threads)
    uint32_t tied = 0;
    for (int n = lo; n < hi; ++n) {
      const float c = in_lds ? C_s[n] : sens[n];
      for (int l = 0; l < L; ++l) tied += step_order(c, factors[l]) == cut ? 1u : 0u;
    }
    uint32_t all;
    const uint32_t upto = block_scan<THREADS>(tied, s_wave, all);
    left = left > all - upto ? left - (all - upto) : 0u;   // minus those of the threads behind this one
    __syncthreads();
  }
  uint32_t sum = 0;
  for (int n = hi - 1; n >= lo; --n) {
    int b = K <= 0 ? initial : 1;
    if (select) {
      const float c = in_lds ? C_s[n] : sens[n];
      uint32_t above = 0, equal = 0;
      for (int l = 0; l < L; ++l) {
        const uint32_t o = step_order(c, factors[l]);
        above += o > cut ? 1u : 0u;
        equal += o == cut ? 1u : 0u;
      }
      const uint32_t taken = equal < left ? equal : left;
      left -= taken;
      b = initial - (int)(above + taken);
    }
    bits[n] = b;
    sum += (uint32_t)b;
  }
  if (prefix) {                                        // exclusive prefix of the widths
    uint32_t all;
    uint32_t at = block_scan<THREADS>(sum, s_wave, all) - sum;
    if (threadIdx.x == 0) prefix[N] = (int32_t)all;
    for (int n = lo; n < hi; ++n) {
      prefix[n] = (int32_t)at;
      at += (uint32_t)bits[n];                         // (written by this thread above)
    }
  }
}

// Thousands of items: a thread owns the items t, t + 1024, ... and all their steps in registers, so that the
// patterns - a double product each, what the one-block kernel is bound by - are evaluated once, the widths
// are counts over registers, and every access to memory is coalesced (the widths change over to runs of
// consecutive items through LDS).  A lane starts with the step its number says, so that the lanes of a
// histogram atomic hold different steps, as above.  Items of like sensitivities, whose steps of one kind share a bin, can
// count in several histograms by their lanes, which all have to be cleared and added up: four for 4097 items and more, one for
// fewer.  us with the sensitivities' pass in front, one / four histograms, for equal sensitivities at 1.5 bits on average, for
// sensitivities within a few percent, and for ones e^(z/2) and e^(4 z) apart (z normal), at 2 bits: 1171 items 12.7 / 12.0,
// 8.4 / 8.2, 9.2 / 9.4, 9.3 / 9.5; 2048 14.8 / 14.0, 9.3 / 9.3, 10.0 / 10.3, 10.0 / 10.3; 4096 24.0 / 21.8, 14.1 / 13.7, 14.9 / 15.1,
// 14.8 / 15.2; 4097 30.1 / 27.3, 18.6 / 18.1, 20.4 / 20.6, 23.0 / 23.2; 6000 37.0 / 33.1, 22.3 / 21.6, 23.8 / 23.9, 23.5 / 23.7;
// 8192 45.1 / 39.9, 27.3 / 25.8, 27.6 / 27.6, 27.4 / 27.6: the larger the batch, the more the like ones gain and the less the others lose.
template <int ITEMS>
__global__ __launch_bounds__(1024) void allocate_many_kernel(const float* __restrict__ sens, int32_t* __restrict__ bits,
                                                             int32_t* __restrict__ prefix, int N, int initial,
                                                             int64_t K) {
  constexpr int kN = 1024, kSteps = 7;
  constexpr int kPer = kBins / kN, kCopies = ITEMS > 4 ? 4 : 1;
  __shared__ double factors[8];
  __shared__ uint32_t hist[kCopies][kBins];
  __shared__ uint32_t s_wave[kN / 64];
  __shared__ uint32_t s_digit, s_above, s_inside;
  __shared__ __align__(16) uint8_t s_width[kN * ITEMS];
  const int t = threadIdx.x;
  const int L = initial - 1;
  const bool select = K > 0 && K < (int64_t)N * L;     // otherwise nothing or everything is taken
  uint32_t cut = 0, left = 0;
  uint32_t key[ITEMS][kSteps];
  if (select) {
    float C[ITEMS];
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) C[k] = t + k * kN < N ? sens[t + k * kN] : 0.0f;
    if (t < L) factors[t] = kStepFactor[initial - t];
#pragma unroll
    for (int k = 0; k < kCopies * kPer; ++k) (&hist[0][0])[k * kN + t] = 0;
    __syncthreads();
    uint32_t* const my_hist = hist[(t >> 3) & (kCopies - 1)];      // (lanes of one step lie 7 apart)
    int l = t % L;
#pragma unroll
    for (int j = 0; j < kSteps; ++j) {
      if (j < L) {
        const double f = factors[l];
#pragma unroll
        for (int k = 0; k < ITEMS; ++k) key[k][j] = step_order(C[k], f);
      }
      l = l + 1 == L ? 0 : l + 1;
    }
    left = (uint32_t)K;
#pragma unroll 1
    for (int pass = 0; pass < 3; ++pass) {
      const int shift = pass == 0 ? 21 : pass == 1 ? 10 : 0, width = pass == 2 ? 10 : 11;
      const uint32_t last = (1u << width) - 1u;
      if (pass > 0) {
#pragma unroll
        for (int k = 0; k < kCopies * kPer; ++k) (&hist[0][0])[k * kN + t] = 0;
        __syncthreads();
      }
#pragma unroll
      for (int j = 0; j < kSteps; ++j) {
        if (j < L) {
#pragma unroll
          for (int k = 0; k < ITEMS; ++k) {
            const uint32_t o = key[k][j];
            // (the dearest steps in the last bin; a shift by 32 is what pass 0 would ask for)
            if (t + k * kN < N && (pass == 0 || (o >> (shift + width)) == cut)) atomicAdd(&my_hist[last - ((o >> shift) & last)], 1u);
          }
        }
      }
      __syncthreads();
      uint32_t h[kPer], mine = 0;
#pragma unroll
      for (int k = 0; k < kPer; ++k) {
        h[k] = 0;
#pragma unroll
        for (int c = 0; c < kCopies; ++c) h[k] += hist[c][t * kPer + k];
        mine += h[k];
      }
      uint32_t all;
      uint32_t before = block_scan<kN>(mine, s_wave, all) - mine;
      if (before < left && left <= before + mine) {    // one thread: the step sought lies in one of its bins
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
          if (before < left && left <= before + h[k]) {
            s_digit = last - (t * kPer + k);
            s_above = before;
            s_inside = h[k];
            before = left;                             // found: it only grows from here, so no later bin compares
          } else {
            before += h[k];
          }
        }
      }
      __syncthreads();
      cut = (cut << width) | s_digit;
      left -= s_above;
      if (left == s_inside) {                          // the whole bin is taken: its lower end is the cut
        cut = (cut << shift) - 1u;                     // (no step has the pattern 0: that is a NaN's)
        left = 0;
        break;
      }
    }
  }
  uint32_t behind = 0;                                 // steps of the cost `cut` that items further back hold
#pragma unroll
  for (int k = ITEMS - 1; k >= 0; --k) {
    int b = K <= 0 ? initial : 1;
    if (select) {
      uint32_t above = 0, equal = 0;
      const bool live = t + k * kN < N;
#pragma unroll
      for (int j = 0; j < kSteps; ++j) {
        if (j < L && live) {
          above += key[k][j] > cut ? 1u : 0u;
          equal += key[k][j] == cut ? 1u : 0u;
        }
      }
      uint32_t taken = 0;
      if (left > 0) {                                  // (the same for all threads) not all of them are taken
        __syncthreads();
        uint32_t all;
        const uint32_t upto = block_scan<kN>(equal, s_wave, all);
        const uint32_t later = behind + (all - upto);
        const uint32_t room = left > later ? left - later : 0u;
        taken = equal < room ? equal : room;
        behind += all;
      }
      b = initial - (int)(above + taken);
    }
    s_width[t + k * kN] = (uint8_t)b;
  }
  __syncthreads();
  // widths and their exclusive prefix, a run of ITEMS consecutive items per thread
  int w[ITEMS];
  uint32_t sum = 0;
#pragma unroll
  for (int k = 0; k < ITEMS; ++k) {
    w[k] = t * ITEMS + k < N ? (int)s_width[t * ITEMS + k] : 0;
    sum += (uint32_t)w[k];
  }
  uint32_t all;
  uint32_t at = block_scan<kN>(sum, s_wave, all) - sum;
#pragma unroll
  for (int k = 0; k < ITEMS; ++k) {
    if (t * ITEMS + k < N) {
      bits[t * ITEMS + k] = w[k];
      if (prefix) prefix[t * ITEMS + k] = (int32_t)at;
      at += (uint32_t)w[k];
    }
  }
  if (prefix && t == 0) prefix[N] = (int32_t)all;
}

// As many threads as have work, and their candidates in registers while they fit.  Measured (bf16, start
// width 8): 64 items 4.2 us, 128 items 4.6 us with 256 threads; 256 items 5.2 us, 512 items 5.6 us (9.3 us
// with 256 threads), 1100 items 7.3 us with 1024; more items: see allocate_many_kernel, up to the 8192 whose
// steps fit the registers of one block.  Beyond those the patterns are evaluated anew in each pass: with the
// sensitivities' pass in front 9362 items take 35.7 us (47.2 with 64 patterns a thread in registers,
// which spill), 16384 items 66 us, from memory 131072 items 694 us; the host routine needs 143, 230 and
// 1610 us and the GPU waits for it.  Ranking every candidate against every other by a grid of blocks, and
// scanning the widths in a launch of its own, took 6.5 + 2.8 us at 32 items, 7.7 + 5.3 us at 256, and
// stopped at 8192 candidates.
int launch_allocate(const float* sens, int32_t* bits, int32_t* prefix, int64_t N, int initial, int64_t target,
                    hipStream_t s) {
  const int64_t K = N * initial - target, candidates = N * (initial > 1 ? initial - 1 : 1);
  if (candidates <= 256 * 4) allocate_kernel<256, 4><<<dim3(1), dim3(256), 0, s>>>(sens, bits, prefix, (int)N, initial, K);
  else if (candidates <= 1024 * 8) allocate_kernel<1024, 8><<<dim3(1), dim3(1024), 0, s>>>(sens, bits, prefix, (int)N, initial, K);
  else if (N <= 2048) allocate_many_kernel<2><<<dim3(1), dim3(1024), 0, s>>>(sens, bits, prefix, (int)N, initial, K);
  else if (N <= 4096) allocate_many_kernel<4><<<dim3(1), dim3(1024), 0, s>>>(sens, bits, prefix, (int)N, initial, K);
  else if (N <= 8192) allocate_many_kernel<8><<<dim3(1), dim3(1024), 0, s>>>(sens, bits, prefix, (int)N, initial, K);
  else allocate_kernel<1024, 0><<<dim3(1), dim3(1024), 0, s>>>(sens, bits, prefix, (int)N, initial, K);
  ACTNN_RETURN_LAUNCH_STATUS();
}

}  // namespace
}  // namespace actnn

extern "C" int actnn_range_sqr(const void* mn, const void* mx, float* out, int64_t N, int64_t G,
                               float factor, const float* mult, int mult_per_sample, int dtype,
                               void* stream) {
  using namespace actnn;
  if (N < 0 || G < 0 || N > 0x7fffffffLL) return ACTNN_EINVAL;
  if (N == 0) return ACTNN_OK;
  if (!out || (G > 0 && (!mn || !mx))) return ACTNN_EINVAL;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int stride = mult_per_sample ? 1 : 0;
  switch (dtype) {
    case ACTNN_F32: return launch_range_sqr<float>(mn, mx, out, N, G, factor, mult, stride, s);
    case ACTNN_F16: return launch_range_sqr<__half>(mn, mx, out, N, G, factor, mult, stride, s);
    case ACTNN_BF16: return launch_range_sqr<bf16_t>(mn, mx, out, N, G, factor, mult, stride, s);
    default: return ACTNN_EDTYPE;
  }
}

extern "C" int actnn_calc_precision_device(const float* C, int32_t* bits, int64_t N, int initial_bits,
                                           int64_t target, void* stream) {
  using namespace actnn;
  if (N < 0) return ACTNN_EINVAL;
  if (N == 0) return ACTNN_OK;
  if (!C || !bits) return ACTNN_EINVAL;
  if (initial_bits < 1 || initial_bits > 8) return ACTNN_EBITS;
  if (N * (initial_bits - 1) > kMaxCand) return ACTNN_EINVAL;           // larger batches take the host routine
  return launch_allocate(C, bits, nullptr, N, initial_bits, target, static_cast<hipStream_t>(stream));
}

namespace actnn {
// actnn_allocate_bits_device; with `fold`, batch norm's partial sums are folded beside the sensitivities.  (N > 0 then.)
int allocate_bits(const void* mn, const void* mx, float factor, const float* mult, int mult_per_sample, float* sensitivity, int32_t* bits,
                  int32_t* prefix, int64_t N, int64_t G, int initial_bits, int64_t target, int dtype, const BnFinalize* fold,
                  hipStream_t s) {
  if (N < 0 || G < 0 || (dtype != ACTNN_F32 && dtype != ACTNN_F16 && dtype != ACTNN_BF16))
    return N < 0 || G < 0 ? ACTNN_EINVAL : ACTNN_EDTYPE;
  if (initial_bits < 1 || initial_bits > 8) return ACTNN_EBITS;
  if (N > kMaxAllocated || N * (initial_bits - 1) > kMaxAllocated) return ACTNN_EINVAL;
  if (!prefix || (N > 0 && (!sensitivity || !bits || (G > 0 && (!mn || !mx))))) return ACTNN_EINVAL;
  if (N > 0) {
    const int stride = mult_per_sample ? 1 : 0;
    const int rc = !fold ? actnn_range_sqr(mn, mx, sensitivity, N, G, factor, mult, mult_per_sample, dtype, s)
                   : dtype == ACTNN_F32 ? launch_range_sqr_and_fold<float>(mn, mx, sensitivity, N, G, factor, mult, stride, *fold, s)
                   : dtype == ACTNN_F16 ? launch_range_sqr_and_fold<__half>(mn, mx, sensitivity, N, G, factor, mult, stride, *fold, s)
                                        : launch_range_sqr_and_fold<bf16_t>(mn, mx, sensitivity, N, G, factor, mult, stride, *fold, s);
    if (rc != ACTNN_OK) return rc;
  }
  return launch_allocate(sensitivity, bits, prefix, N, initial_bits, target, s);
}
}  // namespace actnn

extern "C" int actnn_allocate_bits_device(const void* mn, const void* mx, float factor, const float* mult,
                                          int mult_per_sample, float* sensitivity, int32_t* bits,
                                          int32_t* prefix, int64_t N, int64_t G, int initial_bits,
                                          int64_t target, int dtype, void* stream) {
  return actnn::allocate_bits(mn, mx, factor, mult, mult_per_sample, sensitivity, bits, prefix, N, G, initial_bits, target, dtype, nullptr,
                              static_cast<hipStream_t>(stream));
}
