// Per-row min/max (replaces minimax_cuda_kernel.cu:23-89 of the reference).
//
// HBM-bound streaming read.  A row of D elements is reduced by 16, 32 or 64 lanes so that each
// load instruction of a block covers 4 KiB of consecutive memory (one 16-byte non-temporal
// load per lane; a 256-element fp32 row is exactly one wave-wide load).  Lanes are combined
// with DPP steps (quad_perm, row mirrors, row broadcasts).  Small blocks that each sweep a
// short contiguous run measured faster on MI355X than blocks with many loads in flight per lane;
// eight rows per lane group (32 KiB per block for fp32 rows of 256) measured best.
#include "device_utils.h"

namespace actnn {
namespace {

constexpr int kThreads = 256;
constexpr int kRowGroups = kThreads / 16;     // rows per block in the generic kernel

constexpr int kRowsPerLaneGroup = 8;          // rows per lane group and block (8 measured best)

template <typename T> struct Vec16;           // running min/max over one 16-byte vector of T
template <> struct Vec16<float> {
  static constexpr int kElems = 4;
  static ACTNN_DEV void minmax(const float* p, float& lo, float& hi) { minmax(load16_nt(p), lo, hi); }
  static ACTNN_DEV void minmax(u32x4 u, float& lo, float& hi) {
    const float a = as_float(u.x), b = as_float(u.y), c = as_float(u.z), d = as_float(u.w);
    lo = min3_f32(min3_f32(lo, a, b), c, d);
    hi = max3_f32(max3_f32(hi, a, b), c, d);
  }
};
template <> struct Vec16<__half> {
  static constexpr int kElems = 8;
  static ACTNN_DEV void minmax(const __half* p, float& lo, float& hi) { minmax(load16_nt(p), lo, hi); }
  static ACTNN_DEV void minmax(u32x4 u, float& lo, float& hi) {
    const uint32_t w[4] = {u.x, u.y, u.z, u.w};
    float v[8];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[2 * i] = half_bits_to_float(w[i] & 0xffffu);
      v[2 * i + 1] = half_bits_to_float(w[i] >> 16);
    }
    float l8, h8;
    minmax_of<8>(v, l8, h8);
    lo = min_f32(lo, l8);
    hi = max_f32(hi, h8);
  }
};
template <> struct Vec16<bf16_t> {
  static constexpr int kElems = 8;
  static ACTNN_DEV void minmax(const bf16_t* p, float& lo, float& hi) { minmax(load16_nt(p), lo, hi); }
  static ACTNN_DEV void minmax(u32x4 u, float& lo, float& hi) {
    const uint32_t w[4] = {u.x, u.y, u.z, u.w};
    float v[8];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[2 * i] = as_float(w[i] << 16);
      v[2 * i + 1] = as_float(w[i] & 0xffff0000u);
    }
    float l8, h8;
    minmax_of<8>(v, l8, h8);
    lo = min_f32(lo, l8);
    hi = max_f32(hi, h8);
  }
};

// Vector path: a row is D = LPR * kElems * V elements, read by LPR lanes (16, 32 or 64) with V
// 16-byte loads each, so that every load instruction of a lane group covers LPR * 16
// contiguous bytes and a block sweeps kThreads * 16 contiguous bytes per instruction.  The
// base pointer is 16-byte aligned.  V == 0 means "runtime count" (vecs_per_lane).
template <typename T, int LPR, int V>
__global__ __launch_bounds__(kThreads) void minimax_vec_kernel(const T* __restrict__ data,
                                                               T* __restrict__ mn,
                                                               T* __restrict__ mx, int64_t M,
                                                               int64_t D, int vecs_per_lane) {
  constexpr int E = Vec16<T>::kElems;
  constexpr int kSlots = kThreads / LPR;
  constexpr int R = kRowsPerLaneGroup;
  const int sub = threadIdx.x % LPR;
  const int slot = threadIdx.x / LPR;
  const int64_t row0 = (int64_t)blockIdx.x * (kSlots * R) + slot;
  float lo[R], hi[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    lo[r] = INFINITY;
    hi[r] = -INFINITY;
    const int64_t row = row0 + r * kSlots;
    if (row < M) {
      const T* p = data + row * D + sub * E;
      if (V > 0) {
#pragma unroll
        for (int i = 0; i < V; ++i) Vec16<T>::minmax(p + i * LPR * E, lo[r], hi[r]);
      } else {
        for (int i = 0; i < vecs_per_lane; ++i) Vec16<T>::minmax(p + (int64_t)i * LPR * E, lo[r], hi[r]);
      }
    }
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    float l = lo[r], h = hi[r];
    lanes_minmax<LPR / 16>(l, h);
    const int64_t row = row0 + r * kSlots;
    if (sub == LPR - 1 && row < M) {      // the last lane of the group holds the combined result
      Conv<T>::store(mn, row, l);
      Conv<T>::store(mx, row, h);
    }
  }
}

// Generic path: any D, element-wise loads, one 16-lane group per row.
template <typename T>
__global__ __launch_bounds__(kThreads) void minimax_generic_kernel(const T* __restrict__ data,
                                                                   T* __restrict__ mn,
                                                                   T* __restrict__ mx, int64_t M,
                                                                   int64_t D) {
  const int sub = threadIdx.x & 15;
  const int64_t row = (int64_t)blockIdx.x * kRowGroups + (threadIdx.x >> 4);
  float lo = INFINITY, hi = -INFINITY;
  if (row < M) {
    const T* p = data + row * D;
    for (int64_t i = sub; i < D; i += 16) {
      const float v = Conv<T>::load(p, i);
      lo = min_f32(lo, v);
      hi = max_f32(hi, v);
    }
  }
  lanes_minmax<1>(lo, hi);
  if (sub == 0 && row < M) {
    Conv<T>::store(mn, row, lo);
    Conv<T>::store(mx, row, hi);
  }
}

template <typename T, int LPR>
int launch_vec(const T* d, T* lo, T* hi, int64_t M, int64_t D, int64_t vecs, hipStream_t s) {
  constexpr int kRows = (kThreads / LPR) * kRowsPerLaneGroup;
  const int64_t blocks = (M + kRows - 1) / kRows;
  if (blocks > 0x7fffffffLL || vecs > 0x7fffffffLL) return ACTNN_EINVAL;
  const dim3 grid((unsigned)blocks), blk(kThreads);
  if (vecs == 1) minimax_vec_kernel<T, LPR, 1><<<grid, blk, 0, s>>>(d, lo, hi, M, D, 1);
  else if (vecs == 2) minimax_vec_kernel<T, LPR, 2><<<grid, blk, 0, s>>>(d, lo, hi, M, D, 2);
  else minimax_vec_kernel<T, LPR, 0><<<grid, blk, 0, s>>>(d, lo, hi, M, D, (int)vecs);
  ACTNN_RETURN_LAUNCH_STATUS();
}

template <typename T>
int launch_minimax(const void* data, void* mn, void* mx, int64_t M, int64_t D, hipStream_t s) {
  constexpr int E = Vec16<T>::kElems;
  const T* d = static_cast<const T*>(data);
  T* lo = static_cast<T*>(mn);
  T* hi = static_cast<T*>(mx);
  if (D % (16 * E) == 0 && aligned16(data)) {
    const int64_t nvec = D / E;                       // 16-byte vectors per row, a multiple of 16
    if (nvec % 64 == 0) return launch_vec<T, 64>(d, lo, hi, M, D, nvec / 64, s);
    if (nvec % 32 == 0) return launch_vec<T, 32>(d, lo, hi, M, D, nvec / 32, s);
    return launch_vec<T, 16>(d, lo, hi, M, D, nvec / 16, s);
  }
  const int64_t blocks = (M + kRowGroups - 1) / kRowGroups;
  if (blocks > 0x7fffffffLL) return ACTNN_EINVAL;
  minimax_generic_kernel<T><<<dim3((unsigned)blocks), dim3(kThreads), 0, s>>>(d, lo, hi, M, D);
  ACTNN_RETURN_LAUNCH_STATUS();
}

// Groups of 256 of rows of F elements at any address, the last group of a row padded with zeros (which count).
// As the vector path: 64 lanes (fp32) or 32 lanes own a group with one 16-byte load each, eight groups a lane
// in flight.  Copying the rows to padded ones first was two passes of its own (fp32 [32, 309123]: 16.0 + 8.3 us
// for the copy and its minimax, 9.3 now).
template <typename T>
__global__ __launch_bounds__(kThreads) void minimax_rows_kernel(const T* __restrict__ data, T* __restrict__ mn,
                                                                T* __restrict__ mx, uint32_t M, int64_t F,
                                                                FastDiv groups, const T* last) {
  constexpr int E = 16 / sizeof(T);
  constexpr int LPR = 256 / E;
  constexpr int kSlots = kThreads / LPR;
  constexpr int R = kRowsPerLaneGroup;
  const int sub = threadIdx.x % LPR;
  const uint32_t row0 = blockIdx.x * (kSlots * R) + threadIdx.x / LPR;
  RowVector u[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const uint32_t row = row0 + r * kSlots, n = groups.div(row);
    const int64_t at = (int64_t)(row - n * groups.d) * 256 + sub * E;
    u[r] = load16_row(data + n * F + at, row < M ? part_of_row(F, at) : 0, last);
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    float lo = INFINITY, hi = -INFINITY;
    Vec16<T>::minmax(row_vector_ends<T>(u[r]), lo, hi);
    lanes_minmax<LPR / 16>(lo, hi);
    const uint32_t row = row0 + r * kSlots;
    if (sub == LPR - 1 && row < M) {
      Conv<T>::store(mn, row, lo);
      Conv<T>::store(mx, row, hi);
    }
  }
}

template <typename T>
int launch_minimax_rows(const void* data, void* mn, void* mx, int64_t N, int64_t F, hipStream_t s) {
  constexpr int kRows = kThreads / (256 * (int)sizeof(T) / 16) * kRowsPerLaneGroup;
  const int64_t G = (F + 255) / 256, M = N * G;
  if (M > 0x7fffffffLL - kRows) return ACTNN_EINVAL;
  const T* d = static_cast<const T*>(data);
  minimax_rows_kernel<T><<<dim3((unsigned)((M + kRows - 1) / kRows)), dim3(kThreads), 0, s>>>(
      d, static_cast<T*>(mn), static_cast<T*>(mx), (uint32_t)M, F, FastDiv((uint32_t)G), d + N * F - 16 / sizeof(T));
  ACTNN_RETURN_LAUNCH_STATUS();
}

// Squared L2 norm of every sample (the gradient statistic of the bit allocation, qscheme.py:47-55):
// part[n * B + b] = sum of squares over slice b of row n, fp32, in a fixed order; the caller adds
// the B slices.  Rows are read with 16-byte non-temporal loads; 16-bit types use the dot-product
// instructions (exact products, fp32 accumulation).
template <typename T> ACTNN_DEV float square_sum16(u32x4 u);
template <> ACTNN_DEV float square_sum16<float>(u32x4 u) {
  const float a = as_float(u.x), b = as_float(u.y), c = as_float(u.z), d = as_float(u.w);
  return fmaf(a, a, fmaf(b, b, fmaf(c, c, d * d)));
}
typedef _Float16 f16x2_mm __attribute__((ext_vector_type(2)));
template <> ACTNN_DEV float square_sum16<__half>(u32x4 u) {
  float q = 0.0f;
  const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
  for (int i = 0; i < 4; ++i)
    q = __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2_mm, w[i]), __builtin_bit_cast(f16x2_mm, w[i]), q, false);
  return q;
}
template <> ACTNN_DEV float square_sum16<bf16_t>(u32x4 u) {
  float q = 0.0f;
  const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
  for (int i = 0; i < 4; ++i)
    q = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, w[i]), __builtin_bit_cast(bf16x2_t, w[i]), q, false);
  return q;
}

template <typename T>
__global__ __launch_bounds__(kThreads) void sample_sqnorm_kernel(const T* __restrict__ x, float* __restrict__ part,
                                                                int64_t F, int64_t slice) {
  constexpr int E = Vec16<T>::kElems;
  __shared__ float s_part[kThreads];
  const int64_t n = blockIdx.y;
  const int64_t lo = (int64_t)blockIdx.x * slice;
  const int64_t hi = lo + slice < F ? lo + slice : F;
  const T* row = x + n * F;
  float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  int64_t i = lo + (int64_t)threadIdx.x * E;
  for (; i + 3 * (int64_t)kThreads * E < hi; i += 4 * (int64_t)kThreads * E) {
#pragma unroll
    for (int u = 0; u < 4; ++u) acc[u] += square_sum16<T>(load16_nt(row + i + (int64_t)u * kThreads * E));
  }
  for (; i < hi; i += (int64_t)kThreads * E) acc[0] += square_sum16<T>(load16_nt(row + i));
  s_part[threadIdx.x] = (acc[0] + acc[1]) + (acc[2] + acc[3]);
  __syncthreads();
  for (int w = kThreads / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) s_part[threadIdx.x] += s_part[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[n * gridDim.x + blockIdx.x] = s_part[0];
}

// What a linear layer's backward wants of the gradient of its output, [N, F], from one read: the sum of every
// column (the bias's gradient) and, SQ, the squared norm of every row - the sums of sample_sqnorm_kernel with
// one slice, in its order.  A block takes kSumRows rows and up to 256 * V vectors of columns (SQ: whole
// rows), a thread the same V vectors in every row; column sums go to part[block row][F] and a second kernel
// adds them in a fixed order.  Bound by the read.  Norms, then torch's sum over the rows, took 13.7 + 26.8 us on
// f16 [8192, 4096]; one read takes 15.4 us and the fold 5.4.
constexpr int kSumRows = 16;

template <typename T, int V, bool SQ>
__global__ __launch_bounds__(kThreads) void row_column_sums_kernel(const T* __restrict__ x, float* __restrict__ part,
                                                                  float* __restrict__ sq, int64_t N, int64_t F) {
  constexpr int E = Vec16<T>::kElems;
  constexpr int kBatch = V >= 4 ? 2 : 4;               // rows in flight
  __shared__ float s_part[SQ ? kSumRows * kThreads : 1];
  const int64_t n0 = (int64_t)blockIdx.y * kSumRows;
  const int rows = (int)(N - n0 < kSumRows ? N - n0 : kSumRows);
  const int64_t col = ((int64_t)blockIdx.x * V * kThreads + threadIdx.x) * E;
  float sum[V][E];
#pragma unroll
  for (int v = 0; v < V; ++v)
#pragma unroll
    for (int e = 0; e < E; ++e) sum[v][e] = 0.0f;
  for (int r0 = 0; r0 < rows; r0 += kBatch) {
    u32x4 u[kBatch][V];
#pragma unroll
    for (int r = 0; r < kBatch; ++r)
#pragma unroll
      for (int v = 0; v < V; ++v) {
        const int64_t c = col + (int64_t)v * kThreads * E;
        u[r][v] = (u32x4){0, 0, 0, 0};
        if (c < F && r0 + r < rows) u[r][v] = load16(x + (n0 + r0 + r) * F + c);
      }
#pragma unroll
    for (int r = 0; r < kBatch; ++r) {
      float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int v = 0; v < V; ++v) {
        const uint32_t w[4] = {u[r][v].x, u[r][v].y, u[r][v].z, u[r][v].w};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          if constexpr (sizeof(T) == 4) {
            sum[v][k] += as_float(w[k]);
          } else if constexpr (sizeof(T) == 2) {
            constexpr bool kBf16 = !__is_same(T, __half);
            sum[v][2 * k] += kBf16 ? as_float(w[k] << 16) : half_bits_to_float(w[k] & 0xffffu);
            sum[v][2 * k + 1] += kBf16 ? as_float(w[k] & 0xffff0000u) : half_bits_to_float(w[k] >> 16);
          }
        }
        if (SQ && col + (int64_t)v * kThreads * E < F) {
          // four running sums while four vectors are left, the rest in the first
          const bool four = col + (int64_t)((v & ~3) + 3) * kThreads * E < F && (v | 3) < V;
          const float q = square_sum16<T>(u[r][v]);
          if (four) acc[v & 3] += q;
          else acc[0] += q;
        }
      }
      if (SQ && r0 + r < rows) s_part[(r0 + r) * kThreads + threadIdx.x] = (acc[0] + acc[1]) + (acc[2] + acc[3]);
    }
  }
#pragma unroll
  for (int v = 0; v < V; ++v) {
    const int64_t c = col + (int64_t)v * kThreads * E;
    if (c < F) {
#pragma unroll
      for (int e = 0; e < E; e += 4)
        store16(part + (int64_t)blockIdx.y * F + c + e, (u32x4){as_uint(sum[v][e]), as_uint(sum[v][e + 1]),
                                                                as_uint(sum[v][e + 2]), as_uint(sum[v][e + 3])});
    }
  }
  if constexpr (SQ) {
    __syncthreads();
    const int lane = threadIdx.x & 63;
    for (int r = threadIdx.x >> 6; r < rows; r += kThreads / 64) {      // (folded in halves, as sample_sqnorm_kernel does)
      const float* s = s_part + r * kThreads + lane;
      float v = (s[0] + s[128]) + (s[64] + s[192]);
#pragma unroll
      for (int d = 32; d > 0; d >>= 1) v += __shfl_down(v, d);
      if (lane == 0) sq[n0 + r] = v;
    }
  }
}

// The same sums of 16-bit rows, and the rows turned over on the way: out[column * ld + row], rows up to ld zero, as
// the product of the weight gradient reads its left factor fastest.  A block takes 64 rows of 256 columns
// (store_transposed_tile), sums its columns (part[block row][F]) and the squares of its rows' pieces
// (sq_part[column tile][N]); the second kernel adds both up in a fixed order.  Bound by reading and writing the
// tensor once.
template <typename T>
__global__ __launch_bounds__(kThreads) void row_column_sums_transposed_kernel(
    const T* __restrict__ x, T* __restrict__ out, float* __restrict__ part, float* __restrict__ sq_part, int64_t N,
    int64_t F, int64_t ld, int64_t blocks, FastDiv by_tiles) {
  __shared__ u32x4 s_tile[256 * kTileSamples / 8];
  __shared__ float s_sum[kThreads / 64][256];
  const int64_t block = xcd_block();
  if (block >= blocks) return;
  const uint32_t row = by_tiles.div((uint32_t)block), tile = (uint32_t)block - row * by_tiles.d;
  const uint32_t lane = threadIdx.x & 31u, half = threadIdx.x >> 5;
  const int64_t c = (int64_t)tile * 256 + 8 * lane, n0 = (int64_t)row * kTileSamples + 8 * half;
  uint32_t w[8][4];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    u32x4 u = {0, 0, 0, 0};
    if (c < F && n0 + i < N) u = load16(x + (n0 + i) * F + c);
#pragma unroll
    for (int j = 0; j < 4; ++j) w[i][j] = u[j];
  }
  if (part) {
    constexpr bool kBf16 = !__is_same(T, __half);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float a = 0.0f, b = 0.0f;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        a += kBf16 ? as_float(w[i][j] << 16) : half_bits_to_float(w[i][j] & 0xffffu);
        b += kBf16 ? as_float(w[i][j] & 0xffff0000u) : half_bits_to_float(w[i][j] >> 16);
      }
      a += __shfl_xor(a, 32);
      b += __shfl_xor(b, 32);
      if ((threadIdx.x & 32u) == 0) {
        s_sum[threadIdx.x >> 6][8 * lane + 2 * j] = a;
        s_sum[threadIdx.x >> 6][8 * lane + 2 * j + 1] = b;
      }
    }
  }
  if (sq_part) {
    // eight sums over 32 lanes: each exchange halves the sums a lane still carries, so that lane l ends with
    // that of row l >> 2
    float q[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) q[i] = square_sum16<T>((u32x4){w[i][0], w[i][1], w[i][2], w[i][3]});
    float h[4], g[2];
#pragma unroll
    for (int i = 0; i < 4; ++i) h[i] = ((lane & 16u) ? q[i + 4] : q[i]) + __shfl_xor((lane & 16u) ? q[i] : q[i + 4], 16);
#pragma unroll
    for (int i = 0; i < 2; ++i) g[i] = ((lane & 8u) ? h[i + 2] : h[i]) + __shfl_xor((lane & 8u) ? h[i] : h[i + 2], 8);
    float v = ((lane & 4u) ? g[1] : g[0]) + __shfl_xor((lane & 4u) ? g[0] : g[1], 4);
    v += __shfl_xor(v, 2);
    v += __shfl_xor(v, 1);
    const int64_t n = n0 + (lane >> 2);
    if ((lane & 3u) == 0 && n < N) sq_part[(int64_t)tile * N + n] = v;
  }
  store_transposed_tile(w, s_tile, out, (int64_t)tile * 256, F, (int64_t)row * kTileSamples, ld);
  const int64_t column = (int64_t)tile * 256 + threadIdx.x;
  if (part && column < F)                              // (the barrier inside store_transposed_tile lies between)
    part[(int64_t)row * F + column] = (s_sum[0][threadIdx.x] + s_sum[1][threadIdx.x]) + (s_sum[2][threadIdx.x] + s_sum[3][threadIdx.x]);
}

// out[c] = sum of part[b][c] over the block rows b: 16 threads per vector of four columns, each every 16th
// block row, then folded in halves.  Blocks from column_blocks on: sq[n] = sum of sq_part[t][n] over the tiles t.
template <typename T>
__global__ __launch_bounds__(kThreads) void fold_columns_kernel(const float* __restrict__ part, T* __restrict__ out,
                                                               int64_t F, int64_t B, unsigned column_blocks,
                                                               const float* __restrict__ sq_part, float* __restrict__ sq,
                                                               int64_t N, int tiles) {
  __shared__ float s[16][16][4];
  if (blockIdx.x >= column_blocks) {
    const int64_t n = (int64_t)(blockIdx.x - column_blocks) * kThreads + threadIdx.x;
    if (n < N) {
      float v = 0.0f;
#pragma unroll 4
      for (int t = 0; t < tiles; ++t) v += sq_part[(int64_t)t * N + n];
      sq[n] = v;
    }
    return;
  }
  const int v = threadIdx.x & 15, y = threadIdx.x >> 4;
  const int64_t c = ((int64_t)blockIdx.x * 16 + v) * 4;
  float sum[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  if (c < F) {
#pragma unroll 4
    for (int64_t b = y; b < B; b += 16) {
      const u32x4 u = load16(part + b * F + c);
      sum[0] += as_float(u.x);
      sum[1] += as_float(u.y);
      sum[2] += as_float(u.z);
      sum[3] += as_float(u.w);
    }
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) s[y][v][k] = sum[k];
  __syncthreads();
  for (int w = 8; w > 0; w >>= 1) {
    if (y < w) {
#pragma unroll
      for (int k = 0; k < 4; ++k) s[y][v][k] += s[y + w][v][k];
    }
    __syncthreads();
  }
  if (y == 0 && c < F) {
#pragma unroll
    for (int k = 0; k < 4; ++k) Conv<T>::store(out, c + k, s[0][v][k]);
  }
}

template <typename T>
int launch_sums(const void* x, void* columns, float* sq, float* part, int64_t N, int64_t F, hipStream_t s) {
  constexpr int E = Vec16<T>::kElems;
  const int64_t B = (N + kSumRows - 1) / kSumRows, per = (F / E + kThreads - 1) / kThreads;
  const dim3 blk(kThreads);
  const T* d = static_cast<const T*>(x);
  if (sq) {
    const dim3 grid(1, (unsigned)B);
    if (per <= 1) row_column_sums_kernel<T, 1, true><<<grid, blk, 0, s>>>(d, part, sq, N, F);
    else if (per <= 2) row_column_sums_kernel<T, 2, true><<<grid, blk, 0, s>>>(d, part, sq, N, F);
    else if (per <= 4) row_column_sums_kernel<T, 4, true><<<grid, blk, 0, s>>>(d, part, sq, N, F);
    else return ACTNN_EINVAL;
  } else {
    row_column_sums_kernel<T, 1, false><<<dim3((unsigned)per, (unsigned)B), blk, 0, s>>>(d, part, nullptr, N, F);
  }
  const unsigned column_blocks = (unsigned)((F / 4 + 15) / 16);
  fold_columns_kernel<T><<<dim3(column_blocks), blk, 0, s>>>(part, static_cast<T*>(columns), F, B, column_blocks, nullptr, nullptr, 0, 0);
  ACTNN_RETURN_LAUNCH_STATUS();
}

template <typename T>
int launch_sums_transposed(const void* x, void* columns, float* sq, void* out, float* part, float* sq_part, int64_t N,
                           int64_t F, int64_t ld, hipStream_t s) {
  const int64_t rows = (N + kTileSamples - 1) / kTileSamples, tiles = (F + 255) / 256;
  if (rows > (0x7fffffffLL - kXcds) / tiles) return ACTNN_EINVAL;
  const dim3 blk(kThreads);
  row_column_sums_transposed_kernel<T><<<dim3(xcd_grid(rows * tiles)), blk, 0, s>>>(
      static_cast<const T*>(x), static_cast<T*>(out), columns ? part : nullptr, sq ? sq_part : nullptr, N, F, ld,
      rows * tiles, FastDiv((uint32_t)tiles));
  const unsigned column_blocks = columns ? (unsigned)((F / 4 + 15) / 16) : 0;
  const unsigned row_blocks = sq ? (unsigned)((N + kThreads - 1) / kThreads) : 0;
  if (column_blocks + row_blocks)
    fold_columns_kernel<T><<<dim3(column_blocks + row_blocks), blk, 0, s>>>(part, static_cast<T*>(columns), F, rows, column_blocks,
                                                                           sq_part, sq, N, (int)tiles);
  ACTNN_RETURN_LAUNCH_STATUS();
}

}  // namespace

// minimum and maximum of the groups of [N, F] rows (actnn_quantize_rows has checked the arguments)
int minimax_rows(const void* data, void* mn, void* mx, int64_t N, int64_t F, int dtype, hipStream_t s) {
  switch (dtype) {
    case ACTNN_F32: return launch_minimax_rows<float>(data, mn, mx, N, F, s);
    case ACTNN_F16: return launch_minimax_rows<__half>(data, mn, mx, N, F, s);
    case ACTNN_BF16: return launch_minimax_rows<bf16_t>(data, mn, mx, N, F, s);
    default: return ACTNN_EDTYPE;
  }
}

}  // namespace actnn

extern "C" int actnn_minimax(const void* data, void* mn, void* mx, int64_t M, int64_t D, int dtype,
                             void* stream) {
  using namespace actnn;
  if (M < 0 || D < 1) return ACTNN_EINVAL;
  if (M == 0) return ACTNN_OK;
  if (!data || !mn || !mx) return ACTNN_EINVAL;
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (dtype) {
    case ACTNN_F32: return launch_minimax<float>(data, mn, mx, M, D, s);
    case ACTNN_F16: return launch_minimax<__half>(data, mn, mx, M, D, s);
    case ACTNN_BF16: return launch_minimax<bf16_t>(data, mn, mx, M, D, s);
    default: return ACTNN_EDTYPE;
  }
}

extern "C" int actnn_sample_sqnorm(const void* x, float* part, int64_t N, int64_t F, int slices, int dtype,
                                   void* stream) {
  using namespace actnn;
  if (N < 0 || F < 0 || slices < 1 || slices > 65535 || N > 65535) return ACTNN_EINVAL;
  if (N == 0) return ACTNN_OK;
  if (!x || !part) return ACTNN_EINVAL;
  const int elems = dtype == ACTNN_F32 ? 4 : 8;
  if (F % elems != 0) return ACTNN_EINVAL;
  if (!aligned16(x)) return ACTNN_EALIGN;
  int64_t slice = (F + slices - 1) / slices;
  slice = (slice + elems - 1) / elems * elems;                 // whole 16-byte vectors
  hipStream_t s = static_cast<hipStream_t>(stream);
  const dim3 grid((unsigned)slices, (unsigned)N), blk(kThreads);
  switch (dtype) {
    case ACTNN_F32: sample_sqnorm_kernel<float><<<grid, blk, 0, s>>>(static_cast<const float*>(x), part, F, slice); break;
    case ACTNN_F16: sample_sqnorm_kernel<__half><<<grid, blk, 0, s>>>(static_cast<const __half*>(x), part, F, slice); break;
    case ACTNN_BF16: sample_sqnorm_kernel<bf16_t><<<grid, blk, 0, s>>>(static_cast<const bf16_t*>(x), part, F, slice); break;
    default: return ACTNN_EDTYPE;
  }
  ACTNN_RETURN_LAUNCH_STATUS();
}

extern "C" int actnn_row_column_sums(const void* x, void* columns, float* sqnorm, float* part, int64_t N, int64_t F,
                                     int dtype, void* stream) {
  using namespace actnn;
  if (N <= 0 || F <= 0 || N > 65535 * (int64_t)kSumRows || F > 0x7fffffffLL) return ACTNN_EINVAL;
  const int elems = dtype == ACTNN_F32 ? 4 : 8;
  if (F % elems != 0 || !x || !columns || !part) return ACTNN_EINVAL;
  if (sqnorm && F > 4 * kThreads * elems) return ACTNN_EINVAL;
  if (!aligned16(x) || !aligned16(part)) return ACTNN_EALIGN;
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (dtype) {
    case ACTNN_F32: return launch_sums<float>(x, columns, sqnorm, part, N, F, s);
    case ACTNN_F16: return launch_sums<__half>(x, columns, sqnorm, part, N, F, s);
    case ACTNN_BF16: return launch_sums<bf16_t>(x, columns, sqnorm, part, N, F, s);
    default: return ACTNN_EDTYPE;
  }
}

extern "C" int actnn_row_column_sums_transposed(const void* x, void* columns, float* sqnorm, void* transposed, float* part,
                                                float* sq_part, int64_t N, int64_t F, int64_t ld, int dtype, void* stream) {
  using namespace actnn;
  if (N <= 0 || F <= 0 || F % 8 != 0 || N > 0x7fffffffLL || F > 0x7fffffffLL) return ACTNN_EINVAL;
  if (ld < N || ld % 8 != 0 || ld > (N + kTileSamples - 1) / kTileSamples * kTileSamples) return ACTNN_EINVAL;
  if (!x || !transposed || (columns && !part) || (sqnorm && !sq_part)) return ACTNN_EINVAL;
  if (!aligned16(x) || !aligned16(transposed) || !aligned16(part)) return ACTNN_EALIGN;
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (dtype) {
    case ACTNN_F16: return launch_sums_transposed<__half>(x, columns, sqnorm, transposed, part, sq_part, N, F, ld, s);
    case ACTNN_BF16: return launch_sums_transposed<bf16_t>(x, columns, sqnorm, transposed, part, sq_part, N, F, ld, s);
    default: return ACTNN_EDTYPE;
  }
}
