// ReLU and Dropout with 1-bit masks (replaces quantization_cuda_kernel.cu:411-627).
//
// Mask layout (kept from the reference): elements are cut into blocks of 512; element
// t = 16*j + k of a block is bit j of the block's word k (16 int32 words per block).  Lane j
// of a 32-lane half-wave therefore owns 16 contiguous elements; two blocks fill a 32-bit
// register per lane and one 32x32 bit transpose leaves the 32 mask words of the two blocks in
// lanes 0..31, stored as one contiguous 128-byte run.
#include "device_utils.h"

namespace actnn {
namespace {

constexpr int kThreads = 256;
constexpr int kMaskBlock = 512;

enum class Op { kRelu, kDropout };

// The tensor's last n < 2048 elements (their mask blocks, fully materialised), by one block.
// OP selects the keep rule: x > 0 (ReLU) or Philox r16 >= threshold (Dropout); elem_offset: index of
// x[0] in the tensor.
template <typename T, Op OP>
ACTNN_DEV void mask_forward_rest(const T* __restrict__ x, T* __restrict__ y, int32_t* __restrict__ mask, int64_t n,
                                 uint32_t thr, float keep_div, uint64_t seed, uint64_t offset,
                                 int64_t elem_offset, const T* __restrict__ add) {
  const uint32_t lane = threadIdx.x & 31;
  const int64_t mb0 = (threadIdx.x >> 5) * 2;
  const int64_t n_mask_blocks = (n + kMaskBlock - 1) / kMaskBlock;
  uint32_t acc = 0;
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const int64_t e0 = (mb0 + r) * kMaskBlock + lane * 16;
    if (e0 >= n) continue;
    float v[16];
    const bool full = e0 + 16 <= n;
    if (full) {
      load8(x + e0, reinterpret_cast<float(&)[8]>(v[0]));
      load8(x + e0 + 8, reinterpret_cast<float(&)[8]>(v[8]));
    } else {
#pragma unroll
      for (int k = 0; k < 16; ++k) v[k] = e0 + k < n ? Conv<T>::load(x, e0 + k) : 0.0f;
    }
    if (add) {                                       // the sum as a tensor addition rounds it, then the rule
      float a[16];
      if (full) {
        load8(add + e0, reinterpret_cast<float(&)[8]>(a[0]));
        load8(add + e0 + 8, reinterpret_cast<float(&)[8]>(a[8]));
      } else {
#pragma unroll
        for (int k = 0; k < 16; ++k) a[k] = e0 + k < n ? Conv<T>::load(add, e0 + k) : 0.0f;
      }
#pragma unroll
      for (int k = 0; k < 16; ++k) v[k] = Conv<T>::round(v[k] + a[k]);
    }
    uint32_t bitsr = 0;
    if (OP == Op::kRelu) {
#pragma unroll
      for (int k = 0; k < 16; ++k) {
        const bool keep = v[k] > 0.0f;
        v[k] = keep ? v[k] : 0.0f;
        bitsr |= (uint32_t)keep << k;
      }
    } else {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        uint32_t r16[8];
        philox_octet((uint64_t)((elem_offset + e0) >> 3) + h, seed, offset, r16);
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const bool keep = r16[k] >= thr && e0 + h * 8 + k < n;
          v[h * 8 + k] = keep ? v[h * 8 + k] / keep_div : 0.0f;
          bitsr |= (uint32_t)keep << (h * 8 + k);
        }
      }
    }
    acc |= bitsr << (16 * r);
    if (full) {
      store8(y + e0, reinterpret_cast<const float(&)[8]>(v[0]));
      store8(y + e0 + 8, reinterpret_cast<const float(&)[8]>(v[8]));
    } else {
#pragma unroll
      for (int k = 0; k < 16; ++k)
        if (e0 + k < n) Conv<T>::store(y, e0 + k, v[k]);
    }
  }
  const uint32_t w = transpose32(acc, lane);       // lane p: word p % 16 of mask block mb0 + p / 16
  if (mb0 + (lane >> 4) < n_mask_blocks) mask[mb0 * 16 + lane] = (int32_t)w;
}

template <typename T>
ACTNN_DEV void mask_backward_rest(const T* __restrict__ gout, const int32_t* __restrict__ mask, T* __restrict__ gin,
                                  int64_t n, float keep_div, bool divide, const T* __restrict__ acc) {
  const uint32_t lane = threadIdx.x & 31;
  const int64_t mb0 = (threadIdx.x >> 5) * 2;
  const int64_t n_mask_blocks = (n + kMaskBlock - 1) / kMaskBlock;
  uint32_t w = 0;
  if (mb0 + (lane >> 4) < n_mask_blocks) w = (uint32_t)mask[mb0 * 16 + lane];
  const uint32_t rows = transpose32(w, lane);       // bits 16*r + k: keep flag of element 16*lane + k of block r
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const int64_t e0 = (mb0 + r) * kMaskBlock + lane * 16;
    if (e0 >= n) continue;
    float v[16];
    const bool full = e0 + 16 <= n;
    if (full) {
      load8(gout + e0, reinterpret_cast<float(&)[8]>(v[0]));
      load8(gout + e0 + 8, reinterpret_cast<float(&)[8]>(v[8]));
    } else {
#pragma unroll
      for (int k = 0; k < 16; ++k) v[k] = e0 + k < n ? Conv<T>::load(gout, e0 + k) : 0.0f;
    }
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      const bool keep = (rows >> (16 * r + k)) & 1u;
      v[k] = keep ? (divide ? v[k] / keep_div : v[k]) : 0.0f;
    }
    if (acc) {                                       // the masked gradient added to another, as a tensor addition adds them
      float a[16];
      if (full) {
        load8(acc + e0, reinterpret_cast<float(&)[8]>(a[0]));
        load8(acc + e0 + 8, reinterpret_cast<float(&)[8]>(a[8]));
      } else {
#pragma unroll
        for (int k = 0; k < 16; ++k) a[k] = e0 + k < n ? Conv<T>::load(acc, e0 + k) : 0.0f;
      }
#pragma unroll
      for (int k = 0; k < 16; ++k) v[k] = a[k] + v[k];
    }
    if (full) {
      store8(gin + e0, reinterpret_cast<const float(&)[8]>(v[0]));
      store8(gin + e0 + 8, reinterpret_cast<const float(&)[8]>(v[8]));
    } else {
#pragma unroll
      for (int k = 0; k < 16; ++k)
        if (e0 + k < n) Conv<T>::store(gin, e0 + k, v[k]);
    }
  }
}

// ---------------------------------------------------------------------------------------------
// Whole-line streaming.  A wave handles 4 mask blocks (2048 elements) with wave-wide 16-byte loads and
// stores, so that every instruction covers whole cache lines (a lane that owned the 16 contiguous
// elements of a mask row came back to its line four times in fp32).  What is left of the tensor (< 2048
// elements) is the last block's, in the same launch.  Bound by memory: fp32 [256, 100352] 34 us forward and
// 34 us backward (6 TB/s; 54 and 54 us with a lane per mask row), bf16 [362, 122467] 31 + 30 us (37 + 36 us with
// the remainder in a launch of its own).  fp32 results are stored through the caches, 16-bit ones past them.  For fp32 that
// depends on who reads next (ReLU of 256 MB alone 79 us, 87 past the caches; forward and backward in turn
// 183 and 173; 120 MB 79 and 84; 16 MB 13.7 and 10.5; 512 MB 375 and 346).
constexpr int kTileElems = 4 * kMaskBlock;        // elements per wave
constexpr int kTilesPerBlock = kThreads / 64;

struct RestArgs {                                 // the last block's part
  int64_t tiles;                                  // whole tiles before it
  int64_t tile_blocks;                            // blocks that hold them
  int rest;                                       // elements behind them (0: there is no such block)
};

// MINMAX: also write the minimum and maximum of every group of 256 consecutive outputs (the lower
// and upper 32 lanes of each load own one group each) - what actnn_minimax returns for the output
// viewed as rows of 256, for a consumer that quantises it next.
// ADD: the rule is applied to x + add, rounded to T as the tensor addition it replaces rounds it
// (the closing `relu(out + identity)` of a residual block in one pass over the two operands).
// 16-bit element types: lane l holds elements 8l..8l+7 of each block, i.e. half of the 16 elements a
// mask row belongs to (rows_to_word).
template <typename T, Op OP, bool MINMAX, bool ADD>
ACTNN_DEV void mask_forward_tile(const T* __restrict__ x, T* __restrict__ y, int32_t* __restrict__ mask, int64_t tile,
                                 uint32_t thr, float keep_div, uint64_t seed, uint64_t offset,
                                 T* __restrict__ mn, T* __restrict__ mx, const T* __restrict__ add) {
  const uint32_t lane = threadIdx.x & 63;
  const int64_t e0 = tile * kTileElems + lane * 8;
  float v[4][8];
#pragma unroll
  for (int i = 0; i < 4; ++i) load8_nt(x + e0 + i * kMaskBlock, v[i]);
  if (ADD) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float a[8];
      load8_nt(add + e0 + i * kMaskBlock, a);
#pragma unroll
      for (int k = 0; k < 8; k += 2) {
        v[i][k] += a[k];
        v[i][k + 1] += a[k + 1];
        round_pair<T>(v[i][k], v[i][k + 1]);
      }
    }
  }
  uint32_t m[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    uint32_t r16[8];
    if (OP == Op::kDropout) philox_octet((uint64_t)((e0 + i * kMaskBlock) >> 3), seed, offset, r16);
    m[i] = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const bool keep = OP == Op::kRelu ? v[i][k] > 0.0f : r16[k] >= thr;
      v[i][k] = keep ? (OP == Op::kRelu ? v[i][k] : v[i][k] / keep_div) : 0.0f;
      m[i] |= (uint32_t)keep << k;
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) store8_nt(y + e0 + i * kMaskBlock, v[i]);
  if (MINMAX) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float lo, hi;
      minmax_of<8>(v[i], lo, hi);
      lanes_minmax<2>(lo, hi);
      if ((lane & 31u) == 31u) {
        const int64_t g = tile * (kTileElems / 256) + i * (kMaskBlock / 256) + (lane >> 5);
        Conv<T>::store(mn, g, lo);
        Conv<T>::store(mx, g, hi);
      }
    }
  }
  const uint32_t w = rows_to_word(m, lane);
  // lane 2p+h holds word p % 16 of block 2h + p / 16
  mask[tile * 64 + (lane & 1u) * 32 + (lane >> 1)] = (int32_t)w;
}

// fp32: a wave-wide load is half a mask block, lane l elements 4l..4l+3, so the quad Q = l / 4 holds mask
// row Q (first half of a block) or 16 + Q (second half) and lane l its bits 4 (l & 3) .. + 3.  The four
// lanes of a quad hand each other their nibbles - each ends with the two 16-bit rows of one half u = bit
// 1 of its index and of the blocks 2h, 2h + 1, h = bit 0 of its index - and the two interleaved 32x32 bit
// transposes (the matrices of the even and of the odd lanes) run over the remaining lane bits: row
// bit 4 is lane bit 1, row bits 3..0 are lane bits 5..2.
ACTNN_DEV uint32_t transpose32_quads(uint32_t x, uint32_t lane) {
  auto stage = [&](uint32_t p, int s, uint32_t m, bool hi) {
    const uint32_t u = __builtin_amdgcn_alignbit(p, p, hi ? s : 32 - s);
    const uint32_t sel = hi ? m : ~m;
    x = (x & sel) | (u & ~sel);
  };
  stage(lane_xor<2>(x), 16, 0xFFFF0000u, (lane & 2u) != 0);
  stage((uint32_t)__builtin_amdgcn_ds_bpermute((int)((lane ^ 32u) << 2), (int)x), 8, 0xFF00FF00u, (lane & 32u) != 0);
  stage(lane_xor<16>(x), 4, 0xF0F0F0F0u, (lane & 16u) != 0);
  stage(lane_xor<8>(x), 2, 0xCCCCCCCCu, (lane & 8u) != 0);
  stage(lane_xor<4>(x), 1, 0xAAAAAAAAu, (lane & 4u) != 0);
  return x;
}
// where the lane's word lies in the tile's 64: word p % 16 of block 2h + p / 16, p as the lane bits say
ACTNN_DEV uint32_t quads_word_at(uint32_t lane) {
  const uint32_t p = ((lane & 2u) << 3) | ((lane & 32u) >> 2) | ((lane & 16u) >> 2) | ((lane & 8u) >> 2) | ((lane & 4u) >> 2);
  return (lane & 1u) * 32 + p;
}
// nib[i]: the lane's four keep bits of half block i (blocks i / 2, halves i & 1) -> its mask word
ACTNN_DEV uint32_t nibbles_to_word(const uint32_t (&nib)[8], uint32_t lane) {
  const int sh = 4 * (int)(lane & 3u);
  uint32_t pair[2][2];                             // [h][u]: bits of blocks 2h | 2h + 1 of half u
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int u = 0; u < 2; ++u) pair[h][u] = (nib[4 * h + u] | (nib[4 * h + 2 + u] << 16)) << sh;
  const bool h = lane & 1u, u = lane & 2u;
  uint32_t half[2];
#pragma unroll
  for (int k = 0; k < 2; ++k) half[k] = (h ? pair[1][k] : pair[0][k]) | lane_xor<1>(h ? pair[0][k] : pair[1][k]);
  const uint32_t row = (u ? half[1] : half[0]) | lane_xor<2>(u ? half[0] : half[1]);
  return transpose32_quads(row, lane);
}
// inverse
ACTNN_DEV void word_to_nibbles(uint32_t w, uint32_t lane, uint32_t (&nib)[8]) {
  const int row = (int)transpose32_quads(w, lane);
  const int sh = 4 * (int)(lane & 3u);
  uint32_t quad[4];                                // rows of the quad's lanes: [2u + h]
  quad[0] = (uint32_t)__builtin_amdgcn_update_dpp(0, row, 0x00, 0xF, 0xF, true);
  quad[1] = (uint32_t)__builtin_amdgcn_update_dpp(0, row, 0x55, 0xF, 0xF, true);
  quad[2] = (uint32_t)__builtin_amdgcn_update_dpp(0, row, 0xAA, 0xF, 0xF, true);
  quad[3] = (uint32_t)__builtin_amdgcn_update_dpp(0, row, 0xFF, 0xF, 0xF, true);
#pragma unroll
  for (int i = 0; i < 8; ++i) nib[i] = (quad[2 * (i & 1) + (i >> 2)] >> (16 * ((i >> 1) & 1) + sh)) & 0xfu;
}

template <Op OP, bool ADD>
ACTNN_DEV void mask_forward_tile32(const float* __restrict__ x, float* __restrict__ y, int32_t* __restrict__ mask,
                                   int64_t tile, uint32_t thr, float keep_div, uint64_t seed, uint64_t offset,
                                   const float* __restrict__ add) {
  const uint32_t lane = threadIdx.x & 63;
  const int64_t e0 = tile * kTileElems + lane * 4;
  u32x4 v[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = load16_nt(x + e0 + i * 256);
  if (ADD) {
    u32x4 a[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) a[i] = load16_nt(add + e0 + i * 256);
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int k = 0; k < 4; ++k) v[i][k] = as_uint(as_float(v[i][k]) + as_float(a[i][k]));
  }
  uint32_t nib[8];
#pragma unroll
  for (int i = 0; i < 8; i += 2) {
    uint32_t na[2], nb[2];                         // draws of half blocks i and i + 1, two to a word
    if (OP == Op::kDropout) {
      // lanes 2j and 2j + 1 hold the halves of one octet: the even lane evaluates the octet of half
      // block i, the odd lane that of half block i + 1, and they hand each other the words they do not use
      const bool odd = lane & 1u;
      const Philox4 r = philox_at((uint64_t)((e0 + (i + (odd ? 1 : 0)) * 256) >> 3), seed, offset);
      const uint32_t nx = lane_xor<1>(r.x), ny = lane_xor<1>(r.y), nz = lane_xor<1>(r.z), nw = lane_xor<1>(r.w);
      na[0] = odd ? nz : r.x;
      na[1] = odd ? nw : r.y;
      nb[0] = odd ? r.z : nx;
      nb[1] = odd ? r.w : ny;
    }
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      nib[i + q] = 0;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float f = as_float(v[i + q][k]);
        bool keep;
        if (OP == Op::kRelu) {
          keep = f > 0.0f;
          v[i + q][k] = keep ? as_uint(f) : 0u;
        } else {
          keep = (((q ? nb : na)[k >> 1] >> (16 * (k & 1))) & 0xffffu) >= thr;
          v[i + q][k] = keep ? as_uint(f / keep_div) : 0u;
        }
        nib[i + q] |= (uint32_t)keep << k;
      }
    }
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) store16(y + e0 + i * 256, v[i]);
  mask[tile * 64 + quads_word_at(lane)] = (int32_t)nibbles_to_word(nib, lane);
}

template <typename T, Op OP, bool MINMAX = false, bool ADD = false>
__global__ __launch_bounds__(kThreads) void mask_forward_kernel(const T* __restrict__ x, T* __restrict__ y,
                                                                int32_t* __restrict__ mask, RestArgs part,
                                                                uint32_t thr, float keep_div, uint64_t seed,
                                                                uint64_t offset,
                                                                T* __restrict__ mn = nullptr,
                                                                T* __restrict__ mx = nullptr,
                                                                const T* __restrict__ add = nullptr) {
  if ((int64_t)blockIdx.x >= part.tile_blocks) {
    const int64_t done = part.tiles * kTileElems;
    mask_forward_rest<T, OP>(x + done, y + done, mask + done / 32, part.rest, thr, keep_div, seed, offset, done,
                             ADD ? add + done : nullptr);
    return;
  }
  const int64_t tile = (int64_t)blockIdx.x * kTilesPerBlock + (threadIdx.x >> 6);
  if (tile >= part.tiles) return;                  // whole waves leave together
  if constexpr (sizeof(T) == 4) mask_forward_tile32<OP, ADD>(x, y, mask, tile, thr, keep_div, seed, offset, add);
  else mask_forward_tile<T, OP, MINMAX, ADD>(x, y, mask, tile, thr, keep_div, seed, offset, mn, mx, add);
}

// ACC: gin = acc + masked gradient (rounded to T as the tensor addition of the two rounds it): the
// gradient that arrives at a residual block's input over the skip connection, masked and added to the
// one from the block's first convolution in one pass.
template <typename T, bool ACC>
ACTNN_DEV void mask_backward_tile(const T* __restrict__ gout, const int32_t* __restrict__ mask, T* __restrict__ gin,
                                  int64_t tile, float keep_div, bool divide, const T* __restrict__ acc) {
  const uint32_t lane = threadIdx.x & 63;
  const int64_t e0 = tile * kTileElems + lane * 8;
  float v[4][8];
#pragma unroll
  for (int i = 0; i < 4; ++i) load8_nt(gout + e0 + i * kMaskBlock, v[i]);
  uint32_t m[4];
  word_to_rows((uint32_t)mask[tile * 64 + (lane & 1u) * 32 + (lane >> 1)], lane, m);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const bool keep = (m[i] >> k) & 1u;
      v[i][k] = keep ? (divide ? v[i][k] / keep_div : v[i][k]) : 0.0f;
    }
    if (ACC) {
      float a[8];
      load8_nt(acc + e0 + i * kMaskBlock, a);
#pragma unroll
      for (int k = 0; k < 8; ++k) v[i][k] = a[k] + v[i][k];
    }
    store8_nt(gin + e0 + i * kMaskBlock, v[i]);
  }
}

template <bool ACC>
ACTNN_DEV void mask_backward_tile32(const float* __restrict__ gout, const int32_t* __restrict__ mask,
                                    float* __restrict__ gin, int64_t tile, float keep_div, bool divide,
                                    const float* __restrict__ acc) {
  const uint32_t lane = threadIdx.x & 63;
  const int64_t e0 = tile * kTileElems + lane * 4;
  const uint32_t word = (uint32_t)mask[tile * 64 + quads_word_at(lane)];
  u32x4 v[8], a[ACC ? 8 : 1];
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = load16_nt(gout + e0 + i * 256);
  if (ACC) {
#pragma unroll
    for (int i = 0; i < 8; ++i) a[ACC ? i : 0] = load16_nt(acc + e0 + i * 256);
  }
  uint32_t nib[8];
  word_to_nibbles(word, lane, nib);
#pragma unroll
  for (int i = 0; i < 8; ++i) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float f = as_float(v[i][k]);
      const bool keep = (nib[i] >> k) & 1u;
      const float g = keep ? (divide ? f / keep_div : f) : 0.0f;
      v[i][k] = as_uint(ACC ? as_float(a[ACC ? i : 0][k]) + g : g);
    }
    store16(gin + e0 + i * 256, v[i]);
  }
}

template <typename T, bool ACC = false>
__global__ __launch_bounds__(kThreads) void mask_backward_kernel(const T* __restrict__ gout,
                                                                 const int32_t* __restrict__ mask,
                                                                 T* __restrict__ gin, RestArgs part,
                                                                 float keep_div, bool divide,
                                                                 const T* __restrict__ acc = nullptr) {
  if ((int64_t)blockIdx.x >= part.tile_blocks) {
    const int64_t done = part.tiles * kTileElems;
    mask_backward_rest<T>(gout + done, mask + done / 32, gin + done, part.rest, keep_div, divide,
                          ACC ? acc + done : nullptr);
    return;
  }
  const int64_t tile = (int64_t)blockIdx.x * kTilesPerBlock + (threadIdx.x >> 6);
  if (tile >= part.tiles) return;
  if constexpr (sizeof(T) == 4) mask_backward_tile32<ACC>(gout, mask, gin, tile, keep_div, divide, acc);
  else mask_backward_tile<T, ACC>(gout, mask, gin, tile, keep_div, divide, acc);
}

// -> blocks of the launch, 0 when there are too many for a grid
inline int64_t split_tensor(int64_t n, RestArgs& part) {
  part.tiles = n / kTileElems;
  part.tile_blocks = (part.tiles + kTilesPerBlock - 1) / kTilesPerBlock;
  part.rest = (int)(n - part.tiles * kTileElems);
  const int64_t blocks = part.tile_blocks + (part.rest > 0 ? 1 : 0);
  return blocks > 0x7fffffffLL ? 0 : blocks;
}

template <typename T, Op OP>
int launch_forward(const void* x, void* y, int32_t* mask, int64_t n, uint32_t thr, float keep_div,
                   uint64_t seed, uint64_t offset, hipStream_t s, const void* add = nullptr) {
  const T* xi = static_cast<const T*>(x);
  const T* ai = static_cast<const T*>(add);
  T* yo = static_cast<T*>(y);
  RestArgs part;
  const int64_t blocks = split_tensor(n, part);
  if (blocks == 0) return ACTNN_EINVAL;
  const dim3 grid((unsigned)blocks), blk(kThreads);
  if (OP == Op::kRelu && ai)
    mask_forward_kernel<T, Op::kRelu, false, true><<<grid, blk, 0, s>>>(xi, yo, mask, part, thr, keep_div, seed, offset,
                                                                        nullptr, nullptr, ai);
  else
    mask_forward_kernel<T, OP><<<grid, blk, 0, s>>>(xi, yo, mask, part, thr, keep_div, seed, offset);
  ACTNN_RETURN_LAUNCH_STATUS();
}

template <typename T>
int launch_backward(const void* gout, const int32_t* mask, void* gin, int64_t n, float keep_div,
                    bool divide, hipStream_t s, const void* acc = nullptr) {
  const T* go = static_cast<const T*>(gout);
  const T* ac = static_cast<const T*>(acc);
  T* gi = static_cast<T*>(gin);
  RestArgs part;
  const int64_t blocks = split_tensor(n, part);
  if (blocks == 0) return ACTNN_EINVAL;
  const dim3 grid((unsigned)blocks), blk(kThreads);
  if (ac) mask_backward_kernel<T, true><<<grid, blk, 0, s>>>(go, mask, gi, part, keep_div, divide, ac);
  else mask_backward_kernel<T><<<grid, blk, 0, s>>>(go, mask, gi, part, keep_div, divide);
  ACTNN_RETURN_LAUNCH_STATUS();
}

template <Op OP>
int dispatch_forward(const void* x, void* y, int32_t* mask, int64_t n, uint32_t thr, float keep_div,
                     uint64_t seed, uint64_t offset, int dtype, void* stream, const void* add = nullptr) {
  if (n < 0) return ACTNN_EINVAL;
  if (n == 0) return ACTNN_OK;
  if (!x || !y || !mask) return ACTNN_EINVAL;
  if (!aligned16(x) || !aligned16(y) || !aligned16(add)) return ACTNN_EALIGN;
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (dtype) {
    case ACTNN_F32: return launch_forward<float, OP>(x, y, mask, n, thr, keep_div, seed, offset, s, add);
    case ACTNN_F16: return launch_forward<__half, OP>(x, y, mask, n, thr, keep_div, seed, offset, s, add);
    case ACTNN_BF16: return launch_forward<bf16_t, OP>(x, y, mask, n, thr, keep_div, seed, offset, s, add);
    default: return ACTNN_EDTYPE;
  }
}

int dispatch_backward(const void* gout, const int32_t* mask, void* gin, int64_t n, float keep_div,
                      bool divide, int dtype, void* stream, const void* acc = nullptr) {
  if (n < 0) return ACTNN_EINVAL;
  if (n == 0) return ACTNN_OK;
  if (!gout || !gin || !mask) return ACTNN_EINVAL;
  if (!aligned16(gout) || !aligned16(gin) || !aligned16(acc)) return ACTNN_EALIGN;
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (dtype) {
    case ACTNN_F32: return launch_backward<float>(gout, mask, gin, n, keep_div, divide, s, acc);
    case ACTNN_F16: return launch_backward<__half>(gout, mask, gin, n, keep_div, divide, s, acc);
    case ACTNN_BF16: return launch_backward<bf16_t>(gout, mask, gin, n, keep_div, divide, s, acc);
    default: return ACTNN_EDTYPE;
  }
}

// keep iff r16 >= thr, r16 uniform on [0, 2^16): P(keep) = 1 - thr / 2^16 ~ 1 - p.
inline uint32_t dropout_threshold(float p) {
  double t = (double)p * 65536.0;
  t = t < 0.0 ? 0.0 : (t > 65536.0 ? 65536.0 : t);
  return (uint32_t)(t + 0.5);
}

}  // namespace
}  // namespace actnn

extern "C" int actnn_relu_forward(const void* x, void* y, int32_t* mask, int64_t n, int dtype,
                                  void* stream) {
  return actnn::dispatch_forward<actnn::Op::kRelu>(x, y, mask, n, 0u, 1.0f, 0, 0, dtype, stream);
}

extern "C" int actnn_relu_forward_minmax(const void* x, void* y, int32_t* mask, void* mn, void* mx,
                                         int64_t n, int dtype, void* stream) {
  using namespace actnn;
  if (n < 0 || n % kTileElems != 0) return ACTNN_EINVAL;       // whole tiles of 2048 elements only
  if (dtype != ACTNN_F16 && dtype != ACTNN_BF16) return ACTNN_EDTYPE;
  if (n == 0) return ACTNN_OK;
  if (!x || !y || !mask || !mn || !mx) return ACTNN_EINVAL;
  if (!aligned16(x) || !aligned16(y)) return ACTNN_EALIGN;
  RestArgs part;
  const int64_t blocks = split_tensor(n, part);
  if (blocks == 0) return ACTNN_EINVAL;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const dim3 grid((unsigned)blocks), blk(kThreads);
  if (dtype == ACTNN_F16)
    mask_forward_kernel<__half, Op::kRelu, true><<<grid, blk, 0, s>>>(
        static_cast<const __half*>(x), static_cast<__half*>(y), mask, part, 0u, 1.0f, 0, 0,
        static_cast<__half*>(mn), static_cast<__half*>(mx));
  else
    mask_forward_kernel<bf16_t, Op::kRelu, true><<<grid, blk, 0, s>>>(
        static_cast<const bf16_t*>(x), static_cast<bf16_t*>(y), mask, part, 0u, 1.0f, 0, 0,
        static_cast<bf16_t*>(mn), static_cast<bf16_t*>(mx));
  ACTNN_RETURN_LAUNCH_STATUS();
}

extern "C" int actnn_relu_add_forward(const void* x, const void* residual, void* y, int32_t* mask, void* mn,
                                      void* mx, int64_t n, int dtype, void* stream) {
  using namespace actnn;
  if ((mn == nullptr) != (mx == nullptr)) return ACTNN_EINVAL;
  if (n > 0 && !residual) return ACTNN_EINVAL;
  if (!mn) return dispatch_forward<Op::kRelu>(x, y, mask, n, 0u, 1.0f, 0, 0, dtype, stream, residual);
  if (n < 0 || n % kTileElems != 0) return ACTNN_EINVAL;       // whole tiles of 2048 elements only
  if (dtype != ACTNN_F16 && dtype != ACTNN_BF16) return ACTNN_EDTYPE;
  if (n == 0) return ACTNN_OK;
  if (!x || !y || !mask) return ACTNN_EINVAL;
  if (!aligned16(x) || !aligned16(residual) || !aligned16(y)) return ACTNN_EALIGN;
  RestArgs part;
  const int64_t blocks = split_tensor(n, part);
  if (blocks == 0) return ACTNN_EINVAL;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const dim3 grid((unsigned)blocks), blk(kThreads);
  if (dtype == ACTNN_F16)
    mask_forward_kernel<__half, Op::kRelu, true, true><<<grid, blk, 0, s>>>(
        static_cast<const __half*>(x), static_cast<__half*>(y), mask, part, 0u, 1.0f, 0, 0,
        static_cast<__half*>(mn), static_cast<__half*>(mx), static_cast<const __half*>(residual));
  else
    mask_forward_kernel<bf16_t, Op::kRelu, true, true><<<grid, blk, 0, s>>>(
        static_cast<const bf16_t*>(x), static_cast<bf16_t*>(y), mask, part, 0u, 1.0f, 0, 0,
        static_cast<bf16_t*>(mn), static_cast<bf16_t*>(mx), static_cast<const bf16_t*>(residual));
  ACTNN_RETURN_LAUNCH_STATUS();
}

extern "C" int actnn_relu_backward(const void* grad_out, const int32_t* mask, void* grad_in,
                                   int64_t n, int dtype, void* stream) {
  return actnn::dispatch_backward(grad_out, mask, grad_in, n, 1.0f, false, dtype, stream);
}

extern "C" int actnn_relu_backward_add(const void* grad_out, const int32_t* mask, const void* other,
                                       void* grad_in, int64_t n, int dtype, void* stream) {
  if (n > 0 && !other) return ACTNN_EINVAL;
  return actnn::dispatch_backward(grad_out, mask, grad_in, n, 1.0f, false, dtype, stream, other);
}

extern "C" int actnn_dropout_forward(const void* x, void* y, int32_t* mask, int64_t n, float p,
                                     uint64_t seed, uint64_t offset, int dtype, void* stream) {
  if (!(p >= 0.0f && p <= 1.0f)) return ACTNN_EINVAL;
  const float keep_div = (float)(1.0 - (double)p);     // x / (1.0 - p), .cu:540
  return actnn::dispatch_forward<actnn::Op::kDropout>(x, y, mask, n, actnn::dropout_threshold(p),
                                                      keep_div, seed, offset, dtype, stream);
}

extern "C" int actnn_dropout_backward(const void* grad_out, const int32_t* mask, void* grad_in,
                                      int64_t n, float p, int dtype, void* stream) {
  if (!(p >= 0.0f && p <= 1.0f)) return ACTNN_EINVAL;
  const float keep_div = (float)(1.0 - (double)p);     // .cu:601
  return actnn::dispatch_backward(grad_out, mask, grad_in, n, keep_div, true, dtype, stream);
}
