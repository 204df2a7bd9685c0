// Mixed-precision pack / unpack (replaces quantization_cuda_kernel.cu:22-205).
//
// Stream layout (kept from the reference): sample n with b = bits[n] owns
// b * G * gs / 32 consecutive int32 words starting at prefix[n] * G * gs / 32; inside a group
// of gs = 32 * E elements, bit i of the code of element d = E * j + k is bit j of word
// k * b + i.  So a word is a 32-lane "ballot" over j, where lane j owns the E consecutive
// elements E*j .. E*j+E-1.
//
// gs == 256 fast path: a 32-lane half-wave owns a group; lane j loads its 8 contiguous
// elements (one 16-byte load for 16-bit types, two for f32), quantises them and
// concatenates the 8 codes into 8*b bits of a register (several groups share a register
// when 8*b <= 16).  One 32x32 bit transpose per register (5 exchange stages) then leaves
// word p in lane p, which is stored coalesced.  A wave handles a unit of consecutive groups of
// one sample (4 for f32, 8 for 16-bit types), a 256-thread block four units that follow each
// other; the element loads are issued first, the block's scales are computed by the first
// threads and shared through LDS while the loads are in flight.  unpack mirrors this; its fp32
// stores go through LDS so that each store instruction of a wave writes one whole 1 KiB group.
//
// Other group sizes (multiples of 32 up to 1024) take a simple LDS-staged kernel.
#include "quant_math.h"

namespace actnn {
namespace {

// Groups per half-wave.  fp32: 2 measured best (16 KiB of input per block).
// 16-bit types: a block with 8 KiB of data is dominated by its own latency chain (widths ->
// scales -> data), so they take 4.
template <typename T> struct Gph {
  static constexpr int kPack = sizeof(T) == 2 ? 4 : 2;
  static constexpr int kUnpack = sizeof(T) == 2 ? 4 : 2;
};

constexpr int kThreads = 256;
constexpr int kGs = 256;

template <int BITS, int GPH> struct Tile {
  static constexpr int kWordsPerGroup = 8 * BITS;
  // consecutive groups that share one register (one transpose): as many as fit in 32 bits
  static constexpr int kFit = BITS == 1 ? 4 : BITS == 2 ? 2 : 1;
  static constexpr int kGroupsPerReg = kFit < GPH ? kFit : GPH;
  static constexpr bool kTwoRegs = BITS > 4;                                  // 8*BITS > 32
  // Group (within the wave's unit) that a half of the wave handles in its q-th slot: GPH consecutive
  // groups per half, whatever the bit width, so that loads can be issued before the width is known.
  static __device__ __forceinline__ int group_of(int half, int q) { return half * GPH + q; }
};

// The unit of a wave: `valid` groups of sample n from group gb on (0 behind the last sample, where n
// is a sample that exists all the same).  The units of a sample follow each other and a block takes the
// next four whatever samples they belong to: with whole blocks per sample, short rows left most of a
// block idle (f16 [8192, 4096], 16 groups a row: pack 26.1 and unpack 22.6 us with blocks of 32 groups, 20.3
// and 16.5 us now; fp32 [256, 3136 groups] pack 149 and 145 us).
struct Unit {
  int64_t n, gb;
  int valid;
};
template <int GROUPS> ACTNN_DEV Unit unit_of(uint32_t unit, const FastDiv& per_sample, int64_t N, int64_t G) {
  Unit u;
  const uint32_t n = per_sample.div(unit);
  u.gb = (int64_t)(unit - n * per_sample.d) * GROUPS;
  const int64_t left = G - u.gb;
  u.valid = n >= N ? 0 : left < GROUPS ? (int)left : GROUPS;
  u.n = n >= N ? N - 1 : n;
  return u;
}
constexpr int kWaves = kThreads / 64;
// the wave's number in its block, as a scalar
ACTNN_DEV uint32_t wave_of_block() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); }

// elements of a unit of `groups` groups from element `at` of a row of F on
ACTNN_DEV int unit_count(int64_t F, int64_t at, int groups) {
  const int64_t left = F - at, all = (int64_t)groups * kGs;
  return (int)(left < all ? left : all);
}

// fp32 output of unpack: a lane owns 32 contiguous bytes, which as direct stores would be two
// half-used 16-byte accesses per cache line.  Instead lanes park their 8 values in the wave's
// private LDS slab and the wave stores whole 1 KiB groups with one non-temporal instruction each
// (measured 6.9 instead of 5.3 TB/s, and no dirty lines are left for the next kernel to wait on).
// Only lanes of one wave exchange data, so no block barrier is needed: LDS operations of a wave
// complete in order.  (The same staging for the fp32 loads of pack was measured slower.)
// ROWS: `out` is a row of F elements at any address and elem_base an offset in it; its ends share lines with other rows.
template <int GPH, int ROWS>
ACTNN_DEV void stage_out_f32(float* __restrict__ out, int64_t elem_base, int64_t F, int groups_valid,
                             u32x4* __restrict__ slab, const float (&v)[GPH][8]) {
  const int wl = threadIdx.x & 63;
  const int h = (threadIdx.x >> 5) & 1;
  const uint32_t lane = threadIdx.x & 31;
#pragma unroll
  for (int q = 0; q < GPH; ++q) {
    u32x4 a, b;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      a[k] = as_uint(v[q][k]);
      b[k] = as_uint(v[q][4 + k]);
    }
    slab[(h * GPH + q) * 64 + 2 * lane] = a;
    slab[(h * GPH + q) * 64 + 2 * lane + 1] = b;
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  if constexpr (ROWS == kRowsPast) {
    store_unit_any(out + elem_base, reinterpret_cast<const uint32_t*>(slab), unit_count(F, elem_base, groups_valid));
  } else {
#pragma unroll
    for (int i = 0; i < 2 * GPH; ++i) {
      if (i < groups_valid) {
        const int64_t at = elem_base + (int64_t)i * kGs + wl * 4;
        if constexpr (ROWS == kRowsCached) store16_part<false>(out + at, slab[i * 64 + wl], part_of_row(F, at));
        else store16_nt(out + at, slab[i * 64 + wl]);
      }
    }
  }
}

template <typename T> struct IsF32 { static constexpr bool value = false; };
template <> struct IsF32<float> { static constexpr bool value = true; };
template <typename T> struct IsBf16 { static constexpr bool value = false; };
template <> struct IsBf16<bf16_t> { static constexpr bool value = true; };

// ---------------------------------------------------------------------------- pack (gs = 256)
// Issue the loads of this lane's elements (and noise in deterministic mode) for its GPH groups.
// The elements stay as loaded until their group is packed (16-bit types: 4 registers per group
// rather than 8), which keeps the kernel within the registers of 8 waves per SIMD.
template <typename T, bool DET, int GPH>
ACTNN_DEV void load_groups(const T* __restrict__ data, const T* __restrict__ noise, int64_t elem_base,
                           int groups_valid, Raw8<T> (&v)[GPH], Raw8<T> (&nz)[DET ? GPH : 1]) {
  using TL = Tile<1, GPH>;
  const uint32_t lane = threadIdx.x & 31;
  const int half = (threadIdx.x >> 5) & 1;
#pragma unroll
  for (int q = 0; q < GPH; ++q) {
    const int gl = TL::group_of(half, q);
    if (gl < groups_valid) {
      const int64_t e = elem_base + (int64_t)gl * kGs + lane * 8;
      raw8_load_nt(data + e, v[q]);      // non-temporal for 16-bit types only (one instruction per line)
      if (DET) raw8_load_nt(noise + e, nz[DET ? q : 0]);
    } else {
      raw8_zero(v[q]);
      if (DET) raw8_zero(nz[DET ? q : 0]);
    }
  }
}

template <typename T, int BITS, bool DET>
ACTNN_DEV void pack_groups(const Raw8<T> (&raw)[Gph<T>::kPack], const Raw8<T> (&nzraw)[DET ? Gph<T>::kPack : 1],
                           int32_t* __restrict__ packed, int64_t elem_base, int64_t word_base,
                           int groups_valid, const float* s_mul, const float* s_sub,
                           uint64_t seed, uint64_t offset) {
  constexpr int kGroupsPerHalf = Gph<T>::kPack;
  using TL = Tile<BITS, kGroupsPerHalf>;
  constexpr int R = TL::kGroupsPerReg;
  constexpr int WPG = TL::kWordsPerGroup;
  constexpr float Bf = (float)((1 << BITS) - 1);
  const uint32_t lane = threadIdx.x & 31;
  const int half = (threadIdx.x >> 5) & 1;
  static_assert(kGroupsPerHalf % 2 == 0, "the noise of the groups is drawn in pairs");
  constexpr int NB = R > 2 ? R : 2;                    // groups whose noise is drawn together
  constexpr float kUnit = (float)(1u << (32 - BITS - Noise<T>::kBits));
  uint32_t rw[NB][Noise<T>::kWords];

#pragma unroll
  for (int q0 = 0; q0 < kGroupsPerHalf; q0 += R) {
    uint64_t acc = 0;                                  // DET
    CodeShifter<BITS, TL::kTwoRegs> sh;                // RNG
    if (!DET && q0 % NB == 0) {
      // noise of NB groups, two at a time: the octets of lane ^ 1 in the same two groups are
      // their neighbours (elem_base is a multiple of 256, so octet and lane parity agree)
#pragma unroll
      for (int p = 0; p < NB; p += 2) {
        const uint64_t o = (uint64_t)(elem_base >> 3) + (uint64_t)TL::group_of(half, q0 + p) * 32 + lane;
        Noise<T>::octets(o, o + 32, seed, offset, rw[p], rw[p + 1]);
      }
    }
#pragma unroll
    for (int r = R - 1; r >= 0; --r) {                 // last group first: see CodeShifter
      const int q = q0 + r;
      const int gl = TL::group_of(half, q);
      const float mul = s_mul[gl];
      const float sub = s_sub[gl];
      float v[8], nz[8];
      raw8_widen(raw[q], v);
      if (DET) raw8_widen(nzraw[DET ? q : 0], nz);
#pragma unroll
      for (int k = 7; k >= 0; --k) {
        if (DET) acc |= (uint64_t)det_code<T>(v[k], nz[k], mul, sub, Bf) << (r * WPG + k * BITS);
        else sh.push(RngFixed<T>::word(v[k], Noise<T>::at(rw[q % NB], k), mul, sub, kUnit));
      }
    }
    if (!DET) acc = ((uint64_t)sh.hi << 32) | sh.lo;
    const int glt = TL::group_of(half, q0);            // first group of this register tile
    const int64_t tile_words = word_base + (int64_t)glt * WPG;
    const uint32_t lo = transpose32((uint32_t)acc, lane);
    // each half-wave stores its own 4-byte words (whole 128-byte lines), non-temporally: 3 % faster
    // than plain stores, and no dirty lines are left behind for the next kernel
    int32_t* dst = packed + tile_words;
    if (TL::kTwoRegs) {
      const uint32_t hi = transpose32((uint32_t)(acc >> 32), lane);
      if (glt < groups_valid) {
        __builtin_nontemporal_store((int32_t)lo, dst + lane);
        if ((int)lane < WPG - 32) __builtin_nontemporal_store((int32_t)hi, dst + 32 + lane);
      }
    } else {
      if ((int)lane < R * WPG && glt + (int)lane / WPG < groups_valid)
        __builtin_nontemporal_store((int32_t)lo, dst + lane);
    }
  }
}

// ROWS: rows of F elements at any address, the last group padded with zeros.  S: the type the scales are
// written in; where it is not the tensor's own (bfloat16 for fp32), the minima are written in it as well.
template <typename T, typename S, bool DET, bool ROWS>
__global__ __launch_bounds__(kThreads, DET ? 1 : 8) void pack_mixed_kernel(
    const T* __restrict__ data, const T* __restrict__ mn, const T* __restrict__ mx,
    const int32_t* __restrict__ bits, const int32_t* __restrict__ prefix, S* __restrict__ scale,
    S* __restrict__ mn_out, int32_t* __restrict__ packed, const T* __restrict__ noise, uint64_t seed,
    uint64_t offset, int64_t N, int64_t F, int64_t G, FastDiv per_sample, const T* last) {
  constexpr int GPH = Gph<T>::kPack;
  constexpr int kUnit = 2 * GPH;                                 // groups of a wave
  __shared__ float s_mul[kWaves * kUnit];
  __shared__ float s_sub[kWaves * kUnit];
  const uint32_t wave = wave_of_block();
  const Unit u = unit_of<kUnit>(blockIdx.x * kWaves + wave, per_sample, N, G);
  const int64_t n = u.n, gb = u.gb;
  const int groups_valid = u.valid;
  const int64_t elem_base = (n * G + gb) * kGs;

  // The element loads do not depend on the bit width or the scales: get them in flight first,
  // then compute the block's scales while they travel.
  Raw8<T> v[GPH];
  Raw8<T> nz[DET ? GPH : 1];
  // fp32 in RNG mode: a lane's 8 elements are 32 bytes, so a direct load would touch every cache
  // line with two instructions of the wave.  The wave's groups (4 KiB, contiguous) instead travel
  // straight into LDS, one whole 1 KiB group per instruction and no registers, and each lane then
  // picks its 32 bytes out of LDS.
  constexpr bool kViaLds = sizeof(T) == 4 && !DET;
  __shared__ __align__(16) uint8_t s_stage[kViaLds ? kWaves * kUnit * kGs * 4 : 16];
  uint8_t* stage = s_stage + (kViaLds ? wave * (kUnit * kGs * 4) : 0);
  constexpr int kRowVectors = sizeof(T) == 4 ? 2 * GPH : GPH;
  RowVector st[ROWS ? kRowVectors : 1];                          // ROWS: by way of registers, at any address
  if constexpr (ROWS) {
#pragma unroll
    for (int i = 0; i < kRowVectors; ++i) {
      const int gl = sizeof(T) == 4 ? i : Tile<1, GPH>::group_of((threadIdx.x >> 5) & 1, i);
      const int64_t at = (gb + gl) * kGs + (sizeof(T) == 4 ? (threadIdx.x & 63) * 4 : (threadIdx.x & 31) * 8);
      st[i] = load16_row(data + n * F + at, gl < groups_valid ? part_of_row(F, at) : 0, last);
    }
  } else if constexpr (kViaLds) {
    const uint32_t wl = threadIdx.x & 63;
#pragma unroll
    for (int i = 0; i < kUnit; ++i) {
      if (i < groups_valid)
        load_to_lds16_nt(data + elem_base + (int64_t)i * kGs + wl * 4, stage + i * (kGs * 4));
    }
  } else {
    load_groups<T, DET, GPH>(data, noise, elem_base, groups_valid, v, nz);
  }

  const int b = bits[n];
  if (threadIdx.x < kWaves * kUnit) {
    float mul = 0.0f, sub = 0.0f;
    // thread t: group t % kUnit of wave t / kUnit, which may belong to another sample than this wave's
    const Unit ut = unit_of<kUnit>(blockIdx.x * kWaves + threadIdx.x / kUnit, per_sample, N, G);
    const int gt = (int)threadIdx.x % kUnit;
    if (gt < ut.valid) {
      const int64_t gi = ut.n * G + ut.gb + gt;
      const float lo = Conv<T>::load(mn, gi);
      const float sc = GroupQuant<T, DET>::prepare(lo, Conv<T>::load(mx, gi), bits[ut.n], mul, sub);
      Conv<S>::store(scale, gi, sc);
      if constexpr (sizeof(S) != sizeof(T)) Conv<S>::store(mn_out, gi, lo);
    }
    s_mul[threadIdx.x] = mul;
    s_sub[threadIdx.x] = sub;
  }
  if constexpr (ROWS) {
#pragma unroll
    for (int i = 0; i < kRowVectors; ++i) {
      if constexpr (sizeof(T) == 4)
        *reinterpret_cast<u32x4*>(stage + i * (kGs * 4) + (threadIdx.x & 63) * 16) = row_vector_ends<T>(st[i]);
      else
        v[i].a = row_vector_ends<T>(st[i]);
    }
  }
  __syncthreads();
  if constexpr (kViaLds) {
    if constexpr (!ROWS) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");             // this wave's own groups have landed
    const uint32_t lane = threadIdx.x & 31;
    const int half = (threadIdx.x >> 5) & 1;
#pragma unroll
    for (int q = 0; q < GPH; ++q) {
      const int gl = Tile<1, GPH>::group_of(half, q);
      raw8_zero(v[q]);
      if (gl < groups_valid) {
        const u32x4* src = reinterpret_cast<const u32x4*>(stage + gl * (kGs * 4) + lane * 32);
        v[q].a = src[0];
        v[q].b = src[1];
      }
    }
  }

  const int64_t word_base = (int64_t)prefix[n] * G * 8 + gb * 8 * b;
  switch (b) {
#define ACTNN_CASE(B_)                                                                          \
  case B_:                                                                                      \
    pack_groups<T, B_, DET>(v, nz, packed, elem_base, word_base, groups_valid,                  \
                            s_mul + wave * kUnit, s_sub + wave * kUnit, seed, offset);          \
    break;
    ACTNN_CASE(1) ACTNN_CASE(2) ACTNN_CASE(3) ACTNN_CASE(4)
    ACTNN_CASE(5) ACTNN_CASE(6) ACTNN_CASE(7) ACTNN_CASE(8)
#undef ACTNN_CASE
    default: break;   // bits outside 1..8 are rejected on the host when known; nothing is written
  }
}

// ---------------------------------------------------------------------------- unpack (gs = 256)
// ROWS: `out` is a row of F elements at any address and elem_base an offset in it.
template <typename T, int BITS, int ROWS>
ACTNN_DEV void unpack_groups(const int32_t* __restrict__ packed, T* __restrict__ out,
                             int64_t elem_base, int64_t F, int64_t word_base, int groups_valid,
                             float* s_scale, float* s_min, float my_scale, float my_min, u32x4* slab) {
  constexpr int kGroupsPerHalf = Gph<T>::kUnpack;
  constexpr bool kStage = IsF32<T>::value;
  float vs[kStage ? kGroupsPerHalf : 1][8];
  using TL = Tile<BITS, kGroupsPerHalf>;
  constexpr int R = TL::kGroupsPerReg;
  constexpr int WPG = TL::kWordsPerGroup;
  constexpr uint32_t kMask = (1u << BITS) - 1u;
  const uint32_t lane = threadIdx.x & 31;
  const int half = (threadIdx.x >> 5) & 1;

  uint32_t wlo[kGroupsPerHalf / R], whi[kGroupsPerHalf / R];
#pragma unroll
  for (int t = 0; t < kGroupsPerHalf / R; ++t) {
    const int glt = TL::group_of(half, t * R);
    const int64_t tile_words = word_base + (int64_t)glt * WPG;
    wlo[t] = 0;
    whi[t] = 0;
    if (TL::kTwoRegs) {
      if (glt < groups_valid) {
        wlo[t] = (uint32_t)packed[tile_words + lane];
        if ((int)lane < WPG - 32) whi[t] = (uint32_t)packed[tile_words + 32 + lane];
      }
    } else {
      if ((int)lane < R * WPG && glt + (int)lane / WPG < groups_valid)
        wlo[t] = (uint32_t)packed[tile_words + lane];
    }
  }
  // the wave's scales and minima go to LDS only now, after the word loads have been issued, so
  // that the two global round trips overlap; only lanes of the wave read them
  if ((int)(threadIdx.x & 63) < groups_valid) {
    s_scale[threadIdx.x & 63] = my_scale;
    s_min[threadIdx.x & 63] = my_min;
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
  for (int t = 0; t < kGroupsPerHalf / R; ++t) {
    const int q0 = t * R;
    uint64_t acc = transpose32(wlo[t], lane);
    if (TL::kTwoRegs) acc |= (uint64_t)transpose32(whi[t], lane) << 32;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int gl = TL::group_of(half, q0 + r);
      if (gl < groups_valid) {
        const Dequant<T> dq(s_scale[gl], s_min[gl]);
        if constexpr (sizeof(T) == 2 && BITS <= 2) {
          // A group at 1 or 2 bits has at most four distinct values.  Lane l evaluates level l & 3
          // (once instead of once per element), the four lanes of a quad exchange them (DPP
          // quad_perm broadcasts) into an 8-byte table, and every pair of elements is one byte
          // permute of that table.  Same arithmetic per level, hence the same bits.
          const float mine = dq(lane & 3u);
          const int h = (int)(sizeof(T) == 2 && IsBf16<T>::value ? float_to_bf16_bits(mine) : float_to_half_bits(mine));
          const uint32_t l0 = (uint32_t)__builtin_amdgcn_update_dpp(0, h, 0x00, 0xF, 0xF, true);   // quad_perm [0,0,0,0]
          const uint32_t l1 = (uint32_t)__builtin_amdgcn_update_dpp(0, h, 0x55, 0xF, 0xF, true);   // [1,1,1,1]
          const uint32_t l2 = (uint32_t)__builtin_amdgcn_update_dpp(0, h, 0xAA, 0xF, 0xF, true);   // [2,2,2,2]
          const uint32_t l3 = (uint32_t)__builtin_amdgcn_update_dpp(0, h, 0xFF, 0xF, 0xF, true);   // [3,3,3,3]
          const uint32_t lut_lo = l0 | (l1 << 16), lut_hi = l2 | (l3 << 16);
          const uint32_t a = (uint32_t)(acc >> (r * WPG));
          u32x4 outw;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const uint32_t c0 = (a >> (2 * j * BITS)) & kMask;
            const uint32_t c1 = (a >> ((2 * j + 1) * BITS)) & kMask;
            // bytes 2c, 2c+1 of the table for each of the two elements
            const uint32_t sel = (c0 * 0x0202u + 0x0100u) | ((c1 * 0x0202u + 0x0100u) << 16);
            outw[j] = __builtin_amdgcn_perm(lut_hi, lut_lo, sel);
          }
          const int64_t at = elem_base + (int64_t)gl * kGs + lane * 8;
          if constexpr (ROWS == kRowsPast) slab[gl * 32 + lane] = outw;
          else if constexpr (ROWS == kRowsCached) store16_part<false>(out + at, outw, part_of_row(F, at));
          else store16_nt(out + at, outw);
          continue;
        }
        float v[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = dq((uint32_t)(acc >> (r * WPG + k * BITS)) & kMask);
        if constexpr (kStage) {
#pragma unroll
          for (int k = 0; k < 8; ++k) vs[kStage ? q0 + r : 0][k] = v[k];
        } else if constexpr (ROWS == kRowsPast) {
          slab[gl * 32 + lane] = words_of8(out, v);
        } else if constexpr (ROWS == kRowsCached) {
          const int64_t at = elem_base + (int64_t)gl * kGs + lane * 8;
          store16_part<false>(out + at, words_of8(out, v), part_of_row(F, at));
        } else {
          store8_nt(out + elem_base + (int64_t)gl * kGs + lane * 8, v);
        }
      }
    }
  }
  if constexpr (kStage) {
    stage_out_f32<kGroupsPerHalf, ROWS>(reinterpret_cast<float*>(out), elem_base, F, groups_valid, slab, vs);
  } else if constexpr (ROWS == kRowsPast) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    store_unit_any(out + elem_base, reinterpret_cast<const uint32_t*>(slab), unit_count(F, elem_base, groups_valid));
  }
}

// S: the type the scales and minima are stored in.
template <typename T, typename S, int ROWS>
__global__ __launch_bounds__(kThreads) void unpack_mixed_kernel(
    const int32_t* __restrict__ packed, const int32_t* __restrict__ bits,
    const int32_t* __restrict__ prefix, const S* __restrict__ scale, const S* __restrict__ mn,
    T* __restrict__ out, int64_t N, int64_t F, int64_t G, FastDiv per_sample) {
  constexpr int kUnit = 2 * Gph<T>::kUnpack;                     // groups of a wave
  __shared__ float s_scale[kWaves * kUnit];
  __shared__ float s_min[kWaves * kUnit];
  constexpr bool kStage = IsF32<T>::value || ROWS == kRowsPast;
  constexpr int kSlab = kUnit * kGs * (int)sizeof(T) / 16;
  __shared__ u32x4 s_slab[kStage ? kWaves * kSlab : 1];
  const uint32_t wave = wave_of_block();
  u32x4* slab = s_slab + (kStage ? wave * kSlab : 0);
  const Unit u = unit_of<kUnit>(blockIdx.x * kWaves + wave, per_sample, N, G);
  const int64_t n = u.n, gb = u.gb;
  const int b = bits[n];
  const int groups_valid = u.valid;
  float my_scale = 0.0f, my_min = 0.0f;
  if ((int)(threadIdx.x & 63) < groups_valid) {
    const int64_t gi = n * G + gb + (threadIdx.x & 63);
    my_scale = Conv<S>::load(scale, gi);
    my_min = Conv<S>::load(mn, gi);
  }
  const int64_t elem_base = ROWS ? gb * kGs : (n * G + gb) * kGs;
  if constexpr (ROWS) out += n * F;
  const int64_t word_base = (int64_t)prefix[n] * G * 8 + gb * 8 * b;
  switch (b) {
#define ACTNN_CASE(B_)                                                                          \
  case B_:                                                                                      \
    unpack_groups<T, B_, ROWS>(packed, out, elem_base, F, word_base, groups_valid,              \
                               s_scale + wave * kUnit, s_min + wave * kUnit, my_scale, my_min,  \
                               slab);                                                           \
    break;
    ACTNN_CASE(1) ACTNN_CASE(2) ACTNN_CASE(3) ACTNN_CASE(4)
    ACTNN_CASE(5) ACTNN_CASE(6) ACTNN_CASE(7) ACTNN_CASE(8)
#undef ACTNN_CASE
    default: break;
  }
}

// ---------------------------------------------------------------------------- unpack, transposed
// The rows of a linear layer's input with the samples contiguous, out[feature * ld + sample], as the matrix
// product of its weight gradient reads them fastest: that product sums over the samples, and with both factors
// stored sample by sample its loads run across the rows (the product alone, bf16, go [N, O] and x [N, F], us with x as
// rows / with x like this / with go turned over as well: [8192, 4096] x [8192, 4096] 250 / 198 / 171, [4096, 4096] x
// [4096, 4096] 128 / 103 / 90, [2048, 4096] x [2048, 8192] 137 / 112 / 96, [65536, 1024] x [65536, 1024] 321 / 281 / 258).
// Bound by the write, as unpack: the values are unpack's bit for bit.  A half-wave takes 8 samples of one group (a
// block 64), whose words are loaded before the first is decoded.  The widths of the two halves of a wave
// differ, so the decoders take them at run time: the table of four levels where neither exceeds 2 bits.
template <typename T>
__global__ __launch_bounds__(kThreads) void unpack_mixed_transposed_kernel(
    const int32_t* __restrict__ packed, const int32_t* __restrict__ bits, const int32_t* __restrict__ prefix,
    const T* __restrict__ scale, const T* __restrict__ mn, T* __restrict__ out, int64_t N, int64_t F, int64_t G,
    int64_t ld, int64_t blocks, FastDiv by_groups) {
  __shared__ u32x4 s_tile[kGs * kTileSamples / 8];
  // (the groups of a tile of samples on one XCD: at 2 bits two neighbouring groups share a line of the stream)
  const int64_t block = xcd_block();
  if (block >= blocks) return;
  const uint32_t tile = by_groups.div((uint32_t)block), g = (uint32_t)block - tile * by_groups.d;
  const uint32_t lane = threadIdx.x & 31u, half = threadIdx.x >> 5;
  const int64_t sample0 = (int64_t)tile * kTileSamples, n0 = sample0 + 8 * half;
  // lane l looks up sample l & 7 of the half-wave's eight
  const int64_t nl = n0 + (lane & 7u) < N ? n0 + (lane & 7u) : N - 1;
  const int width = bits[nl];
  const int my_bits = width < 1 || width > 8 ? 0 : width;      // (a width that there is not has no words to read)
  const int my_prefix = prefix[nl];
  const float my_scale = Conv<T>::load(scale, nl * G + g), my_min = Conv<T>::load(mn, nl * G + g);
  uint32_t lo[8], hi[8];
  int b[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    b[i] = __shfl(my_bits, i, 32);
    const int32_t* words = packed + (int64_t)__shfl(my_prefix, i, 32) * G * 8 + (int64_t)g * b[i] * 8;
    lo[i] = (int)lane < 8 * b[i] ? (uint32_t)words[lane] : 0u;
    hi[i] = (int)lane + 32 < 8 * b[i] ? (uint32_t)words[lane + 32] : 0u;
  }
  uint32_t w[8][4];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const Dequant<T> dq(__shfl(my_scale, i, 32), __shfl(my_min, i, 32));
    const uint32_t acc = transpose32(lo[i], lane);
    if (__builtin_amdgcn_ballot_w64(b[i] > 2) == 0) {
      // (as unpack_groups: lane l evaluates level l & 3, a byte permute picks the two values of a word)
      const float mine = dq(lane & 3u);
      const int h = (int)(IsBf16<T>::value ? float_to_bf16_bits(mine) : float_to_half_bits(mine));
      const uint32_t l0 = (uint32_t)__builtin_amdgcn_update_dpp(0, h, 0x00, 0xF, 0xF, true);
      const uint32_t l1 = (uint32_t)__builtin_amdgcn_update_dpp(0, h, 0x55, 0xF, 0xF, true);
      const uint32_t l2 = (uint32_t)__builtin_amdgcn_update_dpp(0, h, 0xAA, 0xF, 0xF, true);
      const uint32_t l3 = (uint32_t)__builtin_amdgcn_update_dpp(0, h, 0xFF, 0xF, 0xF, true);
      const uint32_t lut_lo = l0 | (l1 << 16), lut_hi = l2 | (l3 << 16);
      const uint32_t pair = ((1u << b[i]) - 1u) * 0x00010001u;
      const uint32_t a = acc & 0xffffu, both = a | (a << (16 - b[i]));
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t sel = __umul24((both >> (2 * j * b[i])) & pair, 0x0202u) + 0x01000100u;
        w[i][j] = __builtin_amdgcn_perm(lut_hi, lut_lo, sel);
      }
    } else {
      uint64_t codes = acc;
      if (__builtin_amdgcn_ballot_w64(b[i] > 4) != 0) codes |= (uint64_t)transpose32(hi[i], lane) << 32;
      const uint32_t mask = (1u << b[i]) - 1u;
      float v[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = dq((uint32_t)(codes >> (k * b[i])) & mask);
      const u32x4 packed8 = words_of8(out, v);
#pragma unroll
      for (int j = 0; j < 4; ++j) w[i][j] = packed8[j];
    }
    if (n0 + i >= N) {                                 // the row's end up to ld
#pragma unroll
      for (int j = 0; j < 4; ++j) w[i][j] = 0u;
    }
  }
  store_transposed_tile(w, s_tile, out, (int64_t)g * kGs, F, sample0, ld);
}

// ---------------------------------------------------------------------------- generic group size
// One block per (sample, group); codes staged as bytes in LDS, then thread w assembles word w.
template <typename T, bool DET>
__global__ __launch_bounds__(kThreads) void pack_mixed_generic_kernel(
    const T* __restrict__ data, const T* __restrict__ mn, const T* __restrict__ mx,
    const int32_t* __restrict__ bits, const int32_t* __restrict__ prefix, T* __restrict__ scale,
    int32_t* __restrict__ packed, const T* __restrict__ noise, uint64_t seed, uint64_t offset,
    int64_t G, int gs) {
  __shared__ uint8_t s_code[1024];
  __shared__ float s_par[2];
  const int64_t n = blockIdx.x / G;
  const int64_t g = blockIdx.x % G;
  const int b = bits[n];
  if (b < 1 || b > 8) return;
  const int64_t gi = n * G + g;
  if (threadIdx.x == 0) {
    float mul, sub;
    const float sc = GroupQuant<T, DET>::prepare(Conv<T>::load(mn, gi), Conv<T>::load(mx, gi), b, mul, sub);
    Conv<T>::store(scale, gi, sc);
    s_par[0] = mul;
    s_par[1] = sub;
  }
  __syncthreads();
  const float mul = s_par[0], sub = s_par[1];
  const float Bf = (float)((1 << b) - 1);
  for (int d = threadIdx.x; d < gs; d += kThreads) {
    const int64_t e = gi * gs + d;
    const float x = Conv<T>::load(data, e);
    uint32_t c;
    if (DET) {
      c = det_code<T>(x, Conv<T>::load(noise, e), mul, sub, Bf);
    } else {
      uint32_t w[Noise<T>::kWords];
      Noise<T>::octet((uint64_t)e >> 3, seed, offset, w);
      uint32_t r = Noise<T>::at(w, 0);
#pragma unroll
      for (int k = 1; k < 8; ++k) r = ((int)(e & 7) == k) ? Noise<T>::at(w, k) : r;
      c = RngFixed<T>::word(x, r, mul, sub, RngFixed<T>::unit(b)) >> (32 - b);
    }
    s_code[d] = (uint8_t)c;
  }
  __syncthreads();
  const int E = gs / 32;
  const int L = E * b;
  const int64_t word_base = ((int64_t)prefix[n] * G + (int64_t)b * g) * E;
  for (int w = threadIdx.x; w < L; w += kThreads) {
    const int k = w / b, i = w % b;
    uint32_t word = 0;
    for (int j = 0; j < 32; ++j) word |= ((uint32_t)(s_code[E * j + k] >> i) & 1u) << j;
    packed[word_base + w] = (int32_t)word;
  }
}

template <typename T>
__global__ __launch_bounds__(kThreads) void unpack_mixed_generic_kernel(
    const int32_t* __restrict__ packed, const int32_t* __restrict__ bits,
    const int32_t* __restrict__ prefix, const T* __restrict__ scale, const T* __restrict__ mn,
    T* __restrict__ out, int64_t G, int gs) {
  __shared__ uint32_t s_word[256];   // E * b <= 32 * 8
  const int64_t n = blockIdx.x / G;
  const int64_t g = blockIdx.x % G;
  const int b = bits[n];
  if (b < 1 || b > 8) return;
  const int E = gs / 32;
  const int L = E * b;
  const int64_t word_base = ((int64_t)prefix[n] * G + (int64_t)b * g) * E;
  for (int w = threadIdx.x; w < L; w += kThreads) s_word[w] = (uint32_t)packed[word_base + w];
  __syncthreads();
  const int64_t gi = n * G + g;
  const Dequant<T> dq(Conv<T>::load(scale, gi), Conv<T>::load(mn, gi));
  for (int d = threadIdx.x; d < gs; d += kThreads) {
    const int j = d / E, k = d % E;
    uint32_t c = 0;
    for (int i = 0; i < b; ++i) c |= ((s_word[k * b + i] >> j) & 1u) << i;
    Conv<T>::store(out, gi * gs + d, dq(c));
  }
}

// ---------------------------------------------------------------------------- prefix sum
__global__ __launch_bounds__(1024) void bits_prefix_kernel(const int32_t* __restrict__ bits,
                                                           int32_t* __restrict__ prefix, int64_t N) {
  __shared__ int32_t s_part[1024];
  // thread t owns the contiguous chunk [t * per, (t + 1) * per)
  const int64_t per = (N + 1023) / 1024;
  const int64_t lo = (int64_t)threadIdx.x * per;
  const int64_t hi = lo + per < N ? lo + per : N;
  int32_t sum = 0;
  for (int64_t i = lo; i < hi; ++i) sum += bits[i];
  s_part[threadIdx.x] = sum;
  __syncthreads();
  for (int off = 1; off < 1024; off <<= 1) {           // inclusive Hillis-Steele scan
    int32_t add = threadIdx.x >= (unsigned)off ? s_part[threadIdx.x - off] : 0;
    __syncthreads();
    s_part[threadIdx.x] += add;
    __syncthreads();
  }
  int32_t run = threadIdx.x == 0 ? 0 : s_part[threadIdx.x - 1];
  if (threadIdx.x == 0) prefix[0] = 0;
  for (int64_t i = lo; i < hi; ++i) {
    run += bits[i];
    prefix[i + 1] = run;
  }
}

// Units of `groups` groups per sample and the blocks of four that cover them all.  Numbers of units stay
// below 2^31: a sample of several units holds more than 1024 elements (fp32; 2048 in 16 bits), so that only a tensor
// of 4 TiB has as many, and one of shorter rows has a unit to a row, as it had a block before.
bool unit_grid(int64_t N, int64_t G, int groups, int64_t& per_sample, int64_t& blocks) {
  per_sample = (G + groups - 1) / groups;
  if (per_sample > 0x7fffffffLL / N) return false;
  blocks = (N * per_sample + kWaves - 1) / kWaves;
  return true;
}

template <typename T, typename S, bool DET, bool ROWS>
int launch_pack_groups(const void* data, const void* mn, const void* mx, const int32_t* bits, const int32_t* prefix,
                       void* scale, void* mn_out, int32_t* packed, const void* noise, uint64_t seed, uint64_t offset,
                       int64_t N, int64_t F, hipStream_t s) {
  const int64_t G = (F + kGs - 1) / kGs;
  int64_t per_sample, blocks;
  if (!unit_grid(N, G, 2 * Gph<T>::kPack, per_sample, blocks)) return ACTNN_EINVAL;
  const T* d = static_cast<const T*>(data);
  pack_mixed_kernel<T, S, DET, ROWS><<<dim3((unsigned)blocks), dim3(kThreads), 0, s>>>(
      d, static_cast<const T*>(mn), static_cast<const T*>(mx), bits, prefix,
      static_cast<S*>(scale), static_cast<S*>(mn_out), packed, static_cast<const T*>(noise), seed, offset, N, F, G,
      FastDiv((uint32_t)per_sample), d + N * F - 16 / sizeof(T));
  ACTNN_RETURN_LAUNCH_STATUS();
}

template <typename T, typename S, int ROWS>
int launch_unpack_groups(const int32_t* packed, const int32_t* bits, const int32_t* prefix, const void* scale,
                         const void* mn, void* out, int64_t N, int64_t F, hipStream_t s) {
  const int64_t G = (F + kGs - 1) / kGs;
  int64_t per_sample, blocks;
  if (!unit_grid(N, G, 2 * Gph<T>::kUnpack, per_sample, blocks)) return ACTNN_EINVAL;
  unpack_mixed_kernel<T, S, ROWS><<<dim3((unsigned)blocks), dim3(kThreads), 0, s>>>(
      packed, bits, prefix, static_cast<const S*>(scale), static_cast<const S*>(mn), static_cast<T*>(out), N, F, G,
      FastDiv((uint32_t)per_sample));
  ACTNN_RETURN_LAUNCH_STATUS();
}

template <typename T>
int launch_unpack_transposed(const int32_t* packed, const int32_t* bits, const int32_t* prefix, const void* scale,
                             const void* mn, void* out, int64_t N, int64_t F, int64_t ld, hipStream_t s) {
  const int64_t G = (F + kGs - 1) / kGs, tiles = (N + kTileSamples - 1) / kTileSamples;
  if (tiles > (0x7fffffffLL - kXcds) / G) return ACTNN_EINVAL;
  unpack_mixed_transposed_kernel<T><<<dim3(xcd_grid(tiles * G)), dim3(kThreads), 0, s>>>(
      packed, bits, prefix, static_cast<const T*>(scale), static_cast<const T*>(mn), static_cast<T*>(out), N, F, G, ld,
      tiles * G, FastDiv((uint32_t)G));
  ACTNN_RETURN_LAUNCH_STATUS();
}

// whole groups at an aligned address take the kernels without the row ends
template <typename T, typename S>
int launch_pack_rows(const void* data, const void* mn, const void* mx, const int32_t* bits, const int32_t* prefix,
                     void* scale, void* mn_out, int32_t* packed, uint64_t seed, uint64_t offset, int64_t N, int64_t F,
                     hipStream_t s) {
  if (F % kGs == 0 && aligned16(data))
    return launch_pack_groups<T, S, false, false>(data, mn, mx, bits, prefix, scale, mn_out, packed, nullptr, seed, offset, N, F, s);
  return launch_pack_groups<T, S, false, true>(data, mn, mx, bits, prefix, scale, mn_out, packed, nullptr, seed, offset, N, F, s);
}

template <typename T, typename S>
int launch_unpack_rows(const int32_t* packed, const int32_t* bits, const int32_t* prefix, const void* scale,
                       const void* mn, void* out, int64_t N, int64_t F, hipStream_t s) {
  if (F % kGs == 0) return launch_unpack_groups<T, S, kWholeRows>(packed, bits, prefix, scale, mn, out, N, F, s);
  if (stream_rows(N * F * (int64_t)sizeof(T)))
    return launch_unpack_groups<T, S, kRowsPast>(packed, bits, prefix, scale, mn, out, N, F, s);
  return launch_unpack_groups<T, S, kRowsCached>(packed, bits, prefix, scale, mn, out, N, F, s);
}

template <typename T>
int launch_pack(const void* data, const void* mn, const void* mx, const int32_t* bits,
                const int32_t* prefix, void* scale, int32_t* packed, const void* noise,
                uint64_t seed, uint64_t offset, int64_t N, int64_t G, int64_t gs, hipStream_t s) {
  const T* d = static_cast<const T*>(data);
  const T* nz = static_cast<const T*>(noise);
  if (gs == kGs) {
    if (noise)
      return launch_pack_groups<T, T, true, false>(data, mn, mx, bits, prefix, scale, nullptr, packed, noise, seed, offset, N, G * kGs, s);
    return launch_pack_groups<T, T, false, false>(data, mn, mx, bits, prefix, scale, nullptr, packed, noise, seed, offset, N, G * kGs, s);
  } else {
    if (N * G > 0x7fffffffLL) return ACTNN_EINVAL;
    const dim3 grid((unsigned)(N * G));
    if (noise)
      pack_mixed_generic_kernel<T, true><<<grid, dim3(kThreads), 0, s>>>(
          d, static_cast<const T*>(mn), static_cast<const T*>(mx), bits, prefix,
          static_cast<T*>(scale), packed, nz, seed, offset, G, (int)gs);
    else
      pack_mixed_generic_kernel<T, false><<<grid, dim3(kThreads), 0, s>>>(
          d, static_cast<const T*>(mn), static_cast<const T*>(mx), bits, prefix,
          static_cast<T*>(scale), packed, nz, seed, offset, G, (int)gs);
  }
  ACTNN_RETURN_LAUNCH_STATUS();
}

template <typename T>
int launch_unpack(const int32_t* packed, const int32_t* bits, const int32_t* prefix,
                  const void* scale, const void* mn, void* out, int64_t N, int64_t G, int64_t gs,
                  hipStream_t s) {
  if (gs == kGs) {
    return launch_unpack_groups<T, T, kWholeRows>(packed, bits, prefix, scale, mn, out, N, G * kGs, s);
  } else {
    if (N * G > 0x7fffffffLL) return ACTNN_EINVAL;
    unpack_mixed_generic_kernel<T><<<dim3((unsigned)(N * G)), dim3(kThreads), 0, s>>>(
        packed, bits, prefix, static_cast<const T*>(scale), static_cast<const T*>(mn),
        static_cast<T*>(out), G, (int)gs);
  }
  ACTNN_RETURN_LAUNCH_STATUS();
}

}  // namespace

// pack of [N, F] rows with the scales (and, for bfloat16 of fp32 rows, the minima) written in store_dtype
// (actnn_quantize_rows has checked the arguments)
int pack_mixed_rows(const void* data, const void* mn, const void* mx, const int32_t* bits, const int32_t* prefix,
                    void* scale, void* mn_out, int32_t* packed, uint64_t seed, uint64_t offset, int64_t N, int64_t F,
                    int dtype, int store_dtype, hipStream_t s) {
  if (dtype == ACTNN_F32 && store_dtype == ACTNN_BF16)
    return launch_pack_rows<float, bf16_t>(data, mn, mx, bits, prefix, scale, mn_out, packed, seed, offset, N, F, s);
  if (dtype != store_dtype) return ACTNN_EDTYPE;
  switch (dtype) {
    case ACTNN_F32: return launch_pack_rows<float, float>(data, mn, mx, bits, prefix, scale, mn_out, packed, seed, offset, N, F, s);
    case ACTNN_F16: return launch_pack_rows<__half, __half>(data, mn, mx, bits, prefix, scale, mn_out, packed, seed, offset, N, F, s);
    case ACTNN_BF16: return launch_pack_rows<bf16_t, bf16_t>(data, mn, mx, bits, prefix, scale, mn_out, packed, seed, offset, N, F, s);
    default: return ACTNN_EDTYPE;
  }
}

}  // namespace actnn

extern "C" int actnn_unpack_mixed_rows(const int32_t* packed, const int32_t* bits, const int32_t* prefix,
                                       const void* scale, const void* mn, void* out, int64_t N, int64_t F, int dtype,
                                       int store_dtype, void* stream) {
  using namespace actnn;
  if (N < 0 || F < 0) return ACTNN_EINVAL;
  if (N == 0 || F == 0) return ACTNN_OK;
  if (!packed || !bits || !prefix || !scale || !mn || !out) return ACTNN_EINVAL;
  if (!aligned16(out)) return ACTNN_EALIGN;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dtype == ACTNN_F32 && store_dtype == ACTNN_BF16)
    return launch_unpack_rows<float, bf16_t>(packed, bits, prefix, scale, mn, out, N, F, s);
  if (dtype != store_dtype) return ACTNN_EDTYPE;
  switch (dtype) {
    case ACTNN_F32: return launch_unpack_rows<float, float>(packed, bits, prefix, scale, mn, out, N, F, s);
    case ACTNN_F16: return launch_unpack_rows<__half, __half>(packed, bits, prefix, scale, mn, out, N, F, s);
    case ACTNN_BF16: return launch_unpack_rows<bf16_t, bf16_t>(packed, bits, prefix, scale, mn, out, N, F, s);
    default: return ACTNN_EDTYPE;
  }
}

extern "C" int actnn_unpack_mixed_rows_transposed(const int32_t* packed, const int32_t* bits, const int32_t* prefix,
                                                  const void* scale, const void* mn, void* out, int64_t N, int64_t F,
                                                  int64_t ld, int dtype, void* stream) {
  using namespace actnn;
  if (N < 0 || F < 0 || ld < N || ld % 8 != 0 || ld > (N + kTileSamples - 1) / kTileSamples * kTileSamples) return ACTNN_EINVAL;
  if (N == 0 || F == 0) return ACTNN_OK;
  if (!packed || !bits || !prefix || !scale || !mn || !out) return ACTNN_EINVAL;
  if (!aligned16(out)) return ACTNN_EALIGN;
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (dtype) {
    case ACTNN_F16: return launch_unpack_transposed<__half>(packed, bits, prefix, scale, mn, out, N, F, ld, s);
    case ACTNN_BF16: return launch_unpack_transposed<bf16_t>(packed, bits, prefix, scale, mn, out, N, F, ld, s);
    default: return ACTNN_EDTYPE;
  }
}

extern "C" int actnn_bits_prefix(const int32_t* bits, int32_t* prefix, int64_t N, void* stream) {
  using namespace actnn;
  if (N < 0 || !prefix || (N > 0 && !bits)) return ACTNN_EINVAL;
  bits_prefix_kernel<<<dim3(1), dim3(1024), 0, static_cast<hipStream_t>(stream)>>>(bits, prefix, N);
  ACTNN_RETURN_LAUNCH_STATUS();
}

extern "C" int actnn_pack_mixed(const void* data, const void* mn, const void* mx,
                                const int32_t* bits, const int32_t* prefix, void* scale,
                                int32_t* packed, const void* noise, uint64_t seed, uint64_t offset,
                                int64_t N, int64_t G, int64_t gs, int dtype, void* stream) {
  using namespace actnn;
  if (N < 0 || G < 0 || gs < 32 || gs > 1024 || gs % 32 != 0) return ACTNN_EINVAL;
  if (N == 0 || G == 0) return ACTNN_OK;
  if (!data || !mn || !mx || !bits || !prefix || !scale || !packed) return ACTNN_EINVAL;
  if (!aligned16(data) || (noise && !aligned16(noise))) return ACTNN_EALIGN;
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (dtype) {
    case ACTNN_F32: return launch_pack<float>(data, mn, mx, bits, prefix, scale, packed, noise, seed, offset, N, G, gs, s);
    case ACTNN_F16: return launch_pack<__half>(data, mn, mx, bits, prefix, scale, packed, noise, seed, offset, N, G, gs, s);
    case ACTNN_BF16: return launch_pack<bf16_t>(data, mn, mx, bits, prefix, scale, packed, noise, seed, offset, N, G, gs, s);
    default: return ACTNN_EDTYPE;
  }
}

extern "C" int actnn_unpack_mixed(const int32_t* packed, const int32_t* bits, const int32_t* prefix,
                                  const void* scale, const void* mn, void* out, int64_t N,
                                  int64_t G, int64_t gs, int dtype, void* stream) {
  using namespace actnn;
  if (N < 0 || G < 0 || gs < 32 || gs > 1024 || gs % 32 != 0) return ACTNN_EINVAL;
  if (N == 0 || G == 0) return ACTNN_OK;
  if (!packed || !bits || !prefix || !scale || !mn || !out) return ACTNN_EINVAL;
  if (!aligned16(out)) return ACTNN_EALIGN;
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (dtype) {
    case ACTNN_F32: return launch_unpack<float>(packed, bits, prefix, scale, mn, out, N, G, gs, s);
    case ACTNN_F16: return launch_unpack<__half>(packed, bits, prefix, scale, mn, out, N, G, gs, s);
    case ACTNN_BF16: return launch_unpack<bf16_t>(packed, bits, prefix, scale, mn, out, N, G, gs, s);
    default: return ACTNN_EDTYPE;
  }
}
