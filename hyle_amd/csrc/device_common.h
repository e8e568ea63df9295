// device_common.h -- device-side building blocks shared by the gfx950 kernels:
// storage codecs, 128-bit vector access and wave64 reductions.
//
// Storage codecs follow include/hyle/simd/dtype.h:55-121 of the reference:
// bf16 is RN-even with NaN keeping its upper payload and gaining the quiet bit;
// f16 uses the hardware converters (IEEE RN-even, exact subnormals) with NaN
// forced to mantissa 0x3FF.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace hyle_hip {

constexpr int kBlockThreads = 256;
constexpr int kWaveLanes = 64;

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_element __attribute__((ext_vector_type(4), aligned(2)));  // at any element's address

struct F32 {};
struct F16 {};
struct BF16 {};

__device__ __forceinline__ float bits_f32(uint32_t u) { return __uint_as_float(u); }
__device__ __forceinline__ uint32_t f32_bits(float f) { return __float_as_uint(f); }

// f32 -> bf16 with the gfx950 converter (v_cvt_pk_bf16_f32).  It was compared on the
// device with the reference rule of include/hyle/simd/dtype.h:114-121 (RN-even, NaN keeps
// its upper payload and gains the quiet bit) over all 2^32 f32 patterns: identical.
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
  const f32x2 in = {lo, hi};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(in, bf16x2));
}
__device__ __forceinline__ uint16_t f32_to_bf16(float f) {
  return (uint16_t)(pack_bf16x2(f, 0.0f) & 0xFFFFu);
}
// the value after one trip through bf16 storage
__device__ __forceinline__ float bf16_round_trip(float f) {
  return bits_f32(pack_bf16x2(f, 0.0f) << 16);
}
__device__ __forceinline__ float bf16_lo(uint32_t w) { return bits_f32(w << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t w) { return bits_f32(w & 0xFFFF0000u); }

__device__ __forceinline__ float f16_to_f32(uint16_t h) {
  return (float)__builtin_bit_cast(_Float16, h);
}
// The value is made opaque before it is narrowed: left alone, the compiler fuses a preceding
// multiply by a widened f16 into v_fma_mixlo_f16 (a * b + 0), and that +0 addend turns a
// product of -0 into +0.
__device__ __forceinline__ uint16_t f32_to_f16(float f) {
  asm("" : "+v"(f));
  const uint16_t h = __builtin_bit_cast(uint16_t, (_Float16)f);
  const uint16_t nan = (uint16_t)(((f32_bits(f) >> 16) & 0x8000u) | 0x7FFFu);
  return (f != f) ? nan : h;
}

// Two values narrowed by one v_cvt_pk_f16_f32, under the same rules as f32_to_f16.
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pack_f16x2(float lo, float hi) {
  asm("" : "+v"(lo), "+v"(hi));
  const f32x2 in = {lo, hi};
  const uint32_t pair = __builtin_bit_cast(uint32_t, __builtin_convertvector(in, f16x2));
  const uint32_t nans = ((f32_bits(lo) >> 16) & 0x8000u) | (f32_bits(hi) & 0x80000000u) | 0x7FFF7FFFu;
  const uint32_t take = (lo != lo ? 0x0000FFFFu : 0u) | (hi != hi ? 0xFFFF0000u : 0u);
  return (pair & ~take) | (nans & take);
}

// ---- per-type traits: element size, elements per 16-byte vector, scalar and
// ---- vector load/store through f32 -----------------------------------------
template <class T> struct Traits;

template <> struct Traits<F32> {
  static constexpr int kSize = 4;
  static constexpr int kVec = 4;
  static __device__ __forceinline__ float load(const void *p, size_t i) {
    return static_cast<const float *>(p)[i];
  }
  static __device__ __forceinline__ void store(void *p, size_t i, float v) {
    static_cast<float *>(p)[i] = v;
  }
  static __device__ __forceinline__ float round(float v) { return v; }
  static __device__ __forceinline__ void unpack(u32x4 w, float (&v)[4]) {
    v[0] = bits_f32(w.x); v[1] = bits_f32(w.y); v[2] = bits_f32(w.z); v[3] = bits_f32(w.w);
  }
  static __device__ __forceinline__ u32x4 pack(const float (&v)[4]) {
    u32x4 w;
    w.x = f32_bits(v[0]); w.y = f32_bits(v[1]); w.z = f32_bits(v[2]); w.w = f32_bits(v[3]);
    return w;
  }
};

template <> struct Traits<BF16> {
  static constexpr int kSize = 2;
  static constexpr int kVec = 8;
  static __device__ __forceinline__ float load(const void *p, size_t i) {
    return bits_f32((uint32_t)static_cast<const uint16_t *>(p)[i] << 16);
  }
  static __device__ __forceinline__ void store(void *p, size_t i, float v) {
    static_cast<uint16_t *>(p)[i] = f32_to_bf16(v);
  }
  // value after one trip through storage
  static __device__ __forceinline__ float round(float v) { return bf16_round_trip(v); }
  static __device__ __forceinline__ void unpack(u32x4 w, float (&v)[8]) {
    v[0] = bf16_lo(w.x); v[1] = bf16_hi(w.x); v[2] = bf16_lo(w.y); v[3] = bf16_hi(w.y);
    v[4] = bf16_lo(w.z); v[5] = bf16_hi(w.z); v[6] = bf16_lo(w.w); v[7] = bf16_hi(w.w);
  }
  static __device__ __forceinline__ u32x4 pack(const float (&v)[8]) {
    u32x4 w;
    w.x = pack_bf16x2(v[0], v[1]); w.y = pack_bf16x2(v[2], v[3]);
    w.z = pack_bf16x2(v[4], v[5]); w.w = pack_bf16x2(v[6], v[7]);
    return w;
  }
};

template <> struct Traits<F16> {
  static constexpr int kSize = 2;
  static constexpr int kVec = 8;
  static __device__ __forceinline__ float load(const void *p, size_t i) {
    return f16_to_f32(static_cast<const uint16_t *>(p)[i]);
  }
  static __device__ __forceinline__ void store(void *p, size_t i, float v) {
    static_cast<uint16_t *>(p)[i] = f32_to_f16(v);
  }
  static __device__ __forceinline__ float round(float v) { return f16_to_f32(f32_to_f16(v)); }
  static __device__ __forceinline__ void unpack(u32x4 w, float (&v)[8]) {
    v[0] = f16_to_f32((uint16_t)w.x); v[1] = f16_to_f32((uint16_t)(w.x >> 16));
    v[2] = f16_to_f32((uint16_t)w.y); v[3] = f16_to_f32((uint16_t)(w.y >> 16));
    v[4] = f16_to_f32((uint16_t)w.z); v[5] = f16_to_f32((uint16_t)(w.z >> 16));
    v[6] = f16_to_f32((uint16_t)w.w); v[7] = f16_to_f32((uint16_t)(w.w >> 16));
  }
  static __device__ __forceinline__ u32x4 pack(const float (&v)[8]) {
    u32x4 w;
    w.x = pack_f16x2(v[0], v[1]); w.y = pack_f16x2(v[2], v[3]);
    w.z = pack_f16x2(v[4], v[5]); w.w = pack_f16x2(v[6], v[7]);
    return w;
  }
};

// A fence for the compiler only: the loads written before it are issued before it and no
// later load is hoisted above it, and the named registers must hold their loaded values here.
// Used after a group of independent loads so that they are all in flight together instead of
// being sunk next to their first use, one memory latency after another.
__device__ __forceinline__ void loads_issued(u32x4 &a) { asm volatile("" : "+v"(a) : : "memory"); }
__device__ __forceinline__ void loads_issued(uint32_t &a) { asm volatile("" : "+v"(a) : : "memory"); }

// 16-byte global access.  Streaming data is touched once, so loads and stores
// carry the non-temporal hint; small reused operands use the plain forms.
__device__ __forceinline__ u32x4 load16_stream(const void *base, size_t vec) {
  return __builtin_nontemporal_load(static_cast<const u32x4 *>(base) + vec);
}
__device__ __forceinline__ u32x4 load16(const void *base, size_t vec) {
  return static_cast<const u32x4 *>(base)[vec];
}
__device__ __forceinline__ void store16_stream(void *base, size_t vec, u32x4 w) {
  __builtin_nontemporal_store(w, static_cast<u32x4 *>(base) + vec);
}
__device__ __forceinline__ void store16(void *base, size_t vec, u32x4 w) {
  static_cast<u32x4 *>(base)[vec] = w;
}

// ---- wave64 butterflies ----------------------------------------------------
// The first four steps stay inside a 16-lane DPP row (quad swaps, half-row and
// row mirrors); steps 16 and 32 cross rows through the LDS crossbar without
// touching LDS memory.  Every participating lane ends with the full result.
template <int kCtrl> __device__ __forceinline__ float dpp_move(float v) {
  return __int_as_float(
      __builtin_amdgcn_update_dpp(0, __float_as_int(v), kCtrl, 0xF, 0xF, true));
}
template <int kCtrl> __device__ __forceinline__ int dpp_move(int v) {
  return __builtin_amdgcn_update_dpp(0, v, kCtrl, 0xF, 0xF, true);
}
constexpr int kDppSwap1 = 0xB1;        // quad_perm [1,0,3,2]
constexpr int kDppSwap2 = 0x4E;        // quad_perm [2,3,0,1]
constexpr int kDppHalfMirror = 0x141;  // lane i <-> 7 - i within 8
constexpr int kDppRowMirror = 0x140;   // lane i <-> 15 - i within 16

// The value of the lane kStep places below, as __shfl_up has it but without a trip through LDS (about a hundred
// cycles each, in a row in a scan): neighbours by the wavefront shift, rows of sixteen and halves by the lane
// swaps.  Lanes below kStep come back with some lane's value.
template <int kStep> __device__ __forceinline__ uint32_t lane_up(uint32_t v) {
  static_assert(kStep == 1 || kStep == 2 || kStep == 4 || kStep == 8 || kStep == 16 || kStep == 32, "a step of a scan");
  if constexpr (kStep == 32) {
    return __builtin_amdgcn_permlane32_swap(v, v, false, false)[0];  // the lower half in both
  } else if constexpr (kStep == 16) {
    const auto rows = __builtin_amdgcn_permlane16_swap(v, v, false, false);  // rows 0 0 2 2 and 1 1 3 3
    const auto first = __builtin_amdgcn_permlane32_swap(rows[1], rows[1], false, false);
    return (threadIdx.x & 48u) == 32u ? first[0] : rows[0];
  } else if constexpr (kStep == 8) {
    const uint32_t turned = (uint32_t)dpp_move<0x128>((int)v);  // row_ror:8
    const uint32_t above = lane_up<16>(turned);
    return (threadIdx.x & 8u) != 0 ? turned : above;
  } else {
#pragma unroll
    for (int i = 0; i < kStep; ++i) v = (uint32_t)dpp_move<0x138>((int)v);  // wave_shr:1
    return v;
  }
}
template <int kStep> __device__ __forceinline__ double lane_up(double v) {
  const uint64_t bits = __builtin_bit_cast(uint64_t, v);
  return __builtin_bit_cast(double, ((uint64_t)lane_up<kStep>((uint32_t)(bits >> 32)) << 32) | lane_up<kStep>((uint32_t)bits));
}
// One lane's value, the same lane for the whole wave.
__device__ __forceinline__ float lane_value(float v, int lane) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane)); }
__device__ __forceinline__ double lane_value(double v, int lane) {
  const uint64_t bits = __builtin_bit_cast(uint64_t, v);
  return __builtin_bit_cast(double, ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(bits >> 32), lane) << 32) |
                                        (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)bits, lane));
}
// v of this lane + v of lane ^ kStep (addition commutes: the sums of the two are the same bits)
template <int kStep> __device__ __forceinline__ double add_xor(double v) {
  const uint64_t bits = __builtin_bit_cast(uint64_t, v);
  const uint32_t low = (uint32_t)bits, high = (uint32_t)(bits >> 32);
  auto joined = [](uint32_t h, uint32_t l) { return __builtin_bit_cast(double, ((uint64_t)h << 32) | l); };
  if constexpr (kStep == 32) {
    const auto h = __builtin_amdgcn_permlane32_swap(high, high, false, false), l = __builtin_amdgcn_permlane32_swap(low, low, false, false);
    return joined(h[0], l[0]) + joined(h[1], l[1]);
  } else if constexpr (kStep == 16) {
    const auto h = __builtin_amdgcn_permlane16_swap(high, high, false, false), l = __builtin_amdgcn_permlane16_swap(low, low, false, false);
    return joined(h[0], l[0]) + joined(h[1], l[1]);
  } else {
    auto moved = [](uint32_t w) {
      if constexpr (kStep == 1) return (uint32_t)dpp_move<kDppSwap1>((int)w);
      else if constexpr (kStep == 2) return (uint32_t)dpp_move<kDppSwap2>((int)w);
      else if constexpr (kStep == 4) return (uint32_t)dpp_move<0x1B>(dpp_move<kDppHalfMirror>((int)w));  // and quad_perm [3,2,1,0]
      else return (uint32_t)dpp_move<0x128>((int)w);                                                     // row_ror:8
    };
    return v + joined(moved(high), moved(low));
  }
}

// The sum over a wave, the same in every lane.
__device__ __forceinline__ double wave_sum(double v) {
  return add_xor<32>(add_xor<16>(add_xor<8>(add_xor<4>(add_xor<2>(add_xor<1>(v))))));
}

// The sum over a wave of f32 values, its last three steps in 64 bits: those before them round at an eighth of the sum and below.
__device__ __forceinline__ double wave_sum_of_eighths(float v) {
  v += __int_as_float(dpp_move<kDppSwap1>(__float_as_int(v)));
  v += __int_as_float(dpp_move<kDppSwap2>(__float_as_int(v)));
  v += __int_as_float(dpp_move<kDppHalfMirror>(__float_as_int(v)));
  return add_xor<32>(add_xor<16>(add_xor<8>((double)v)));
}

// Lanes 0 to 31: a of this lane + a of the lane 32 above; lanes 32 to 63: b of the lane 32 below + b of this lane.
__device__ __forceinline__ double add_halves_apart(double a, double b) {
  const uint64_t first = __builtin_bit_cast(uint64_t, a), second = __builtin_bit_cast(uint64_t, b);
  const auto h = __builtin_amdgcn_permlane32_swap((uint32_t)(first >> 32), (uint32_t)(second >> 32), false, false);
  const auto l = __builtin_amdgcn_permlane32_swap((uint32_t)first, (uint32_t)second, false, false);
  return __builtin_bit_cast(double, ((uint64_t)h[0] << 32) | l[0]) + __builtin_bit_cast(double, ((uint64_t)h[1] << 32) | l[1]);
}
// The same for rows of sixteen lanes: rows 0 and 2 add their a and the next row's, rows 1 and 3 the previous row's b and theirs.
__device__ __forceinline__ double add_rows_apart(double a, double b) {
  const uint64_t first = __builtin_bit_cast(uint64_t, a), second = __builtin_bit_cast(uint64_t, b);
  const auto h = __builtin_amdgcn_permlane16_swap((uint32_t)(first >> 32), (uint32_t)(second >> 32), false, false);
  const auto l = __builtin_amdgcn_permlane16_swap((uint32_t)first, (uint32_t)second, false, false);
  return __builtin_bit_cast(double, ((uint64_t)h[0] << 32) | l[0]) + __builtin_bit_cast(double, ((uint64_t)h[1] << 32) | l[1]);
}

// Combine across `kLanes` adjacent lanes (4, 8, 16, 32 or 64) with `op`.
template <int kLanes, class V, class Op>
__device__ __forceinline__ V group_reduce(V v, Op op) {
  static_assert(kLanes == 4 || kLanes == 8 || kLanes == 16 || kLanes == 32 || kLanes == 64, "group width");
  v = op(v, v.template moved<kDppSwap1>());
  v = op(v, v.template moved<kDppSwap2>());
  if constexpr (kLanes >= 8) v = op(v, v.template moved<kDppHalfMirror>());
  if constexpr (kLanes >= 16) v = op(v, v.template moved<kDppRowMirror>());
  if constexpr (kLanes >= 32) v = op(v, v.shuffled_xor(16));
  if constexpr (kLanes >= 64) v = op(v, v.shuffled_xor(32));
  return v;
}

struct LaneF32 {
  float x;
  template <int kCtrl> __device__ __forceinline__ LaneF32 moved() const {
    return {dpp_move<kCtrl>(x)};
  }
  __device__ __forceinline__ LaneF32 shuffled_xor(int mask) const {
    return {__shfl_xor(x, mask, kWaveLanes)};
  }
};
struct LaneArg {  // (value, index) candidate of an arg-extremum
  float value;
  int index;
  template <int kCtrl> __device__ __forceinline__ LaneArg moved() const {
    return {dpp_move<kCtrl>(value), dpp_move<kCtrl>(index)};
  }
  __device__ __forceinline__ LaneArg shuffled_xor(int mask) const {
    return {__shfl_xor(value, mask, kWaveLanes), __shfl_xor(index, mask, kWaveLanes)};
  }
};

template <int kLanes> __device__ __forceinline__ float group_sum(float v) {
  return group_reduce<kLanes>(LaneF32{v}, [](LaneF32 a, LaneF32 b) { return LaneF32{a.x + b.x}; }).x;
}
// Plain maximum of NaN-free values.
template <int kLanes> __device__ __forceinline__ float group_max(float v) {
  return group_reduce<kLanes>(LaneF32{v}, [](LaneF32 a, LaneF32 b) {
    return LaneF32{a.x > b.x ? a.x : b.x};
  }).x;
}

// A row handled by `kLanes` adjacent lanes of a block: a slice of a wave, one wave, or
// several whole waves.  Waves of one row meet through `joint` (one float per wave of the
// block) and one block barrier; each call needs its own `joint` array.
template <int kLanes, class Op>
__device__ __forceinline__ float row_reduce(float v, float *joint, Op op) {
  constexpr int kGroup = kLanes < kWaveLanes ? kLanes : kWaveLanes;
  v = group_reduce<kGroup>(LaneF32{v}, [op](LaneF32 a, LaneF32 b) { return LaneF32{op(a.x, b.x)}; }).x;
  if constexpr (kLanes > kWaveLanes) {
    constexpr int kWavesPerRow = kLanes / kWaveLanes;
    if ((threadIdx.x & (kWaveLanes - 1)) == 0) joint[threadIdx.x / kWaveLanes] = v;
    __syncthreads();
    const int first = (threadIdx.x / kLanes) * kWavesPerRow;
    v = joint[first];
#pragma unroll
    for (int w = 1; w < kWavesPerRow; ++w) v = op(v, joint[first + w]);
  }
  return v;
}
template <int kLanes> __device__ __forceinline__ float row_sum(float v, float *joint) {
  return row_reduce<kLanes>(v, joint, [](float a, float b) { return a + b; });
}
template <int kLanes> __device__ __forceinline__ float row_max(float v, float *joint) {
  return row_reduce<kLanes>(v, joint, [](float a, float b) { return a > b ? a : b; });
}
// Whether `mine` holds in any thread of a block of kThreads: a ballot per wave and one barrier.  At most
// one call per kernel (the words are not protected against the next).  (The runtime's own
// block votes reduce over the block size that they read from the implicit arguments.)
template <int kThreads> __device__ __forceinline__ bool block_any(bool mine) {
  constexpr int kWaves = kThreads / kWaveLanes;
  __shared__ uint32_t seen[kWaves];
  const uint64_t lanes = __ballot(mine);
  if (threadIdx.x % kWaveLanes == 0) seen[threadIdx.x / kWaveLanes] = lanes != 0 ? 1u : 0u;
  __syncthreads();
  uint32_t any = 0;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) any |= seen[w];
  return any != 0;
}
// NaN-propagating extrema of the reference's Reduce
// (src/compute_provider_native/reduction.cc:34-47): the first NaN met sticks;
// +0 ranks above -0 (tests/simd/search_test.cc:203-206).
__device__ __forceinline__ float max_propagate(float a, float b) {
  if (a != a) return a;
  if (b != b) return b;
  if (a == b) return (f32_bits(a) & 0x80000000u) ? b : a;
  return a > b ? a : b;
}
__device__ __forceinline__ float min_propagate(float a, float b) {
  if (a != a) return a;
  if (b != b) return b;
  if (a == b) return (f32_bits(a) & 0x80000000u) ? a : b;
  return a < b ? a : b;
}

// TopK(count = 1, largest) ordering of src/compute_provider_cuda/collectives.cu:478-495:
// a number beats NaN, a larger number beats a smaller one, otherwise (equal,
// -0 vs +0, NaN vs NaN) the lower index wins.  index < 0 marks "no candidate".
__device__ __forceinline__ LaneArg arg_best(LaneArg a, LaneArg b) {
  if (a.index < 0) return b;
  if (b.index < 0) return a;
  const bool a_nan = a.value != a.value, b_nan = b.value != b.value;
  if (a_nan != b_nan) return a_nan ? b : a;
  if (!a_nan && a.value != b.value) return a.value > b.value ? a : b;
  return a.index < b.index ? a : b;
}

}  // namespace hyle_hip
