// Row Softmax / LogSoftmax over rows that are no whole number of 16-byte vectors, or start at an
// address that is none (an odd number of keys, a mask row of odd length, a view one element in):
// the last axis of a dense tensor, any width from one vector on, arithmetic and the invalid-row
// rule as in softmax.hip but for the exponential of narrow types (row_exp), which is nearer to exp.
//
// A lane takes whole 16-byte vectors at element-aligned addresses (gfx950 loads and stores them
// like any others, a wave's 64 neighbours still cover whole lines), and the vector that would pass
// the row's end is moved back to end there: no scalar tail, every access inside the row.  The two
// vectors then share elements, which both compute and store alike and only one counts in the sum.
// The loads are plain ones, since neighbours share the lines at their seams; the stores stream
// (bf16 [24, 777, 1013] 1.8 us less than with plain stores).  Bound by HBM from about 1000
// elements a row on, below that by the vector instructions of a wave's two reductions, which is why
// short rows share a wave.  MI355X, without a mask / Boolean / additive, before (softmax_general,
// which walks the strides of every element in three passes) and here:
//   bf16 [24, 777, 1013]  177 / 189 / 190 -> 13.4 / 14.5 / 15.4 us (5640 / 5300 / 5000 GB/s)
//   f32  [24, 777, 1013]  180 -> 27.5 us (5500 GB/s)    f32 [12, 777, 7001] Boolean 658 -> 91.0 us (5800 GB/s)
//   bf16 [24, 777, 3001]  491 -> 35.1 us (6380 GB/s; an aligned row of 3000 in softmax.hip: 45.4)
//   f16  [24, 777, 100]    42 ->  4.0 us               f32 [8, 1, 1271] 12.7 -> 2.6 us
//   f32  [1, 777] 10.3 -> 2.2 us, [6, 129] 4.4 -> 1.9 us, [1, 5] 4.1 -> 1.8 us: no call is too small for it
// Running the heads of a mask row next to each other on one XCD, which pays for 64 MiB masks
// (softmax.hip), loses here: bf16 [24, 777, 1013] additive 17.5 -> 20.2 us, f32 [32, 1777, 1777]
// 149 -> 161 us.
#include "softmax_math.h"

namespace hyle_hip {
namespace {

// 16 bytes (or the mask bytes of one vector) at any element's address.
typedef uint32_t words4_any __attribute__((ext_vector_type(4), aligned(1)));
typedef uint32_t word_any __attribute__((aligned(1)));

// exp(t) * 2^32 for t <= 0.  Narrow types: 2^(t * log2(e)) as a power of two, which goes into the exponent
// field, and the rest in [-0.5, 0.5], which is exact up to one rounding.  Root of the mean square error:
// 5e-8 for t in (-5, 0), 7e-7 in (-66, -45); exp_scaled, one instruction longer, has 4e-7 and 7e-7, a single
// fused multiply-add into exp2, two instructions, 4e-7 and 1.1e-6 (bf16 [24, 777, 1013] unmasked / Boolean /
// additive with it 13.3 / 13.0 / 13.6 us, with exp_scaled 15.7 / 16.1 / 16.6, here 13.2 / 14.7 / 14.3).  The
// lower end keeps the exponent field above zero; what lies below it is a zero of either narrow type once it
// is divided by a sum of at least one.
// kLog: the exponentials only meet in the sum, to which those far below the maximum, where the single
// multiply-add falls behind, add nothing: rows of 67 to 8145 normal values of standard deviation 1 to 12 have
// sums with an error of 3.6e-8 to 9.3e-8 with it and 3.7e-8 to 9.2e-8 with exp_scaled (bf16 [2048, 20001] Boolean
// 107 us, with the exponential above 143).  -inf is a zero there, for the logarithm of a sum of one element.
template <class T, bool kLog> __device__ __forceinline__ float row_exp(float t) {
  if constexpr (Traits<T>::kSize == 4) {
    return exp_scaled(t);
  } else {
    constexpr float kLog2e = 1.44269504088896340736f;
    if constexpr (kLog) return __builtin_amdgcn_exp2f(__builtin_fmaf(t, kLog2e, 32.0f));
    constexpr float kWhole = 12582912.0f + 32.0f;  // 1.5 * 2^23 + 32: the sum's low bits are round(t * log2(e)) + 32
    t = fmaxf(t, -108.0f);
    const float shifted = __builtin_fmaf(t, kLog2e, kWhole);
    const float rest = __builtin_fmaf(t, kLog2e, kWhole - shifted);
    return bits_f32(f32_bits(__builtin_amdgcn_exp2f(rest)) + (f32_bits(shifted) << 23));
  }
}

// kShared: rows `inner` apart have the same mask row (the heads of a layer), and a lane takes up to `each` of them one after
// another: the mask is loaded once, and a row's loads are under way while the row before is worked on.
template <class T, int kLanes, int kVpl, int kThreads, int kMask, bool kLog, bool kShared>
__global__ __launch_bounds__(kThreads) void softmax_rows_unaligned(const char *x, const char *mask, char *y, uint32_t rows,
                                                                  uint32_t width, float scale, MaskRows mrows, uint32_t inner, uint32_t each) {
  constexpr uint32_t kVec = Traits<T>::kVec, kSize = Traits<T>::kSize;
  constexpr int kWords = kVec / 4;
  constexpr int kGroupsPerBlock = kThreads / kLanes;
  constexpr int kWaves = kThreads / kWaveLanes;
  __shared__ float joint_max[kWaves], joint_sum[kWaves];
  const uint32_t lane = threadIdx.x % kLanes;
  uint32_t group = threadIdx.x / kLanes;
  if constexpr (kLanes >= kWaveLanes) group = __builtin_amdgcn_readfirstlane(group);  // the row's address stays scalar
  const uint32_t wanted_row = blockIdx.x * kGroupsPerBlock + group;
  const uint32_t places = kShared ? inner : rows;
  const bool row_ok = wanted_row < places;
  uint32_t row = row_ok ? wanted_row : places - 1, left = 1;
  if constexpr (kShared) {
    row += blockIdx.y * each * inner;
    left = min(each, rows / inner - blockIdx.y * each);
  }
  const char *mask_row = nullptr;
  if constexpr (kMask != kMaskNone) mask_row = mask + mask_row_offset(mrows, row);
  const char *row_x = x + (size_t)row * width * kSize;

  // Vector `lane + k * kLanes` of the row, moved back to end at the row's end where it would pass
  // it: `skip` of its elements belong to the vector before it (all of them: nothing is left).
  uint32_t start[kVpl], skip[kVpl];
#pragma unroll
  for (int k = 0; k < kVpl; ++k) {
    const uint32_t own = (lane + k * kLanes) * kVec;
    start[k] = own < width - kVec ? own : width - kVec;
    skip[k] = own - start[k];
  }
  uint32_t bits[kVpl][kWords];
  if constexpr (kMask == kMaskBoolean) {
#pragma unroll
    for (int k = 0; k < kVpl; ++k)
#pragma unroll
      for (int q = 0; q < kWords; ++q) bits[k][q] = reinterpret_cast<const word_any *>(mask_row + start[k])[q];
  }
  u32x4 raw[kVpl], added[kVpl];
  uint32_t from[kVpl];
#pragma unroll
  for (int k = 0; k < kVpl; ++k) {
    from[k] = start[k];
    if constexpr (kMask == kMaskBoolean) {
      uint32_t any = 0;
#pragma unroll
      for (int q = 0; q < kWords; ++q) any |= bits[k][q];
      from[k] = any != 0 ? from[k] : 0u;  // nothing kept: no new line is asked for
    }
    raw[k] = *reinterpret_cast<const words4_any *>(row_x + (size_t)from[k] * kSize);
    if constexpr (kMask == kMaskAdditive) added[k] = *reinterpret_cast<const words4_any *>(mask_row + (size_t)start[k] * kSize);
  }
#pragma unroll
  for (int k = 0; k < kVpl; ++k) loads_issued(raw[k]);

  while (true) {
    float v[kVpl][kVec];
    if constexpr (kShared) {
#pragma unroll
      for (int k = 0; k < kVpl; ++k) Traits<T>::unpack(raw[k], v[k]);
      row_x += (size_t)inner * width * kSize;
      if (left > 1) {
#pragma unroll
        for (int k = 0; k < kVpl; ++k) raw[k] = *reinterpret_cast<const words4_any *>(row_x + (size_t)from[k] * kSize);
        asm volatile("" ::: "memory");
      }
    }
    float peak = -INFINITY;
#pragma unroll
    for (int k = 0; k < kVpl; ++k) {
      if constexpr (!kShared) Traits<T>::unpack(raw[k], v[k]);
      if constexpr (kMask == kMaskAdditive) {
        float addend[kVec];
        Traits<T>::unpack(added[k], addend);
#pragma unroll
        for (int j = 0; j < (int)kVec; ++j) v[k][j] = v[k][j] * scale + addend[j];
      } else if constexpr (kMask == kMaskBoolean) {
#pragma unroll
        for (int j = 0; j < (int)kVec; ++j) {
          const bool keep = ((bits[k][j / 4] >> (8 * (j % 4))) & 0xFFu) != 0;
          v[k][j] = keep ? v[k][j] * scale : -INFINITY;
        }
      } else {
#pragma unroll
        for (int j = 0; j < (int)kVec; ++j) v[k][j] *= scale;
      }
#pragma unroll
      for (int j = 0; j < (int)kVec; j += 2) {
        peak = __builtin_elementwise_maximum(__builtin_elementwise_maximum(v[k][j], v[k][j + 1]), peak);  // a NaN stays
      }
    }
    // an infinite maximum of either sign marks the row: +inf poisoned, -inf nothing finite
    peak = row_max<kLanes>(peak != peak ? INFINITY : peak, joint_max);
    const bool invalid = __builtin_fabsf(peak) == INFINITY;
    float total = 0.0f, maxima = 0.0f;
#pragma unroll
    for (int k = 0; k < kVpl; ++k) {
      float sum = 0.0f, count = 0.0f;
#pragma unroll
      for (int j = 0; j < (int)kVec; ++j) {
        const float shifted = v[k][j] - peak;
        if constexpr (kLog) {  // the maxima are counted, not summed (src/compute_provider_cuda/reduction_kernel.cu:178-196)
          const bool at_peak = shifted == 0.0f;
          sum += at_peak ? 0.0f : row_exp<T, kLog>(shifted);
          count += at_peak ? 1.0f : 0.0f;
          v[k][j] = shifted;
        } else {
          v[k][j] = row_exp<T, kLog>(shifted);
          sum += v[k][j];
        }
      }
      if (skip[k] != 0) {  // the row's last vectors: elements of two vectors count once
        sum = 0.0f;
        count = 0.0f;
#pragma unroll
        for (int j = 0; j < (int)kVec; ++j) {
          const bool mine = (uint32_t)j >= skip[k];
          if constexpr (kLog) {
            sum += mine && v[k][j] != 0.0f ? row_exp<T, kLog>(v[k][j]) : 0.0f;
            count += mine && v[k][j] == 0.0f ? 1.0f : 0.0f;
          } else {
            sum += mine ? v[k][j] : 0.0f;
          }
        }
      }
      total += sum;
      maxima += count;
    }
    total = row_sum<kLanes>(total, joint_sum);  // = 2^32 * sum(exp)
    // joint_max is free again: every wave read it before the barrier of the sum above
    if constexpr (kLog) maxima = row_sum<kLanes>(maxima, joint_max);
    float normaliser = kLog ? log1pf((maxima - 1.0f) + total * 2.3283064365386963e-10f) : 1.0f / total;
    if (invalid) normaliser = __builtin_nanf("");
    char *row_y = y + (size_t)row * width * kSize;
#pragma unroll
    for (int k = 0; k < kVpl; ++k) {
      if (row_ok && skip[k] < kVec) {
        float out[kVec];
#pragma unroll
        for (int j = 0; j < (int)kVec; ++j) out[j] = kLog ? v[k][j] - normaliser : v[k][j] * normaliser;
        const u32x4 packed = Traits<T>::pack(out);
        __builtin_nontemporal_store(packed, reinterpret_cast<words4_any *>(row_y + (size_t)start[k] * kSize));
      }
    }
    if constexpr (!kShared) break;
    if (--left == 0) break;  // the same for the whole block
    row += inner;
    if constexpr (kLanes > kWaveLanes) __syncthreads();  // the joint words are free again
  }
}

// softmax_unaligned/<lanes>x<vectors per lane>/<threads per block>/<mask>[#shared: several rows to a mask row]
template <int kLanes, int kVpl, int kThreads, int kMask, bool kShared> struct UnalignedTag {
  static std::string text() {
    return "softmax_unaligned/" + std::to_string(kLanes) + "x" + std::to_string(kVpl) + "/" + std::to_string(kThreads) + "/" + mask_word(kMask) +
           (kShared ? "#shared" : "");
  }
};

// Three rows to a mask row in large launches of masked rows of several waves: the mask is asked for once instead of three times,
// and a row's loads are under way during the exponentials of the row before.  us, one row / three: additive bf16
// [19, 1932, 6908] 216 / 181, [16, 1500, 5001] 126 / 110, [46, 1495, 2094] 118 / 109, f16 [9, 3800, 4081] 116 / 107, f32
// [16, 1500, 2501] 102 / 87; Boolean bf16 [19, 1932, 6908] 183 / 169, [24, 2200, 3100] 119 / 111.  Not below 100 MB, where it
// leaves too few waves (bf16 [16, 800, 2201] 28.2 / 30.6, [64, 260, 2500] 32.9 / 35.6), nor with a mask that every
// L2 holds beside the rows ([64, 300, 2700] 40.1 / 40.8); rows of one wave gain nothing
// (bf16 [30, 2000, 1700] 77 / 82 with five vectors a lane, [24, 777, 1013] 18.4 / 19.5), nor do rows without a mask ([24, 777, 2094] 30.9 / 32.6).
constexpr uint32_t kSharedRows = 3;
constexpr uint64_t kSharedBytes = 100000000, kSharedMask = 2000000;
// Rows between two that have the same mask row (0: none that a launch could share).
inline uint32_t shared_inner(const SoftmaxParams &p, uint32_t size) {
  if ((int)p.mask_kind == kMaskNone || (uint64_t)p.shape.rows * p.shape.width * size < kSharedBytes) return 0;
  uint64_t outer = 1;
  for (int i = 0; i < p.outer_rank && (p.mask_outer_strides[i] == 0 || p.outer_dims[i] == 1); ++i) outer *= p.outer_dims[i];
  const uint64_t inner = p.shape.rows / outer, mask_bytes = inner * p.shape.width * ((int)p.mask_kind == kMaskBoolean ? 1 : size);
  return outer >= kSharedRows && mask_bytes >= kSharedMask && (outer + kSharedRows - 1) / kSharedRows <= 65535u ? (uint32_t)inner : 0u;
}

template <class T, int kLanes, int kVpl, int kThreads, int kMask, bool kShared = false>
void run_mask(const SoftmaxParams &p, const MaskRows &m, const void *x, const void *mask, void *y, hipStream_t s) {
  constexpr uint32_t kGroupsPerBlock = kThreads / kLanes;
  const uint32_t rows = (uint32_t)p.shape.rows, inner = kShared ? shared_inner(p, Traits<T>::kSize) : rows, outer = rows / inner;
  const dim3 grid((inner + kGroupsPerBlock - 1) / kGroupsPerBlock, kShared ? (outer + kSharedRows - 1) / kSharedRows : 1);
  const char *in = static_cast<const char *>(x), *in_mask = static_cast<const char *>(mask);
  char *out = static_cast<char *>(y);
  note_variant<UnalignedTag<kLanes, kVpl, kThreads, kMask, kShared>>();
  if (p.log)
    hipLaunchKernelGGL((softmax_rows_unaligned<T, kLanes, kVpl, kThreads, kMask, true, kShared>), grid, dim3(kThreads), 0, s, in, in_mask, out, rows,
                       p.shape.width, p.scale, m, inner, kSharedRows);
  else
    hipLaunchKernelGGL((softmax_rows_unaligned<T, kLanes, kVpl, kThreads, kMask, false, kShared>), grid, dim3(kThreads), 0, s, in, in_mask, out, rows,
                       p.shape.width, p.scale, m, inner, kSharedRows);
}

inline MaskRows mask_rows(const SoftmaxParams &p) {
  MaskRows m{};
  m.outer_rank = p.outer_rank;
  for (int i = 0; i < kMaxRank; ++i) {
    m.outer_dims[i] = p.outer_dims[i];
    m.outer_strides[i] = p.mask_outer_strides[i];
  }
  m.inner_stride = p.mask_inner_stride;
  return m;
}

template <class T, int kLanes, int kVpl, int kThreads>
void run_shape(const SoftmaxParams &p, const void *x, const void *mask, void *y, hipStream_t s) {
  const MaskRows m = mask_rows(p);
  if constexpr (kLanes == 128 || kLanes == 256) {
    if (shared_inner(p, Traits<T>::kSize) != 0) {
      if ((int)p.mask_kind == kMaskBoolean) return run_mask<T, kLanes, kVpl, kThreads, kMaskBoolean, true>(p, m, x, mask, y, s);
      return run_mask<T, kLanes, kVpl, kThreads, kMaskAdditive, true>(p, m, x, mask, y, s);
    }
  }
  switch ((int)p.mask_kind) {
    case kMaskBoolean: return run_mask<T, kLanes, kVpl, kThreads, kMaskBoolean>(p, m, x, mask, y, s);
    case kMaskAdditive: return run_mask<T, kLanes, kVpl, kThreads, kMaskAdditive>(p, m, x, mask, y, s);
    default: return run_mask<T, kLanes, kVpl, kThreads, kMaskNone>(p, m, x, mask, y, s);
  }
}

// Lanes x vectors for a row of that many vectors, the tightest measured: three vectors a lane where
// two would leave a third of the lanes idle (bf16 601 additive 64 x 2 14.9 us, 32 x 3 13.4; 3001
// unmasked 128 x 4 40.0, 128 x 3 39.0), two rows per wave below 64 vectors (f16 203: 64 x 1 7.7 us,
// 32 x 1 5.3, 16 x 2 5.1; 503 additive 64 x 1 11.7, 32 x 2 11.0), but one row per wave at 65-128
// (1013 additive 64 x 2 17.9, 32 x 4 19.8).
template <class T> void run_width(const SoftmaxParams &p, const void *x, const void *mask, void *y, hipStream_t s) {
  const uint32_t vectors = (p.shape.width + Traits<T>::kVec - 1) / Traits<T>::kVec;
  if (vectors <= 8) return run_shape<T, 8, 1, 256>(p, x, mask, y, s);
  if (vectors <= 16) return run_shape<T, 16, 1, 256>(p, x, mask, y, s);
  if (vectors <= 32) return run_shape<T, 16, 2, 256>(p, x, mask, y, s);
  if (vectors <= 64) return run_shape<T, 32, 2, 256>(p, x, mask, y, s);
  if (vectors <= 96) return run_shape<T, 32, 3, 256>(p, x, mask, y, s);
  if (vectors <= 128) return run_shape<T, 64, 2, 256>(p, x, mask, y, s);
  if (vectors <= 192) return run_shape<T, 64, 3, 256>(p, x, mask, y, s);
  if (vectors <= 256) return run_shape<T, 64, 4, 256>(p, x, mask, y, s);
  if (vectors <= 384) return run_shape<T, 128, 3, 256>(p, x, mask, y, s);
  if (vectors <= 512) return run_shape<T, 128, 4, 256>(p, x, mask, y, s);
  if (vectors <= 768) return run_shape<T, 256, 3, 256>(p, x, mask, y, s);
  if (vectors <= 1024) return run_shape<T, 256, 4, 256>(p, x, mask, y, s);
  if (vectors <= 1536) return run_shape<T, 512, 3, 512>(p, x, mask, y, s);
  if (vectors <= 2048) return run_shape<T, 512, 4, 512>(p, x, mask, y, s);
  return run_shape<T, 1024, 8, 1024>(p, x, mask, y, s);
}

}  // namespace

bool softmax_unaligned_serves(Elem type, const SoftmaxParams &p) {
  const uint32_t kvec = (uint32_t)elem_vec(type);
  if (p.shape.width < kvec || p.shape.width > 8u * 1024u * kvec) return false;
  // A launch has fewer than 2^32 threads, which needs no line here: admission takes at most 2^31 - 1 elements, and a
  // row of more than one vector has less than two lanes to an element.
  const int64_t unit = (int)p.mask_kind == kMaskBoolean ? 1 : elem_size(type);
  return (int)p.mask_kind == kMaskNone || p.mask_inner_stride == unit;
}

hipError_t launch_softmax_unaligned(Elem type, const SoftmaxParams &p, const void *x, const void *mask, void *y, hipStream_t stream) {
  switch (type) {
    case Elem::kF32: run_width<F32>(p, x, mask, y, stream); break;
    case Elem::kF16: run_width<F16>(p, x, mask, y, stream); break;
    case Elem::kBF16: run_width<BF16>(p, x, mask, y, stream); break;
  }
  return hipGetLastError();
}

}  // namespace hyle_hip
