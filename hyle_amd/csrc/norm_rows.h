// The row kernel of RMSNorm and LayerNorm and what its launchers share: included by norm.hip (the
// launch shapes that mask lanes and rows outside the tensor), by norm_exact_rms.hip /
// norm_exact_layer.hip (the shapes that cover it exactly) and by norm_tail_rms.hip /
// norm_tail_layer.hip (one wave per row, only the last vector masked), which are separate files so
// that their many instantiations compile side by side.
#pragma once

#include <type_traits>

#include "device_common.h"
#include "kernels.h"

namespace hyle_hip {
namespace {

template <class W, int kVec>
__device__ __forceinline__ void load_weight(const void *w, uint32_t vec, float (&out)[kVec]) {
  if constexpr (Traits<W>::kVec == kVec) {
    Traits<W>::unpack(load16(w, vec), out);
  } else {  // f32 parameters under a narrow input: two vectors per input vector
    float lo[4], hi[4];
    Traits<F32>::unpack(load16(w, 2 * (size_t)vec), lo);
    Traits<F32>::unpack(load16(w, 2 * (size_t)vec + 1), hi);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      out[j] = lo[j];
      out[4 + j] = hi[j];
    }
  }
}

template <int kVec> __device__ __forceinline__ float tree_sum(const float (&v)[kVec]) {
  if constexpr (kVec == 8) return ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
  else return (v[0] + v[1]) + (v[2] + v[3]);
}

// row_sum with the sums of a row's waves added in pairs: one after the other they round at the size of the whole row more than
// once, which a LayerNorm's mean shows (f32 [500, 4096] about 3, 256 lanes: 1.42e-7 off the 64-bit result (2-norm), 1.21e-7 in pairs; with
// two waves to a row 1.21e-7; [64, 16384], 1024 lanes, 2.0e-7 and 1.2e-7).
template <int kLanes> __device__ __forceinline__ float norm_sum(float v, float *joint) {
  if constexpr (kLanes <= 2 * kWaveLanes) {
    return row_sum<kLanes>(v, joint);
  } else {
    constexpr int kWaves = kLanes / kWaveLanes;
    v = group_sum<kWaveLanes>(v);
    if ((threadIdx.x & (kWaveLanes - 1)) == 0) joint[threadIdx.x / kWaveLanes] = v;
    __syncthreads();
    const int first = (threadIdx.x / kLanes) * kWaves;
    float parts[kWaves];
#pragma unroll
    for (int w = 0; w < kWaves; ++w) parts[w] = joint[first + w];
#pragma unroll
    for (int half = kWaves / 2; half > 0; half /= 2)
#pragma unroll
      for (int w = 0; w < half; ++w) parts[w] += parts[w + half];
    return parts[0];
  }
}

enum : int { kPlain = 0, kScale = 1, kScaleBias = 2 };  // learned parameters of a launch

// `kRows` consecutive rows share one group of lanes.  Loads carry no branches (a lane outside
// the row, or a row outside the tensor, reads a clamped, valid address and zeroes the value).
// The rows are loaded one after another (the kVpl loads of a row together, the next row once
// they have arrived), the parameter vectors are fetched once for all rows, and every store
// follows the last load: a block reads in one phase and writes in another, which for tensors of
// a few tens of MB measured 10-15 % faster on MI355X than issuing all loads of a lane at once.
// `kExact` launches cover the tensor exactly (every lane a vector of every row of its group), so
// nothing is masked -- not even a group's second row by one comparison for the whole group: with
// that, LayerNorm over [8192, 2048] bf16 measured 14.5 us against 11.7 us -- and `kParameters` is
// fixed per instantiation: per element the bf16 LayerNorm is ten vector instructions instead of
// sixteen.  One such instruction per element is 0.44 us of every SIMD's time for 16.7 M
// elements, which the loads do not hide once all waves of a launch are resident together and
// move through their phases side by side.
// `kTail` launches (norm_tail.h) cover their rows, and only the last vector of a lane is masked.
template <class T, class W, int kLanes, int kVpl, int kThreads, int kRows, bool kLayer, int kParameters, bool kExact,
          bool kTail>
__device__ __forceinline__ void norm_group(const void *x, const void *w, const void *b, void *y, uint32_t first_row, uint32_t rows,
                                           uint32_t row_vectors, float width, float epsilon) {
  constexpr int parameters = kParameters;
  constexpr int kVec = Traits<T>::kVec;
  __shared__ float joint[kLayer ? 2 : 1][kRows][kThreads / kWaveLanes];
  const uint32_t lane = threadIdx.x % kLanes;

  u32x4 raw[kRows][kVpl];
  uint32_t vec[kVpl];
#pragma unroll
  for (int k = 0; k < kVpl; ++k) {
    const uint32_t wanted = lane + k * kLanes;
    vec[k] = kExact || (kTail && k < kVpl - 1) || wanted < row_vectors ? wanted : row_vectors - 1;
  }
#pragma unroll
  for (int r = 0; r < kRows; ++r) {
    const uint32_t row = kExact || kTail || first_row + r < rows ? first_row + r : rows - 1;
    const size_t row_base = (size_t)row * row_vectors;
#pragma unroll
    for (int k = 0; k < kVpl; ++k) raw[r][k] = load16_stream(x, row_base + vec[k]);
#pragma unroll
    for (int k = 0; k < kVpl; ++k) loads_issued(raw[r][k]);
  }
  float scale[kVpl][kVec], bias[kVpl][kVec];
  if constexpr (parameters != kPlain) {
#pragma unroll
    for (int k = 0; k < kVpl; ++k) load_weight<W, kVec>(w, vec[k], scale[k]);
  }
  if constexpr (kLayer && parameters == kScaleBias) {
#pragma unroll
    for (int k = 0; k < kVpl; ++k) load_weight<W, kVec>(b, vec[k], bias[k]);
  }
  // Row by row: measured on MI355X, reducing the statistics of both rows behind one barrier
  // is slower (RMSNorm over [8192, 2048] bf16: 13.5 us against 11.4 us).
  float v[kRows][kVpl][kVec];
  float inverse[kRows];
#pragma unroll
  for (int r = 0; r < kRows; ++r) {
    bool ok[kVpl];
#pragma unroll
    for (int k = 0; k < kVpl; ++k) {
      ok[k] = kExact || (kTail && k < kVpl - 1) || ((kTail || first_row + r < rows) && lane + k * kLanes < row_vectors);
      Traits<T>::unpack(raw[r][k], v[r][k]);
    }
    if constexpr (kLayer) {
      float sum = 0.0f;
      if constexpr (kTail) {  // a sum per element of a vector: shorter chains, and fewer roundings in each
        float sums[kVec] = {};
#pragma unroll
        for (int k = 0; k < kVpl; ++k)
#pragma unroll
          for (int j = 0; j < kVec; ++j) sums[j] += ok[k] ? v[r][k][j] : 0.0f;
        sum = tree_sum(sums);
      } else {
#pragma unroll
        for (int k = 0; k < kVpl; ++k)
#pragma unroll
          for (int j = 0; j < kVec; ++j) sum += ok[k] ? v[r][k][j] : 0.0f;
      }
      const float mean = norm_sum<kLanes>(sum, joint[1][r]) / width;
#pragma unroll
      for (int k = 0; k < kVpl; ++k)
#pragma unroll
        for (int j = 0; j < kVec; ++j) v[r][k][j] -= mean;
    }
    float squares = 0.0f, parts[kVec] = {};
#pragma unroll
    for (int k = 0; k < kVpl; ++k)
#pragma unroll
      for (int j = 0; j < kVec; ++j) {
        v[r][k][j] = ok[k] ? v[r][k][j] : 0.0f;
        float &sum = kTail ? parts[j] : squares;
        sum = __builtin_fmaf(v[r][k][j], v[r][k][j], sum);
      }
    if constexpr (kTail) squares = tree_sum(parts);
    squares = norm_sum<kLanes>(squares, joint[0][r]);
    inverse[r] = 1.0f / sqrtf(squares / width + epsilon);
  }
#pragma unroll
  for (int r = 0; r < kRows; ++r) {
    const uint32_t row = first_row + r;
    const size_t row_base = (size_t)row * row_vectors;
#pragma unroll
    for (int k = 0; k < kVpl; ++k) {
      if (kExact || (kTail && k < kVpl - 1) || ((kTail || row < rows) && lane + k * kLanes < row_vectors)) {
        float out[kVec];
#pragma unroll
        for (int j = 0; j < kVec; ++j) {
          out[j] = v[r][k][j] * inverse[r];
          if constexpr (kLayer && parameters == kScaleBias) out[j] = __builtin_fmaf(out[j], scale[k][j], bias[k][j]);
          else if constexpr (parameters != kPlain) out[j] = out[j] * scale[k][j];
        }
        store16_stream(y, row_base + vec[k], Traits<T>::pack(out));
      }
    }
  }
}

template <class T, class W, int kLanes, int kVpl, int kThreads, int kRows, bool kLayer, int kParameters, bool kExact, bool kTail = false>
__global__ __launch_bounds__(kThreads) void norm_rows(const void *x, const void *w, const void *b,
                                                      void *y, uint32_t rows, uint32_t row_vectors,
                                                      float width, float epsilon) {
  constexpr int kGroupsPerBlock = kThreads / kLanes;
  uint32_t group = blockIdx.x * kGroupsPerBlock + threadIdx.x / kLanes;
  if constexpr (kTail) {
    static_assert(!kExact && kLanes == kWaveLanes, "a wave goes its own way: no barrier follows");
    group = __builtin_amdgcn_readfirstlane(group);
    const uint32_t first_row = group * kRows;
    if (first_row >= rows) return;
    if (kRows > 1 && first_row + kRows > rows) {  // the last rows one by one
      for (uint32_t row = first_row; row < rows; ++row)
        norm_group<T, W, kLanes, kVpl, kThreads, 1, kLayer, kParameters, false, true>(x, w, b, y, row, rows, row_vectors, width, epsilon);
      return;
    }
  }
  norm_group<T, W, kLanes, kVpl, kThreads, kRows, kLayer, kParameters, kExact, kTail>(x, w, b, y, group * kRows, rows, row_vectors,
                                                                                      width, epsilon);
}

struct Bound {
  const void *x, *w, *b;
  void *y;
};

// <family>/<rms|layer>/<lanes>x<vectors per lane>/<threads per block>/<rows per lane group>[/<ragged|exact>]
template <bool kLayer, int kLanes, int kVpl, int kThreads, int kRows, int kForm> struct NormTag {  // kForm: 0 exact-only shape, 1 ragged, 2 exact
  static std::string text() {
    return std::string(kForm == 0 ? "norm_rows_exact/" : "norm_rows/") + (kLayer ? "layer/" : "rms/") + std::to_string(kLanes) + "x" +
           std::to_string(kVpl) + "/" + std::to_string(kThreads) + "/" + std::to_string(kRows) +
           (kForm == 1 ? "/ragged" : (kForm == 2 ? "/exact" : ""));
  }
};

// A launch shape used only when it covers the tensor exactly (no masked variant is built for it).
template <class T, class W, bool kLayer, int kLanes, int kVpl, int kThreads, int kRows>
bool run_exact(const NormParams &p, const Bound &io, int parameters, hipStream_t s) {
  constexpr int kRowsPerBlock = kThreads / kLanes * kRows;
  const uint32_t rows = (uint32_t)p.shape.rows, row_vectors = p.shape.width / Traits<T>::kVec;
  if (rows % kRowsPerBlock != 0 || row_vectors != (uint32_t)(kLanes * kVpl)) return false;
  note_variant<NormTag<kLayer, kLanes, kVpl, kThreads, kRows, 0>>();
  const dim3 grid(rows / kRowsPerBlock), block(kThreads);
  const float width = (float)p.shape.width;
  if (parameters == kPlain)
    hipLaunchKernelGGL((norm_rows<T, W, kLanes, kVpl, kThreads, kRows, kLayer, kPlain, true>), grid, block, 0, s, io.x, io.w,
                       io.b, io.y, rows, row_vectors, width, p.epsilon);
  else if (kLayer && parameters == kScaleBias)
    hipLaunchKernelGGL((norm_rows<T, W, kLanes, kVpl, kThreads, kRows, kLayer, kLayer ? kScaleBias : kScale, true>), grid, block,
                       0, s, io.x, io.w, io.b, io.y, rows, row_vectors, width, p.epsilon);
  else
    hipLaunchKernelGGL((norm_rows<T, W, kLanes, kVpl, kThreads, kRows, kLayer, kScale, true>), grid, block, 0, s, io.x, io.w,
                       io.b, io.y, rows, row_vectors, width, p.epsilon);
  return true;
}

}  // namespace

// Launches the shape that covers [rows, width] exactly, if there is one (norm_exact.h lists them:
// rows of 16 to 128 vectors in multiples of a block's rows, an even number of rows of 64 n, 128 n
// or 256 n vectors).  False: nothing was launched, take the masked shapes.
bool launch_norm_exact_rms(Elem type, const NormParams &p, const void *x, const void *w, void *y, hipStream_t stream);
bool launch_norm_exact_layer(Elem type, const NormParams &p, const void *x, const void *w, const void *b, void *y,
                             hipStream_t stream);
// Rows of 65 to 768 vectors (norm_tail.h).  False: nothing was launched.
bool launch_norm_tail_rms(Elem type, const NormParams &p, const void *x, const void *w, void *y, hipStream_t stream);
bool launch_norm_tail_layer(Elem type, const NormParams &p, const void *x, const void *w, const void *b, void *y,
                            hipStream_t stream);

}  // namespace hyle_hip
