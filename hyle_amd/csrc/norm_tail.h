// Launch shapes of RMSNorm / LayerNorm for rows of 65 to 768 vectors, any width and any number of rows: one wave
// per row, or per two rows one after the other, with ceil(vectors / 64) vectors per lane, of which only the last can be
// missing in some lanes.  The masked shapes of norm.hip round a row up to 128, 256, 512 or 1024 vectors instead (a row of
// 640 keeps 640 of 1024 places busy and waits for a barrier).
//
// Two rows per wave where the launch holds the chip about once: its reads then end before its writes begin.  A smaller
// launch wants all its loads at once, a larger one has reads and writes side by side in any case, and a LayerNorm of
// narrow elements has no registers for two rows beside its parameters.  MI355X, us, masked / one row / two rows:
//   LayerNorm f32 [5003, 2560] 21.6 / 19.8 / 19.0   [4626, 1552] 13.0 / 12.5 / 10.3   [8001, 1040] 15.1 / 14.7 / 13.2
//     [1501, 2560] 8.2 / 5.3 / 5.7   [801, 2304] 4.5 / 3.7 / 4.3
//   LayerNorm bf16 [5003, 2560] 13.0 / 8.3 / 8.9   [8191, 5000] 33.2 / 31.3 / 35.3   f16 [2301, 5000] 11.9 / 9.4 / 14.9
//   RMSNorm bf16 [8191, 2560] 16.2 / 15.4 / 13.1   [4000, 4992] 16.1 / 14.7 / 13.2   [64, 2048] 3.2 / 2.2 / 2.7
//   RMSNorm f32 [5001, 1600] 13.0 / 11.5 / 10.3   [7001, 3008] 29.6 / 28.6 / 30.7   [2001, 1088] 4.7 / 3.9 / 4.3
// RMSNorm of 193 to 256 vectors at two rows is norm.hip's masked shape (bf16 [8191, 2048] 10.7 / 12.7 / 11.0).
// Rows of 65 to 128 vectors come four to a block of four waves, which are dispatched faster than as many blocks of one
// (RMSNorm bf16 [5000, 704] 3.7 against 4.6).  Each lane sums per element of a vector, so that its chains are no longer
// than those of the masked shapes with their more lanes.
#pragma once

#include "norm_rows.h"

namespace hyle_hip {
namespace {

// Too few rows for the waves of a row to be better spent on other rows: a row of more than 256 vectors is 256 lanes'
// there (us, there / here: RMSNorm bf16 [5, 5120] 2.5 / 2.7, [1, 5120] 2.4 / 2.5; LayerNorm f32 [16, 3000] 2.9 / 2.75).
// Up to 512 vectors a row is a wave's here however few there are, there of two rows: RMSNorm bf16 [1, 2048] 2.55 / 2.0, f32
// [1, 1024] 2.3 / 1.9, bf16 [5, 2560] 2.8 / 2.2, f32 [15, 1280] 3.0 / 2.2, [2, 2048] 2.5 / 2.1, LayerNorm f32 [15, 1792] 3.2 / 2.3;
// one after another in a graph RMSNorm bf16 [3, 2048] 2.7 / 1.8, [3, 4096] 2.4 / 2.2, LayerNorm f32 [3, 1024] 2.7 / 1.7.
// Rows of narrow elements of nine vectors a lane and more are the masked shapes' from 32 rows up to as many as a wave for each
// vector wants (bf16 [64, 5600] 3.0 / 3.25, [501, 4112] 3.95 / 4.1, [700, 5600] 4.3 / 4.55, [1000, 5600] 5.4 / 5.2).
inline bool enough_rows(uint64_t rows, uint32_t per_lane, int size) {
  if (size == 2 && per_lane >= 9 && rows >= 32 && rows < 64u * per_lane) return false;
  return per_lane <= 8 || rows >= 16;
}

template <bool kLayer, int kVpl, int kThreads, int kRows> struct TailTag {
  static std::string text() {
    return std::string("norm_rows_tail/") + (kLayer ? "layer" : "rms") + "/64x" + std::to_string(kVpl) + "/" + std::to_string(kThreads) + "/" +
           std::to_string(kRows);
  }
};

template <class T, class W, bool kLayer, int kVpl, int kThreads, int kRows>
void launch_tail(const NormParams &p, const Bound &io, int parameters, hipStream_t s) {
  constexpr uint32_t kRowsPerBlock = kThreads / kWaveLanes * kRows;
  const uint32_t rows = (uint32_t)p.shape.rows, row_vectors = p.shape.width / Traits<T>::kVec;
  note_variant<TailTag<kLayer, kVpl, kThreads, kRows>>();
  const dim3 grid((rows + kRowsPerBlock - 1) / kRowsPerBlock), block(kThreads);
  const float width = (float)p.shape.width;
  if (parameters == kPlain)
    hipLaunchKernelGGL((norm_rows<T, W, kWaveLanes, kVpl, kThreads, kRows, kLayer, kPlain, false, true>), grid, block, 0, s, io.x, io.w, io.b,
                       io.y, rows, row_vectors, width, p.epsilon);
  else if (kLayer && parameters == kScaleBias)
    hipLaunchKernelGGL((norm_rows<T, W, kWaveLanes, kVpl, kThreads, kRows, kLayer, kLayer ? kScaleBias : kScale, false, true>), grid, block, 0,
                       s, io.x, io.w, io.b, io.y, rows, row_vectors, width, p.epsilon);
  else
    hipLaunchKernelGGL((norm_rows<T, W, kWaveLanes, kVpl, kThreads, kRows, kLayer, kScale, false, true>), grid, block, 0, s, io.x, io.w, io.b,
                       io.y, rows, row_vectors, width, p.epsilon);
}

// False: nothing was launched, the masked shapes are the faster.
template <class T, class W, bool kLayer, int kVpl>
bool run_tail(const NormParams &p, const Bound &io, int parameters, hipStream_t s) {
  const uint64_t rows = p.shape.rows, bytes = rows * p.shape.width * Traits<T>::kSize;
  // two rows per wave also where a smaller launch has more rows than waves find room at once (f32 LayerNorm [5000, 520],
  // masked / one row / two rows 5.6 / 6.3 / 5.3, [5000, 1000] 8.3 / 9.6 / 7.8, [9001, 520] 8.3 / 9.5 / 8.0; [2500, 520] 4.6 / 4.0 / 4.2)
  const bool once = (bytes >= (20ull << 20) || rows >= (Traits<T>::kSize == 4 ? 4000u : 7000u)) && bytes <= (64ull << 20);
  if constexpr (kVpl == 2) {
    // 2048 blocks of four rows find room at once, of a LayerNorm in f32 1536, and a launch of a few more is the masked shape's, of
    // two rows per wave, up to 20 MiB (masked / here: RMSNorm f32 [9001, 512] 7.0 / 7.75, [12000, 400] 7.2 / 8.5, [12000, 508] 11.3 / 10.1, [20001, 508]
    // 19.4 / 15.4, [5500, 508] 5.8 / 5.2; LayerNorm bf16 [9001, 1024] 7.7 / 8.8, f32 [7000, 400] 5.35 / 6.1)
    if (rows > (kLayer && Traits<T>::kSize == 4 ? 6144u : 8192u) && bytes < (20ull << 20)) return false;
    launch_tail<T, W, kLayer, kVpl, 256, 1>(p, io, parameters, s);
  } else if constexpr (!kLayer && kVpl == 4) {
    if (once) return false;
    launch_tail<T, W, kLayer, kVpl, 64, 1>(p, io, parameters, s);
  } else if constexpr (!kLayer || Traits<T>::kSize == 4) {
    if (once) launch_tail<T, W, kLayer, kVpl, 64, 2>(p, io, parameters, s);
    else launch_tail<T, W, kLayer, kVpl, 64, 1>(p, io, parameters, s);
  } else {
    // 5120 waves of these find room at once (masked / here: bf16 [6001, 1600] 7.9 / 9.4, [6001, 2000] 9.8 / 11.2, [5000, 2000]
    // 8.7 / 8.3, [7101, 2000] alike)
    if (kVpl == 4 && rows > 5120 && rows <= 6656) return false;
    launch_tail<T, W, kLayer, kVpl, 64, 1>(p, io, parameters, s);
  }
  return true;
}

template <class T, class W, bool kLayer>
bool run_tail_shape(const NormParams &p, const Bound &io, hipStream_t s) {
  constexpr uint32_t kVec = Traits<T>::kVec;
  if (p.shape.width % kVec != 0) return false;
  const uint32_t per_lane = (p.shape.width / kVec + kWaveLanes - 1) / kWaveLanes;
  if (!enough_rows(p.shape.rows, per_lane, Traits<T>::kSize)) return false;
  const int parameters = !p.has_weight ? kPlain : (kLayer && p.has_bias ? kScaleBias : kScale);
  switch (per_lane) {
    case 2: return run_tail<T, W, kLayer, 2>(p, io, parameters, s);
    case 3: return run_tail<T, W, kLayer, 3>(p, io, parameters, s);
    case 4: return run_tail<T, W, kLayer, 4>(p, io, parameters, s);
    case 5: return run_tail<T, W, kLayer, 5>(p, io, parameters, s);
    case 6: return run_tail<T, W, kLayer, 6>(p, io, parameters, s);
    case 7: return run_tail<T, W, kLayer, 7>(p, io, parameters, s);
    case 8: return run_tail<T, W, kLayer, 8>(p, io, parameters, s);
    case 9: return run_tail<T, W, kLayer, 9>(p, io, parameters, s);
    case 10: return run_tail<T, W, kLayer, 10>(p, io, parameters, s);
    case 11: return run_tail<T, W, kLayer, 11>(p, io, parameters, s);
    case 12: return run_tail<T, W, kLayer, 12>(p, io, parameters, s);
    default: return false;
  }
}

template <bool kLayer>
bool run_tail_typed(Elem type, const NormParams &p, const Bound &io, hipStream_t stream) {
  switch (type) {
    case Elem::kF32: return run_tail_shape<F32, F32, kLayer>(p, io, stream);
    case Elem::kF16:
      return p.weight_f32 ? run_tail_shape<F16, F32, kLayer>(p, io, stream) : run_tail_shape<F16, F16, kLayer>(p, io, stream);
    case Elem::kBF16:
      return p.weight_f32 ? run_tail_shape<BF16, F32, kLayer>(p, io, stream) : run_tail_shape<BF16, BF16, kLayer>(p, io, stream);
  }
  return false;
}

}  // namespace
}  // namespace hyle_hip
