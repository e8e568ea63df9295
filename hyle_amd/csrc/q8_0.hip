// q8_0.hip -- Q8_0 block dequant to bf16 fused with the per-row sum of squares,
// for gfx950.
//
// Block layout (src/compute_ops/low_precision.cc:28-29 of the reference; ggml
// block_q8_0): 34 bytes = little-endian fp16 scale d followed by 32 int8 quants.
// A weight [K, N] is stored as N physical rows of K/32 blocks
// (src/compute_ops/low_precision.cc:269-297).  Decode is y = (float)q * (float)d:
// an 8-bit by 11-bit significand product, exact in f32, so the bf16 store is one
// RN-even rounding and the result is bit-identical on every implementation.
//
// Blocks are only 2-byte aligned, so a wave parks its row in LDS with 16-byte global loads
// (every cache line requested once) and re-slices it there; output leaves as 16-byte bf16x8
// stores, 1 KiB of consecutive bf16 per store instruction of a wave.  Each row's sum of squares
// of the exact products is reduced with a wave64 butterfly.
//
// Three kernels: rows made of whole 16-byte vectors (K = 256 n) take one wave per row
// with a region of LDS that only this wave touches and no block barrier (q8_0_lines: aligned
// 32-bit LDS words joined by byte-wise funnel shifts), or, where a launch of rows of no whole spans is resident at
// once, whole rows staged by blocks (q8_0_rows); anything else reads bytes (q8_0_rows_bytes).
#include <algorithm>
#include <type_traits>

#include "device_common.h"
#include "gguf_decode.h"
#include "kernels.h"

namespace hyle_hip {
namespace {

constexpr int kBlockBytes = 34;
constexpr int kBlockElems = 32;

// Rows of whole 16-byte vectors (K = 256 n), 16-byte aligned: one wave per row, no barrier.
// A span of 2048 values is 64 blocks = 2176 bytes = 136 vectors: two per lane and a third for
// the first eight lanes (the others repeat the span's last vector, one request for all of them), the row's last
// span what is left of it: 17 vectors to 256 values;
// plain loads: the non-temporal hint costs 10 % here, while the stores keep it.
// The vectors are parked in LDS that only this wave touches (LDS executes one wave's
// instructions in order); lane l then decodes output vectors l, l + 64, l + 128, l + 192 of
// the span: eight quants at a 2-byte aligned offset come out of three aligned words and two
// funnel shifts, the block's scale out of one 16-bit read.  The next span's loads are in flight
// while this one is decoded.
// (kWhole: rows of whole spans, which then have no bounds to look at: [2048 x 1024] 3.0 us, 3.1 with them)
template <int kWaves, bool kWhole>
__global__ __launch_bounds__(kWaves *kWaveLanes) void q8_0_lines(const unsigned char *blocks, void *out,
                                                                float *sumsq, uint32_t rows, uint32_t k,
                                                                uint64_t row_stride) {
  constexpr uint32_t kSpan = 2048;
  constexpr uint32_t kVectors = kSpan / kBlockElems * kBlockBytes / 16;  // 136
  constexpr int kLoads = (kVectors + kWaveLanes - 1) / kWaveLanes;       // 3
  __shared__ __align__(16) unsigned char slots[kWaves][kLoads * kWaveLanes * 16];
  const uint32_t lane = threadIdx.x % kWaveLanes;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWaveLanes);
  const uint32_t row = blockIdx.x * kWaves + wave;
  if (row >= rows) return;
  unsigned char *slot = slots[wave];
  const unsigned char *source = blocks + (size_t)row * row_stride;
  const uint32_t steps = (k + kSpan - 1) / kSpan;
  u32x4 raw[kLoads];
  auto load = [&](uint32_t step) {
    const uint32_t last = (kWhole ? kVectors : min(kVectors, (k - step * kSpan) / 256 * 17)) - 1;
#pragma unroll
    for (int i = 0; i < kLoads; ++i) raw[i] = load16(source, (size_t)step * kVectors + min(lane + i * kWaveLanes, last));
  };
  load(0);
  float squares = 0.0f;
  for (uint32_t step = 0; step < steps; ++step) {
#pragma unroll
    for (int i = 0; i < kLoads; ++i) *reinterpret_cast<u32x4 *>(slot + (size_t)(lane + i * kWaveLanes) * 16) = raw[i];
    if (step + 1 < steps) load(step + 1);  // uniform across the wave
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const uint32_t values = k - step * kSpan;
    auto decode = [&](auto whole) {  // a whole span has no branch, so that its LDS reads go out together
#pragma unroll
      for (uint32_t i = 0; i < kSpan / (kWaveLanes * 8); ++i) {
        const uint32_t j = i * kWaveLanes + lane;  // output vector of the span: block j / 4, quants 8 (j % 4) ..
        if (!decltype(whole)::value && 8 * j >= values) break;
        const uint32_t block_offset = (j / 4) * kBlockBytes;
        const float d = f16_to_f32(*reinterpret_cast<const uint16_t *>(slot + block_offset));
        uint32_t q[2];
        lds_piece(slot, block_offset + 2 + 8 * (j % 4), q);
        float y[8];
#pragma unroll
        for (int w = 0; w < 2; ++w)
#pragma unroll
          for (int t = 0; t < 4; ++t) y[4 * w + t] = (float)(int)(signed char)(q[w] >> (8 * t)) * d;
        squares += sum_of_squares(y);
        store16_stream(out, ((size_t)row * k + (size_t)step * kSpan) / 8 + j, Traits<BF16>::pack(y));
      }
    };
    if (kWhole || values >= kSpan) decode(std::true_type{});
    else decode(std::false_type{});
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
  const double total = wave_sum_of_eighths(squares);
  if (lane == 0) sumsq[row] = (float)total;
}

// Rows of whole 16-byte vectors, 16-byte aligned: a block stages a whole row for each of its waves, and decodes once all
// are there.  Few registers, and no piece of a row left over: where all blocks of a launch are resident at once, their reads end
// before their writes begin, and a short last span does not cost a step of its own.
template <int kWaves>
__global__ __launch_bounds__(kWaves *kWaveLanes) void q8_0_rows(const unsigned char *blocks, void *out, float *sumsq, uint32_t rows, uint32_t k,
                                                               uint64_t row_stride) {
  extern __shared__ __align__(16) unsigned char staged[];
  const uint32_t wave = threadIdx.x / kWaveLanes, lane = threadIdx.x % kWaveLanes;
  const uint32_t row = blockIdx.x * kWaves + wave;
  const uint32_t row_vectors = k / 256 * 17, out_vectors = k / 8;
  unsigned char *mine = staged + (size_t)wave * row_vectors * 16;
  if (row < rows) {
    const unsigned char *source = blocks + (size_t)row * row_stride;
    for (uint32_t v = lane; v < row_vectors; v += kWaveLanes) reinterpret_cast<u32x4 *>(mine)[v] = load16_stream(source, v);
  }
  __syncthreads();
  float squares = 0.0f;
  if (row < rows) {
    for (uint32_t j = lane; j < out_vectors; j += kWaveLanes) {  // block j / 4, quants 8 (j % 4) ..
      const unsigned char *block = mine + (size_t)(j / 4) * kBlockBytes;
      const float d = f16_to_f32(*reinterpret_cast<const uint16_t *>(block));
      const uint16_t *q = reinterpret_cast<const uint16_t *>(block + 2 + 8 * (j % 4));
      float y[8];
#pragma unroll
      for (int h = 0; h < 4; ++h) {
        const uint32_t pair = q[h];
        y[2 * h] = (float)(int8_t)(pair & 0xFFu) * d;
        y[2 * h + 1] = (float)(int8_t)(pair >> 8) * d;
      }
      squares += sum_of_squares(y);
      store16_stream(out, (size_t)row * out_vectors + j, Traits<BF16>::pack(y));
    }
  }
  const double total = wave_sum_of_eighths(squares);
  if (row < rows && lane == 0) sumsq[row] = (float)total;
}

// Any k (multiple of 32), any stride or alignment: one wave per row, byte loads.
__global__ __launch_bounds__(kBlockThreads) void q8_0_rows_bytes(const uint8_t *blocks, uint16_t *out,
                                                                 float *sumsq, uint32_t rows,
                                                                 uint32_t k, uint64_t row_stride) {
  const uint32_t wave = threadIdx.x / kWaveLanes, lane = threadIdx.x % kWaveLanes;
  const uint32_t row = blockIdx.x * (kBlockThreads / kWaveLanes) + wave;
  const bool row_ok = row < rows;
  float squares = 0.0f;
  if (row_ok) {
    const uint8_t *src = blocks + (size_t)row * row_stride;
    for (uint32_t e = lane; e < k; e += kWaveLanes) {
      const uint8_t *block = src + (size_t)(e / kBlockElems) * kBlockBytes;
      const float d = f16_to_f32((uint16_t)(block[0] | ((uint16_t)block[1] << 8)));
      const float y = (float)(int8_t)block[2 + e % kBlockElems] * d;
      squares = __builtin_fmaf(y, y, squares);
      out[(size_t)row * k + e] = f32_to_bf16(y);
    }
  }
  squares = group_sum<kWaveLanes>(squares);
  if (row_ok && lane == 0) sumsq[row] = squares;
}

template <bool kWhole> struct LinesTag {
  static std::string text() { return kWhole ? "q8_0_lines" : "q8_0_lines/pieces"; }
};
struct RowsTag {
  static std::string text() { return "q8_0_rows"; }
};
struct BytesTag {
  static std::string text() { return "q8_0_rows_bytes"; }
};

// Where q8_0_rows is the faster one: rows of more than one span and no whole number of them, in launches that are resident at once
// (a compute unit holds eight blocks of four waves, or as many as have room in its LDS) and have more than four blocks to a unit, three
// and a half of rows of more than two spans.  MI355X, us, lines / rows: [2304 x 6144] 9.8 / 8.3, [2816 x 4352] 8.2 / 6.9, [4608 x 8192] 22.3 / 20.3,
// [4864 x 7168] 21.9 / 19.9, [5888 x 6144] 22.2 / 20.3, [7424 x 3584] 17.0 / 16.0; one block more than fit: [4608 x 8448] 22.9 / 24.7,
// [4864 x 7680] 23.0 / 23.9, [6656 x 6144] 24.9 / 26.3; fewer: [3072 x 3072] 6.4 / 7.2, [8960 x 3073] 17.0 / 19.6, [8960 x 3328] alike.
constexpr uint32_t kUnitLds = 160 * 1024;
inline bool rows_pay(const Q8Params &p, int compute_units) {
  if (p.k <= 2048 || p.k % 2048 == 0) return false;
  const uint32_t fit = std::min(8u, kUnitLds / (4 * (p.k / kBlockElems) * kBlockBytes));
  const uint64_t units = compute_units > 0 ? (uint64_t)compute_units : 256u, blocks = (p.rows + 3) / 4;
  return (p.k <= 4096 ? blocks > 4 * units : 2 * blocks >= 7 * units) && blocks <= fit * units;
}

}  // namespace

hipError_t launch_q8_0_dequant(const Q8Params &p, const void *blocks, void *out, float *sumsq,
                               bool vectorised, int compute_units, hipStream_t stream) {
  if (p.rows == 0) return hipSuccess;
  const uint32_t rows = (uint32_t)p.rows;
  if (vectorised && p.k != 0 && p.k % 256 == 0 && p.row_stride % 16 == 0) {
    // Measured on MI355X for W[6144 x 2048] (38.6 MB of traffic, buffers rotated): 6.7 us with
    // plain loads and non-temporal stores; 7.4 us with non-temporal loads too; 8.6 / 10.5 us with
    // plain stores; a wave that walks several rows with the next row in flight 7.3 - 9.3 us.  Widths that are no multiple
    // of 2048, in blocks that stage their rows / like this: [1280 x 14080] 13.1 / 9.4 us, [3840 x 1024] 5.2 / 3.8, [5120 x 16000] 49 / 40.
    constexpr int kWaves = 4;
    const dim3 grid((rows + kWaves - 1) / kWaves), block(kWaves * kWaveLanes);
    const unsigned char *in = static_cast<const unsigned char *>(blocks);
    if (rows_pay(p, compute_units)) {
      note_variant<RowsTag>();
      hipLaunchKernelGGL((q8_0_rows<kWaves>), grid, block, (size_t)kWaves * (p.k / kBlockElems) * kBlockBytes, stream, in, out, sumsq, rows, p.k,
                         p.row_stride);
    } else if (p.k % 2048 == 0) {
      note_variant<LinesTag<true>>();
      hipLaunchKernelGGL((q8_0_lines<kWaves, true>), grid, block, 0, stream, in, out, sumsq, rows, p.k, p.row_stride);
    } else {
      note_variant<LinesTag<false>>();
      hipLaunchKernelGGL((q8_0_lines<kWaves, false>), grid, block, 0, stream, in, out, sumsq, rows, p.k, p.row_stride);
    }
    return hipGetLastError();
  }
  constexpr int kWaves = kBlockThreads / kWaveLanes;
  note_variant<BytesTag>();
  hipLaunchKernelGGL(q8_0_rows_bytes, dim3((rows + kWaves - 1) / kWaves), dim3(kBlockThreads), 0,
                     stream, static_cast<const uint8_t *>(blocks), static_cast<uint16_t *>(out),
                     sumsq, rows, p.k, p.row_stride);
  return hipGetLastError();
}

}  // namespace hyle_hip
