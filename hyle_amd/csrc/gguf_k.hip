// GGUF Q4_K and Q6_K rows -> bf16 [rows, k] plus the f32 row sums of squares of the exact f32
// values, the K-quant siblings of q8_0.hip.
//
// Geometry from the reference (src/compute_ops/low_precision.cc:22-27: 256 elements in 144 and
// 210 bytes); the decode is ggml's dequantize_row_q4_K / dequantize_row_q6_K, restated from the
// published block layouts, checked against the two readings of these formats the reference
// tree holds (third_party/ggml_q4k_apple/ggml_q4k_apple.h:9-38;
// tests/compute_models/qwen27_original_nextn_reference.h:74-86,262-287):
//   Q4_K  {f16 d; f16 dmin; u8 scales[12]; u8 qs[128]}   y = (d * sc) * q - (dmin * m)
//   Q6_K  {u8 ql[128]; u8 qh[64]; i8 scales[16]; f16 d}  y = (d * scale) * (q - 32)
// with separate f32 roundings for the products and the subtraction, as the source writes them.
//
// Two kernels.  Q4_K rows on 16-byte boundaries and Q6_K rows at even addresses (the usual case)
// take a wave or a block per row, whole cache lines into wave-private LDS and word-wise decoding
// (k_quant_lines, measured 5.9 / 6.3 us for Q4_K / Q6_K [6144 x 2048] on MI355X).  Anything else, Q4_K rows off a
// 16-byte boundary and Q6_K rows at odd addresses or an odd number of bytes apart,
// takes the general kernel: a block of 256 threads takes four rows at a time, eight super-blocks
// of each (at most 1680 bytes) are staged in LDS per step with the widest loads the row's
// address allows, and a thread decodes eight neighbouring values from LDS bytes (Q4_K [6144 x 2048] four bytes off 10.8 us,
// Q6_K one byte off 17.1).  Both store eight values as one 16-byte vector.
#include <type_traits>

#include "device_common.h"
#include "gguf_decode.h"
#include "kernels.h"

namespace hyle_hip {
namespace {

constexpr int kChunkBlocks = kBlockThreads * 8 / kSuper;  // super-blocks decoded per step: 8

// Bytes -> LDS with the widest loads the address allows: words, pairs or single bytes for Q4_K rows, whatever boundary they are
// off; single bytes for a chunk of Q6_K blocks at an odd address, pairs for the rows between whose addresses are even.
__device__ __forceinline__ void stage(unsigned char *to, const unsigned char *from, uint32_t bytes) {
  if (((reinterpret_cast<uintptr_t>(from) | bytes) & 3u) == 0) {
    for (uint32_t i = threadIdx.x; i < bytes / 4; i += kBlockThreads)
      reinterpret_cast<uint32_t *>(to)[i] = __builtin_nontemporal_load(reinterpret_cast<const uint32_t *>(from) + i);
  } else if (((reinterpret_cast<uintptr_t>(from) | bytes) & 1u) == 0) {
    for (uint32_t i = threadIdx.x; i < bytes / 2; i += kBlockThreads)
      reinterpret_cast<uint16_t *>(to)[i] = __builtin_nontemporal_load(reinterpret_cast<const uint16_t *>(from) + i);
  } else {
    for (uint32_t i = threadIdx.x; i < bytes; i += kBlockThreads) to[i] = from[i];
  }
}

// kRows rows per block: their chunks are staged together, so kRows times the bytes are in flight
// per barrier and each thread has kRows independent decodes.
template <int kKind, int kRows>  // 0 = Q4_K, 1 = Q6_K
__global__ __launch_bounds__(kBlockThreads) void k_quant_rows(const unsigned char *blocks, void *out,
                                                              float *sumsq, uint32_t rows, uint32_t k,
                                                              uint64_t row_stride) {
  constexpr uint32_t kBlockBytes = kKind == 0 ? 144 : 210;
  constexpr uint32_t kSlot = (kChunkBlocks * kBlockBytes + 15) / 16 * 16;
  __shared__ __align__(16) unsigned char staged[kRows][kSlot];
  __shared__ float joint[kRows][kBlockThreads / kWaveLanes];
  const uint32_t first_row = blockIdx.x * kRows;
  const uint32_t super_blocks = k / kSuper;
  float acc[kRows];
#pragma unroll
  for (int r = 0; r < kRows; ++r) acc[r] = 0.0f;
  for (uint32_t first = 0; first < super_blocks; first += kChunkBlocks) {
    const uint32_t count = min((uint32_t)kChunkBlocks, super_blocks - first);
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
      const uint32_t row = min(first_row + r, rows - 1);  // a row past the end re-reads the last one
      stage(staged[r], blocks + (size_t)row * row_stride + (size_t)first * kBlockBytes, count * kBlockBytes);
    }
    __syncthreads();
    const uint32_t local = threadIdx.x * 8;  // position within the chunk
    if (local < count * kSuper) {
#pragma unroll
      for (int r = 0; r < kRows; ++r) {
        const unsigned char *blk = staged[r] + (local / kSuper) * kBlockBytes;
        float y[8];
        if constexpr (kKind == 0) decode_q4_k(blk, local % kSuper, y);
        else decode_q6_k(blk, local % kSuper, y);
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[r] = __builtin_fmaf(y[j], y[j], acc[r]);
        if (first_row + r < rows) {
          const size_t element = (size_t)(first_row + r) * k + (size_t)first * kSuper + local;
          store16_stream(out, element / 8, Traits<BF16>::pack(y));
        }
      }
    }
    __syncthreads();  // the next step overwrites the staging
  }
#pragma unroll
  for (int r = 0; r < kRows; ++r) {
    const float total = row_sum<kBlockThreads>(acc[r], joint[r]);
    if (threadIdx.x == 0 && first_row + r < rows) sumsq[first_row + r] = total;
  }
}

// One wave per row, or kShare waves where rows are few and wide; no barrier before the row's last.
// The wave reads 2048 values' worth of blocks (1152 or 1680 bytes, the row's last piece what is left of it) as
// aligned 16-byte vectors, one per lane and request, so that every cache line is asked for once; parks them in a
// region of LDS that only this wave touches (LDS executes one wave's instructions in order); and each lane
// decodes eight neighbouring values at a time from aligned 32-bit words, so that a store
// instruction of the wave writes 1 KiB of consecutive bf16.  The next piece is on its
// way while this one is decoded.  A Q6_K row may start at any even address: its vectors start at the 16-byte boundary
// at or below it, as far below for every piece (1680 = 105 * 16), and the decoder joins words anyway.  (Q4_K headers
// are read as words: rows on 16-byte boundaries.)  The loads are plain ones: with the non-temporal hint
// [6144 x 2048] took 8.0 / 9.3 us instead of 5.9 / 6.3 us (the bf16 stores keep the hint).
// Bound by HBM.  MI355X, us, before (a block to four rows, below) / here:
//   Q4_K [1280 x 2048] 6.2 / 3.5  [2560 x 6144] 15.6 / 7.8  [5120 x 14080] 52.5 / 30.0 (6160 GB/s)
//   Q6_K [1024 x 5120] 7.7 / 4.1  [3328 x 1280] 15.9 / 4.0  [17408 x 2048] 56.8 / 17.1 (5870 GB/s)
// (kWhole: rows of whole pieces, which then have no bounds to look at: [2048 x 1024] 3.3 us, 3.4 with them)
template <int kKind, int kShare, bool kWhole>  // 0 = Q4_K, 1 = Q6_K
__global__ __launch_bounds__(kBlockThreads) void k_quant_lines(const unsigned char *blocks, void *out, float *sumsq,
                                                               uint32_t rows, uint32_t k, uint64_t row_stride) {
  constexpr uint32_t kBlockBytes = kKind == 0 ? 144 : 210;
  constexpr uint32_t kSpan = 2048, kSpanBytes = kSpan / kSuper * kBlockBytes;  // values and bytes per step: 72 or 105 vectors
  constexpr int kLoads = 2;                                                    // at most 106 vectors
  constexpr int kWaves = kBlockThreads / kWaveLanes;
  __shared__ __align__(16) unsigned char slots[kWaves][kLoads * kWaveLanes * 16];
  __shared__ double joint[kShare];
  const uint32_t lane = threadIdx.x % kWaveLanes;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWaveLanes);
  const uint32_t wanted_row = blockIdx.x * (kWaves / kShare) + wave / kShare, member = wave % kShare;
  if (kShare == 1 && wanted_row >= rows) return;
  const uint32_t row = min(wanted_row, rows - 1);  // (waves that share a row all have one)
  unsigned char *slot = slots[wave];
  const unsigned char *source = blocks + (size_t)row * row_stride;
  const uint32_t below = kKind == 0 ? 0u : (uint32_t)reinterpret_cast<uintptr_t>(source) & 15u;
  source -= below;
  const uint32_t steps = (k + kSpan - 1) / kSpan;
  u32x4 raw[kLoads];
  auto load = [&](uint32_t step) {
    const uint32_t bytes = kWhole ? kSpanBytes : min(kSpan, k - step * kSpan) / kSuper * kBlockBytes, last = (below + bytes - 1) / 16;
#pragma unroll
    for (int i = 0; i < kLoads; ++i)  // past the piece: its last vector again (parked, never read)
      raw[i] = load16(source + (size_t)step * kSpanBytes, min(lane + i * kWaveLanes, last));
  };
  load(min(member, steps - 1));
  float squares = 0.0f;
  for (uint32_t step = member; step < steps; step += kShare) {
#pragma unroll
    for (int i = 0; i < kLoads; ++i) *reinterpret_cast<u32x4 *>(slot + (size_t)(lane + i * kWaveLanes) * 16) = raw[i];
    load(min(step + kShare, steps - 1));
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const uint32_t values = k - step * kSpan;
    auto decode = [&](auto whole) {  // a whole piece has no branch, so that its LDS reads go out together
#pragma unroll
      for (uint32_t i = 0; i < kSpan / (kWaveLanes * 8); ++i) {
        const uint32_t p = (i * kWaveLanes + lane) * 8;  // position within the span
        if (!decltype(whole)::value && p >= values) break;
        float y[8];
        if constexpr (kKind == 0) decode_q4_k_words(slot, (p / kSuper) * kBlockBytes, p % kSuper, y);
        else decode_q6_k_words(slot, below + (p / kSuper) * kBlockBytes, p % kSuper, y);
        squares += sum_of_squares(y);
        store16_stream(out, ((size_t)row * k + (size_t)step * kSpan + p) / 8, Traits<BF16>::pack(y));
      }
    };
    if (kWhole || values >= kSpan) decode(std::true_type{});
    else decode(std::false_type{});
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
  double total = wave_sum_of_eighths(squares);
  if constexpr (kShare == 1) {
    if (lane == 0) sumsq[row] = (float)total;
  } else {
    static_assert(kShare == kWaves, "a row to a block");
    if (lane == 0) joint[wave] = total;
    __syncthreads();
    total = joint[0];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) total += joint[w];
    if (threadIdx.x == 0) sumsq[row] = (float)total;
  }
}

}  // namespace

namespace {
enum : int { kGeneral = 0, kWholePieces = 1, kPieces = 2, kShared = 3 };  // a wave to a row, or (kShared) a block
template <int kKind, int kForm> struct KQuantTag {
  static std::string text() {
    return std::string(kForm == kGeneral ? "k_quant_rows/" : "k_quant_lines/") + (kKind == 0 ? "q4_k" : "q6_k") +
           (kForm == kShared ? "/shared" : (kForm == kPieces ? "/pieces" : ""));
  }
};

template <int kKind>
hipError_t run_lines(const KQuantParams &p, const unsigned char *in, void *out, float *sumsq, int compute_units, hipStream_t stream) {
  constexpr uint32_t kWaves = kBlockThreads / kWaveLanes;
  const uint32_t rows = (uint32_t)p.rows;
  // A block to a row of more than one piece where the compute units find room for all rows at once, eight to a unit; Q4_K
  // rows, with more to decode per byte, gain up to seven of one or two pieces, seven and a half of three or four, six and a half of more (us, a
  // wave / a block: Q6_K [17408 x 512] 9.1 / 5.55, [6144 x 1280] 6.4 / 4.9, [3840 x 2048] 5.5 / 5.0, [3840 x 2560] 5.9 / 6.1; Q4_K
  // [5120 x 1024] 4.9 / 3.9, [4096 x 1792] 4.6 / 4.5, [4096 x 2048] 4.8 / 5.5, [2304 x 2048] 4.1 / 4.8, [6144 x 1793] 6.0 / 5.7,
  // [6144 x 2047] 6.2 / 6.4, [9728 x 1537] 8.5 / 7.7, [17408 x 1793] 13.8 / 14.8).
  const uint32_t halves = kKind == 1 ? 16 : (p.k <= 4096 ? 14 : (p.k <= 8192 ? 15 : 13));
  const bool shared = p.k > 2048 && rows <= halves * (compute_units > 0 ? (uint32_t)compute_units : 256u) / 2;
  const dim3 waves((rows + kWaves - 1) / kWaves), block(kBlockThreads);
  if (shared) {
    note_variant<KQuantTag<kKind, kShared>>();
    hipLaunchKernelGGL((k_quant_lines<kKind, kWaves, false>), dim3(rows), block, 0, stream, in, out, sumsq, rows, p.k, p.row_stride);
  } else if (p.k % 2048 != 0) {
    note_variant<KQuantTag<kKind, kPieces>>();
    hipLaunchKernelGGL((k_quant_lines<kKind, 1, false>), waves, block, 0, stream, in, out, sumsq, rows, p.k, p.row_stride);
  } else {
    note_variant<KQuantTag<kKind, kWholePieces>>();
    hipLaunchKernelGGL((k_quant_lines<kKind, 1, true>), waves, block, 0, stream, in, out, sumsq, rows, p.k, p.row_stride);
  }
  return hipGetLastError();
}
}  // namespace

hipError_t launch_k_quant_dequant(const KQuantParams &p, const void *blocks, void *out, float *sumsq, int compute_units,
                                  hipStream_t stream) {
  if (p.rows == 0) return hipSuccess;
  const unsigned char *in = static_cast<const unsigned char *>(blocks);
  // whole blocks on 16-byte (Q6_K: even) boundaries
  const uint64_t together = reinterpret_cast<uintptr_t>(blocks) | p.row_stride;
  if (p.k != 0 && p.k % kSuper == 0 && (together & (p.kind == 0 ? 15u : 1u)) == 0)
    return p.kind == 0 ? run_lines<0>(p, in, out, sumsq, compute_units, stream) : run_lines<1>(p, in, out, sumsq, compute_units, stream);
  constexpr int kRows = 4;
  const dim3 grid(((uint32_t)p.rows + kRows - 1) / kRows), block(kBlockThreads);
  if (p.kind == 0) note_variant<KQuantTag<0, kGeneral>>();
  else note_variant<KQuantTag<1, kGeneral>>();
  if (p.kind == 0)
    hipLaunchKernelGGL((k_quant_rows<0, kRows>), grid, block, 0, stream, in, out, sumsq, (uint32_t)p.rows, p.k,
                       p.row_stride);
  else
    hipLaunchKernelGGL((k_quant_rows<1, kRows>), grid, block, 0, stream, in, out, sumsq, (uint32_t)p.rows, p.k,
                       p.row_stride);
  return hipGetLastError();
}

}  // namespace hyle_hip
