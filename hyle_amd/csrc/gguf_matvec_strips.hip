// y[m][n] = MatMul(x, W) on the ggml route (8-bit activation blocks, integer dots; the arithmetic is
// described in gguf_matvec_q8.hip) for one to eight activation rows against many weight rows: any
// width of whole runs of 256 values, rows at any even address, every dot on the matrix unit.
//
// v_mfma_i32_16x16x64_i8: lane (c, p) = c + 16 p gives sixteen int8 of row c of A and of column c of
// B at k-slots 16 p .. 16 p + 15, and gets D[4 p .. 4 p + 3][c] back.  A column is a weight row.  Of
// every run of 256 values lane (c, p) decodes whole scale groups of row c:
//   Q8_0  blocks p and 4 + p of the run's eight
//   Q6_K  the 16-value groups of half p / 2 at positions 16 (p % 2) .. + 15 of each 32
//   Q4_K  sub-blocks 2 p and 2 p + 1
// Row 4 q + t of A carries activation row t's codes at the k-slots of lanes p == q and zeros at the
// others, so the four values that lane (c, p) gets back are the dots of *its own* group of weight
// row c against activation rows 0 .. 3: the scales it needs are the ones it holds, and a second set
// of A rows serves activation rows 4 .. 7 from the same weight registers.  A lane that carries zeros
// reads them from a row of zeros in LDS: its address does not advance.
//
// Q8_0 rows of whole 16-byte vectors need no decoding: a run's 272 bytes go to the matrix unit as they
// lie, a wave's five windows of four vectors at a time (the fifth holds the seventeenth vector), and the codes
// are laid out to match, each block's 32 in 48 bytes of LDS at the place its quants have in the three vectors
// that hold them, zeros round them (at the scale, and at the neighbours' bytes).  Row 4 q + t of A holds the codes of
// block 4 g + q for the g-th half of a run, so three windows give a lane the dots of one block again; its scale
// comes out of the windows with two lane swaps.
//
// A block of sixteen waves (eight where the codes leave no room for more slots) has a compute unit's
// LDS, quantises the activation rows once, while its first weight bytes are on their way, and walks its
// share of the weight rows in tiles of at most sixteen; `split` waves share a tile, each
// taking every split-th run, and the first adds the shares.  A lane's chain of up to 224 runs, the sums
// over the lanes of a column and the sum over the shares run in 64 bits: in 32, a chain that is several times as long
// as one of the kernels that spread a row over 64 lanes was further from the 64-bit sum than theirs in a third of the
// shapes (f32 Q8_0 [5120 -> 2304] x 6 9.6e-8 relative against 8.4e-8 there, Q4_K [4096 -> 6656] x 4 7.6e-8 against 7.1e-8;
// in 64 bits 3.5e-8 for both, at most 4.3e-8 over 300 shapes, for about 1 % of the time).  Q8_0 and Q6_K runs are loaded as the aligned vectors that cover them and
// redistributed through a wave-private slot: lanes that load their own 16 bytes at 2-byte addresses keep the
// memory pipe busy several times as long (Q8_0 [2048 -> 151936] 111 us that way, 63 us through the slot), and lanes
// that load their own aligned vectors ask for sixteen half lines at a time (in place, [5120 -> 17408] x 4 24.6 us,
// through the slot 21.6: the direct form serves where the codes leave no room for slots).  A Q4_K row is whole
// vectors and goes straight into the lanes (52 us through the slot, 43 us straight).  The loads are plain ones: a run's
// last line is the next run's first, which another wave asks for (non-temporal: 24.0 us).
//
// A wave has one run on its way while it works on the one before.  More are slower: sixteen waves with two or three
// runs each ask for several times what the first-level cache holds, and the lines at the seams of neighbouring runs,
// which another wave asks for at about the same time, are gone by then (a bare read of Q8_0 [5120 -> 17408] in this pattern
// 20.6 us with two runs a wave, two neighbouring runs at once and nothing behind them 18.1; lane-contiguous 15.6).
//
// Bound by HBM in that pattern from about 50 MB of weights on, and by what stands round the stream: of the 23.3 us of Q8_0
// [5120 -> 17408] x 5 quantising takes 1.5, at [17408 -> 5120] 4.8 of 25.9, of the 5 to 6 us of a few MB 1 to 1.5.
// MI355X, bf16 activations, us (weights of 600 MB in turn); before: two or three runs on their way, loads of an address that
// had been an integer (flat ones, which every wait for LDS waits for), a power of two waves to a tile:
//   Q8_0 [5120 -> 17408] x 5   24.8 -> 23.3 (4060 GB/s)    [17408 -> 5120] x 5   27.7 -> 25.9
//   Q6_K [5120 -> 17408] x 5   24.1 -> 20.3                [13056 -> 5120] x 2   17.5 -> 16.6
//   Q4_K [5120 -> 17408] x 5   20.7 -> 16.3                [5120 -> 13056] x 2   12.5 -> 10.6    [14080 -> 3328] x 1   10.5 -> 9.3
//   Q8_0 [2304 -> 7936] x 2 8.5 -> 7.2    Q4_K [2816 -> 2304] x 6 6.3 -> 5.9    Q6_K [1280 -> 3328] x 8 6.1 -> 5.5
#include <type_traits>

#include "device_common.h"
#include "gguf_q8_math.h"
#include "gguf_q8_quantise.h"
#include "kernels.h"

namespace hyle_hip {
namespace {

constexpr uint32_t kStripRows = 16, kMostWaves = 16;
constexpr size_t kStripLds = 160 * 1024;  // of a compute unit, and the most one block can have
constexpr uint32_t kZeroBytes = 384;      // a lane's operands of one run lie within 384 bytes of its base
constexpr uint32_t kCodePad = 16;         // between activation rows: neighbours start on other LDS banks

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// kWords words of LDS from any even offset.
template <int kWords> __device__ __forceinline__ void lds_even(const unsigned char *slot, uint32_t offset, uint32_t *out) {
  const uint32_t *words = reinterpret_cast<const uint32_t *>(slot + (offset & ~3u));
  uint32_t w[kWords + 1];
#pragma unroll
  for (int i = 0; i <= kWords; ++i) w[i] = words[i];
#pragma unroll
  for (int i = 0; i < kWords; ++i) out[i] = __builtin_amdgcn_alignbyte(w[i + 1], w[i], offset & 2u);
}

// The aligned 16-byte vectors that cover a run of a tile's sixteen rows, as a wave loads and parks
// them: kVectors per row (a run starts up to 14 bytes into its first), rows an odd number of vectors
// apart in LDS, so that the sixteen rows of a column start on different banks.
template <uint32_t kBytes> struct StripStage {
  static constexpr bool kParked = true, kWhole = false;
  static constexpr uint32_t kRunBytes = kBytes, kVectors = (kBytes + 14 + 15) / 16, kPitch = (kVectors | 1u) * 16;
  static constexpr uint32_t kLoads = (kStripRows * kVectors + kWaveLanes - 1) / kWaveLanes, kSlotBytes = kStripRows * kPitch;
  struct Pending {
    u32x4 v[kLoads];
  };
};

// What a lane decodes of one run of its weight row, from the wave's slot; `at`: the run's first byte.
template <int kKind> struct Strip;
template <> struct Strip<0> {  // rows are whole 16-byte vectors as a rule: loaded straight into the lanes
  static constexpr bool kParked = false, kWhole = false;
  // one piece per lane of its own row
  static constexpr uint32_t kRunBytes = 144, kVectors = 1, kLoads = 1, kSlotBytes = 0;
  using Pending = Strip;
  u32x4 head, q[2];
  __device__ __forceinline__ void load(const unsigned char *at, uint32_t part) {
    head = *reinterpret_cast<const u32x4_element *>(at);
#pragma unroll
    for (int s = 0; s < 2; ++s) q[s] = *reinterpret_cast<const u32x4_element *>(at + 16 + 32 * part + 16 * s);
  }
};
template <> struct Strip<1> : StripStage<210> {
  u32x4 low, high, top;
  uint32_t scales[2];
  uint16_t d;
  __device__ __forceinline__ void take(const unsigned char *slot, uint32_t at, uint32_t part) {
    const uint32_t half = part / 2, sub = part % 2;
    uint32_t words[4];
    lds_even<4>(slot, at + 64 * half + 16 * sub, words);
    low = u32x4{words[0], words[1], words[2], words[3]};
    lds_even<4>(slot, at + 64 * half + 32 + 16 * sub, words);
    high = u32x4{words[0], words[1], words[2], words[3]};
    lds_even<4>(slot, at + 128 + 32 * half + 16 * sub, words);
    top = u32x4{words[0], words[1], words[2], words[3]};
    lds_even<2>(slot, at + 192 + 8 * half, scales);
    d = *reinterpret_cast<const uint16_t *>(slot + at + 208);
  }
};
template <> struct Strip<2> : StripStage<272> {
  u32x4 q[4];
  uint16_t d[2];
  __device__ __forceinline__ void take(const unsigned char *slot, uint32_t at, uint32_t part) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      // the block's nine words hold its scale in front of the quants, or half a word later
      const uint32_t block = at + 34 * (4 * j + part);
      const uint32_t *words = reinterpret_cast<const uint32_t *>(slot + (block & ~3u));
      const bool late = (block & 2u) != 0;
      const uint32_t select = late ? 0x07060504u : 0x05040302u;
      uint32_t w[9];
#pragma unroll
      for (int i = 0; i < 9; ++i) w[i] = words[i];
      d[j] = (uint16_t)(late ? w[0] >> 16 : w[0]);
#pragma unroll
      for (int i = 0; i < 8; ++i) q[2 * j + i / 4][i % 4] = __builtin_amdgcn_perm(w[i + 1], w[i], select);
    }
  }
};

// Q8_0 rows of whole 16-byte vectors, as they lie in memory: lane (c, p) holds vectors 4 w + p of the run's seventeen
// (the seventeenth alone in the fifth window, in every part).  Strip<4> loads a tile's runs one after another and parks
// them, Strip<3> loads straight into the lanes and needs no slots.
struct StripInPlace {
  static constexpr uint32_t kRunBytes = 272;
  u32x4 v[5];
  __device__ __forceinline__ void take(const unsigned char *at, uint32_t part) {
#pragma unroll
    for (int w = 0; w < 4; ++w) v[w] = load16(at + 16 * part, 4 * w);
    v[4] = load16(at, 16);
  }
};
template <> struct Strip<3> : StripInPlace {
  static constexpr bool kParked = false, kWhole = false;
  static constexpr uint32_t kVectors = 1, kLoads = 1, kSlotBytes = 0;
  using Pending = Strip;
  __device__ __forceinline__ void load(const unsigned char *at, uint32_t part) { take(at, part); }
};
template <> struct Strip<4> : StripInPlace {
  static constexpr bool kParked = true, kWhole = true;
  static constexpr uint32_t kVectors = 17, kPitch = kVectors * 16, kLoads = (kStripRows * kVectors + kWaveLanes - 1) / kWaveLanes, kSlotBytes = kStripRows * kPitch;
  struct Pending {
    u32x4 v[kLoads];
  };
  __device__ __forceinline__ void take(const unsigned char *slot, uint32_t at, uint32_t part) { StripInPlace::take(slot + at, part); }
};

// LDS of a block: zeros | codes [m][k + pad] | scales [activation blocks][4 sets] |
// Q4_K: sums [sub-blocks][4 sets] | shares [waves][sets][64] | slots [waves]
struct StripLayout {
  uint32_t scales, sums, shares, slots, bytes;
};
// Bytes of an activation row's codes; of a run's.
__host__ __device__ inline uint32_t strip_run_codes(int kind) { return kind >= 3 ? 384u : 256u; }
__host__ __device__ inline uint32_t strip_code_pitch(int kind, uint32_t k) { return k / 256 * strip_run_codes(kind) + kCodePad; }
__host__ __device__ inline StripLayout strip_layout(int kind, uint32_t m, uint32_t k, uint32_t waves) {
  const uint32_t sets = m > 4 ? 2 : 1;
  StripLayout at;
  at.scales = kZeroBytes + m * strip_code_pitch(kind, k);
  at.sums = at.scales + (kind >= 2 ? k / 32 : k / 256) * 16 * sets;
  at.shares = at.sums + (kind == 0 ? k / 32 * 16 * sets : 0);
  at.slots = at.shares + waves * sets * kWaveLanes * 4;
  at.bytes = at.slots + waves * (kind == 1 ? Strip<1>::kSlotBytes : (kind == 2 ? Strip<2>::kSlotBytes : (kind == 4 ? Strip<4>::kSlotBytes : 0u)));
  return at;
}

// The same value, which the compiler can no longer tell: what is worked out from it once a tile is worked
// out there and takes no register through the runs (one that spills waits for every load in flight when
// it comes back: Q8_0 [1536 -> 77056] x 8 39 us with nine spilled, 31 us).
__device__ __forceinline__ uint32_t opaque(uint32_t value) {
  asm volatile("" : "+v"(value));
  return value;
}

// The dots of one run, closed: totals[set][i] gains activation row 4 set + i's part of the lane's groups.
// `codes`: the lane's operand bases, `scales` / `sums`: the run's, at the lane's first group.
template <int kKind, int kSets> struct StripDot;
// The lane's A row has codes at its k-slots; where they start.
template <int kStep> struct StripFaces {
  static constexpr int kBases = 1;
  static __device__ __forceinline__ bool faces(int, uint32_t column, uint32_t part) { return column / 4 == part; }
};
template <int kSets> struct StripDot<2, kSets> : StripFaces<0> {
  static constexpr uint32_t first_chunk(uint32_t, uint32_t part) { return 2 * part; }
  static __device__ __forceinline__ void add(const Strip<2> &w, uint32_t part, const unsigned char *const (&codes)[1][kSets],
                                             const float *scales, const int *, uint32_t run, double (&totals)[kSets][4]) {
#pragma unroll
    for (uint32_t j = 0; j < 2; ++j) {
      const float d = f16_to_f32(w.d[j]);
#pragma unroll
      for (int set = 0; set < kSets; ++set) {
        i32x4 dots = {0, 0, 0, 0};
#pragma unroll
        for (uint32_t s = 0; s < 2; ++s) {
          const u32x4 operand = *reinterpret_cast<const u32x4 *>(codes[0][set] + (8 * j + s) * 16);
          dots = __builtin_amdgcn_mfma_i32_16x16x64_i8((i32x4)operand, (i32x4)w.q[2 * j + s], dots, 0, 0, 0);
        }
        const f32x4 a = *reinterpret_cast<const f32x4 *>(scales + ((size_t)(8 * run + 4 * j + part) * kSets + set) * 4);
#pragma unroll
        for (int i = 0; i < 4; ++i) totals[set][i] = __builtin_fma((double)(d * a[i]), (double)dots[i], totals[set][i]);
      }
    }
  }
};
template <int kSets> struct StripDot<1, kSets> : StripFaces<0> {
  static constexpr uint32_t first_chunk(uint32_t, uint32_t part) { return 8 * (part / 2) + part % 2; }
  static __device__ __forceinline__ void add(const Strip<1> &w, uint32_t part, const unsigned char *const (&codes)[1][kSets],
                                             const float *scales, const int *, uint32_t run, double (&totals)[kSets][4]) {
    const u32x4 top = w.top ^ 0xAAAAAAAAu;  // q - 32 modulo 64: bytes of 4 (q - 32) as int8
    const u32x4 q[4] = {((w.low << 2) & 0x3C3C3C3Cu) | ((top << 6) & 0xC0C0C0C0u), ((w.high << 2) & 0x3C3C3C3Cu) | ((top << 4) & 0xC0C0C0C0u),
                        ((w.low >> 2) & 0x3C3C3C3Cu) | ((top << 2) & 0xC0C0C0C0u), ((w.high >> 2) & 0x3C3C3C3Cu) | (top & 0xC0C0C0C0u)};
    const double step = (double)(f16_to_f32(w.d) * 0.25f);
    int scale[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) scale[g] = (int)(signed char)(w.scales[g / 2] >> (16 * (g % 2) + 8 * (part % 2)));
#pragma unroll
    for (int set = 0; set < kSets; ++set) {
      int whole[4] = {0, 0, 0, 0};
#pragma unroll
      for (uint32_t g = 0; g < 4; ++g) {
        const u32x4 operand = *reinterpret_cast<const u32x4 *>(codes[0][set] + 2 * g * 16);
        const i32x4 zero = {0, 0, 0, 0};
        const i32x4 dots = __builtin_amdgcn_mfma_i32_16x16x64_i8((i32x4)operand, (i32x4)q[g], zero, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) whole[i] = mad24(scale[g], dots[i], whole[i]);
      }
      const f32x4 a = *reinterpret_cast<const f32x4 *>(scales + ((size_t)run * kSets + set) * 4);
#pragma unroll
      for (int i = 0; i < 4; ++i) totals[set][i] = __builtin_fma(step * (double)a[i], (double)whole[i], totals[set][i]);
    }
  }
};
template <int kSets> struct StripDot<0, kSets> : StripFaces<0> {
  static constexpr uint32_t first_chunk(uint32_t, uint32_t part) { return 4 * part; }
  static __device__ __forceinline__ void add(const Strip<0> &w, uint32_t part, const unsigned char *const (&codes)[1][kSets],
                                             const float *scales, const int *sums, uint32_t run, double (&totals)[kSets][4]) {
    // sub-blocks 2 p and 2 p + 1: neighbouring bytes of the table, whole six bits below sub-block 4,
    // from there on four bits in a nibble and two in the top of an earlier byte
    const uint32_t shift = 16 * (part % 2);
    const uint32_t first = w.head.y >> shift, second = w.head.z >> shift, third = w.head.w >> shift;
    const bool packed = part >= 2;
    const uint32_t sc = packed ? (third & 0x0F0Fu) | ((first >> 2) & 0x3030u) : first & 0x3F3Fu;
    const uint32_t mn = packed ? ((third >> 4) & 0x0F0Fu) | ((second >> 2) & 0x3030u) : second & 0x3F3Fu;
    const int sc_low = (int)(sc & 0xFFu), sc_high = (int)((sc >> 8) & 0xFFu), mn_low = (int)(mn & 0xFFu), mn_high = (int)((mn >> 8) & 0xFFu);
    const double d = (double)f16_to_f32((uint16_t)w.head.x), dmin = (double)f16_to_f32((uint16_t)(w.head.x >> 16));
#pragma unroll
    for (int set = 0; set < kSets; ++set) {
      i32x4 low = {0, 0, 0, 0}, high = {0, 0, 0, 0};
#pragma unroll
      for (uint32_t s = 0; s < 2; ++s) {
        const u32x4 for_low = *reinterpret_cast<const u32x4 *>(codes[0][set] + s * 16);
        const u32x4 for_high = *reinterpret_cast<const u32x4 *>(codes[0][set] + (2 + s) * 16);
        low = __builtin_amdgcn_mfma_i32_16x16x64_i8((i32x4)for_low, (i32x4)(w.q[s] & 0x0F0F0F0Fu), low, 0, 0, 0);
        high = __builtin_amdgcn_mfma_i32_16x16x64_i8((i32x4)for_high, (i32x4)((w.q[s] >> 4) & 0x0F0F0F0Fu), high, 0, 0, 0);
      }
      const f32x4 a = *reinterpret_cast<const f32x4 *>(scales + ((size_t)run * kSets + set) * 4);
      const int *of_low = sums + ((size_t)(8 * run + 2 * part) * kSets + set) * 4;
      const i32x4 sum_low = *reinterpret_cast<const i32x4 *>(of_low), sum_high = *reinterpret_cast<const i32x4 *>(of_low + kSets * 4);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int scaled = mad24(sc_low, low[i], __mul24(sc_high, high[i]));
        const int minima = mad24(mn_low, sum_low[i], __mul24(mn_high, sum_high[i]));
        totals[set][i] = __builtin_fma((double)a[i], __builtin_fma(d, (double)scaled, -(dmin * (double)minima)), totals[set][i]);
      }
    }
  }
};

template <int kSets> struct StripDotInPlace {
  static constexpr int kBases = 3;
  static __device__ __forceinline__ bool faces(int j, uint32_t column, uint32_t part) { return part + 4 * j - 2 * (column / 4) <= 2u; }
  static constexpr uint32_t first_chunk(uint32_t column, uint32_t part) { return column / 4 + part; }
  static __device__ __forceinline__ void add(const StripInPlace &w, uint32_t part, const unsigned char *const (&codes)[3][kSets],
                                             const float *scales, const int *, uint32_t run, double (&totals)[kSets][4]) {
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      const auto halves = __builtin_amdgcn_permlane32_swap(w.v[2 * g][2 * g], w.v[2 * g + 1][2 * g + 1], false, false);
      const auto rows = __builtin_amdgcn_permlane16_swap(halves[0], halves[1], false, false);
      const float d = f16_to_f32((uint16_t)(rows[0] >> (16 * (part % 2))));
#pragma unroll
      for (int set = 0; set < kSets; ++set) {
        i32x4 dots = {0, 0, 0, 0};
#pragma unroll
        for (int j = 0; j < 3; ++j) {
          const u32x4 operand = *reinterpret_cast<const u32x4 *>(codes[j][set] + (12 * g + 4 * j) * 16);
          dots = __builtin_amdgcn_mfma_i32_16x16x64_i8((i32x4)operand, (i32x4)w.v[2 * g + j], dots, 0, 0, 0);
        }
        const f32x4 a = *reinterpret_cast<const f32x4 *>(scales + ((size_t)(8 * run + 4 * g + part) * kSets + set) * 4);
#pragma unroll
        for (int i = 0; i < 4; ++i) totals[set][i] = __builtin_fma((double)(d * a[i]), (double)dots[i], totals[set][i]);
      }
    }
  }
};

template <int kSets> struct StripDot<3, kSets> : StripDotInPlace<kSets> {};
template <int kSets> struct StripDot<4, kSets> : StripDotInPlace<kSets> {};

// Orders a wave's own LDS accesses.
__device__ __forceinline__ void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <int kKind, class TX, int kSets>
__global__ __launch_bounds__(kMostWaves * kWaveLanes) void gguf_matvec_q8_strips(const unsigned char *weights, const void *x, void *y, uint32_t rows,
                                                                        uint64_t row_stride, uint32_t k, uint32_t m, uint32_t block_rows,
                                                                        uint32_t tile_rows, uint32_t split, uint32_t split_inverse) {
  using Held = Strip<kKind>;
  using Dot = StripDot<kKind, kSets>;
  extern __shared__ __align__(16) unsigned char shared[];
  const StripLayout layout = strip_layout(kKind, m, k, blockDim.x / kWaveLanes);
  float *scales = reinterpret_cast<float *>(shared + layout.scales);
  int *sums = reinterpret_cast<int *>(shared + layout.sums);
  const uint32_t lane = threadIdx.x % kWaveLanes;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWaveLanes);
  const uint32_t column = lane % 16, part = lane / 16;
  const uint32_t runs = k / 256;

  // ---- the (tile, run) pairs of this wave, in order ------------------------------------------------
  // wave / split = wave * split_inverse >> 8 for fewer than 17 waves; slots * split waves have a place, those behind them none
  const uint32_t slots = (blockDim.x / kWaveLanes * split_inverse) >> 8, slot = (wave * split_inverse) >> 8, member = wave - slot * split;
  const uint32_t row_begin = blockIdx.x * block_rows, row_end = min(row_begin + block_rows, rows);  // begin < rows
  const uint32_t tiles = (row_end - row_begin + tile_rows - 1) / tile_rows, rounds = (tiles + slots - 1) / slots;
  const uint32_t own_tiles = slot < min(tiles, slots) ? (tiles - slot + slots - 1) / slots : 0u;
  const uint32_t own_runs = (runs - member + split - 1) / split;  // split <= runs: at least one
  const uint32_t items = own_tiles * own_runs;
  auto row_of = [&](uint32_t tile, uint32_t r) { return row_begin + tile * tile_rows + r; };
  auto tile_end = [&](uint32_t tile) { return min(row_begin + (tile + 1) * tile_rows, row_end); };
  // rows past a tile's last one are that row again and are not stored
  // (bytes from the block's first row: below 2^32, see gguf_matvec_strips_serve)
  // a pointer throughout: an address that went through an integer is a flat one to the compiler, and a wait for LDS is
  // a wait for every flat load in flight
  const unsigned char *own = weights + (uint64_t)row_begin * row_stride;
  const uint32_t own_offset = (uint32_t)reinterpret_cast<uintptr_t>(own) & 15u;
  auto row_at = [&](uint32_t tile, uint32_t r) { return (min(row_of(tile, r), tile_end(tile) - 1) - row_begin) * (uint32_t)row_stride; };
  uint32_t load_tile = slot, load_run = member, loads_left = items;
  // what a wave loads of a run: each lane its own part, or whole vectors, vector `piece` of the stage
  // being vector piece % kVectors of row piece / kVectors
  using Pending = typename Held::Pending;
  uint32_t load_row[Held::kLoads];
  auto aim = [&]() {
    const uint32_t lane = opaque(threadIdx.x % kWaveLanes), column = lane % 16;
#pragma unroll
    for (uint32_t i = 0; i < Held::kLoads; ++i)
      load_row[i] = row_at(load_tile, Held::kParked ? min((lane + i * kWaveLanes) / Held::kVectors, kStripRows - 1) : column) +
                    (Held::kWhole ? (lane + i * kWaveLanes) % Held::kVectors * 16 : 0u);
  };
  auto next_load = [&](Pending &into) {
    if constexpr (Held::kWhole) {
#pragma unroll
      for (uint32_t i = 0; i < Held::kLoads; ++i) into.v[i] = load16(own + (load_row[i] + load_run * Held::kRunBytes), 0);
    } else if constexpr (Held::kParked) {
#pragma unroll
      for (uint32_t i = 0; i < Held::kLoads; ++i) {
        // bytes from the 16-byte boundary at or below the block's first row
        const uint32_t begin = own_offset + load_row[i] + load_run * Held::kRunBytes;
        const uint32_t wanted = (lane + i * kWaveLanes) % Held::kVectors * 16, last = (begin & 15u) + Held::kRunBytes - 1;
        // a vector past the run's last byte is the last one again
        into.v[i] = load16(own - own_offset + ((begin & ~15u) + min(wanted, last & ~15u)), 0);
      }
    } else {
      into.load(own + (load_row[0] + load_run * Held::kRunBytes), part);
    }
    if (loads_left <= 1) return;  // past the wave's last run: that run again, whose bytes go unused
    --loads_left;
    load_run += split;
    if (load_run >= runs) {
      load_run = member;
      load_tile += slots;
      aim();
    }
  };

  // ---- the activation rows, quantised once per block -----------------------------------------------
  // Four runs at a time per wave, kBatch times on their way: the loads of the first are asked for before the weights',
  // the wave's first run of weights before they are there.
  constexpr int kBatch = Traits<TX>::kSize == 2 ? 2 : 1;
  const uint32_t units = m * runs, step = blockDim.x / 16, u = lane % 16;
  const uint32_t inverse = (1u << 20) / runs + 1;  // unit / runs = unit * inverse >> 20 while units * runs < 2^20 (units <= 8 runs, runs <= 224)
  // a unit past the last is the last one again: the same values to the same places
  auto fetch = [&](uint32_t first, BlockValues<TX> &into) { into.load(x, (size_t)min(first + lane / 16, units - 1) * 256 + 16 * u); };  // rows are dense
  uint32_t unit = 4 * wave;  // of the wave's first sixteen lanes
  BlockValues<TX> ahead[kBatch];
#pragma unroll
  for (int j = 0; j < kBatch; ++j)
    if (unit + j * step < units) fetch(unit + j * step, ahead[j]);
  // (a wave without an item loads all the same, its block's last row: a load that only some waves make leaves the
  // compiler unsure how many are in flight, and it waits for all of them)
  Pending pending;
  aim();
  next_load(pending);
  {
    // zeros round the codes where they lie as the weights do, otherwise only the row of zeros
    const uint32_t clear = (kKind >= 3 ? layout.scales : kZeroBytes) / 16;
    for (uint32_t i = threadIdx.x; i < clear; i += blockDim.x) reinterpret_cast<u32x4 *>(shared)[i] = u32x4{0u, 0u, 0u, 0u};
    if constexpr (kKind >= 3) lds_barrier();
  }
  while (unit < units) {
#pragma unroll
    for (int j = 0; j < kBatch; ++j) {
      if (unit >= units) break;
      const BlockValues<TX> now = ahead[j];
      if (unit + kBatch * step < units) fetch(unit + kBatch * step, ahead[j]);
      const uint32_t mine = min(unit + lane / 16, units - 1), token = __umul24(mine, inverse) >> 20, run = mine - __umul24(token, runs);
      quantise_block<kKind, TX>(now, lane, shared + kZeroBytes + __umul24(token, strip_code_pitch(kKind, k)) + __umul24(run, strip_run_codes(kKind)),
                                scales + (size_t)(kKind >= 2 ? 8 * run : run) * kSets * 4 + token, kSets * 4,
                                sums + (size_t)8 * run * kSets * 4 + token, kSets * 4);
      unit += step;
    }
  }
  lds_barrier();

  // ---- the weight rows -----------------------------------------------------------------------------
  // a lane's operands of a run: its activation row's codes from its first chunk on, or, where its A row has none at
  // its k-slots, the zeros at the start
  uint32_t base[kSets], faces[Dot::kBases];
#pragma unroll
  for (int j = 0; j < Dot::kBases; ++j) faces[j] = Dot::faces(j, column, part) ? 0xFFFFFFFFu : 0u;
#pragma unroll
  for (uint32_t set = 0; set < (uint32_t)kSets; ++set)  // activation rows past the last repeat it and are not stored
    base[set] = kZeroBytes + min(column % 4 + 4 * set, m - 1) * strip_code_pitch(kKind, k) + Dot::first_chunk(column, part) * 16;
  double totals[kSets][4] = {};
  uint32_t run = member, tile = slot;
  uint32_t own_row = items != 0 ? (uint32_t)row_at(slot, column) : 0u;  // the lane's weight row
  unsigned char *parked = shared + layout.slots + wave * Held::kSlotBytes;
  uint32_t round = 0;
  // Lane (c, p) of the tile's first wave ends with activation row 4 set + p against weight row c.
  auto finish = [&]() {
    const uint32_t lane = opaque(threadIdx.x % kWaveLanes), column = lane % 16, part = lane / 16;
    // 64-bit sums over the lanes of a column, one rounding for a share and one for the product (with the lanes' sums rounded
    // first: Q4_K [2304 -> 12800] x 3 6.2e-8 off the 64-bit product in f32, 3.5e-8 like this)
    double mine[kSets];
#pragma unroll
    for (int set = 0; set < kSets; ++set) {
      mine[set] = add_rows_apart(add_halves_apart(totals[set][0], totals[set][2]), add_halves_apart(totals[set][1], totals[set][3]));
#pragma unroll
      for (int i = 0; i < 4; ++i) totals[set][i] = 0.0;
    }
    if (split != 1) {
      // the wave's own share; those of the waves behind it follow, kSets * kWaveLanes apart
      float *share = reinterpret_cast<float *>(shared + opaque(layout.shares + (wave * kSets * kWaveLanes + lane) * 4));
      if (member != 0) {
#pragma unroll
        for (int set = 0; set < kSets; ++set) share[set * kWaveLanes] = (float)mine[set];
      }
      lds_barrier();
      if (member == 0) {
#pragma unroll
        for (int set = 0; set < kSets; ++set)
          for (uint32_t other = 1; other < split; ++other) mine[set] += (double)share[(other * kSets + set) * kWaveLanes];
      }
      if (++round < rounds) lds_barrier();  // before the shares of the next round
    }
    const uint32_t row = row_of(tile, column);
    if (member == 0 && row < tile_end(tile)) {
#pragma unroll
      for (uint32_t set = 0; set < (uint32_t)kSets; ++set)
        if (4 * set + part < m) Traits<TX>::store(y, (size_t)(4 * set + part) * rows + row, (float)mine[set]);
    }
  };
  for (uint32_t done = 0; done < items; ++done) {
    Held held;
    if constexpr (Held::kParked) {
#pragma unroll
      for (uint32_t i = 0; i < Held::kLoads; ++i) {
        // (pieces past the last repeat the last row's)
        const uint32_t piece = lane + i * kWaveLanes;
        *reinterpret_cast<u32x4 *>(parked + min(piece / Held::kVectors, kStripRows - 1) * Held::kPitch + piece % Held::kVectors * 16) = pending.v[i];
      }
      next_load(pending);
      wave_fence();
      held.take(parked, column * Held::kPitch + (Held::kWhole ? 0u : (own_offset + own_row + run * Held::kRunBytes) & 15u), part);
      wave_fence();
    } else {
      held = pending;
      next_load(pending);
    }
    const unsigned char *codes[Dot::kBases][kSets];
#pragma unroll
    for (int j = 0; j < Dot::kBases; ++j)
#pragma unroll
      for (int set = 0; set < kSets; ++set) codes[j][set] = shared + ((base[set] + run * strip_run_codes(kKind)) & faces[j]);
    Dot::add(held, part, codes, scales, sums, run, totals);
    run += split;
    if (run >= runs) {
      finish();
      run = member;
      tile += slots;
      own_row = (uint32_t)row_at(min(tile, tiles - 1), opaque(threadIdx.x % kWaveLanes) % 16);
    }
  }
  if (split != 1) {
    while (round < rounds) {  // the last round has no tile for these waves, or none has: its barriers
      lds_barrier();
      if (++round < rounds) lds_barrier();
    }
  }
}

inline const char *strip_word(int kind) { return kind == 0 ? "q4_k" : (kind == 1 ? "q6_k" : "q8_0"); }
// gguf_matvec_q8_strips/<format>/<activation rows>-tokens/<waves of a block: 16, 8, or 8 where two share a compute
// unit>-waves[/shared: several waves to a tile].  Eight waves for want of LDS nearly always share: one label.
enum : int { kSixteen = 0, kSixteenShared = 1, kEight = 2, kTwice = 3, kTwiceShared = 4 };
template <int kKind, int kSets, int kForm> struct StripsTag {
  static std::string text() {
    static const char *const forms[] = {"16-waves", "16-waves/shared", "8-waves", "2x8-waves", "2x8-waves/shared"};
    return std::string("gguf_matvec_q8_strips/") + strip_word(kKind) + "/" + std::to_string(4 * kSets) + "-tokens/" + forms[kForm] + (kKind == 3 ? "/in-place" : (kKind == 4 ? "/in-place/parked" : ""));
  }
};

// Waves of a block whose buffers fit beside the codes of m activation rows: sixteen, eight, or none.
uint32_t strip_waves(int kind, uint32_t m, uint32_t k) {
  for (uint32_t waves = kMostWaves; waves >= 8; waves /= 2)
    if (strip_layout(kind, m, k, waves).bytes <= kStripLds) return waves;
  return 0;
}
// Activation rows of one launch: all of them, or as many as fit a block's LDS.
uint32_t strip_group(int kind, uint32_t m, uint32_t k) {
  while (m > 1 && strip_waves(kind, m, k) == 0) --m;
  return m;
}

template <int kKind, class TX, int kSets>
hipError_t run_strips(const MatVecParams &p, uint32_t m, const void *w, const void *x, void *y, uint32_t units, hipStream_t s) {
  const uint32_t runs = p.k / 256, rows = (uint32_t)p.rows;
  // One block per compute unit, where the activation rows are quantised once; two of eight waves where
  // that is little beside the weight rows, which then hide each other's tile ends (us, one / two:
  // Q4_K [2048 -> 151936] x 2 47.7 / 39.5, Q6_K [1280 -> 100000] x 5 32.7 / 26.4, Q8_0 [5120 -> 17408] x 1 21.6 / 19.9,
  // [3328 -> 14080] x 4 13.4 / 12.1; but Q8_0 [2048 -> 6144] x 4 6.5 / 6.9).  Q4_K and Q6_K rows of eight runs or more that
  // are no vocabulary's share better among sixteen waves: [2560 -> 9728] x 2 6.0 / 7.3 and 8.3 / 9.5, [5120 -> 17408] x 1
  // 12.7 / 15.4 and 17.2 / 20.2 ([3072 -> 32000] x 2 13.7 / 13.7 and 18.0 / 17.9).
  const uint32_t codes = m * p.k;
  const bool little = (codes <= 16384 && rows >= 8192 && (kKind >= 2 || p.k < 2048 || rows >= 32768)) || (codes <= 32768 && rows >= 65536);
  const bool twice = little && 2 * strip_layout(kKind, m, p.k, 8).bytes <= kStripLds;
  const uint32_t waves = twice ? 8 : strip_waves(kKind, m, p.k);
  const uint32_t wanted = units * (twice ? 2u : 1u);
  const uint32_t block_rows = (rows + wanted - 1) / wanted;
  const uint32_t grid = (rows + block_rows - 1) / block_rows;
  const uint32_t tiles = (block_rows + kStripRows - 1) / kStripRows, tile_rows = (block_rows + tiles - 1) / tiles;
  // waves to a tile: the fewest of those whose busiest wave has the fewest runs, whatever their number (Q8_0 [5120 -> 17408]
  // has five tiles of twenty runs to a block: seven runs with three waves to a tile, nine with eight; 24.3 -> 24.0 us, Q6_K
  // 23.5 -> 21.7); joining the shares of a round counts as a quarter of a run (Q8_0 [1792 -> 105243] x 7, thirteen tiles of seven
  // runs to a block of eight waves: 48.4 one wave to a tile, 50.6 with eight)
  uint32_t split = 1, least = 0xFFFFFFFFu;
  for (uint32_t candidate = 1; candidate <= waves && candidate <= runs; ++candidate) {
    const uint32_t slots = waves / candidate;
    const uint32_t cost = ((tiles + slots - 1) / slots) * (4 * ((runs + candidate - 1) / candidate) + (candidate > 1 ? 1 : 0));
    if (cost < least) {
      least = cost;
      split = candidate;
    }
  }
  // No more waves than have a tile's runs to walk or activations to quantise: a wave without an item loads as much as another,
  // and up to fifteen of them keep a compute unit's memory pipe for 0.2 to 0.8 us (sixteen waves always / like this: Q8_0
  // [1024 -> 768] x 4 4.6 / 3.8, [1536 -> 1280] x 3 4.9 / 4.3, [2048 -> 2816] x 2 5.15 / 4.5, Q4_K [1792 -> 1792] x 3 4.2 / 4.0).
  const uint32_t busy = std::min(tiles, waves / split) * split, quantising = (m * runs + 3) / 4;
  const uint32_t block_waves = std::min(waves, std::max(busy, quantising)), shared = strip_layout(kKind, m, p.k, block_waves).bytes;
  if constexpr (kKind == 3) {
    note_variant<StripsTag<kKind, kSets, kSixteen>>();
  } else {
    if constexpr (kKind != 4) {
      if (!twice && waves == 8) note_variant<StripsTag<kKind, kSets, kEight>>();
    }
    if (twice && split != 1) note_variant<StripsTag<kKind, kSets, kTwiceShared>>();
    else if (twice) note_variant<StripsTag<kKind, kSets, kTwice>>();
    else if (waves == kMostWaves && split != 1) note_variant<StripsTag<kKind, kSets, kSixteenShared>>();
    else if (waves == kMostWaves) note_variant<StripsTag<kKind, kSets, kSixteen>>();
  }
  hipLaunchKernelGGL((gguf_matvec_q8_strips<kKind, TX, kSets>), dim3(grid), dim3(block_waves * kWaveLanes), shared, s, static_cast<const unsigned char *>(w), x, y,
                     rows, p.row_stride, p.k, m, block_rows, tile_rows, split, (255 + split) / split);
  return hipGetLastError();
}

template <int kKind, class TX> hipError_t run_groups(const MatVecParams &p, const void *w, const void *x, void *y, hipStream_t s) {
  const uint32_t launches = (p.m + strip_group(kKind, p.m, p.k) - 1) / strip_group(kKind, p.m, p.k);
  const uint32_t group = (p.m + launches - 1) / launches, units = p.compute_units != 0 ? p.compute_units : 256;
  for (uint32_t done = 0; done < p.m; done += group) {
    const uint32_t m = p.m - done < group ? p.m - done : group;
    const void *xs = static_cast<const char *>(x) + (size_t)done * p.k * Traits<TX>::kSize;
    void *ys = static_cast<char *>(y) + (size_t)done * p.rows * Traits<TX>::kSize;
    const hipError_t err = m <= 4 ? run_strips<kKind, TX, 1>(p, m, w, xs, ys, units, s) : run_strips<kKind, TX, 2>(p, m, w, xs, ys, units, s);
    if (err != hipSuccess) return err;
  }
  return hipSuccess;
}

inline bool in_place_serves(const MatVecParams &p, const void *w) {
  return p.row_stride % 16 == 0 && (reinterpret_cast<uintptr_t>(w) & 15u) == 0 && strip_waves(3, p.m, p.k) == kMostWaves;
}

template <class TX> hipError_t run_strips_kind(const MatVecParams &p, const void *w, const void *x, void *y, hipStream_t s) {
  switch (p.kind) {
    case 0: return run_groups<0, TX>(p, w, x, y, s);
    case 1: return run_groups<1, TX>(p, w, x, y, s);
    case 2:
      if (in_place_serves(p, w)) return strip_waves(4, p.m, p.k) == kMostWaves ? run_groups<4, TX>(p, w, x, y, s) : run_groups<3, TX>(p, w, x, y, s);
      [[fallthrough]];
    default: return run_groups<2, TX>(p, w, x, y, s);
  }
}

}  // namespace

bool gguf_matvec_strips_serve(const MatVecParams &p) {
  const uint64_t units = p.compute_units != 0 ? p.compute_units : 256;
  return p.m >= 1 && p.m <= 8 && p.k >= 256 && p.k % 256 == 0 && p.k / 256 <= 224 && p.rows >= 512 && p.rows <= 0x7FFFFFFFu &&
         strip_waves(p.kind, 1, p.k) != 0 && ((p.rows + units - 1) / units + kStripRows) * p.row_stride < 0xFFFFFFFFull;
}
uint32_t gguf_matvec_strips_dispatches(const MatVecParams &p) {
  if (p.kind == 2 && in_place_serves(p, nullptr)) return 1;
  const uint32_t group = strip_group(p.kind, p.m, p.k);
  return (p.m + group - 1) / group;
}
hipError_t launch_gguf_matvec_strips(Elem x_type, const MatVecParams &p, const void *weights, const void *x, void *y, hipStream_t stream) {
  switch (x_type) {
    case Elem::kF32: return run_strips_kind<F32>(p, weights, x, y, stream);
    case Elem::kF16: return run_strips_kind<F16>(p, weights, x, y, stream);
    case Elem::kBF16: return run_strips_kind<BF16>(p, weights, x, y, stream);
  }
  return hipErrorInvalidValue;
}

}  // namespace hyle_hip
