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
// A block of sixteen waves (eight where the codes leave no room for more slots) has a compute unit's
// LDS, quantises the activation rows once, while its first weight bytes are on their way, and walks its
// share of the weight rows in tiles of at most sixteen; `1 << split_log2` waves share a tile, each
// taking every split-th run, and the first adds the shares.  A lane's chain of up to 224 runs, and the
// sum over the shares, run in 64 bits: in 32, a chain that is several times as long as one of the
// kernels that spread a row over 64 lanes was further from the 64-bit sum than theirs in a third of
// the shapes (f32 Q8_0 [5120 -> 2304] x 6 9.6e-8 relative against 8.2e-8 there, Q4_K [4096 -> 6656] x 4
// 7.6e-8 against 6.2e-8; in 64 bits 5.3e-8 and 4.5e-8, at most 0.75 of theirs over 87 shapes, for about
// 1 % of the time).  Q8_0 and Q6_K runs are
// loaded as the aligned vectors that cover them and redistributed through a wave-private slot: lanes
// that load their own 16 bytes at 2-byte addresses keep the memory pipe busy several times as long
// (Q8_0 [2048 -> 151936] 111 us that way, 63 us through the slot).  A Q4_K row is whole vectors and
// goes straight into the lanes (52 us through the slot, 43 us straight).
//
// Bound by HBM for a vocabulary.  Below about 100 MB of weights by latency and vector instructions together: at
// five rows of Q8_0 [5120 -> 17408] a SIMD issues vector instructions in 38 % of the cycles and matrix ones in 4 %, LDS
// conflicts take 16 % of them and a wave waits for 36 % of its time; at [17408 -> 5120], where the codes leave room for
// eight waves, vector 43 %, two fifths of it quantising, and HBM delivers 2.5 of 6.8 TB/s.  MI355X, bf16
// activations, us, the kernels that these shapes took before and here:
//   Q8_0 [5120 -> 17408] x 5   65.6 -> 28.8 (3290 GB/s)    [17408 -> 5120] x 5   99.9 -> 34.1 (2780 GB/s)
//   Q6_K [5120 -> 17408] x 5   70.3 -> 27.3                [17408 -> 5120] x 5  112.5 -> 35.7
//   Q4_K [5120 -> 17408] x 5   44.0 -> 21.4                [17408 -> 5120] x 5  115.3 -> 31.3
//   [1536 -> 77056] x 8: Q8_0 104.9 -> 31.2 (4030 GB/s)    Q6_K 117.4 -> 29.0
//   Q6_K [5120 -> 32768] x 1   38.3 -> 31.9
#include "device_common.h"
#include "gguf_q8_math.h"
#include "kernels.h"

namespace hyle_hip {
namespace {

constexpr uint32_t kStripRows = 16, kMostWaves = 16;
constexpr size_t kStripLds = 160 * 1024;  // of a compute unit, and the most one block can have
constexpr uint32_t kZeroBytes = 256;      // a lane's operands of one run lie within 256 bytes of its base
constexpr uint32_t kCodePad = 16;         // between activation rows: neighbours start on other LDS banks

// 16 bytes at any even address.
typedef uint32_t words4_even __attribute__((ext_vector_type(4), aligned(2)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef short short2v __attribute__((ext_vector_type(2)));
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
  static constexpr bool kParked = true;
  static constexpr uint32_t kRunBytes = kBytes, kVectors = (kBytes + 14 + 15) / 16, kPitch = (kVectors | 1u) * 16;
  static constexpr uint32_t kLoads = (kStripRows * kVectors + kWaveLanes - 1) / kWaveLanes, kSlotBytes = kStripRows * kPitch;
  struct Pending {
    u32x4 v[kLoads];
  };
};

// What a lane decodes of one run of its weight row, from the wave's slot; `at`: the run's first byte.
template <int kKind> struct Strip;
template <> struct Strip<0> {  // rows are whole 16-byte vectors as a rule: loaded straight into the lanes
  static constexpr bool kParked = false;
  // one piece per lane of its own row
  static constexpr uint32_t kRunBytes = 144, kVectors = 1, kLoads = 1, kSlotBytes = 0;
  using Pending = Strip;
  u32x4 head, q[2];
  __device__ __forceinline__ void load(const unsigned char *at, uint32_t part) {
    head = *reinterpret_cast<const words4_even *>(at);
#pragma unroll
    for (int s = 0; s < 2; ++s) q[s] = *reinterpret_cast<const words4_even *>(at + 16 + 32 * part + 16 * s);
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

// LDS of a block: zeros | codes [m][k + pad] | scales [activation blocks][4 sets] |
// Q4_K: sums [sub-blocks][4 sets] | shares [waves][sets][64] | slots [waves]
struct StripLayout {
  uint32_t scales, sums, shares, slots, bytes;
};
__host__ __device__ inline StripLayout strip_layout(int kind, uint32_t m, uint32_t k, uint32_t waves) {
  const uint32_t sets = m > 4 ? 2 : 1;
  StripLayout at;
  at.scales = kZeroBytes + m * (k + kCodePad);
  at.sums = at.scales + (kind == 2 ? k / 32 : k / 256) * 16 * sets;
  at.shares = at.sums + (kind == 0 ? k / 32 * 16 * sets : 0);
  at.slots = at.shares + waves * sets * kWaveLanes * 4;
  at.bytes = at.slots + waves * (kind == 0 ? Strip<0>::kSlotBytes : (kind == 1 ? Strip<1>::kSlotBytes : Strip<2>::kSlotBytes));
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
template <int kSets> struct StripDot<2, kSets> {
  static constexpr uint32_t first_chunk(uint32_t part) { return 2 * part; }
  static __device__ __forceinline__ void add(const Strip<2> &w, uint32_t part, const unsigned char *const (&codes)[kSets],
                                             const float *scales, const int *, uint32_t run, double (&totals)[kSets][4]) {
#pragma unroll
    for (uint32_t j = 0; j < 2; ++j) {
      const float d = f16_to_f32(w.d[j]);
#pragma unroll
      for (int set = 0; set < kSets; ++set) {
        i32x4 dots = {0, 0, 0, 0};
#pragma unroll
        for (uint32_t s = 0; s < 2; ++s) {
          const u32x4 operand = *reinterpret_cast<const u32x4 *>(codes[set] + (8 * j + s) * 16);
          dots = __builtin_amdgcn_mfma_i32_16x16x64_i8((i32x4)operand, (i32x4)w.q[2 * j + s], dots, 0, 0, 0);
        }
        const f32x4 a = *reinterpret_cast<const f32x4 *>(scales + ((size_t)(8 * run + 4 * j + part) * kSets + set) * 4);
#pragma unroll
        for (int i = 0; i < 4; ++i) totals[set][i] = __builtin_fma((double)(d * a[i]), (double)dots[i], totals[set][i]);
      }
    }
  }
};
template <int kSets> struct StripDot<1, kSets> {
  static constexpr uint32_t first_chunk(uint32_t part) { return 8 * (part / 2) + part % 2; }
  static __device__ __forceinline__ void add(const Strip<1> &w, uint32_t part, const unsigned char *const (&codes)[kSets],
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
        const u32x4 operand = *reinterpret_cast<const u32x4 *>(codes[set] + 2 * g * 16);
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
template <int kSets> struct StripDot<0, kSets> {
  static constexpr uint32_t first_chunk(uint32_t part) { return 4 * part; }
  static __device__ __forceinline__ void add(const Strip<0> &w, uint32_t part, const unsigned char *const (&codes)[kSets],
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
        const u32x4 for_low = *reinterpret_cast<const u32x4 *>(codes[set] + s * 16);
        const u32x4 for_high = *reinterpret_cast<const u32x4 *>(codes[set] + (2 + s) * 16);
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

// Eight neighbouring values of an activation row at any element's address.
template <class TX> struct StripValues {
  static constexpr int kVectors = Traits<TX>::kVec == 8 ? 1 : 2;
  u32x4 raw[kVectors];
  __device__ __forceinline__ void load(const void *x, size_t first) {
#pragma unroll
    for (int h = 0; h < kVectors; ++h)
      raw[h] = *reinterpret_cast<const words4_even *>(static_cast<const char *>(x) + first * Traits<TX>::kSize + 16 * h);
  }
  __device__ __forceinline__ void values(float (&v)[8]) const {
    if constexpr (kVectors == 1) {
      Traits<TX>::unpack(raw[0], v);
    } else {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        float piece[4];
        Traits<TX>::unpack(raw[h], piece);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[4 * h + e] = piece[e];
      }
    }
  }
};

// Half a wave quantises a run of 256 values of an activation row, eight values per lane u: one Q8_K
// block, or eight Q8_0 blocks of four lanes each.
template <int kKind, class TX>
__device__ __forceinline__ void strip_quantise(const StripValues<TX> &fetched, uint32_t lane, uint32_t *codes, float *scale, uint32_t scale_step,
                                               int *sums, uint32_t sum_step) {
  const uint32_t u = lane % 32;
  float v[8];
  fetched.values(v);
  float largest = 0.0f;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    largest = __builtin_fmaxf(largest, __builtin_fabsf(v[e]));  // a NaN is no candidate
  }
  const float top = group_max<kKind == 2 ? 4 : 32>(largest);
  float factor = 0.0f, stored = 0.0f;
  if constexpr (kKind == 2) {
    if (top != 0.0f) {
      stored = f16_to_f32(f32_to_f16(top / 127.0f));
      factor = 127.0f / top;
    }
  } else {
    // the sign of the block's first value of that magnitude: of the lowest lane that has one
    bool negative = false;
#pragma unroll
    for (int e = 7; e >= 0; --e) negative = __builtin_fabsf(v[e]) == top ? v[e] < 0.0f : negative;
    const uint64_t has = __ballot(largest == top), below = __ballot(negative);
    const uint32_t own_has = (uint32_t)(has >> (lane & 32u)), own_below = (uint32_t)(below >> (lane & 32u));
    if (top != 0.0f) {
      const float value = (own_below >> __builtin_ctz(own_has)) & 1u ? -top : top;
      factor = -127.0f / value;
      stored = 1.0f / factor;
    }
  }
  // nearest integer, ties to even, at most 127 (a block of zeros: factor 0); only the low bytes are kept
  uint32_t words[2];
#pragma unroll
  for (int w = 0; w < 2; ++w) {
    int code[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) code[e] = (int)__builtin_rintf(v[4 * w + e] * factor);
    const short2v most = {127, 127};
    const short2v low = __builtin_elementwise_min(__builtin_bit_cast(short2v, __builtin_amdgcn_cvt_pk_i16(code[0], code[1])), most);
    const short2v high = __builtin_elementwise_min(__builtin_bit_cast(short2v, __builtin_amdgcn_cvt_pk_i16(code[2], code[3])), most);
    words[w] = __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, high), __builtin_bit_cast(uint32_t, low), 0x06040200u);
  }
  codes[2 * u] = words[0];
  codes[2 * u + 1] = words[1];
  if constexpr (kKind == 0) {
    int sum = dot4(0x01010101u, words[0], dot4(0x01010101u, words[1], 0));
    sum += dpp_move<kDppSwap1>(sum);
    sum += dpp_move<kDppSwap2>(sum);  // the four lanes of a sub-block
    if (u % 4 == 0) sums[(u / 4) * sum_step] = sum;
  }
  if constexpr (kKind == 2) {
    if (u % 4 == 0) scale[(u / 4) * scale_step] = stored;
  } else {
    if (u == 0) *scale = stored;
  }
}

// Orders a wave's own LDS accesses.
__device__ __forceinline__ void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <int kKind, class TX, int kSets>
__global__ __launch_bounds__(kMostWaves * kWaveLanes) void gguf_matvec_q8_strips(const unsigned char *weights, const void *x, void *y, uint32_t rows,
                                                                        uint64_t row_stride, uint32_t k, uint32_t m, uint32_t block_rows,
                                                                        uint32_t tile_rows, uint32_t split_log2) {
  using Held = Strip<kKind>;
  using Dot = StripDot<kKind, kSets>;
  constexpr int kDepth = Held::kParked ? 2 : 3;  // runs of a wave in flight
  extern __shared__ __align__(16) unsigned char shared[];
  const StripLayout layout = strip_layout(kKind, m, k, blockDim.x / kWaveLanes);
  float *scales = reinterpret_cast<float *>(shared + layout.scales);
  int *sums = reinterpret_cast<int *>(shared + layout.sums);
  const uint32_t lane = threadIdx.x % kWaveLanes;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWaveLanes);
  const uint32_t column = lane % 16, part = lane / 16;
  const uint32_t runs = k / 256;

  // ---- the (tile, run) pairs of this wave, in order ------------------------------------------------
  const uint32_t split = 1u << split_log2, member = wave & (split - 1), slot = wave >> split_log2, slots = (blockDim.x / kWaveLanes) >> split_log2;
  const uint32_t row_begin = blockIdx.x * block_rows, row_end = min(row_begin + block_rows, rows);  // begin < rows
  const uint32_t tiles = (row_end - row_begin + tile_rows - 1) / tile_rows, rounds = (tiles + slots - 1) / slots;
  const uint32_t own_tiles = slot < tiles ? (tiles - slot + slots - 1) / slots : 0u;
  const uint32_t own_runs = (runs - member + split - 1) / split;  // split <= runs: at least one
  const uint32_t items = own_tiles * own_runs;
  auto row_of = [&](uint32_t tile, uint32_t r) { return row_begin + tile * tile_rows + r; };
  auto tile_end = [&](uint32_t tile) { return min(row_begin + (tile + 1) * tile_rows, row_end); };
  // rows past a tile's last one are that row again and are not stored
  // (bytes from the block's first row: below 2^32, see gguf_matvec_strips_serve)
  const uintptr_t own = reinterpret_cast<uintptr_t>(weights) + (uint64_t)row_begin * row_stride;
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
      load_row[i] = row_at(load_tile, Held::kParked ? min((lane + i * kWaveLanes) / Held::kVectors, kStripRows - 1) : column);
  };
  auto next_load = [&](Pending &into) {
    if constexpr (Held::kParked) {
#pragma unroll
      for (uint32_t i = 0; i < Held::kLoads; ++i) {
        const uintptr_t begin = own + (load_row[i] + load_run * Held::kRunBytes);
        const uint32_t wanted = (lane + i * kWaveLanes) % Held::kVectors * 16, last = ((uint32_t)begin & 15u) + Held::kRunBytes - 1;
        // a vector past the run's last byte is the last one again
        into.v[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>((begin & ~(uintptr_t)15) + min(wanted, last & ~15u)));
      }
    } else {
      into.load(reinterpret_cast<const unsigned char *>(own + (load_row[0] + load_run * Held::kRunBytes)), part);
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
  // runs go round the block's half waves; the next kBatch of a half wave are on their way
  constexpr int kBatch = StripValues<TX>::kVectors == 1 ? 4 : 2;
  const uint32_t halves = blockDim.x / 32;
  const uint32_t units = m * runs, u = lane % 32;
  const uint32_t inverse = (1u << 20) / runs + 1;  // unit / runs = unit * inverse >> 20 while units * runs < 2^20 (units <= 8 runs, runs <= 224)
  auto fetch_batch = [&](uint32_t first, StripValues<TX> (&into)[kBatch]) {
#pragma unroll
    for (int j = 0; j < kBatch; ++j) into[j].load(x, (size_t)min(first + j * halves, units - 1) * 256 + 8 * u);  // rows are dense
  };
  const uint32_t half = threadIdx.x / 32;
  StripValues<TX> ahead[kBatch];
  fetch_batch(half, ahead);
  Pending ring[kDepth];
  if (items != 0) {
    aim();
#pragma unroll
    for (int d = 0; d < kDepth; ++d) next_load(ring[d]);
  }
  if (threadIdx.x < kZeroBytes / 16) reinterpret_cast<u32x4 *>(shared)[threadIdx.x] = u32x4{0u, 0u, 0u, 0u};
  for (uint32_t first = half; first - half < units; first += kBatch * halves) {  // the same trips for both halves of a wave
    StripValues<TX> now[kBatch];
#pragma unroll
    for (int j = 0; j < kBatch; ++j) now[j] = ahead[j];
    fetch_batch(first + kBatch * halves, ahead);
#pragma unroll
    for (int j = 0; j < kBatch; ++j) {
      // a unit past the last is the last one again: the same values to the same places
      const uint32_t unit = min(first + j * halves, units - 1), token = (unit * inverse) >> 20, run = unit - token * runs;
      strip_quantise<kKind, TX>(now[j], lane, reinterpret_cast<uint32_t *>(shared + kZeroBytes + (size_t)token * (k + kCodePad) + run * 256),
                                scales + (size_t)(kKind == 2 ? 8 * run : run) * kSets * 4 + token, kSets * 4,
                                sums + (size_t)8 * run * kSets * 4 + token, kSets * 4);
    }
  }
  lds_barrier();

  // ---- the weight rows -----------------------------------------------------------------------------
  const bool faces = column / 4 == part;  // the lane's A row has codes at the lane's k-slots
  uint32_t base[kSets];
  const uint32_t advance = faces ? 256u : 0u;
#pragma unroll
  for (uint32_t set = 0; set < (uint32_t)kSets; ++set)  // activation rows past the last repeat it and are not stored
    base[set] = faces ? kZeroBytes + min(column % 4 + 4 * set, m - 1) * (k + kCodePad) + Dot::first_chunk(part) * 16 : 0u;
  double totals[kSets][4] = {};
  uint32_t run = member, tile = slot;
  uint32_t own_row = items != 0 ? (uint32_t)row_at(slot, column) : 0u;  // the lane's weight row
  unsigned char *parked = shared + layout.slots + wave * Held::kSlotBytes;
  // Lane (c, p) of the tile's first wave ends with activation row 4 set + p against weight row c.
  auto finish = [&]() {
    const uint32_t lane = opaque(threadIdx.x % kWaveLanes), column = lane % 16, part = lane / 16;
    float mine[kSets];
#pragma unroll
    for (int set = 0; set < kSets; ++set) {
      const bool upper = part >= 2, odd = part % 2 != 0;
      float own_sum[4], pair[2];
#pragma unroll
      for (int i = 0; i < 4; ++i) own_sum[i] = (float)totals[set][i];
#pragma unroll
      for (int i = 0; i < 2; ++i)
        pair[i] = (upper ? own_sum[2 + i] : own_sum[i]) + __shfl_xor(upper ? own_sum[i] : own_sum[2 + i], 32, kWaveLanes);
      mine[set] = (odd ? pair[1] : pair[0]) + __shfl_xor(odd ? pair[0] : pair[1], 16, kWaveLanes);
#pragma unroll
      for (int i = 0; i < 4; ++i) totals[set][i] = 0.0;
    }
    if (split_log2 != 0) {
      // the wave's own share; those of the waves behind it follow, kSets * kWaveLanes apart
      float *share = reinterpret_cast<float *>(shared + opaque(layout.shares + (wave * kSets * kWaveLanes + lane) * 4));
#pragma unroll
      for (int set = 0; set < kSets; ++set) share[set * kWaveLanes] = mine[set];
      lds_barrier();
      if (member == 0) {
#pragma unroll
        for (int set = 0; set < kSets; ++set) {
          double whole = (double)mine[set];
          for (uint32_t other = 1; other < split; ++other) whole += (double)share[(other * kSets + set) * kWaveLanes];
          mine[set] = (float)whole;
        }
      }
      lds_barrier();
    }
    const uint32_t row = row_of(tile, column);
    if (member == 0 && row < tile_end(tile)) {
#pragma unroll
      for (uint32_t set = 0; set < (uint32_t)kSets; ++set)
        if (4 * set + part < m) Traits<TX>::store(y, (size_t)(4 * set + part) * rows + row, mine[set]);
    }
  };
  for (uint32_t done = 0; done < items; done += kDepth) {
#pragma unroll
    for (int d = 0; d < kDepth; ++d) {
      if (done + d >= items) break;
      Held held;
      if constexpr (Held::kParked) {
#pragma unroll
        for (uint32_t i = 0; i < Held::kLoads; ++i) {
          const uint32_t piece = lane + i * kWaveLanes;
          if (piece < kStripRows * Held::kVectors)
            *reinterpret_cast<u32x4 *>(parked + piece / Held::kVectors * Held::kPitch + piece % Held::kVectors * 16) = ring[d].v[i];
        }
        next_load(ring[d]);
        wave_fence();
        held.take(parked, column * Held::kPitch + (((uint32_t)own + own_row + run * Held::kRunBytes) & 15u), part);
        wave_fence();
      } else {
        held = ring[d];
        next_load(ring[d]);
      }
      const unsigned char *codes[kSets];
#pragma unroll
      for (int set = 0; set < kSets; ++set) codes[set] = shared + base[set] + run * advance;
      Dot::add(held, part, codes, scales, sums, run, totals);
      run += split;
      if (run >= runs) {
        finish();
        run = member;
        tile += slots;
        own_row = (uint32_t)row_at(min(tile, tiles - 1), opaque(threadIdx.x % kWaveLanes) % 16);
      }
    }
  }
  if (split_log2 != 0 && own_tiles < rounds) {  // the last round has no tile for these waves: its two barriers
    lds_barrier();
    lds_barrier();
  }
}

inline const char *strip_word(int kind) { return kind == 0 ? "q4_k" : (kind == 1 ? "q6_k" : "q8_0"); }
// gguf_matvec_q8_strips/<format>/<activation rows>-tokens/<waves of a block: 16, 8, or 8 where two share a compute
// unit>-waves[/shared: several waves to a tile].  Eight waves for want of LDS nearly always share: one label.
enum : int { kSixteen = 0, kSixteenShared = 1, kEight = 2, kTwice = 3, kTwiceShared = 4 };
template <int kKind, int kSets, int kForm> struct StripsTag {
  static std::string text() {
    static const char *const forms[] = {"16-waves", "16-waves/shared", "8-waves", "2x8-waves", "2x8-waves/shared"};
    return std::string("gguf_matvec_q8_strips/") + strip_word(kKind) + "/" + std::to_string(4 * kSets) + "-tokens/" + forms[kForm];
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
  // Q8_0 [1280 -> 77056] x 4 29.4 / 26.5, Q4_K [3072 -> 77056] x 4 41.0 / 31.8 and x 8 43.9 / 38.3; but
  // Q8_0 [1280 -> 2048] x 4 7.7 / 8.4, [3072 -> 17408] x 8 19.8 / 22.2).
  const uint32_t codes = m * p.k;
  const bool little = (codes <= 16384 && rows >= 8192) || (codes <= 32768 && rows >= 65536);
  const bool twice = little && 2 * strip_layout(kKind, m, p.k, 8).bytes <= kStripLds;
  const uint32_t waves = twice ? 8 : strip_waves(kKind, m, p.k), shared = strip_layout(kKind, m, p.k, waves).bytes;
  const uint32_t wanted = units * (twice ? 2u : 1u);
  const uint32_t block_rows = (rows + wanted - 1) / wanted;
  const uint32_t grid = (rows + block_rows - 1) / block_rows;
  const uint32_t tiles = (block_rows + kStripRows - 1) / kStripRows, tile_rows = (block_rows + tiles - 1) / tiles;
  // waves to a tile: the fewest of those whose busiest wave has the fewest runs
  uint32_t split_log2 = 0, least = 0xFFFFFFFFu;
  for (uint32_t log2 = 0; (1u << log2) <= waves && (1u << log2) <= runs; ++log2) {
    const uint32_t split = 1u << log2, slots = waves / split;
    const uint32_t cost = ((tiles + slots - 1) / slots) * ((runs + split - 1) / split);
    if (cost < least) {
      least = cost;
      split_log2 = log2;
    }
  }
  if (twice && split_log2 != 0) note_variant<StripsTag<kKind, kSets, kTwiceShared>>();
  else if (twice) note_variant<StripsTag<kKind, kSets, kTwice>>();
  else if (waves == 8) note_variant<StripsTag<kKind, kSets, kEight>>();
  else if (split_log2 != 0) note_variant<StripsTag<kKind, kSets, kSixteenShared>>();
  else note_variant<StripsTag<kKind, kSets, kSixteen>>();
  hipLaunchKernelGGL((gguf_matvec_q8_strips<kKind, TX, kSets>), dim3(grid), dim3(waves * kWaveLanes), shared, s, static_cast<const unsigned char *>(w), x, y,
                     rows, p.row_stride, p.k, m, block_rows, tile_rows, split_log2);
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

template <class TX> hipError_t run_strips_kind(const MatVecParams &p, const void *w, const void *x, void *y, hipStream_t s) {
  switch (p.kind) {
    case 0: return run_groups<0, TX>(p, w, x, y, s);
    case 1: return run_groups<1, TX>(p, w, x, y, s);
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
