// Decode-phase attention over compressed caches on the 16-bit matrix cores, for key and value widths of 2, 3 and 4
// bits (one dimension and one kind of caches per object file: PITCH_DIM = 64 or 128, PITCH_KIND below).
//
// The algebra is that of pitch_attention.hip: no token is decoded, the query is rotated once and the weighted values
// are rotated back once. What differs is how the two contractions run. pitch_attention.hip looks a code *pair* up in
// one table that all lanes share, whose random reads conflict (about three LDS passes each), and multiplies in
// float32 (4 x 4 x 1). Here
//   * a code pair is looked up in a table of 32 copies, one per two LDS banks, so that no read conflicts. An entry
//     holds each of the pair's two values twice over: its float16 rounding and the float16 rounding of the rest, 22 bits
//     and a sign;
//   * the two halves are neighbours on the contraction axis of v_mfma_f32_16x16x32_f16, with the other operand
//     doubled, so the looked-up words are operand words as they are: sum_k (hi_k + lo_k) q_k in one instruction;
//   * the other operand (rotated queries, softmax weights) is split too, its parts on rows that the few query heads
//     of a KV head leave empty: row 4 part + head for up to four heads (three parts of the query, two of the
//     weights), row 8 part + head for up to eight (two parts). The parts' products are summed in float32.
// Two float16 parts hold a table value, a cos or sin value or (five to eight heads) a query to 2^-23, three a query to
// 2^-33; a weight is held to 2^-22 down to 2^-28 of the largest of its tile. Error against float64 (relative L2, mean over
// 4 seeds x 2 methods x 4 width pairs x 700, 5000 and 40000 tokens), the float32 kernels' -> these: d = 128, up to four
// heads 9.4e-7 -> 6.6e-7, five to eight 7.8e-7 -> 6.5e-7; d = 64 7.5e-7 -> 6.5e-7, 6.6e-7 -> 6.2e-7; key-bias term, d =
// 128 1.29e-6 -> 9.1e-7, 1.25e-6 -> 8.8e-7; per-channel keys (40 seeds each), d = 128, four heads 1.2 - 1.7e-6 -> 5.1 -
// 7.7e-7, eight 1.3 - 1.8e-6 -> 0.8 - 1.0e-6. Single calls scatter by a factor of three around these, either way.
// Per-channel keys need no table: a code is exact in bfloat16, so a group's query products q_j step_j are split into
// three bfloat16 parts (24 bits) and the codes are converted in registers (v_mfma_f32_16x16x32_bf16).
//
// Work split: a wave takes tiles of 64 tokens by itself (scores, online softmax, weighted values), so no barrier
// separates the phases and the waves of a SIMD hide each other's loads; a workgroup's waves merge through LDS at the
// end and attn_combine merges the workgroups. Weighted values are added up per tile, scores of table keys per two steps,
// in float32 on the VALU: the matrix cores truncate what they align to a running sum, which a long chain would feel
// (one chain per score: mean 6.3e-7 and at most 1.35e-6 of ten seeds, pairs of steps 4.9e-7 and 6.2e-7; same time). Scores
// of per-channel keys are one chain of d / 32 steps, twice as many for five to eight heads: starting each step from zero
// changes nothing for four heads (per-head mean 3.26e-7 and 3.24e-7 at d = 128) and takes eight from 4.2e-7 to 3.4e-7.
//
// Bound: long calls by their reads (Llama-3-8B layer, 8 KV x 4 queries, b = 4, token-major, us per call in a graph with
// the float32 kernels -> here: 131072 tokens 64.7 -> 46.5, 3.0 TB/s; with every tile read from the same few, so out of
// L2, 8 less, without the loads 16 less), the rest by fixed latency: launch, tables, one tile and the second launch are
// 10 - 12 us. Same layer: 16000 tokens 23.4 -> 14.2, 32768 tokens 23.4 -> 18.6; per-channel keys of four bits and values of
// three, 131072 tokens 73.5 -> 44.7; key-bias term, 2 KV x 6, 2000 tokens 21.2 -> 17.8, 4 KV x 4, 48606 tokens 203 -> 36.
#include "pitch_attn_shared.h"

#ifndef PITCH_DIM
#error "compile with -DPITCH_DIM=<dim>"
#endif
#ifndef PITCH_KIND
#error "compile with -DPITCH_KIND=<kind>"
#endif

namespace pitch {
namespace {

constexpr int kTile = (int)kTileTokens;
constexpr float kTabScale = 4096.f;   // table values are stored times 2^12: the rest's float16 stays normal
constexpr float kLoScale = 2048.f;    // a weight's rest is stored times 2^11, in a row (an accumulator) of its own
constexpr int kWRow = kTile + 4;  // row of staged weights (dwords): rows start on other banks, 16-byte aligned

typedef float v4f __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t w4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) uint32_t lds_u32;
typedef uint32_t u32_any __attribute__((aligned(1)));

__device__ __forceinline__ v4f mfma_f16(w4 a, w4 b, v4f c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}
__device__ __forceinline__ v4f mfma_bf16(w4 a, w4 b, v4f c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// x as (float16 rounding, float16 rounding of the rest), the first in the low half.
__device__ __forceinline__ uint32_t split2(float x) {
  const _Float16 hi = (_Float16)x;
  const _Float16 lo = (_Float16)(x - (float)hi);
  return (uint32_t)__builtin_bit_cast(uint16_t, hi) | ((uint32_t)__builtin_bit_cast(uint16_t, lo) << 16);
}
__device__ __forceinline__ uint32_t twice(_Float16 x) {
  const uint32_t h = __builtin_bit_cast(uint16_t, x);
  return h | (h << 16);
}

// Largest of a and b over the lane pair at distance 32 (16): of a in the lower lane of the pair, of b in the upper one.
__device__ __forceinline__ float max32(float a, float b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return fmax_hw(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float max16(float a, float b) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return fmax_hw(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
// Largest value over each row of 16 lanes, in all its lanes.
__device__ __forceinline__ float row_max(float x) {
  x = fmax_hw(x, xchg<1>(x));
  x = fmax_hw(x, xchg<2>(x));
  x = fmax_hw(x, xchg<4>(x));
  return fmax_hw(x, xchg<8>(x));
}
// x, opaque to the compiler: what follows from it is formed where it is used (in a loop, instead of being kept in a
// register per row offset).
__device__ __forceinline__ uint32_t in_loop(uint32_t x) {
  asm volatile("" : "+s"(x));
  return x;
}
// A wave-uniform value, moved to a scalar register.
__device__ __forceinline__ float uniform(float x) {
  return __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(x)));
}
__device__ __forceinline__ float lane_value(float x, int lane) {
  return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(x), lane));
}
// Largest value over the wave (uniform).
__device__ __forceinline__ float wave_max(float x) { return lane_value(row_max(max16(max32(x, x), max32(x, x))), 0); }
// The same of four values: one reduction of a register whose rows hold the four.
__device__ __forceinline__ void wave_max4(const float (&x)[4], float (&m)[4]) {
  const float r = row_max(max16(max32(x[0], x[1]), max32(x[2], x[3])));
  m[0] = lane_value(r, 0);
  m[1] = lane_value(r, 32);
  m[2] = lane_value(r, 16);
  m[3] = lane_value(r, 48);
}
// The same of every head's value.
template <int NH>
__device__ __forceinline__ void wave_max_heads(const float (&x)[NH], float (&m)[NH]) {
#pragma unroll
  for (int h = 0; h < NH; h += 4) {
    const float x4[4] = {x[h], x[h + 1], x[h + 2], x[h + 3]};
    float m4[4];
    wave_max4(x4, m4);
#pragma unroll
    for (int k = 0; k < 4; ++k) m[h + k] = m4[k];
  }
}
__device__ __forceinline__ float wave_sum(float x) {
  x += xchg<1>(x);
  x += xchg<2>(x);
  x += xchg<4>(x);
  x += xchg<8>(x);
  {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  }
  {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  }
  return x;
}
// (a, b) -> per lane, the sum of one operand over the lane pair at distance 32 (16): a for the lower lane of the
// pair, b for the upper one.
__device__ __forceinline__ float fold32(float a, float b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float fold16(float a, float b) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// 2^e as a float32, -126 <= e <= 127.
__device__ __forceinline__ float pow2i(int e) { return __uint_as_float((uint32_t)(e + 127) << 23); }
// floor(log2 |x|) of a normal x (-127 for 0 and subnormals).
__device__ __forceinline__ int exponent_of(float x) { return (int)((__float_as_uint(x) >> 23) & 255u) - 127; }

__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The bits [pos, pos + width) of the lane's words w, moved to [at, at + width) of the result, with other bits around
// them (pos, width, at constants).
template <int NW>
__device__ __forceinline__ uint32_t bits_at(const uint32_t (&w)[NW], int pos, int width, int at) {
  const int wi = pos >> 5, q = pos & 31;
  if (q + width > 32) {
    const uint32_t next = w[wi + 1 < NW ? wi + 1 : wi];
    return q >= at ? __builtin_amdgcn_alignbit(next, w[wi], q - at) : (next << (at - q)) | (w[wi] >> (32 - (at - q)));
  }
  return q >= at ? w[wi] >> (q - at) : w[wi] << (at - q);
}

// The bits of word k of a code stream that are the top bit of a code.
template <int B>
constexpr uint32_t top_bits(int k) {
  uint32_t x = 0;
  for (int i = 0; i < 32; ++i)
    if ((32 * k + i) % B == B - 1) x |= 1u << i;
  return x;
}

// b where the mask's bits are set, a elsewhere. (A choice between two elements of a private array by a lane's condition
// is compiled into an indexed load, which puts the array into scratch memory.)
__device__ __forceinline__ float pick(uint32_t mask, float a, float b) {
  return __uint_as_float((__float_as_uint(a) & ~mask) | (__float_as_uint(b) & mask));
}

// (x & mask) | rest in one instruction.
__device__ __forceinline__ uint32_t and_or(uint32_t x, uint32_t mask, uint32_t rest) {
  uint32_t r;
  asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(x), "s"(mask), "v"(rest));
  return r;
}

// Table of a code pair's two values (TurboQuant: two centroids; PolarQuant: radius times cosine and sine) in LDS: entry
// (pair, copy) of 8 bytes at byte 256 pair + 8 copy, 32 copies; lane l reads copy l mod 32, so the 32 lanes that one
// pass of an 8-byte read serves never share a bank. 64 KB at four bits, 16 KB at three, 4 KB at two.
// Addresses are most of what the VALU does per value: at four bits a pair is a byte of the row, and one v_perm puts it
// above the lane's byte (the table is at LDS address 0); other widths take a shift and a v_and_or.
template <int D, int B, bool POLAR>
struct PairTab {
  static constexpr int L = 1 << B, kPairs = L * L, C = 32, kShift = 8;
  static constexpr int kWords = kPairs * C * 2;

  // The constants an entry is made of, kept in LDS while the table is built (source s of kSources).
  static constexpr int kSources = POLAR ? 3 * L : L;
  __device__ static __forceinline__ float source(int s) {
    if constexpr (POLAR) {
      constexpr int off = pitch_polar_offset(B);
      return s < L ? pitch_polar_radius_tab[off + s]
                   : s < 2 * L ? pitch_polar_cos_tab[off + s - L] : pitch_polar_sin_tab[off + s - 2 * L];
    } else {
      return pitch_codebook_tab[pitch_codebook_offset(ilog2(D), B) + s];
    }
  }
  // 16 lanes write an entry's 32 copies.
  __device__ static __forceinline__ void build(uint32_t* tab, const float* src, int tid, int threads) {
    for (int i = tid; i < kPairs * 16; i += threads) {
      const int p = i >> 4, c0 = p & (L - 1), c1 = p >> B;
      const float x = POLAR ? src[c0] * src[L + c1] : src[c0], y = POLAR ? src[c0] * src[2 * L + c1] : src[c1];
      const uint32_t u = split2(x * kTabScale), v = split2(y * kTabScale);
      *(w4*)(tab + i * 4) = w4{u, v, u, v};
    }
  }
  // This lane's byte offset within an entry, plus the table's LDS address (a multiple of the table's size).
  __device__ static __forceinline__ uint32_t lane_byte(const uint32_t* tab, int lane) {
    return (uint32_t)(uintptr_t)(const lds_u32*)tab | (uint32_t)(lane & (C - 1)) * 8u;
  }
  // The values of codes j and j + 1 (j even, a constant) of the lane's words.
  template <int NW>
  __device__ static __forceinline__ uint2 pair(const uint32_t (&w)[NW], int j, uint32_t lb) {
    typedef uint32_t u2 __attribute__((ext_vector_type(2)));
    typedef __attribute__((address_space(3))) const u2 lds_u2;
    uint32_t at;
    if constexpr (2 * B == 8)
      at = __builtin_amdgcn_perm(lb, w[(B * j) >> 5], 0x0C0C0004u | (uint32_t)(((B * j) & 31) >> 3) << 8);
    else
      at = and_or(bits_at(w, B * j, 2 * B, kShift), (uint32_t)(kPairs - 1) << kShift, lb);
    const u2 v = *(lds_u2*)(uintptr_t)at;
    return make_uint2(v.x, v.y);
  }
};

// What the caches of an object file hold: keys TurboQuant, PolarQuant (each also with the key-bias term) or
// per-channel, values TurboQuant or PolarQuant.
constexpr bool kChanKeys = PITCH_KIND == kAttnKindChanTurbo || PITCH_KIND == kAttnKindChanPolar;
constexpr bool kBias = PITCH_KIND == kAttnKindTurboBias || PITCH_KIND == kAttnKindPolarBias;
constexpr bool kKeyPolar = PITCH_KIND == kAttnKindPolar || PITCH_KIND == kAttnKindPolarBias;
constexpr bool kValPolar = kKeyPolar || PITCH_KIND == kAttnKindChanPolar;

// Most waves of a workgroup, one workgroup per compute unit: four per SIMD (128 registers each) for up to four heads, two
// (256) for five to eight and with the key-bias term, whose accumulators would spill.
constexpr uint32_t max_waves(bool q8) { return q8 || kBias ? 8 : kAttnCodesWaves; }

template <int D, int KB, int VB, bool Q8>
struct Shape {
  static constexpr int NH = Q8 ? 8 : 4;         // query heads, padded
  static constexpr int KS = kChanKeys ? D / 32 : D / 16;  // score instructions per 16 tokens
  using KT = PairTab<D, KB, kKeyPolar>;
  using VT = PairTab<D, VB, kValPolar>;
  static constexpr bool kOneTab = !kChanKeys && KB == VB && kKeyPolar == kValPolar;
  // LDS (dwords): key table, value table, query operand (per-channel keys: float32 queries), key-bias operands,
  // per-wave space (staged weights, a group's query operand, or the wave's accumulators), per-wave maxima and sums
  static constexpr int kTabK = kChanKeys ? 0 : KT::kWords;
  static constexpr int kTabV = kOneTab ? 0 : VT::kWords;
  static constexpr int kQ = kChanKeys ? NH * D : KS * 256;
  static constexpr int kBiasQ = kBias ? (D / 16) * 256 : 0;
  static constexpr int KOPS = kChanKeys && Q8 ? 2 : 1;  // operands of a group's query products (the third part of eight)
  static constexpr int kW = 2 * NH * kWRow, kAcc = NH * D, kGq = kChanKeys ? KOPS * KS * 256 : 0;
  static constexpr int kWave = kW > kAcc ? (kW > kGq ? kW : kGq) : (kAcc > kGq ? kAcc : kGq);
  static constexpr int kStat = 2 * NH + 16;      // per wave: maxima, sums (and the tables' constants before)
  static constexpr int kHead = 2 * NH;          // per head: the query operand's and the bias operand's scale
  __host__ __device__ static constexpr uint32_t bytes(uint32_t waves) {
    return 4u * (uint32_t)(kTabK + kTabV + kQ + kBiasQ + kHead) + 4u * waves * (uint32_t)(kWave + kStat);
  }
};

// Stores the parts of x (coordinate c, head h) into a doubled score operand: three float16 parts for up to four
// heads (the fourth row group is zero), two for up to eight.
template <bool Q8, int GC>
__device__ __forceinline__ void put_query(uint32_t* s_q, int c, int h, float x) {
  // coordinate c belongs to lane group c / GC (GC consecutive coordinates), instruction (c % GC) / 4, word c % 4
  const int base = (((c % GC) >> 2) * 64 + (c / GC) * 16 + h) * 4 + (c & 3);
  const _Float16 p0 = (_Float16)x;
  const float r0 = x - (float)p0;
  const _Float16 p1 = (_Float16)r0;
  s_q[base] = twice(p0);
  if constexpr (Q8) {
    s_q[base + 8 * 4] = twice(p1);
  } else {
    const _Float16 p2 = (_Float16)(r0 - (float)p1);
    s_q[base + 4 * 4] = twice(p1);
    s_q[base + 8 * 4] = twice(p2);
    s_q[base + 12 * 4] = 0u;
  }
}

template <int D, int KB, int VB, bool Q8>
__global__ __launch_bounds__(64 * max_waves(Q8)) void attn_codes(AttnArgs a) {
  using S = Shape<D, KB, VB, Q8>;
  using KT = typename S::KT;
  using VT = typename S::VT;
  constexpr int NH = S::NH, KS = S::KS, E = D / 64;
  constexpr int GC = D / 4;                               // codes of a token row that one lane group holds
  constexpr int KNW = D * KB / 32, VNW = D * VB / 32;      // words of a row
  constexpr int KW = (GC * KB + 31) / 32;                  // words a lane loads of a key row
  constexpr int RC = D / 16;                               // value codes of a token that one lane holds
  extern __shared__ __attribute__((aligned(16))) uint32_t s_mem[];
  // the larger table first, so that each lies at a multiple of its size (s_mem is at LDS address 0)
  uint32_t* const s_ktab = S::kTabV > S::kTabK ? s_mem + S::kTabV : s_mem;
  uint32_t* const s_vtab = S::kTabV > S::kTabK || S::kOneTab ? s_mem : s_mem + S::kTabK;
  uint32_t* const s_q = s_mem + S::kTabK + S::kTabV;
  uint32_t* const s_bq = s_q + S::kQ;
  float* const s_hs = (float*)(s_bq + S::kBiasQ);
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, g = lane >> 4;
  const int waves = blockDim.x >> 6, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  uint32_t* const s_wave0 = (uint32_t*)(s_hs + S::kHead);
  float* const s_stat = (float*)(s_wave0 + waves * S::kWave);
  uint32_t* const s_w = s_wave0 + wid * S::kWave;

  // Workgroups go to the eight XCDs in turn, and each XCD has an L2 of its own. In a token-major cache the rows of one
  // token's heads share cache lines, so a chunk's heads are put on one XCD (a.spread: 8 chunks x heads, chunk fastest).
  uint32_t kv, c;
  if (a.spread) {
    const uint32_t per = 8u * a.kv_heads, i = blockIdx.x / per, r = blockIdx.x % per;
    kv = r >> 3;
    c = 8u * i + (r & 7u);
    if (c >= a.chunks) return;
  } else {
    kv = blockIdx.x / a.chunks;
    c = blockIdx.x % a.chunks;
  }
  const uint64_t t0 = (uint64_t)c * a.chunk;
  const uint32_t nt = (uint32_t)min((uint64_t)a.chunk, a.tokens - t0);
  const uint32_t tiles = (nt + kTile - 1) / kTile;
  const uint64_t row0 = t0 * a.token_stride + (uint64_t)kv * a.head_stride;  // vector index of the first token
  const uint32_t ts = (uint32_t)a.token_stride;  // bounded by the launcher: 64 rows span less than 2^31 bytes
  const uint64_t groups_per_head = kChanKeys ? a.head_stride / a.k_group : 0;

  // ---- a tile's rows: a uniform address plus a 32-bit lane offset. A row past the chunk's end reads the last token
  // instead (its weight is zero), by a minimum on the offset; there is no branch, so that the compiler knows how many
  // loads are in flight and waits for none that it need not.
  const uint32_t kstep = ts * (uint32_t)(KNW * 4), vstep = ts * (uint32_t)(VNW * 4);
  const uint32_t kbyte = (uint32_t)((GC * KB * g) >> 5) * 4u;  // first word of this lane's part of a key row
  const uint32_t ksh = (uint32_t)((GC * KB * g) & 31);         // its codes start at this bit (d = 64, odd widths)
  const uint32_t koff = (uint32_t)n * kstep + kbyte;
  constexpr int RE = kChanKeys ? E : 1;
  uint32_t kw[4][KW];
  uint16_t rlo[RE], rhi[RE];  // per-channel keys: the tile's group's ranges of this lane's coordinates
  auto load_keys = [&](uint32_t tile, uint32_t last) {
    const uint32_t kstep = in_loop(ts) * (uint32_t)(KNW * 4);
    const uint64_t r = row0 + (uint64_t)tile * kTile * ts;
    const char* base = (const char*)(a.k_codes + r * KNW);
    const uint32_t end = last * kstep + kbyte;
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      const uint32_t* q = (const uint32_t*)(base + min(koff + (uint32_t)(16 * m) * kstep, end));
      int k = 0;
#pragma unroll
      for (; k + 4 <= KW; k += 4) {
        const u32x4 v = *(const u32x4*)(q + k);
        kw[m][k] = v.x; kw[m][k + 1] = v.y; kw[m][k + 2] = v.z; kw[m][k + 3] = v.w;
      }
      if constexpr (KW % 4 == 3) {
        const u32x3 v = *(const u32x3*)(q + k);
        kw[m][k] = v.x; kw[m][k + 1] = v.y; kw[m][k + 2] = v.z;
      } else if constexpr (KW % 4 == 2) {
        const u32x2 v = *(const u32x2*)(q + k);
        kw[m][k] = v.x; kw[m][k + 1] = v.y;
      } else if constexpr (KW % 4 == 1) {
        kw[m][k] = q[k];
      }
    }
    if constexpr (kChanKeys) {
      const uint16_t* rg = a.k_ranges + ((uint64_t)kv * groups_per_head + (t0 + (uint64_t)tile * kTile) / a.k_group) * 2u * D;
#pragma unroll
      for (int e = 0; e < RE; ++e) {
        rlo[e] = rg[lane * E + e];
        rhi[e] = rg[D + lane * E + e];
      }
    }
  };
  // the lane's value codes: bits [RC VB n, RC VB (n + 1)) of a row, read as one word at a byte that keeps the read
  // inside the row, and shifted
  const uint32_t vbyte = (uint32_t)min((RC * VB * n) >> 3, VNW * 4 - 4);
  const uint32_t vsh = (uint32_t)(RC * VB * n) - 8u * vbyte;
  const uint32_t voff = (uint32_t)(4 * g) * vstep + vbyte;
  constexpr bool kShiftV = (RC * VB) % 8 != 0 || (RC * VB) < 32;
  static_assert(RC * VB <= 32, "one word holds a lane's value codes");
  uint32_t vw[16];
  float nv, nk = 0.f;
  auto load_values = [&](uint32_t tile, int m) {
    const uint32_t vstep = in_loop(ts) * (uint32_t)(VNW * 4);
    const uint64_t r = row0 + (uint64_t)tile * kTile * ts;
    const uint32_t last = min(nt - 1u - tile * kTile, (uint32_t)kTile - 1u);
    const char* base = (const char*)(a.v_codes + r * VNW);
    const uint32_t end = last * vstep + vbyte;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      vw[4 * m + j] = *(const u32_any*)(base + min(voff + (uint32_t)(16 * m + j) * vstep, end));
  };
  auto load_scales = [&](uint32_t tile) {
    const uint64_t r = row0 + (uint64_t)tile * kTile * ts;
    const uint32_t soff = min((uint32_t)lane, nt - 1u - tile * kTile) * ts * 4u;
    nv = *(const float*)((const char*)(a.v_scales + r) + soff);
    if constexpr (!kChanKeys) nk = *(const float*)((const char*)(a.k_scales + r) + soff);
  };

  {
    const uint32_t first = min((uint32_t)wid, tiles - 1u);
    load_keys(first, min(nt - 1u - first * kTile, (uint32_t)kTile - 1u));
  }

  // ---- tables and the query operand
  // (the tables' constants first: their loads are the first to return, and the tables are built after a barrier)
  constexpr int kSrcK = kChanKeys || S::kOneTab ? 0 : KT::kSources, kSrcV = VT::kSources;
  static_assert(kSrcK + kSrcV <= 2 * 64, "two constants per lane of the first wave");
  float* const s_src = s_stat;  // free until the waves merge
  static_assert(S::kStat * 4 >= kSrcK + kSrcV, "constants fit the space of four waves");
  for (int i = tid; i < kSrcK + kSrcV; i += blockDim.x) s_src[i] = i < kSrcV ? VT::source(i) : KT::source(i - kSrcV);
  for (int h = wid; h < NH; h += waves) {
    float v[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int j = lane * E + e;
      v[e] = h < (int)a.nq ? a.q[((uint64_t)kv * a.nq + h) * D + j] : 0.f;
    }
    if constexpr (kChanKeys) {
#pragma unroll
      for (int e = 0; e < E; ++e) ((float*)s_q)[h * D + lane * E + e] = v[e] * a.kscale;
    } else {
      float u[E], x[E];
      if constexpr (kBias) {
        // q . o_t = sum_j (q_j b_j) cos_tj + (q_j rotate_half(b)_j) sin_tj; the two products' parts, scaled alike
        const float* bb = a.kb_bias + (uint64_t)kv * D;
        float mx = 0.f;
#pragma unroll
        for (int e = 0; e < E; ++e) {
          const int j = lane * E + e;
          const float rh = j < D / 2 ? -bb[j + D / 2] : bb[j - D / 2];
          u[e] = v[e] * bb[j] * a.kscale;
          x[e] = v[e] * rh * a.kscale;
          mx = fmaxf(mx, fmaxf(__builtin_fabsf(u[e]), __builtin_fabsf(x[e])));
        }
        const int eb = max(exponent_of(wave_max(mx)), -100);
        const float sc = pow2i(14 - eb > 127 ? 127 : 14 - eb);
#pragma unroll
        for (int e = 0; e < E; ++e) {
          // pairs of coordinates share a word: head rows as in put_query, instruction j / 32 (cos, then sin)
          const int j = lane * E + e;
#pragma unroll
          for (int half = 0; half < 2; ++half) {
            const float y = (half ? x[e] : u[e]) * sc;
            const int k = half * D + j;                       // position on the contraction axis (2 D long)
            uint16_t* dst = (uint16_t*)s_bq + (((k >> 5) * 64 + ((k >> 2) & 3) * 16 + h) * 4 + ((k & 31) >> 4) * 2) * 2 + (k & 3);
            const _Float16 p0 = (_Float16)y;
            const float r0 = y - (float)p0;
            const _Float16 p1 = (_Float16)r0;
            dst[0] = __builtin_bit_cast(uint16_t, p0);
            if constexpr (Q8) {
              dst[8 * 8] = __builtin_bit_cast(uint16_t, p1);
            } else {
              dst[4 * 8] = __builtin_bit_cast(uint16_t, p1);
              dst[8 * 8] = __builtin_bit_cast(uint16_t, (_Float16)(r0 - (float)p1));
              dst[12 * 8] = 0;
            }
          }
        }
        if (lane == 0) s_hs[NH + h] = pow2i(eb - 14);
      }
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const int j = lane * E + e;
        v[e] = sign_is_negative(a.kseed, (uint32_t)j) ? -v[e] : v[e];
      }
      fwht_contig<E, 64, float>(v, lane);
      float mx = 0.f;
#pragma unroll
      for (int e = 0; e < E; ++e) {
        v[e] *= a.qscale;
        mx = fmaxf(mx, __builtin_fabsf(v[e]));
      }
      const int eq = max(exponent_of(wave_max(mx)), -100);
      const float sc = pow2i(14 - eq > 127 ? 127 : 14 - eq);
#pragma unroll
      for (int e = 0; e < E; ++e) put_query<Q8, GC>(s_q, lane * E + e, h, v[e] * sc);
      if (lane == 0) s_hs[h] = pow2i(eq - 14) * (1.f / kTabScale);
    }
  }
  __syncthreads();
  VT::build(s_vtab, s_src, tid, blockDim.x);
  if constexpr (kSrcK > 0) KT::build(s_ktab, s_src + kSrcV, tid, blockDim.x);
  __syncthreads();

  const uint32_t klb = KT::lane_byte(s_ktab, lane), vlb = VT::lane_byte(s_vtab, lane);
  float qs[NH], bs[NH];
  if constexpr (!kChanKeys) {
#pragma unroll
    for (int h = 0; h < NH; ++h) {
      qs[h] = uniform(s_hs[h]);
      bs[h] = kBias ? uniform(s_hs[NH + h]) : 0.f;
    }
  }
  // The running maxima start at the lowest finite value: a score of minus infinity then weighs nothing, also in a tile,
  // a wave or a chunk without any other (relative to a maximum of minus infinity it would weigh NaN).
  float M[NH], l[NH];
#pragma unroll
  for (int h = 0; h < NH; ++h) {
    M[h] = -__FLT_MAX__;
    l[h] = 0.f;
  }
  constexpr int NA = Q8 ? RC : RC / 2;  // accumulators (four heads: a pair's two coordinates on one's rows)
  v4f acc[NA];
#pragma unroll
  for (int i = 0; i < NA; ++i) acc[i] = v4f{0.f, 0.f, 0.f, 0.f};
  const uint32_t even = n < 8 ? ~0u : 0u;  // this lane weighs (row n) a pair's first coordinate
  const uint32_t odd = g & 1 ? ~0u : 0u;   // eight heads: this lane accumulates heads 4 - 7

  // Key-bias term: a tile's cos rows, then its sin rows, in steps of 32 coordinates, loaded two steps ahead of their
  // products (the first two ahead of the tile's scores).
  constexpr int BS = D / 16;
  f32x4 row[kBias ? 3 : 1][4][2];
  auto load_step = [&](int k, uint32_t tile) {
    const uint64_t p0 = a.kb_first + t0 + (uint64_t)tile * kTile;
    const float* tab = (k >= BS / 2 ? a.kb_sin : a.kb_cos) + p0 * D + 32 * (k % (BS / 2)) + 4 * g;
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      const float* p = tab + min((uint32_t)(16 * m + n), nt - 1u - tile * kTile) * (uint32_t)D;
      row[k % 3][m][0] = *(const f32x4*)p;
      row[k % 3][m][1] = *(const f32x4*)(p + 16);
    }
  };

  for (uint32_t tile = (uint32_t)wid; tile < tiles; tile += waves) {
    if constexpr (kBias) {
      load_step(0, tile);
      load_step(1, tile);
    }
    load_scales(tile);
#pragma unroll
    for (int m = 0; m < 4; ++m) load_values(tile, m);
    const bool in = (uint32_t)lane < nt - tile * kTile;  // this lane's token is one of the chunk's

    // ---- scores: c[m] of lane (n, g) = rows 4 g .. 4 g + 3 (parts and heads) of token 16 m + n
    // (table keys: pairs of steps start from zero and are added on the VALU, see above)
    v4f cs[4], co[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) cs[m] = v4f{0.f, 0.f, 0.f, 0.f};
    if constexpr (GC * KB % 32 != 0) {
#pragma unroll
      for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int k = 0; k < KW; ++k) kw[m][k] = __builtin_amdgcn_alignbit(k + 1 < KW ? kw[m][k + 1] : 0u, kw[m][k], ksh);
    }
    float sb[NH];  // per head: the bias term, or the per-channel keys' q . lo
    if constexpr (kChanKeys) {
      // the group's operand: lane holds coordinates E lane .. E lane + E - 1 of every head
      constexpr float levels = (float)((1 << KB) - 1);
      float mid[E], step[E];  // the decode of code 2^(b - 1), and the step
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const float lo = widen1<1>(rlo[e]);
        step[e] = (widen1<1>(rhi[e]) - lo) / levels;
        step[e] = step[e] == 0.f ? 1.f : step[e];
        mid[e] = __builtin_fmaf((float)(1 << (KB - 1)), step[e], lo);
      }
      uint16_t* gq = (uint16_t*)s_w;
#pragma unroll
      for (int h = 0; h < NH; ++h) {
        sb[h] = 0.f;
#pragma unroll
        for (int e = 0; e < E; ++e) {
          const int j = lane * E + e;
          const float q = ((const float*)s_q)[h * D + j];
          sb[h] = __builtin_fmaf(q, mid[e], sb[h]);
          const float y = q * step[e];
          // three bfloat16 parts by truncation: exact
          const uint32_t p0 = __float_as_uint(y) & 0xFFFF0000u;
          const float r0 = y - __uint_as_float(p0);
          const uint32_t p1 = __float_as_uint(r0) & 0xFFFF0000u;
          const float r1 = r0 - __uint_as_float(p1);
          uint16_t* dst = gq + ((((j % GC) >> 3) * 64 + (j / GC) * 16 + h) * 8 + (j & 7));
          dst[0] = (uint16_t)(p0 >> 16);
          if constexpr (Q8) {
            // eight heads fill the rows with two parts: the third is a second operand, whose products add to the
            // first part's rows
            dst[8 * 8] = (uint16_t)(p1 >> 16);
            dst[KS * 512] = (uint16_t)(__float_as_uint(r1) >> 16);
            dst[KS * 512 + 8 * 8] = 0;
          } else {
            dst[4 * 8] = (uint16_t)(p1 >> 16);
            dst[8 * 8] = (uint16_t)(__float_as_uint(r1) >> 16);
            dst[12 * 8] = 0;
          }
        }
        sb[h] = wave_sum(sb[h]);
      }
      wave_lds_fence();
#pragma unroll
      for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int k = 0; k < KW; ++k) kw[m][k] ^= top_bits<KB>(k);
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const w4 qa = *(const w4*)(s_w + (s * 64 + lane) * 4);
        w4 qb = qa;
        if constexpr (Q8) qb = *(const w4*)(s_w + ((KS + s) * 64 + lane) * 4);
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          w4 b;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            // the top halves of float32(code - 2^(b - 1)): the code's top bit is flipped, so it is a signed field
            const int p = KB * (8 * s + 2 * i);
            const int x0 = (int)bits_at(kw[m], p, KB, 32 - KB) >> (32 - KB);
            const int x1 = (int)bits_at(kw[m], p + KB, KB, 32 - KB) >> (32 - KB);
            b[i] = __builtin_amdgcn_perm(__float_as_uint((float)x1), __float_as_uint((float)x0), 0x07060302u);
          }
          cs[m] = mfma_bf16(qa, b, cs[m]);
          if constexpr (Q8) cs[m] = mfma_bf16(qb, b, cs[m]);
        }
      }
      wave_lds_fence();
    } else {
      // half a step's table reads (two sub-tiles) are issued ahead of the products of the half before
      w4 qa[2], t[2][2];
      auto look = [&](int k) {
        const int s = k >> 1, m0 = 2 * (k & 1);
        if ((k & 1) == 0) qa[s & 1] = *(const w4*)(s_q + (s * 64 + lane) * 4);
#pragma unroll
        for (int m = 0; m < 2; ++m) {
          const uint2 x = KT::pair(kw[m0 + m], 4 * s, klb), y = KT::pair(kw[m0 + m], 4 * s + 2, klb);
          t[k & 1][m] = w4{x.x, x.y, y.x, y.y};
        }
      };
      look(0);
#pragma unroll
      for (int k = 0; k < 2 * KS; ++k) {
        if (k + 1 < 2 * KS) look(k + 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int m = 0; m < 2; ++m) {
          v4f& sum = co[2 * (k & 1) + m];
          sum = mfma_f16(qa[(k >> 1) & 1], t[k & 1][m], (k >> 1) & 1 ? sum : v4f{0.f, 0.f, 0.f, 0.f});
        }
        __builtin_amdgcn_sched_barrier(0);
        if ((k >> 1) & 1) {
#pragma unroll
          for (int m = 0; m < 2; ++m) cs[2 * (k & 1) + m] += co[2 * (k & 1) + m];
        }
      }
    }
    float s[NH];
    auto gather = [&](const v4f (&cc)[4], float (&out)[NH]) {
      // sums the parts and gives lane l the scores of token l (tile m = g), one or two registers per head
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const float x = fold32(cc[0][v], cc[2][v]), y = fold32(cc[1][v], cc[3][v]);
        if constexpr (Q8) {
          const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(y), false, false);
          out[v] = __uint_as_float(r[0]);
          out[4 + v] = __uint_as_float(r[1]);
        } else {
          out[v] = fold16(x, y);
        }
      }
    };
    gather(cs, s);
    // the score of head h is s f + sb, rounded once where the maximum is subtracted from it
    float sf[NH];
#pragma unroll
    for (int h = 0; h < NH; ++h) {
      sf[h] = kChanKeys ? 1.f : qs[h] * nk;  // a power of two times the token's scale: exact
      if constexpr (!kChanKeys && !kBias) sb[h] = 0.f;
    }
    if constexpr (kBias) {
      // the bias term: cos and sin rows of the tile's positions split into two float16 parts, the rest's times 2^11
      v4f bh[4], bl[4];
#pragma unroll
      for (int m = 0; m < 4; ++m) bh[m] = bl[m] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < BS; ++k) {
        if (k + 2 < BS) load_step(k + 2, tile);
        __builtin_amdgcn_sched_barrier(0);
        const w4 qa = *(const w4*)(s_bq + (k * 64 + lane) * 4);
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          f16x8 hi, lo;
#pragma unroll
          for (int r = 0; r < 8; ++r) {
            const float f = row[k % 3][m][r >> 2][r & 3];
            hi[r] = (_Float16)f;
            lo[r] = (_Float16)((f - (float)hi[r]) * kLoScale);
          }
          bh[m] = mfma_f16(qa, __builtin_bit_cast(w4, hi), bh[m]);
          bl[m] = mfma_f16(qa, __builtin_bit_cast(w4, lo), bl[m]);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int m = 0; m < 4; ++m) bh[m] += bl[m] * (1.f / kLoScale);
      gather(bh, sb);
#pragma unroll
      for (int h = 0; h < NH; ++h) sb[h] *= bs[h];
    }
    // the next tile's keys, while this tile's softmax and values run; after the last tile all lanes read one row again,
    // which costs next to nothing (a branch would leave the compiler unsure of the loads in flight)
    const bool more = tile + (uint32_t)waves < tiles;
    const uint32_t next = more ? tile + (uint32_t)waves : tile;
    load_keys(next, more ? min(nt - 1u - next * kTile, (uint32_t)kTile - 1u) : 0u);

    // ---- online softmax; the tile's weights w = p n_t relative to the largest of them per head, in two float16 parts
    const float n_t = in ? nv : 0.f;
    float sv[NH], mx[NH], al[NH], w[NH], fx[NH];
#pragma unroll
    for (int h = 0; h < NH; ++h) sv[h] = in ? __builtin_fmaf(s[h], sf[h], sb[h]) : -__builtin_inff();
    wave_max_heads(sv, mx);
#pragma unroll
    for (int h = 0; h < NH; ++h) {
      const float m = uniform(fmax_hw(M[h], mx[h]));
      al[h] = __builtin_amdgcn_exp2f(M[h] - m);
      M[h] = m;
      const float p = in ? __builtin_amdgcn_exp2f(__builtin_fmaf(s[h], sf[h], sb[h] - m)) : 0.f;
      l[h] = __builtin_fmaf(l[h], al[h], p);
      w[h] = p * n_t;
      sv[h] = __builtin_fabsf(w[h]);
    }
    float fa[4], ft[4];  // factors of the accumulators and of the tile's sums
#pragma unroll
    for (int v = 0; v < 4; ++v) fa[v] = Q8 ? pick(odd, al[v], al[NH - 4 + v]) : al[v];
    wave_max_heads(sv, mx);
#pragma unroll
    for (int h = 0; h < NH; ++h) {
      const int e = max(exponent_of(mx[h]), -100);
      fx[h] = pow2i(e - 14 - 12);  // 2^14 of the weights, 2^12 of the table
      const float y = w[h] * pow2i(14 - e);
      const _Float16 hi = (_Float16)y;
      const _Float16 lo = (_Float16)((y - (float)hi) * kLoScale);
      s_w[h * kWRow + lane] = twice(hi);
      s_w[(NH + h) * kWRow + lane] = twice(lo);
    }
    wave_lds_fence();
#pragma unroll
    for (int v = 0; v < 4; ++v) ft[v] = Q8 ? pick(odd, fx[v], fx[NH - 4 + v]) : fx[v];

    // ---- weighted values. A step takes two tokens of each lane group and a code pair, whose two values lie side by
    // side on the contraction axis as the table read returns them; the weights are zero at the other value's place:
    // rows 0 - 7 weigh the pair's first coordinate and rows 8 - 15 its second (four heads), or one instruction each.
    // A code pair of one sub-tile at a time, its table reads issued ahead of the products of the one before.
    constexpr int NP = RC / 2;
    const uint32_t* const s_row = s_w + (n % (2 * NH)) * kWRow + 4 * g;
    w4 t[2][2], wa[2];
    auto look = [&](int k) {
      const int m = k / NP, p = k % NP;
      if (p == 0) {
        wa[m & 1] = *(const w4*)(s_row + 16 * m);
        if constexpr (kShiftV) {
#pragma unroll
          for (int j = 0; j < 4; ++j) vw[4 * m + j] >>= vsh;
        }
      }
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const uint32_t w0[1] = {vw[4 * m + 2 * j]}, w1[1] = {vw[4 * m + 2 * j + 1]};
        const uint2 x = VT::pair(w0, 2 * p, vlb), y = VT::pair(w1, 2 * p, vlb);
        t[k & 1][j] = w4{x.x, x.y, y.x, y.y};
      }
    };
    look(0);
    v4f x[NP], y[Q8 ? NP : 1];
    w4 a0[2], a1[2];
#pragma unroll
    for (int k = 0; k < 4 * NP; ++k) {
      const int m = k / NP, p = k % NP;
      if (k + 1 < 4 * NP) look(k + 1);
      __builtin_amdgcn_sched_barrier(0);
      if (m == 0) {
        x[p] = v4f{0.f, 0.f, 0.f, 0.f};
        if constexpr (Q8) y[p] = x[p];
      }
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        if (p == 0) {
          const uint32_t w0 = wa[m & 1][2 * j], w1 = wa[m & 1][2 * j + 1];
          if constexpr (Q8) {
            a0[j] = w4{w0, 0u, w1, 0u};
            a1[j] = w4{0u, w0, 0u, w1};
          } else {
            a0[j] = w4{w0 & even, w0 & ~even, w1 & even, w1 & ~even};
          }
        }
        x[p] = mfma_f16(a0[j], t[k & 1][j], x[p]);
        if constexpr (Q8) y[p] = mfma_f16(a1[j], t[k & 1][j], y[p]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int p = 0; p < NP; ++p)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        if constexpr (Q8) {
          acc[2 * p][v] = __builtin_fmaf(acc[2 * p][v], fa[v], x[p][v] * ft[v]);
          acc[2 * p + 1][v] = __builtin_fmaf(acc[2 * p + 1][v], fa[v], y[p][v] * ft[v]);
        } else {
          acc[p][v] = __builtin_fmaf(acc[p][v], fa[v], x[p][v] * ft[v]);
        }
      }
    wave_lds_fence();
  }

  // ---- the workgroup's waves merge through LDS
#pragma unroll
  for (int h = 0; h < NH; ++h) l[h] = wave_sum(l[h]);
  if (lane == 0) {
    float* st = s_stat + wid * S::kStat;
#pragma unroll
    for (int h = 0; h < NH; ++h) {
      st[h] = M[h];
      st[NH + h] = l[h];
    }
  }
  // the parts' rows add up: four heads, lane groups 0 + 1 (a pair's first coordinate) and 2 + 3 (its second); eight,
  // groups 0 + 2 (heads 0 - 3) and 1 + 3 (heads 4 - 7)
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    float* const dst = (float*)s_w + (Q8 ? 4 * g + v : v) * D + RC * n + (Q8 ? 0 : g >> 1);
#pragma unroll
    for (int i = 0; i < NA; ++i) {
      const uint32_t u = __float_as_uint(acc[i][v]);
      const auto r = Q8 ? __builtin_amdgcn_permlane32_swap(u, u, false, false)
                        : __builtin_amdgcn_permlane16_swap(u, u, false, false);
      const float o = __builtin_fmaf(__uint_as_float(r[1]), 1.f / kLoScale, __uint_as_float(r[0]));
      if (Q8 ? g < 2 : (g & 1) == 0) dst[Q8 ? i : 2 * i] = o;
    }
  }
  __syncthreads();
  float* const s_out = (float*)s_q;  // heads x D: the query operand's space, no longer read
  static_assert(S::kQ >= NH * D, "merged heads fit the query operand's space");
  const int nqh = (int)a.nq;
  for (int x = tid; x < nqh * D; x += blockDim.x) {
    const int h = x / D, j = x % D;
    float m = -__builtin_inff();
    for (int w = 0; w < waves; ++w) m = fmaxf(m, s_stat[w * S::kStat + h]);
    float ls = 0.f, o = 0.f;
    for (int w = 0; w < waves; ++w) {
      const float* st = s_stat + w * S::kStat;
      const float e = __builtin_amdgcn_exp2f(st[h] - m);
      ls = __builtin_fmaf(st[NH + h], e, ls);
      o = __builtin_fmaf(((const float*)(s_wave0 + w * S::kWave))[h * D + j], e, o);
    }
    if (a.chunks > 1) {
      a.ws[a.ws_acc + (((uint64_t)kv * a.nqp + h) * a.chunks + c) * D + j] = o;
      if (j == 0) {
        float* ml = a.ws + a.ws_ml + (((uint64_t)kv * a.nqp + h) * a.chunks + c) * 2;
        ml[0] = m;
        ml[1] = ls;
      }
    } else {
      s_out[x] = o / ls;
      if (j == 0 && a.lse) a.lse[(uint64_t)kv * a.nq + h] = (m + log2f(ls)) * kLn2;
    }
  }
  if (a.chunks > 1) return;
  // one workgroup per KV head: rotate back and write the output here
  __syncthreads();
  for (int h = wid; h < nqh; h += waves) {
    float y[E];
#pragma unroll
    for (int e = 0; e < E; ++e) y[e] = s_out[h * D + lane * E + e];
    fwht_contig<E, 64, float>(y, lane);
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int j = lane * E + e;
      const float o = y[e] * a.oscale;
      a.out[((uint64_t)kv * a.nq + h) * D + j] = sign_is_negative(a.vseed, (uint32_t)j) ? -o : o;
    }
  }
}

template <int KB, int VB, bool Q8>
hipError_t launch_one(const AttnArgs& a, uint32_t waves, hipStream_t s) {
  using S = Shape<PITCH_DIM, KB, VB, Q8>;
  constexpr uint32_t kMostBytes = S::bytes(max_waves(Q8));
  static_assert(kMostBytes <= 160u * 1024u, "LDS of one workgroup");
  waves = waves < max_waves(Q8) ? waves : max_waves(Q8);
  const uint32_t bytes = S::bytes(waves);
  // More than 64 KB of LDS have to be allowed for the kernel. That is a property of the kernel, not of the launch, so
  // every call sets what the largest launch takes: a value of its own could be lowered by a shorter call of another
  // thread between this call's setting and its launch.
  if (bytes > 65536u) {
    const hipError_t e = hipFuncSetAttribute((const void*)attn_codes<PITCH_DIM, KB, VB, Q8>,
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMostBytes);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL((attn_codes<PITCH_DIM, KB, VB, Q8>), dim3(a.spread ? (a.chunks + 7) / 8 * 8 * a.kv_heads : a.chunks * a.kv_heads), dim3(64 * waves), bytes, s, a);
  return hipSuccess;
}
template <int KB, int VB>
hipError_t launch_q(const AttnArgs& a, uint32_t waves, hipStream_t s) {
  return a.nq <= 4 ? launch_one<KB, VB, false>(a, waves, s) : launch_one<KB, VB, true>(a, waves, s);
}
template <int KB>
hipError_t launch_v(const AttnArgs& a, uint32_t waves, hipStream_t s) {
  switch (a.vbits) {
    case 2: return launch_q<KB, 2>(a, waves, s);
    case 3: return launch_q<KB, 3>(a, waves, s);
    case 4: return launch_q<KB, 4>(a, waves, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace

#define PITCH_CAT4_(a, b, c, d) a##b##c##d
#define PITCH_CAT4(a, b, c, d) PITCH_CAT4_(a, b, c, d)
hipError_t PITCH_CAT4(launch_attn_codes_d, PITCH_DIM, _k, PITCH_KIND)(const AttnArgs& a, uint32_t waves, hipStream_t s) {
  switch (a.kbits) {
    case 2: return launch_v<2>(a, waves, s);
    case 3: return launch_v<3>(a, waves, s);
    case 4: return launch_v<4>(a, waves, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace pitch
