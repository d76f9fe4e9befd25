// Causal GQA prefill over quantized K/V caches (gfx950), head_dim 256: every
// pair of f16, q8_0, q4_0, q5_0 and q4_1 except f16/f16 (attn_prefill_mfma.hip).
//
// Reference semantics: the batched path of graph.cuh:1473-1535 over a quantized
// cache (attn_split_batch_launch, include/rdna4/attn.cuh:958-1049): query token
// i at position p_i attends keys 0..min(p_i, kmax), dequantized as kv_load<>
// (kv.h:174-368), f32 softmax and accumulation, then the optional sigmoid gate.
//
// Precision: f32 sums, and the error of f32 operands or less, on f16 matrix
// instructions. Every operand enters as an f16 hi part plus the f16 remainder (22
// bits where f32 has 24):
//   * a query row is scaled by a power of two (its largest |q * scale * log2e|
//     comes to [2^8, 2^9)) and split, q' = qh + ql: 22 bits of a value down to 2^-10
//     of the row's largest, below that 2^-34 of the largest. Rows with 8 consecutive
//     dims all below 2^-10 (and not zero), or with an infinity, take f32 scores;
//   * a quantized key row is scaled by a power of two (its largest block scale
//     comes to [2^7, 2^8)) and split: d * int has at most 19 significant bits, so
//     K' = kh + kl exactly (blocks down to 2^-21 of the row's largest scale);
//   * S = kl.qh + kh.ql + kh.qh (q4_1: + kl.ql), f32 accumulation, then times both powers of two;
//     the scores of a key row that this does not hold (scales further apart, values
//     that are not finite) are formed in f32 from the row itself;
//   * value rows are scaled by a power of two 2^e of the CTA (its block of 32 keys
//     has its largest block scale between 1 and 2^8; a block that has not moves e,
//     and O with it) and split like keys, exactly for blocks down to 2^-14;
//   * p stays f32 for the row sum l; p * 2^7 is split for O += vl.ph + vh.pl + vh.ph (q4_1: + vl.pl):
//     22 bits of a p down to 2^-10 of the row's largest, below that 2^-32 of the
//     largest;
//   * V blocks that this does not hold (scales further apart, or not finite) enter
//     the products as zeros and are added in f32 for the rows that attend them.
// f16 rows have no remainder part (and no scaling): two products instead of three.
// Relative error against 64 bits, the VALU kernel (attn_generic.hip), which took
// these calls before, in brackets, for q8_0: 1.2e-7 (1.3e-7) at 33 queries over 33
// keys, 2.1e-7 (2.6e-7) over 233, 3.5e-7 (8.8e-7) over 8064; 0.23 to 0.98 times that
// kernel's in 300 calls of 25 to 2300 queries over up to 32768 keys, queries and caches
// near N(0, 1). (Queries of 0.2 over 28 to 100 q8_0 or q4_0 keys: 1.03 to 1.07, where
// vl.pl, left out, shows beside few other roundings.) What it takes: the
// large products of S in four sums and the small ones in a fifth (one sum for
// all: 2.0 times the error at 233 keys), the p split near 2^7 (near 1: 1.5
// times), and O rounded once per block where a CTA sums most of a row (BSUM below). V's power of two is no part of p (a row's own exponent in p, as 2^e of it:
// rows 2^17 smaller than another lost percents of what they add where the other's
// dims are zero).
//
// Work decomposition: rows r = query * group + head of one kv head as in the
// f16 kernel; CTA = 8 waves x 16 rows, 32-key blocks. Each wave owns 8 key rows of
// a block (waves 0-3 K, 4-7 V): it brings their raw cache bytes to its own LDS
// area by DMA two blocks ahead, and a block ahead converts them, 8 lanes per row
// and one 32-value block per lane, into the hi / lo stage that all waves read.
// Two stages, one CTA barrier per block. Waves w and w + 4 share a SIMD:
// waves 0-3 convert before their products, 4-7 after, so that one's conversion
// runs beside the other's matrix instructions.
// What bounds it: LDS reads (64 KiB per wave and block, 0.5 MiB per CTA, 1.1 us
// of a block's 3.0) and the matrix pipe (192 products per SIMD and block, 1.5 us),
// which two waves per SIMD overlap in part; the conversion is 0.6 us of it. 512
// queries over 8192 q8_0 keys, 24 / 4 heads: 6120 us in the VALU kernel, 342 us
// here (0.29 PFLOP/s, 0.87 counted as issued). Conversion pieces between the
// products of a block, one pair after each fragment, were slower than in one go
// at opposite ends of the block for the two waves of a SIMD (350 against 340 us).
#include <algorithm>
#include <cstdlib>
#include <type_traits>

#include "kv_quant.hpp"
#include "prefill.hpp"

namespace rd4 {

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef short short4v __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) short4v lds_short4;
typedef __attribute__((address_space(3))) const u32x4 lds_u32x4;

constexpr int kHD = 256;
constexpr int kBN = 32;            // keys per block
constexpr int kW = 8;              // waves per CTA
constexpr int kBM = 16 * kW;       // rows per CTA
constexpr int kPart = kBN * kHD * 2;  // one f16 part of a block's K or V rows
constexpr float kLog2e = 1.4426950408889634f;
// the largest p * 2^kPShift of a row is kept between 2^kPShift and 2^(kPShift + 8):
// terms 2^-10 of it still have normal f16 remainder parts
constexpr int kPShift = 7;
// A V block's largest scale, as scaled, is kept between 2^0 and 2^(kVTop + 1)
// (times 127 it is below f16's largest, and steps of the scales' exponents up to
// kVMid either way leave e alone), placed at 2^kVMid when it is not.
constexpr int kVTop = 7, kVMid = 4;
constexpr int kKTop = 7;  // a K row's largest scale, as scaled, is in [2^kKTop, 2^(kKTop + 1))

// LDS: two stages of [K hi][K lo][V hi][V lo] (lo parts of quantized types
// only), each wave's raw rows, then the per-key tables of both stages.
template <bool KLO, bool VLO>
struct Lds {
  static constexpr int KH = 0, KL = kPart, VH = (1 + KLO) * kPart, VL = VH + kPart;
  static constexpr int kStage = (2 + KLO + VLO) * kPart;
  // 8 rows of a wave in whole 1 KiB DMA instructions: f16 4096 B, else at most 3072
  static constexpr int kRawK = KLO ? 3072 : 4096, kRawV = VLO ? 3072 : 4096;
  static constexpr int kRaw = 2 * kStage;
  static constexpr int kTab = kRaw + 4 * (kRawK + kRawV);
  // per stage: f32 2^e of K rows, one byte per V row with a bit for each of its
  // blocks that is outside the products, the same per K row, and V's exponent e
  static constexpr int kNf = kBN * 4, kKm = kNf + kBN, kE = kKm + kBN;
  static constexpr int kTabStage = kE + 16;
  static constexpr int kBytes = kTab + 2 * kTabStage;
  static_assert(kBytes <= 160 * 1024, "LDS of a CU");
};

// LDS swizzle of a 512-byte f16 row: 16-byte chunk c of key r sits in slot
// c ^ swz(r) (the f16 prefill kernel's map, conflict-free for the b128 operand
// reads and for the transposing reads).
__device__ __forceinline__ int swz(int r) {
  return ((r & 1) ? 8 : 0) ^ ((r & 2) ? 7 : 0) ^ ((r & 4) ? 2 : 0) ^ ((r & 8) ? 4 : 0);
}

__device__ __forceinline__ half2v as_h2(uint32_t v) { return __builtin_bit_cast(half2v, v); }
__device__ __forceinline__ uint32_t as_u32(half2v v) { return __builtin_bit_cast(uint32_t, v); }

// max over lanes l, l ^ 16, l ^ 32, l ^ 48
__device__ __forceinline__ float max_groups4(float x) {
  float a = x, b = x;
  __asm__("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(a), "+v"(b));
  float c = fmaxf(a, b), d = c;
  __asm__("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(c), "+v"(d));
  return fmaxf(c, d);
}
// Row and block of a lane in the conversion of a wave's 8 rows: 16 consecutive
// lanes hold blocks 4h .. 4h + 3 of rows 0, 2, 4, 6 (or 1, 3, 5, 7), whose chunks
// i of the 16-byte swizzle fall in 16 different slots: the stage writes meet no
// bank conflict (8 lanes per row in order: 2-way).
__device__ __forceinline__ int conv_row(int lane) { return ((lane >> 4) & 1) | (((lane >> 2) & 3) << 1); }
__device__ __forceinline__ int conv_block(int lane) { return (lane & 3) | ((lane >> 5) << 2); }
// unsigned max over the wave
__device__ __forceinline__ uint32_t max_wave_u32(uint32_t x) {
  int v = (int)x;
  v = max(v, __builtin_amdgcn_update_dpp(v, v, 0xB1, 0xF, 0xF, false));   // quad_perm 1,0,3,2
  v = max(v, __builtin_amdgcn_update_dpp(v, v, 0x4E, 0xF, 0xF, false));   // quad_perm 2,3,0,1
  v = max(v, __builtin_amdgcn_update_dpp(v, v, 0x141, 0xF, 0xF, false));  // row_half_mirror
  v = max(v, __builtin_amdgcn_update_dpp(v, v, 0x140, 0xF, 0xF, false));  // row_mirror
  int a = v, b = v;
  __asm__("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(a), "+v"(b));
  a = max(a, b), b = a;
  __asm__("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(a), "+v"(b));
  return __builtin_amdgcn_readfirstlane((uint32_t)max(a, b));
}
// unsigned max over the 8 lanes of a row
__device__ __forceinline__ uint32_t max_row_u32(uint32_t x) {
  int v = (int)x;
  v = max(v, __builtin_amdgcn_update_dpp(v, v, 0xB1, 0xF, 0xF, false));  // quad_perm 1,0,3,2
  v = max(v, __builtin_amdgcn_update_dpp(v, v, 0x4E, 0xF, 0xF, false));  // quad_perm 2,3,0,1
  int c = v, d = v;
  __asm__("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(c), "+v"(d));
  return (uint32_t)max(c, d);
}

// 16 bytes per lane from sbase + voff into LDS at lds + 16 * lane (asm, so the
// compiler puts no wait for it in front of other LDS reads; the kernel waits)
__device__ __forceinline__ void dma16(const uint8_t *sbase, uint32_t voff, uint32_t lds) {
  __asm__ volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                   :
                   : "v"(voff), "s"(sbase), "s"(lds)
                   : "memory", "m0");
}
__device__ __forceinline__ uint32_t lds_addr(const uint8_t *p) {
  return __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(const __attribute__((address_space(3))) uint8_t *)p);
}
__device__ __forceinline__ const uint8_t *uniform_ptr(const uint8_t *ptr) {
  const uint64_t a = (uint64_t)ptr;
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)a), hi = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32));
  return (const uint8_t *)(((uint64_t)hi << 32) | lo);
}

// The kernel's arguments read again where they are used (the f32 paths), and a
// pointer among them: held in scalar registers through the loop they spill (12 of
// them, read back in each block: 338 -> 347 us at 512 queries over 8192 keys).
__device__ __forceinline__ PrefillArgs args_again() {
  const __attribute__((address_space(4))) PrefillArgs *a =
      (const __attribute__((address_space(4))) PrefillArgs *)__builtin_amdgcn_kernarg_segment_ptr();
  __asm__ volatile("" : "+s"(a));
  PrefillArgs r;
  __builtin_memcpy(&r, (const PrefillArgs *)a, sizeof(r));
  return r;
}
template <typename T>
__device__ __forceinline__ const T *global_ptr(const T *x) {
  return (const T *)(const __attribute__((address_space(1))) T *)x;
}

// Two integers as an f16 pair times the block scale -> hi pair and exact
// remainder pair (an f16 product's rounding error is itself an f16).
__device__ __forceinline__ void split_mul(half2v q, half2v d, uint32_t &hi, uint32_t &lo) {
  const half2v h = q * d;
  hi = as_u32(h);
  lo = as_u32(__builtin_elementwise_fma(q, d, -h));
}
// The same with q4_1's offset: d * q + m, the sum's rounding error recovered by
// a two-sum.
__device__ __forceinline__ void split_mul_add(half2v q, half2v d, half2v m, uint32_t &hi, uint32_t &lo) {
  const half2v h = q * d, l = __builtin_elementwise_fma(q, d, -h);
  const half2v s = h + m, bb = s - h;
  const half2v err = (h - (s - bb)) + (m - bb);
  hi = as_u32(s);
  lo = as_u32(err + l);
}

// The words of 32-value block b of a row (4-byte aligned; blocks start 2 bytes off a
// word where b is odd, except q4_1's): *dm its scale d (q4_1: d | offset m << 16), w
// the data behind it (q5_0: the high bits, then the nibbles; q4_1: the nibbles).
template <int T>
__device__ __forceinline__ void block_words(const uint8_t *row, int b, uint32_t *w, uint32_t *dm) {
  constexpr int BB = block_bytes(T);
  constexpr int NW = T == Q8_0 ? 8 : T == Q5_0 ? 5 : 4;
  const uint32_t *p = (const uint32_t *)(row + ((BB * b) & ~3));
  if constexpr (T == Q4_1) {
    *dm = p[0];
#pragma unroll
    for (int i = 0; i < NW; ++i) w[i] = p[i + 1];
  } else {
    uint32_t x[NW + 1];
#pragma unroll
    for (int i = 0; i <= NW; ++i) x[i] = p[i];
    const bool odd = b & 1;
    *dm = odd ? x[0] >> 16 : x[0] & 0xffffu;
    // even blocks: data starts 2 bytes into x[0]; odd blocks: at x[1]
    const uint32_t sel = odd ? 0x07060504u : 0x05040302u;
#pragma unroll
    for (int i = 0; i < NW; ++i) w[i] = __builtin_amdgcn_perm(x[i + 1], x[i], sel);
  }
}

// Elements 2f, 2f + 1 of the block whose words block_words read: an f16 pair of
// the integers (exact), T's bias taken off.
template <int T>
__device__ __forceinline__ half2v block_pair(const uint32_t *w, int f) {
  if constexpr (T == Q8_0) {  // f16 1024 + 128 + byte, less 1152
    const half2v c = {(_Float16)-1152.0f, (_Float16)-1152.0f};
    return as_h2(__builtin_amdgcn_perm(0u, w[f >> 1], (f & 1) ? 0x0c030c02u : 0x0c010c00u) ^ 0x64806480u) + c;
  } else {
    constexpr float kBias = T == Q4_0 ? -1032.0f : T == Q5_0 ? -1040.0f : -1024.0f;
    const half2v c = {(_Float16)kBias, (_Float16)kBias};
    const int half = f >> 3, i = f & 7;  // low nibbles: elements 0..15, high: 16..31
    const uint32_t by = __builtin_amdgcn_perm(0u, w[(T == Q5_0 ? 1 : 0) + (i >> 1)], (i & 1) ? 0x0c030c02u : 0x0c010c00u);
    uint32_t n = (half ? by >> 4 : by) & 0x000f000fu;
    if constexpr (T == Q5_0) {
      const uint32_t hb = w[0] >> (16 * half + 2 * i);  // bits of the two elements
      n |= ((hb & 1u) << 4) | ((hb & 2u) << 19);
    }
    return as_h2(n | 0x64006400u) + c;
  }
}

// 32-dim block b of a cache row as block_words reads it (f16: its values), and the
// values 4 c .. 4 c + 3 of it.
template <int T>
struct RowBlock {
  uint32_t w[T == F16 ? 16 : 8], dm;
  __device__ __forceinline__ void read(const uint8_t *row, int b) {
    if constexpr (T == F16) {
#pragma unroll
      for (int i = 0; i < 4; ++i) *(u32x4 *)(w + 4 * i) = *(const u32x4 *)(row + 64 * b + 16 * i);
    } else {
      block_words<T>(row, b, w, &dm);
    }
  }
  __device__ __forceinline__ void values(int c, float v[4]) const {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      half2v q;
      if constexpr (T == F16) q = as_h2(w[2 * c + i]);
      else q = block_pair<T>(w, 2 * c + i);
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        float x = (float)q[e];
        if constexpr (T != F16) x = mul_rn(h2f((uint16_t)dm), x);
        if constexpr (T == Q4_1) x = add_rn(x, h2f((uint16_t)(dm >> 16)));
        v[2 * i + e] = x;
      }
    }
  }
};

// Exponent of f16 magnitude bits (subnormals: that of the smallest normal), and the
// larger finite magnitude of a block's scale d and, of q4_1, offset m (dm: d | m << 16).
__device__ __forceinline__ int mag_exponent(uint32_t mag) { return max((int)(mag >> 10), 1) - 15; }
__device__ __forceinline__ uint32_t finite_mag(uint32_t dm, bool with_m) {
  const uint32_t d = dm & 0x7fffu, m = with_m ? (dm >> 16) & 0x7fffu : 0u;
  return max(d >= 0x7c00u ? 0u : d, m >= 0x7c00u ? 0u : m);
}

// Convert the wave's 8 raw rows (lane: row conv_row, block conv_block; rb bytes per
// row) into the stage rows at hi_st (their lo parts kPart bytes on) and the tables:
// for K pw2_tab[key] = 2^e, e the row's exponent; V comes with its exponent ev.
// nf_tab[key] = the mask of the row's blocks that are outside the products: V's are
// zeros in the stage, a K row with any is left to the f32 path as a whole.
template <int T, bool V>
__device__ __forceinline__ void convert_rows(const uint8_t *raw, int key0, int lane, uint8_t *hi_st, float *pw2_tab,
                                             uint8_t *nf_tab, int ev) {
  const int r = conv_row(lane), b = conv_block(lane), key = key0 + r, sz = swz(key & 15);
  uint8_t *dst = hi_st + key * (kHD * 2);
  bool out = false;
  if constexpr (T == F16) {
    bool nonfin = false;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      u32x4 x = *(const u32x4 *)(raw + r * 512 + 64 * b + 16 * i);
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const bool lo = (x[c] & 0x7c00u) == 0x7c00u, hi = (x[c] & 0x7c000000u) == 0x7c000000u;
        nonfin |= lo || hi;
        if (V) x[c] &= (lo ? 0xffff0000u : 0xffffffffu) & (hi ? 0x0000ffffu : 0xffffffffu);
      }
      *(u32x4 *)(dst + 16 * ((4 * b + i) ^ sz)) = x;
    }
    out = nonfin;
  } else {
    uint32_t w[8], dm, ch[4], cl[4];
    block_words<T>(raw + r * (8 * block_bytes(T)), b, w, &dm);
    // K: the row's power of two from its largest scale (q4_1: or offset) magnitude.
    const int e = V ? ev : mag_exponent(max_row_u32(finite_mag(dm, T == Q4_1))) - kKTop;
    _Float16 d = __builtin_amdgcn_ldexph(__builtin_bit_cast(_Float16, (uint16_t)dm), -e);
    _Float16 m = T == Q4_1 ? __builtin_amdgcn_ldexph(__builtin_bit_cast(_Float16, (uint16_t)(dm >> 16)), -e) : (_Float16)0.0f;
    // outside: not finite, or d or m, as scaled, below the normal f16 range, where it
    // may lose bits
    auto lost = [](uint32_t before, _Float16 x) {  // scaled: not normal, and not from a zero
      return __builtin_amdgcn_classh(x, 0x2f7) && (before & 0x7fffu) != 0;
    };
    out = lost(dm, d) || (T == Q4_1 && lost(dm >> 16, m));
    if (V && out) d = (_Float16)0.0f, m = (_Float16)0.0f;
#pragma unroll
    for (int f = 0; f < 16; ++f) {
      const half2v q = block_pair<T>(w, f);
      if constexpr (T == Q4_1) split_mul_add(q, half2v{d, d}, half2v{m, m}, ch[f & 3], cl[f & 3]);
      else split_mul(q, half2v{d, d}, ch[f & 3], cl[f & 3]);
      if ((f & 3) == 3) {
        uint8_t *at = dst + 16 * ((4 * b + (f >> 2)) ^ sz);
        *(u32x4 *)at = u32x4{ch[0], ch[1], ch[2], ch[3]};
        *(u32x4 *)(at + kPart) = u32x4{cl[0], cl[1], cl[2], cl[3]};
      }
    }
    if (!V && b == 0) pw2_tab[key] = __builtin_ldexpf(1.0f, e);
  }
  const uint64_t nf = __ballot(out);
  if (b == 0) nf_tab[key] = (uint8_t)(((nf >> (lane & 0x1c)) & 15u) | (((nf >> ((lane & 0x1c) + 32)) & 15u) << 4));
}

}  // namespace

// The kernel's lambdas are its own text: outlined, they put what they capture in scratch.
#define RD4_INLINE __attribute__((always_inline))

// K fragments and V operand pairs in registers or in flight ahead of their products
constexpr int kRing = 3;  // (2 to 5: within 1%)

// KT, VT: the cache types, or -1 for a type read at run time. KLO, VLO: the rows
// have remainder parts (all but f16); VFULL: q4_1 values, whose remainders are as
// full as p's, take the fourth product vl.pl too (at 120 queries over 120 keys the
// error is 1.04 times the VALU kernel's without it, 0.88 with); q4_1 keys take
// kl.ql likewise (1 query over 31 keys 1.23 times, 0.94 with it; 512 over 8192 385 us,
// 414 with it). BSUM: a block's products with V are summed from zero and added to O once,
// one tile behind, so that O is rounded once per block and not at each product: 64 adds
// per block that no product hides. For calls of one or two splits, whose CTAs sum half of
// a row's keys or more: 990 q4_0 queries over 4051 keys have 1.19 times the VALU
// kernel's error without it, 0.56 with (374 us, 399 with it), rows 780 to 827 of 1660
// from position 0 (two splits, theirs the first) 1.14 and 0.79 (103, 108 us). Shorter sums stay below that kernel's without it
// (512 over 8192 in five splits: 0.6 times; 345 us, 365 with it).
template <int T>
using type_c = std::integral_constant<int, T>;
template <int KT, int VT, bool KLO, bool VLO, bool VFULL, bool BSUM>
__global__ __launch_bounds__(64 * kW, 1) void prefill_quant_kernel(PrefillArgs p) {
  using L = Lds<KLO, VLO>;
  extern __shared__ __align__(512) uint8_t smem[];  // (512: the operand addresses XOR the low bits)
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int n = lane & 15, g = lane >> 4;
  const int grp = p.n_head / p.n_head_kv;
  const int n_rows = p.n_q * grp;
  const int n_rb = (n_rows + kBM - 1) / kBM;
  const int total = n_rb * p.n_head_kv;
  const int ksp = p.n_ksplit > 1 ? (int)blockIdx.x / total : 0;
  const int Lb = (int)blockIdx.x - ksp * total;
  // as in the f16 kernel: a kv head's row blocks share the XCDs (and L2s) of that head
  int kvh, rbp;
  if (8 % p.n_head_kv == 0 && total % 8 == 0) {
    const int X = 8 / p.n_head_kv, xcd = Lb % 8, j = Lb / 8;
    kvh = xcd % p.n_head_kv;
    rbp = j * X + xcd / p.n_head_kv;
  } else {
    kvh = Lb / n_rb;
    rbp = Lb - kvh * n_rb;
  }
  const int r0 = (n_rb - 1 - rbp) * kBM;  // heaviest (latest queries) first

  auto limit_of = [&](int row) RD4_INLINE -> int {
    if (row >= n_rows) return -1;
    const int q = row / grp;
    return min(p.pos0 + q, p.kmax);
  };
  int kend;  // last key that any row of the CTA attends
  {
    int lim = max(limit_of(r0 + lane), limit_of(r0 + 64 + lane));
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) lim = max(lim, __shfl_xor(lim, m, 64));
    kend = __builtin_amdgcn_readfirstlane(lim);
  }
  const int n_blocks = (kend + kBN) / kBN;
  const int b0 = p.n_ksplit > 1 ? ksp * p.ksplit_blocks : 0;
  const int nbk = p.n_ksplit > 1 ? max(0, min(n_blocks, b0 + p.ksplit_blocks) - b0) : n_blocks;

  // ---- raw rows of this wave: 8 consecutive keys of each block, K (waves 0-3) or V
  const bool isv = w >= 4;
  const int my_t = isv ? p.vt : p.kt;
  const int rb = __builtin_amdgcn_readfirstlane((int)row_bytes(my_t, kHD)), nch = rb >> 4;
  const int n_dma = (8 * nch + 63) >> 6;
  const uint8_t *my_base = (isv ? p.v : p.k) + (int64_t)kvh * rb;
  const int my_stride = p.n_head_kv * rb;
  uint8_t *raw = smem + L::kRaw + (isv ? 4 * L::kRawK + (w - 4) * L::kRawV : w * L::kRawK);
  uint32_t c_at[4];  // key in the block (high half) and byte in its row of each 16-byte chunk
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int c = min(64 * i + lane, 8 * nch - 1);  // (surplus lanes repeat the last chunk into the padding)
    c_at[i] = (uint32_t)(8 * (w & 3) + c / nch) << 16 | (uint32_t)(16 * (c % nch));
  }
  // V waves: scale (q4_1: and offset) of 4 of a block's 256 (key, 32 dims) pairs,
  // loaded beside its rows: each V wave needs the exponent of all 32 keys before it
  // converts its own 8
  uint32_t v_dm[4];
  int e_v = 0;
  auto issue = [&](int bi) RD4_INLINE {
    const int j0 = (b0 + bi) * kBN;
    if (VLO && isv) {
      const uint8_t *at = my_base + (int64_t)j0 * my_stride + (lane & 7) * (rb >> 3);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint8_t *x = at + (int64_t)min(8 * i + (lane >> 3), kend - j0) * my_stride;
        if (VT == Q4_1 || (VT < 0 && VFULL)) v_dm[i] = *(const uint32_t *)x;
        else v_dm[i] = ld_u16(x);
      }
    }
    const uint8_t *src = uniform_ptr(my_base + (int64_t)j0 * my_stride);
#pragma unroll
    for (int i = 0; i < 4; ++i)  // keys past kend re-read a valid row (masked later)
      if (i < n_dma) dma16(src, (uint32_t)(min((int)(c_at[i] >> 16), kend - j0) * my_stride) + (c_at[i] & 0xffffu), lds_addr(raw + 1024 * i));
  };
  auto tab = [&](int st) RD4_INLINE { return (float *)(smem + L::kTab + st * L::kTabStage); };
  auto convert_as = [&](auto type, auto is_v, int st) RD4_INLINE {
    float *t = tab(st);
    uint8_t *sb = smem + st * L::kStage;
    constexpr int T = decltype(type)::value;
    if constexpr (decltype(is_v)::value) {
      if (VLO) {  // e_v: the same in the four V waves
        uint32_t mag = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) mag = max(mag, max(v_dm[i] & 0x7fffu, T == Q4_1 ? (v_dm[i] >> 16) & 0x7fffu : 0u));
        mag = max_wave_u32(mag);
        if (mag >= 0x7c00u) {  // (uniform) the largest finite one counts
          mag = 0;
#pragma unroll
          for (int i = 0; i < 4; ++i) mag = max(mag, finite_mag(v_dm[i], T == Q4_1));
          mag = max_wave_u32(mag);
        }
        const int top = mag_exponent(mag) - e_v;
        if (mag && (top < 0 || top > kVTop)) e_v += top - kVMid;
        if (w == 4 && lane == 0) *(int *)((uint8_t *)t + L::kE) = e_v;
      }
      convert_rows<T, true>(raw, 8 * (w & 3), lane, sb + L::VH, nullptr, (uint8_t *)t + L::kNf, e_v);
    } else
      convert_rows<T, false>(raw, 8 * (w & 3), lane, sb + L::KH, t, (uint8_t *)t + L::kKm, 0);
  };
  // this wave's rows into stage st: K for waves 0-3, V for 4-7
  auto convert_k = [&](int st) RD4_INLINE {
    if constexpr (KT >= 0) convert_as(type_c<KT>{}, std::false_type{}, st);
    else if constexpr (!KLO) convert_as(type_c<F16>{}, std::false_type{}, st);
    else switch (p.kt) {
      case Q8_0: convert_as(type_c<Q8_0>{}, std::false_type{}, st); break;
      case Q4_0: convert_as(type_c<Q4_0>{}, std::false_type{}, st); break;
      default: convert_as(type_c<Q5_0>{}, std::false_type{}, st); break;
    }
  };
  auto convert_v = [&](int st) RD4_INLINE {
    if constexpr (VT >= 0) convert_as(type_c<VT>{}, std::true_type{}, st);
    else if constexpr (!VLO) convert_as(type_c<F16>{}, std::true_type{}, st);
    else if constexpr (VFULL) convert_as(type_c<Q4_1>{}, std::true_type{}, st);
    else switch (p.vt) {
      case Q8_0: convert_as(type_c<Q8_0>{}, std::true_type{}, st); break;
      case Q4_0: convert_as(type_c<Q4_0>{}, std::true_type{}, st); break;
      default: convert_as(type_c<Q5_0>{}, std::true_type{}, st); break;
    }
  };
  if (nbk > 0) issue(0);

  // ---- this wave's query rows (row n of the wave is r0 + 16 w + n): scaled, split
  const int row = r0 + 16 * w + n;
  const int lim_row = limit_of(row);
  half8 qh[8], ql[8];
  float c_row;  // 2^-k: the power of two taken out of the row
  uint32_t q_out;  // the wave's rows (bit n) that the split does not hold
  {
    const bool on = row < n_rows;
    const int q = on ? row / grp : 0, head = kvh * grp + (on ? row % grp : 0);
    const int64_t qoff = ((int64_t)q * p.n_head + head) * kHD + 8 * g;
    const float sl2 = on ? p.scale * kLog2e : 0.0f;
    float x[8][8];
    if (p.q_f16) {
#pragma unroll
      for (int b = 0; b < 8; ++b) {
        const half8 h = *(const half8 *)((const uint16_t *)p.q + qoff + 32 * b);
#pragma unroll
        for (int i = 0; i < 8; ++i) x[b][i] = (float)h[i];
      }
    } else {
#pragma unroll
      for (int b = 0; b < 8; ++b) {
        const floatx4 u = *(const floatx4 *)((const float *)p.q + qoff + 32 * b);
        const floatx4 v = *(const floatx4 *)((const float *)p.q + qoff + 32 * b + 4);
#pragma unroll
        for (int i = 0; i < 4; ++i) x[b][i] = u[i], x[b][4 + i] = v[i];
      }
    }
    float mx = 0.0f, least = INFINITY;  // of the lane's 8-dim groups that are not zero, the least maximum
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      float mb = 0.0f;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        x[b][i] *= sl2;
        mb = fmaxf(mb, fabsf(x[b][i]));
      }
      mx = fmaxf(mx, mb);
      if (mb > 0.0f) least = fminf(least, mb);
    }
    mx = max_groups4(mx);
    const uint64_t far = __ballot(least < mx * 0x1p-10f || mx == INFINITY);
    q_out = (uint32_t)(far | far >> 16 | far >> 32 | far >> 48) & 0xffffu;
    // exponent that brings mx to [2^8, 2^9); zero rows and infinities stay as they are
    const int ex = (int)(__builtin_bit_cast(uint32_t, mx) >> 23) - 127;
    const int k = (mx > 0.0f && ex < 128) ? min(126, 8 - ex) : 0;
    c_row = __builtin_ldexpf(1.0f, -k);
#pragma unroll
    for (int b = 0; b < 8; ++b)
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float y = __builtin_ldexpf(x[b][i], k);
        const _Float16 h = (_Float16)y;
        qh[b][i] = h;
        ql[b][i] = (_Float16)(y - (float)h);
      }
  }
  int wave_min_lim = lim_row;  // blocks whose last key is <= it need no mask
#pragma unroll
  for (int m = 1; m < 64; m <<= 1) wave_min_lim = min(wave_min_lim, __shfl_xor(wave_min_lim, m, 64));

  floatx4 o[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) o[i] = floatx4{0.f, 0.f, 0.f, 0.f};
  float m_run = -INFINITY, l_run = 0.0f;
  int e_o = 0;  // O is in units of 2^(e_o - kPShift)

  // transposing V reads (as in the f16 kernel): source lane s of a 16-lane group
  // points at key 4g + s/4, dims 4(s%4)..+3 of a 16-dim tile
  const int tr_kx = 4 * g + (n >> 2);
  const int tr_off = tr_kx * (kHD * 2) + 8 * (n & 1);
  const int tr_m = 16 * ((n >> 1 & 1) ^ swz(tr_kx));
  // LDS address of fragment 0 in stage 0; the others differ in XORed bits (the
  // stages are 512-byte aligned), which costs an instruction at each read and no
  // registers
  auto lds_of = [](const uint8_t *x) RD4_INLINE { return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) uint8_t *)x; };
  const uint32_t v_at = lds_of(smem + L::VH) + tr_off + tr_m;
  const uint32_t k_at = lds_of(smem + L::KH) + n * (kHD * 2) + 16 * (g ^ swz(n));

  // the first block's rows: converted before the loop
  if (nbk > 0) {
    __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (isv) convert_v(0);
    else convert_k(0);
    __asm__ volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // raw rows read before they are overwritten
    if (nbk > 1) issue(1);
  }

  for (int bi = 0; bi < nbk; ++bi) {
    const int st = bi & 1;
    const int j0 = (b0 + bi) * kBN;
    // this wave's conversion of block bi is written; past the barrier so is every
    // wave's, and all are done reading the other stage. (Raw rows are waited for by
    // the wave that converts them: K's here, V's, which were requested a moment
    // ago, after the products.)
    __asm__ volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    const bool more = bi + 1 < nbk;
    auto landed = [&]() RD4_INLINE { __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory"); };
    auto refill = [&]() RD4_INLINE {
      __asm__ volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // raw rows read before they are overwritten
      if (bi + 2 < nbk) issue(bi + 2);
    };
    if (more && !isv) {
      landed();
      convert_k(st ^ 1);
      refill();
    }
    const uint32_t k_st = k_at + st * L::kStage, v_st = v_at + st * L::kStage;
    const float *tb = tab(st);

    // ---- S^T of the two 16-key tiles: fragment f = (tile f / 8, dim block f % 8).
    // (The small products go to a sum of their own and the large ones to four, so
    // that few roundings happen at the size of the whole sum.)
    floatx4 s[2];
    const uint32_t km_lane = ((const uint8_t *)tb + L::kKm)[lane & 31];
    {
      constexpr int D = kRing;
      u32x4 fh[D], fl[D];
      floatx4 sc[5];
      auto read_k = [&](int f) RD4_INLINE {
        const uint32_t a = (k_st ^ (64u * (f & 7))) + (f >> 3) * 16 * (kHD * 2);
        fh[f % D] = *(lds_u32x4 *)a;
        if (KLO) fl[f % D] = *(lds_u32x4 *)(a + kPart);
        __builtin_amdgcn_sched_barrier(0);
      };
#pragma unroll
      for (int f = 0; f < D - 1; ++f) read_k(f);
#pragma unroll
      for (int f = 0; f < 16; ++f) {
        if (f + D - 1 < 16) read_k(f + D - 1);
        const int b = f & 7, kt = f >> 3;
        if (b == 0) {
#pragma unroll
          for (int i = 0; i < 5; ++i) sc[i] = floatx4{0.f, 0.f, 0.f, 0.f};
        }
        const half8 kh = __builtin_bit_cast(half8, fh[f % D]);
        if (KLO) sc[4] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, fl[f % D]), qh[b], sc[4], 0, 0, 0);
        sc[b & 3] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kh, qh[b], sc[b & 3], 0, 0, 0);
        sc[4] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kh, ql[b], sc[4], 0, 0, 0);
        if (KT == Q4_1) sc[4] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, fl[f % D]), ql[b], sc[4], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        if (b == 7) s[kt] = ((sc[0] + sc[1]) + (sc[2] + sc[3])) + sc[4];
      }
    }
    // ---- online softmax: lane = row n, keys 16 kt + 4 g + i. The running max
    // (m_run, in log2) follows s, to within 8.
    half8 ph, pl;
    float pf[2][4];
    const uint8_t *nf = (const uint8_t *)tb + L::kNf;
    const uint32_t nf_lane = nf[lane & 31];  // (read here, used after the products)
    const int e_st = VLO ? *(const int *)((const uint8_t *)tb + L::kE) : 0;
    {
      if (KLO) {
#pragma unroll
        for (int kt = 0; kt < 2; ++kt) {
          const floatx4 ks = *(const floatx4 *)(tb + 16 * kt + 4 * g);
#pragma unroll
          for (int i = 0; i < 4; ++i) s[kt][i] *= ks[i];
        }
      }
      // K rows outside the products (for queries outside them, all): their scores on
      // the f32 matrix instruction, K from the cache and q as it came. Lane (n, g)
      // brings dims 64 g .. 64 g + 63 of key n of a tile and of its row. (512 queries
      // over 4096 keys that are all such: 0.95 ms; the VALU kernel 2.9, the same by FMA
      // with each lane on its own row 3.7 to 7.8.)
      const uint32_t out_keys = (uint32_t)__ballot(km_lane != 0);
      if (out_keys | q_out) {
        const PrefillArgs pa = args_again();
        const uint8_t *pk = global_ptr(pa.k), *pq = global_ptr((const uint8_t *)pa.q);
        const int k_rb = (int)row_bytes(pa.kt, kHD), k_stride = pa.n_head_kv * k_rb;
        const int ga = pa.n_head / pa.n_head_kv;
        int rr = min(row, pa.n_q * ga - 1), d0 = 64 * g;
        __asm__ volatile("" : "+v"(rr), "+v"(d0));  // (addresses formed here, not held through the loop)
        const int64_t qat = ((int64_t)(rr / ga) * pa.n_head + kvh * ga + rr % ga) * kHD + d0;
        const float sl2 = pa.scale * kLog2e, up = 1.0f / c_row;  // (up: a power of two)
        const uint32_t mine = ((q_out >> n) & 1 ? ~0u : out_keys) >> (4 * g);
#pragma unroll 1
        for (int kt = 0; kt < 2; ++kt) {
          if (!(q_out | ((out_keys >> (16 * kt)) & 0xffffu)) || j0 + 16 * kt > kend) continue;
          // (keys past kend re-read a valid row: masked below)
          const uint8_t *kr = pk + (int64_t)(j0 + min(16 * kt + n, kend - j0)) * k_stride + (int64_t)kvh * k_rb;
          floatx4 f[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
          constexpr bool kTight = KLO && KT < 0;
          auto block = [&](auto type, int h) RD4_INLINE {
            RowBlock<decltype(type)::value> kb;
            kb.read(kr, (d0 >> 5) + h);
#pragma unroll
            for (int c = 0; c < 8; ++c) {  // 4 dims at a time (few registers beside O and q)
              float x[4], kv[4];
              if (pa.q_f16) load4<F16>(pq + 2 * qat, 32 * h + 4 * c, x);
              else load4<F32>(pq + 4 * qat, 32 * h + 4 * c, x);
              kb.values(c, kv);
#pragma unroll
              for (int i = 0; i < 4; ++i)
                f[i & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(kv[i], x[i] * sl2 * up, f[i & 1], 0, 0, 0);
              if (kTight || (c & 1)) __builtin_amdgcn_sched_barrier(0);
            }
          };
#pragma unroll 1
          for (int h = 0; h < 2; ++h) {
            if constexpr (KT >= 0) block(type_c<KT>{}, h);
            else if constexpr (!KLO) block(type_c<F16>{}, h);
            else if (pa.kt == Q8_0) block(type_c<Q8_0>{}, h);
            else if (pa.kt == Q4_0) block(type_c<Q4_0>{}, h);
            else block(type_c<Q5_0>{}, h);
          }
#pragma unroll
          for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i)
              if (t == kt && ((mine >> (16 * t + i)) & 1)) s[t][i] = f[0][i] + f[1][i];
        }
      }
      if (j0 + kBN - 1 > wave_min_lim) {  // wave-uniform
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (j0 + 16 * kt + 4 * g + i > lim_row) s[kt][i] = -INFINITY;
      }
      float tmax = -INFINITY;
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int i = 0; i < 4; ++i) tmax = fmaxf(tmax, s[kt][i] * c_row);
      tmax = max_groups4(tmax);
      const bool bump = tmax > m_run + 8.0f;
      if (__any(bump)) {
        const float m_new = bump ? tmax : m_run;
        const float corr = (m_run == -INFINITY) ? 0.0f : __builtin_amdgcn_exp2f(m_run - m_new);
        l_run *= corr;
#pragma unroll
        for (int i = 0; i < 16; ++i) o[i] *= corr;
        m_run = m_new;
      }
      const float m_use = (m_run == -INFINITY) ? 0.0f : m_run;
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float pv = __builtin_amdgcn_exp2f(fmaf(s[kt][i], c_row, -m_use));
          pf[kt][i] = pv;
          const float pp = pv * (float)(1 << kPShift);
          const _Float16 h = (_Float16)pp;
          ph[4 * kt + i] = h;
          pl[4 * kt + i] = (_Float16)(pp - (float)h);
        }
      l_run += ((pf[0][0] + pf[0][1]) + (pf[0][2] + pf[0][3])) + ((pf[1][0] + pf[1][1]) + (pf[1][2] + pf[1][3]));
    }

    // ---- O^T += V^T P^T: 16 dim tiles, two transposing loads per operand
    if (VLO) {
      const int e = __builtin_amdgcn_readfirstlane(e_st);
      if (e != e_o) {  // (uniform)
        const float f = __builtin_ldexpf(1.0f, e_o - e);
#pragma unroll
        for (int i = 0; i < 16; ++i) o[i] *= f;
        e_o = e;
      }
    }
    {
      constexpr int D = kRing;
      half8 fh[D], fl[D];
      auto read_v = [&](int dt) RD4_INLINE {
        const uint32_t a = v_st ^ (32u * dt);
        auto tr = [](uint32_t x) RD4_INLINE {
          const short4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4 *)x);
          const short4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4 *)(x + 16 * (kHD * 2)));
          return __builtin_bit_cast(half8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        };
        fh[dt % D] = tr(a);
        if (VLO) fl[dt % D] = tr(a + kPart);
        __builtin_amdgcn_sched_barrier(0);
      };
#pragma unroll
      for (int t = 0; t < D - 1; ++t) read_v(t);
      floatx4 c;
      auto add = [&](int t) RD4_INLINE {
        o[t] += c;
        __asm__ volatile("" : "+v"(o[t]));  // (here: moved to the block's end the sums spill)
      };
#pragma unroll
      for (int t = 0; t < 16; ++t) {
        if (t + D - 1 < 16) read_v(t + D - 1);
        floatx4 x = BSUM ? floatx4{0.f, 0.f, 0.f, 0.f} : o[t];
        if (VFULL) x = __builtin_amdgcn_mfma_f32_16x16x32_f16(fl[t % D], pl, x, 0, 0, 0);
        if (VLO) x = __builtin_amdgcn_mfma_f32_16x16x32_f16(fl[t % D], ph, x, 0, 0, 0);
        x = __builtin_amdgcn_mfma_f32_16x16x32_f16(fh[t % D], pl, x, 0, 0, 0);
        x = __builtin_amdgcn_mfma_f32_16x16x32_f16(fh[t % D], ph, x, 0, 0, 0);
        if (BSUM && t > 0) add(t - 1);
        if (BSUM) c = x;
        else o[t] = x;
        __builtin_amdgcn_sched_barrier(0);
      }
      if (BSUM) add(15);
    }
    if (more && isv) {
      landed();
      convert_v(st ^ 1);
      refill();
    }
    // What entered as zeros (f16 values that are not finite, blocks of a quantized
    // cache outside the scaled range) is added here, for the rows that attend the key.
    // (512 queries over 4096 keys: 1.0 ms with one block of each row such, 2.7 with
    // nearly all; the VALU kernel 2.9.)
    if (__any(nf_lane != 0)) {
      const PrefillArgs pa = args_again();
      const uint8_t *pv = global_ptr(pa.v);
      const int v_rb = (int)row_bytes(pa.vt, kHD), v_stride = pa.n_head_kv * v_rb;
      auto load_v = [&](const uint8_t *vr, int d, float v[4]) RD4_INLINE {
        if constexpr (VT >= 0) load4<VT>(vr, d, v);
        else if constexpr (VFULL) load4<Q4_1>(vr, d, v);
        else if (pa.vt == Q8_0) load4<Q8_0>(vr, d, v);
        else if (pa.vt == Q4_0) load4<Q4_0>(vr, d, v);
        else load4<Q5_0>(vr, d, v);
      };
#pragma unroll 1
      for (int key = 0; key < kBN; ++key) {
        const uint32_t blocks = __builtin_amdgcn_readfirstlane((uint32_t)nf[key]);
        if (blocks == 0 || j0 + key > kend) continue;  // (past kend a valid row was read again)
        float x = 0.0f;
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (16 * kt + i == (key & 0x13)) x = pf[kt][i];
        x = __builtin_ldexpf(__shfl(x, 4 * (key & 12) + n, 64), kPShift - e_o);
        const uint8_t *vr = pv + (int64_t)(j0 + key) * v_stride + (int64_t)kvh * v_rb;
        const bool on = j0 + key <= lim_row;
        constexpr int kTiles = VT >= 0 || VFULL ? 4 : 2;  // (4 where the type is read at run time spills)
#pragma unroll
        for (int d4 = 0; d4 < 16; d4 += kTiles) {  // kTiles dim tiles' loads in flight together
          if (!((blocks >> (d4 >> 1)) & (kTiles == 4 ? 3 : 1))) continue;  // (uniform)
          int g4 = 4 * g;
          __asm__ volatile("" : "+v"(g4)::"memory");  // (addresses formed here, not held through the loop)
          float v[kTiles][4];
#pragma unroll
          for (int i = 0; i < kTiles; ++i) load_v(vr, 16 * (d4 + i) + g4, v[i]);
#pragma unroll
          for (int i = 0; i < kTiles; ++i)
            if (on && ((blocks >> ((d4 + i) >> 1)) & 1)) {
#pragma unroll
              for (int c = 0; c < 4; ++c)
                if (VLO || !(fabsf(v[i][c]) < INFINITY)) o[d4 + i][c] = fmaf(x, v[i][c], o[d4 + i][c]);
            }
        }
      }
    }
  }

  // ---- epilogue: l over the 4 key groups, then the record of a key split, or
  // normalize, gate, store
  float Ls = l_run;
  Ls += __shfl_xor(Ls, 16, 64);
  Ls += __shfl_xor(Ls, 32, 64);
  const PrefillArgs pe = args_again();
  const int ge = pe.n_head / pe.n_head_kv;
  if (row >= pe.n_q * ge) return;
  const int q = row / ge, head = kvh * ge + row % ge;
  const float o_pw2 = __builtin_ldexpf(1.0f, e_o - kPShift);
  if (pe.n_ksplit > 1) {
    const int64_t nr = (int64_t)pe.n_q * pe.n_head, rr = (int64_t)ksp * nr + (int64_t)q * pe.n_head + head;
    float *rec = pe.part + rr * kHD;
#pragma unroll
    for (int dt = 0; dt < 16; ++dt)
      if (nbk > 0) *(floatx4 *)(rec + 16 * dt + 4 * g) = o[dt] * o_pw2;  // (the merge drops the record of an empty split)
    if (g == 0)  // (l = -1: the row attends no key of the split)
      *(float2 *)(pe.part + (int64_t)pe.n_ksplit * nr * kHD + 2 * rr) = make_float2(m_run, lim_row < b0 * kBN ? -1.0f : Ls);
    return;
  }
  const float inv = (m_run == -INFINITY || !(Ls > 0.0f)) ? 0.0f : o_pw2 / Ls;
  const int64_t ob = ((int64_t)q * pe.n_head + head) * kHD;
#pragma unroll
  for (int dt = 0; dt < 16; ++dt) {
    const int d = 16 * dt + 4 * g;
    float v[4] = {o[dt][0] * inv, o[dt][1] * inv, o[dt][2] * inv, o[dt][3] * inv};
    if (pe.gate) {
      float4 gv = *(const float4 *)(pe.gate + ob + d);
      float gs[4] = {gv.x, gv.y, gv.z, gv.w};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        gs[i] = 1.0f / (1.0f + expf(-gs[i]));
        v[i] *= gs[i];
      }
      *(float4 *)(pe.gate + ob + d) = make_float4(gs[0], gs[1], gs[2], gs[3]);
    }
    *(float4 *)(pe.out + ob + d) = make_float4(v[0], v[1], v[2], v[3]);
  }
}

bool prefill_quant_supported(int kt, int vt, int n_head, int n_head_kv, int head_dim) {
  const char *e = std::getenv("RD4_PREFILL_GENERIC");
  if (e && std::atoi(e) != 0) return false;
  return kt != F32 && vt != F32 && !(kt == F16 && vt == F16) && head_dim == kHD && n_head_kv > 0 &&
         n_head % n_head_kv == 0;
}


template <int KT, int VT, bool KLO = KT != F16, bool VLO = VT != F16, bool VFULL = VT == Q4_1>
static void launch(const PrefillArgs &q, dim3 grid, hipStream_t st) {
  constexpr size_t lds = Lds<KLO, VLO>::kBytes;
  if (q.n_ksplit <= 2)
    hipLaunchKernelGGL((prefill_quant_kernel<KT, VT, KLO, VLO, VFULL, true>), grid, dim3(64 * kW), lds, st, q);
  else
    hipLaunchKernelGGL((prefill_quant_kernel<KT, VT, KLO, VLO, VFULL, false>), grid, dim3(64 * kW), lds, st, q);
}

hipError_t prefill_quant_launch(int kt, int vt, const PrefillArgs &p, hipStream_t st) {
  PrefillArgs q = p;
  q.kt = kt;
  q.vt = vt;
  const int grp = p.n_head / p.n_head_kv;
  const int total = (p.n_q * grp + kBM - 1) / kBM * p.n_head_kv;
  prefill_set_ksplits(q, prefill_ksplits(p, kt, vt, p.part_floats), kBN);
  dim3 grid((unsigned)(total * q.n_ksplit));
  // the pairs that caches are made of have their conversion built in; the others
  // switch on the type in each block (q8_0, 512 queries over 8192 keys: 350 us
  // built in, 384 switched)
  if (kt == Q8_0 && vt == Q8_0) launch<Q8_0, Q8_0>(q, grid, st);
  else if (kt == Q4_0 && vt == Q4_0) launch<Q4_0, Q4_0>(q, grid, st);
  else if (kt == Q5_0 && vt == Q5_0) launch<Q5_0, Q5_0>(q, grid, st);
  else if (kt == Q4_1 && vt == Q4_1) launch<Q4_1, Q4_1>(q, grid, st);
  else if (kt == Q5_0 && vt == Q4_1) launch<Q5_0, Q4_1>(q, grid, st);
  else if (kt == Q4_1 && vt == F16) launch<Q4_1, F16>(q, grid, st);
  else if (kt == Q4_1) launch<Q4_1, -1, true, true, false>(q, grid, st);
  else if (kt == F16 && vt == Q4_1) launch<F16, -1, false, true, true>(q, grid, st);
  else if (kt == F16) launch<F16, -1, false, true, false>(q, grid, st);
  else if (vt == F16) launch<-1, F16, true, false, false>(q, grid, st);
  else if (vt == Q4_1) launch<-1, -1, true, true, true>(q, grid, st);
  else launch<-1, -1, true, true, false>(q, grid, st);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess || q.n_ksplit == 1) return e;
  return prefill_merge_launch(q, st);
}

}  // namespace rd4
