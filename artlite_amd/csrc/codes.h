// The bf16 MFMA products' operands over raw GGUF blocks (experts.hip, stream.hip): a block's integer codes as bf16, exact
// (128 + code), with the scales that the sums take in fp32.
#pragma once

#include "common.h"

namespace artlite {

typedef short bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4 mfma(const u32x4& a, const u32x4& b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                  0, 0);
}

__device__ __forceinline__ uint32_t lds_u32(const uint8_t* p) {
  uint32_t v;
  __builtin_memcpy(&v, p, 4);
  return v;
}

__device__ __forceinline__ uint32_t lds_u16(const uint8_t* p) {
  uint16_t v;
  __builtin_memcpy(&v, p, 2);
  return v;
}

__device__ __forceinline__ float h2f(uint32_t h) { return float(__builtin_bit_cast(_Float16, uint16_t(h))); }

// eight nibbles (the bytes of v0, v1, each < 16) -> the B operand's four dwords of bf16 128 + q
__device__ __forceinline__ u32x4 nib8(uint32_t v0, uint32_t v1) {
  return u32x4{__builtin_amdgcn_perm(0x43434343u, v0, 0x04010400u), __builtin_amdgcn_perm(0x43434343u, v0, 0x04030402u),
               __builtin_amdgcn_perm(0x43434343u, v1, 0x04010400u), __builtin_amdgcn_perm(0x43434343u, v1, 0x04030402u)};
}

// two bf16 of the unsigned bytes 2 j, 2 j + 1 of v (exact: < 256)
__device__ __forceinline__ uint32_t byte2(uint32_t v, int j) {
  const uint32_t f0 = __float_as_uint(float((v >> (16 * j)) & 0xFFu));
  const uint32_t f1 = __float_as_uint(float((v >> (16 * j + 8)) & 0xFFu));
  return __builtin_amdgcn_perm(f1, f0, 0x07060302u);
}

// eight unsigned bytes -> the B operand's four dwords of bf16
__device__ __forceinline__ u32x4 byte8(uint32_t v0, uint32_t v1) {
  return u32x4{byte2(v0, 0), byte2(v0, 1), byte2(v1, 0), byte2(v1, 1)};
}

// Per format: a block's bytes and 32-value groups; the groups of one K-range of k_gemm_decode (a stage: ~300..600 bytes of each row,
// so a 16-row stage is 16 long runs; a straddled cache line is read again by the next range of the same wave, from
// L2) and its bytes; the offset of the codes' bf16 encoding (the B operand holds 128 + c for a code byte c, or
// 128 + IQ4[c], so OFF = 128 + the format's zero point); whether the format has a min term (w = s q - m: Q4_1,
// Q4_K, Q5_K); whether its scales cover 16 values (Q3_K, Q6_K: one MFMA per half of a group, each with the other
// half's B lanes zero).
template <int BB, int GPB_, int KR_, int OFF_, bool MIN_ = false, bool SUB16_ = false>
struct FmtT {
  static constexpr int BLOCK_BYTES = BB;
  static constexpr int GPB = GPB_;  // 32-value groups per block (1 or 8)
  static constexpr int GROUP_BYTES = GPB_ == 1 ? BB : 0;  // (32-value blocks only)
  static constexpr int KR = KR_;
  static constexpr int RUN = KR_ / GPB_ * BB;  // bytes of a row's K-range
  static constexpr float OFF = float(OFF_);
  static constexpr bool MIN = MIN_;
  static constexpr bool SUB16 = SUB16_;
  static_assert(KR_ % GPB_ == 0, "K-ranges of whole blocks");
};
template <int QT>
struct Fmt;
template <>
struct Fmt<ARTLITE_Q4_0> : FmtT<18, 1, 32, 136> {};  // (128 + q) - (q - 8)
template <>
struct Fmt<ARTLITE_Q4_1> : FmtT<20, 1, 24, 128, true> {};
template <>
struct Fmt<ARTLITE_Q8_0> : FmtT<34, 1, 16, 128> {};  // (q + 128 through an unsigned byte)
template <>
struct Fmt<ARTLITE_Q3_K> : FmtT<112, 8, 32, 132, false, true> {};  // (128 + q) - (q - 4)
template <>
struct Fmt<ARTLITE_Q4_K> : FmtT<144, 8, 32, 128, true> {};
template <>
struct Fmt<ARTLITE_Q5_K> : FmtT<176, 8, 24, 128, true> {};
template <>
struct Fmt<ARTLITE_Q6_K> : FmtT<224, 8, 16, 160, false, true> {};  // (128 + q) - (q - 32); the layer's padded blocks
template <>
struct Fmt<ARTLITE_IQ4_NL> : FmtT<18, 1, 32, 128> {};
template <>
struct Fmt<ARTLITE_IQ4_XS> : FmtT<144, 8, 32, 128> {};  // (the layer's padded blocks)

// four codes (bytes < 16) -> the bytes 128 + IQ4[code] (the int8 values with the top bit flipped)
__device__ __forceinline__ uint32_t iq4_bytes(uint32_t c) { return iq4_int8(c) ^ 0x80808080u; }

// Q4_K / Q5_K's 6-bit scale and min of group g from the 12 bytes at s6
__device__ __forceinline__ void k_scale_min(const uint8_t* s6, int g, int& q6, int& m6) {
  q6 = g < 4 ? s6[g] & 63 : (s6[8 + g - 4] & 15) | ((s6[g - 4] >> 6) << 4);
  m6 = g < 4 ? s6[4 + g] & 63 : (s6[8 + g - 4] >> 4) | ((s6[4 + g - 4] >> 6) << 4);
}

// Q3_K's scale of sub-block sb (of 16), minus 32, from the 12 bytes at s
__device__ __forceinline__ int q3k_scale(const uint8_t* s, int sb) {
  const int lo = sb < 8 ? s[sb] & 15 : s[sb - 8] >> 4, hi = (s[8 + (sb & 3)] >> (2 * (sb >> 2))) & 3;
  return (lo | (hi << 4)) - 32;
}

// B operand of group gl of a row's run (row: its first byte in LDS) for lane group lg (values 8 lg .. + 8 of the
// group): 8 codes as 4 dwords of bf16, and the scales: sc (the whole group's, or SUB16: its first half's, with sc2
// the second half's) and, for the formats with a min, mn with w = sc q - mn (Q4_1's w = d q + m: mn = -m)
template <int QT>
__device__ __forceinline__ u32x4 b_operand(const uint8_t* row, int gl, int lg, float& sc, float& mn, float& sc2) {
  using F = Fmt<QT>;
  const uint8_t* blk = row + F::BLOCK_BYTES * (gl / F::GPB);
  const int g = gl % F::GPB;
  if constexpr (QT == ARTLITE_Q4_0 || QT == ARTLITE_Q4_1 || QT == ARTLITE_IQ4_NL) {
    constexpr int QS = QT == ARTLITE_Q4_1 ? 4 : 2;
    sc = h2f(lds_u16(blk));
    if constexpr (QT == ARTLITE_Q4_1) mn = -h2f(lds_u16(blk + 2));
    const int sh = 4 * (lg >> 1);
    const uint32_t u0 = (lds_u32(blk + QS + 8 * (lg & 1)) >> sh) & 0x0F0F0F0Fu;
    const uint32_t u1 = (lds_u32(blk + QS + 4 + 8 * (lg & 1)) >> sh) & 0x0F0F0F0Fu;
    if constexpr (QT == ARTLITE_IQ4_NL) return byte8(iq4_bytes(u0), iq4_bytes(u1));
    return nib8(u0, u1);
  } else if constexpr (QT == ARTLITE_Q8_0) {
    sc = h2f(lds_u16(blk));
    return byte8(lds_u32(blk + 2 + 8 * lg) ^ 0x80808080u, lds_u32(blk + 6 + 8 * lg) ^ 0x80808080u);
  } else if constexpr (QT == ARTLITE_Q4_K || QT == ARTLITE_Q5_K) {  // group g of the super-block
    int q6, m6;
    k_scale_min(blk + 4, g, q6, m6);
    sc = __fmul_rn(h2f(lds_u16(blk)), float(q6));
    mn = __fmul_rn(h2f(lds_u16(blk + 2)), float(m6));
    const uint8_t* qs = blk + (QT == ARTLITE_Q5_K ? 48 : 16) + 32 * (g >> 1) + 8 * lg;
    const int sh = 4 * (g & 1);
    uint32_t u0 = (lds_u32(qs) >> sh) & 0x0F0F0F0Fu, u1 = (lds_u32(qs + 4) >> sh) & 0x0F0F0F0Fu;
    if constexpr (QT == ARTLITE_Q5_K) {  // bit g of qh[l] (at 16) is the code's bit 4
      u0 |= ((lds_u32(blk + 16 + 8 * lg) >> g) & 0x01010101u) << 4;
      u1 |= ((lds_u32(blk + 20 + 8 * lg) >> g) & 0x01010101u) << 4;
    }
    return nib8(u0, u1);
  } else if constexpr (QT == ARTLITE_Q6_K) {  // group g = 4 h + jj: value l at ql[64 h + 32 (jj % 2) + l], qh[32 h + l]
    const int h = g >> 2, jj = g & 3;
    const float d = h2f(lds_u16(blk + 208));
    sc = __fmul_rn(float(int8_t(blk[192 + 2 * g])), d);
    sc2 = __fmul_rn(float(int8_t(blk[193 + 2 * g])), d);
    const uint8_t *ql = blk + 64 * h + 32 * (jj & 1) + 8 * lg, *qh = blk + 128 + 32 * h + 8 * lg;
    const int sh = jj < 2 ? 0 : 4;
    const uint32_t u0 = ((lds_u32(ql) >> sh) & 0x0F0F0F0Fu) | (((lds_u32(qh) >> (2 * jj)) & 0x03030303u) << 4);
    const uint32_t u1 = ((lds_u32(ql + 4) >> sh) & 0x0F0F0F0Fu) | (((lds_u32(qh + 4) >> (2 * jj)) & 0x03030303u) << 4);
    return nib8(u0, u1);
  } else if constexpr (QT == ARTLITE_Q3_K) {  // group g = 4 n + j: value 16 h + l at qs[32 n + 16 h + l], hm[16 h + l]
    const int n = g >> 2, j = g & 3;
    const float d = h2f(lds_u16(blk + 108));
    sc = __fmul_rn(d, float(q3k_scale(blk + 96, 2 * g)));
    sc2 = __fmul_rn(d, float(q3k_scale(blk + 96, 2 * g + 1)));
    const uint8_t *qs = blk + 32 + 32 * n + 8 * lg, *hm = blk + 8 * lg;
    const int hb = 4 * n + j;
    const uint32_t u0 = ((lds_u32(qs) >> (2 * j)) & 0x03030303u) | (((lds_u32(hm) >> hb) & 0x01010101u) << 2);
    const uint32_t u1 = ((lds_u32(qs + 4) >> (2 * j)) & 0x03030303u) | (((lds_u32(hm + 4) >> hb) & 0x01010101u) << 2);
    return nib8(u0, u1);
  } else {  // IQ4_XS (a layer's 144-byte block: the 8-byte header padded to 16): group g's codes at 16 + 16 g, its
            // scale d (ls - 32)
    const int ls = ((blk[4 + g / 2] >> (4 * (g & 1))) & 15) | (((int(lds_u16(blk + 2)) >> (2 * g)) & 3) << 4);
    sc = __fmul_rn(h2f(lds_u16(blk)), float(ls - 32));
    const uint8_t* qs = blk + 16 + 16 * g + 8 * (lg & 1);
    const int sh = 4 * (lg >> 1);
    return byte8(iq4_bytes((lds_u32(qs) >> sh) & 0x0F0F0F0Fu), iq4_bytes((lds_u32(qs + 4) >> sh) & 0x0F0F0F0Fu));
  }
}

}  // namespace artlite
