// MFMA, LDS and bf16-split helpers of the kernels that multiply fp32 values
// as bf16 hi + lo parts on v_mfma_f32_16x16x32_bf16.
#pragma once

#include "wkv7_common.h"

namespace wkv7 {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// LDS layouts. Every operand array is [token][64 channels] with unpadded
// 128 B rows whose 16 B chunks are XOR-swizzled by the row (chunk c of row r
// sits at c ^ (r & 7)): the MFMA operand loads (16 rows x 4 chunks per
// ds_read_b128) are then free of bank conflicts on gfx950, which 144 B padded
// rows are not (measured with the LDS bank-conflict counters). Transposed
// operands come from the same arrays through the LDS transpose reads (ld_tr),
// so nothing is stored twice.
constexpr int kPR = kHead;  // [row][64] arrays: 128 B rows, chunk-swizzled
// element offset of channel e (0..63) of row r of a [row][64] array
__device__ __forceinline__ int rk_off(int r, int e) {
  return r * kPR + ((((e >> 3) ^ r) & 7) << 3) + (e & 7);
}

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

// LDS transpose read (ds_read_b64_tr_b16). Inside each 16-lane group, lane
// lam reads the 4 consecutive bf16 at its address, D[lam][0..3], and receives
// D[4 j + lam / 4][lam % 4] as element j. A lane that reads row r0 + lam / 4
// of a row-major [row][col] array at column c0 + 4 (lam % 4) therefore gets
// column c0 + lam at rows r0 .. r0 + 3: a 16-row fragment of the transpose.
__device__ __forceinline__ uint2 ld_tr(const uint16_t* p) {
  const s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p));
  return __builtin_bit_cast(uint2, v);
}

// x = hi + lo: hi = bf16(x) and lo = bf16(x - hi), both rounded to nearest
// even; |x - hi - lo| <= 2^-18 |x|. The difference comes from one
// v_dot2_f32_bf16 with {-1, 0} or {0, -1}, one instruction where unpacking hi
// and subtracting take two. It is exact in fp32 (x - hi has at most 16
// significant bits), except that the pair's other half enters times 0: one that
// is not finite makes the difference NaN, so the two values of a pair belong
// to one value column of the state, or to one token. The constants
// must be registers: as literals the compiler encodes {-1, 0} as the inline
// constant -1.0, which the instruction reads as {0, -1}.
struct Neg {
  uint32_t lo, hi;  // {-1, 0} and {0, -1} as packed bf16
};
__device__ __forceinline__ Neg neg_consts() {
  Neg n;
  asm volatile("s_mov_b32 %0, 0xbf80\n\ts_mov_b32 %1, 0xbf800000" : "=s"(n.lo), "=s"(n.hi));
  return n;
}
// x - (element of the packed pair that `neg` selects)
__device__ __forceinline__ float sub_bf16(float x, uint32_t pair, uint32_t neg) {
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, pair),
                                         __builtin_bit_cast(bf16x2_t, neg), x, false);
}
// Two values per call, packed as bf16 pairs (first value in the low half).
__device__ __forceinline__ void split2(float a, float b, uint32_t& hi, uint32_t& lo,
                                       const Neg& n) {
  hi = pack_bf16(a, b);
  lo = pack_bf16(sub_bf16(a, hi, n.lo), sub_bf16(b, hi, n.hi));
}

__device__ __forceinline__ void pack_split(const f32x4& x, uint2& hi, uint2& lo, const Neg& n) {
  split2(x[0], x[1], hi.x, lo.x, n);
  split2(x[2], x[3], hi.y, lo.y, n);
}

__device__ __forceinline__ uint4 ld16(const uint16_t* p) { return *reinterpret_cast<const uint4*>(p); }

__device__ __forceinline__ f32x4 mma32(const uint4& a, const uint4& b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
// (The legacy 16x16x16 bf16 instruction is not used: its results read back by
// VALU came out nondeterministically wrong on gfx950 with this toolchain's
// wait-state insertion.)
// (ah + al)(bh + bl) without the lo*lo term, small terms first.
__device__ __forceinline__ f32x4 mma32x3(const uint4& ah, const uint4& al, const uint4& bh,
                                         const uint4& bl, f32x4 c) {
  c = mma32(al, bh, c);
  c = mma32(ah, bl, c);
  return mma32(ah, bh, c);
}

// element m of eight packed bf16
__device__ __forceinline__ float elem(const uint4& x, int m) {
  const uint32_t p = m < 2 ? x.x : m < 4 ? x.y : m < 6 ? x.z : x.w;
  return (m & 1) ? bf16_hi(p) : bf16_lo(p);
}

__device__ __forceinline__ void st16(uint16_t* p, const uint4& x) {
  *reinterpret_cast<uint4*>(p) = x;
}

__device__ __forceinline__ void split8(const float (&x)[8], uint4& hi, uint4& lo, const Neg& n) {
  split2(x[0], x[1], hi.x, lo.x, n);
  split2(x[2], x[3], hi.y, lo.y, n);
  split2(x[4], x[5], hi.z, lo.z, n);
  split2(x[6], x[7], hi.w, lo.w, n);
}

}  // namespace
}  // namespace wkv7
