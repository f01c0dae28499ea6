// Device helpers shared by the packed-KV attention kernels (decode split /
// combine in tq_attn.hip, prefill in tq_prefill.hip): fp16 packing, exp2,
// 3-bit code decode with v_perm_b32 table lookups, and reductions over the
// four lane groups of a wave.
#pragma once

#include "kernels.h"

namespace lkv {
namespace {

__device__ __forceinline__ uint32_t pack2h(float lo, float hi) {
  return static_cast<uint32_t>(f2h(lo)) | (static_cast<uint32_t>(f2h(hi)) << 16);
}

// fp16(a b) in the low half, fp16(c d) in the high half, each product rounded once: v_fma_mixlo / mixhi_f16, by the
// compiler.  No arithmetic here is inline asm: the wait states that gfx950 needs between a v_exp_f32 and the vector
// instruction that reads its result, a vector write and an MFMA or permlane swap that reads it, and an MFMA and a
// reader of its result are put in by the compiler, and only around instructions that it knows.
__device__ __forceinline__ uint32_t mul2h(float a, float b, float c, float d) {
  typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, f16x2{static_cast<_Float16>(fmaf(a, b, 0.f)), static_cast<_Float16>(fmaf(c, d, 0.f))});
}

// 2^x on the hardware exp (v_exp_f32); arguments here are <= 0 and results
// below 2^-126 flush to 0, which only drops contributions < 1e-38 of the max.
__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// 3-bit codes decoded on the VALU: one code dword = 8 nibbles (dims 0..7)
// becomes 4 dwords of fp16 pairs in the dim order [0,2 | 4,6 | 1,3 | 5,7].
// tab[0..1] hold the low bytes of the 8 fp16 centroids, tab[2..3] the high
// bytes; v_perm_b32 picks 4 of those 8 bytes per instruction (selector bytes
// 0..7 address {S0: bytes 4-7, S1: bytes 0-3}), so a lookup is 4 nibbles per
// instruction with no LDS traffic.  The query operand uses the same dim
// order, so each MFMA sees the same fp16 products as with natural order.
__device__ __forceinline__ void decode8(uint32_t w, const uint32_t (&tab)[4], uint32_t (&d)[4]) {
  const uint32_t lo = w & 0x0F0F0F0Fu;         // codes of dims 0, 2, 4, 6 (one per byte)
  const uint32_t hi = (w >> 4) & 0x0F0F0F0Fu;  // dims 1, 3, 5, 7
  const uint32_t llo = __builtin_amdgcn_perm(tab[1], tab[0], lo), hlo = __builtin_amdgcn_perm(tab[3], tab[2], lo);
  const uint32_t lhi = __builtin_amdgcn_perm(tab[1], tab[0], hi), hhi = __builtin_amdgcn_perm(tab[3], tab[2], hi);
  d[0] = __builtin_amdgcn_perm(hlo, llo, 0x05010400u);  // dims 0, 2
  d[1] = __builtin_amdgcn_perm(hlo, llo, 0x07030602u);  // dims 4, 6
  d[2] = __builtin_amdgcn_perm(hhi, lhi, 0x05010400u);  // dims 1, 3
  d[3] = __builtin_amdgcn_perm(hhi, lhi, 0x07030602u);  // dims 5, 7
}
// Position p of a decoded group holds dim kPermDim[p].
__device__ constexpr int kPermDim[8] = {0, 2, 4, 6, 1, 3, 5, 7};

// PERM: decode8 (3-bit codes).  Otherwise a 256-entry LDS table maps one
// code byte to the fp16 pair (c[lo nibble], c[hi nibble]) in natural order.
template <bool PERM>
__device__ __forceinline__ void decode_dw(uint32_t w, const uint32_t (&tab)[4], const uint32_t* s_lut,
                                          uint32_t (&d)[4]) {
  if constexpr (PERM) {
    decode8(w, tab, d);
  } else {
    d[0] = s_lut[w & 0xffu];
    d[1] = s_lut[(w >> 8) & 0xffu];
    d[2] = s_lut[(w >> 16) & 0xffu];
    d[3] = s_lut[w >> 24];
  }
}
// Pairs 2*half and 2*half + 1 of decode_dw (the value pass decodes in two
// halves to halve the live registers).
template <bool PERM>
__device__ __forceinline__ void decode_half(uint32_t w, int half, const uint32_t (&tab)[4], const uint32_t* s_lut,
                                            uint32_t (&d)[2]) {
  if constexpr (PERM) {
    const uint32_t c = (half ? (w >> 4) : w) & 0x0F0F0F0Fu;
    const uint32_t lo = __builtin_amdgcn_perm(tab[1], tab[0], c), hi = __builtin_amdgcn_perm(tab[3], tab[2], c);
    d[0] = __builtin_amdgcn_perm(hi, lo, 0x05010400u);
    d[1] = __builtin_amdgcn_perm(hi, lo, 0x07030602u);
  } else {
    d[0] = s_lut[(w >> (16 * half)) & 0xffu];
    d[1] = s_lut[(w >> (16 * half + 8)) & 0xffu];
  }
}

// Code rows by stored width CB: 4 = nibble rows (3- and 4-bit codes, 64 B per
// token), 2 = four 2-bit codes per byte (32 B), 1 = eight 1-bit codes per byte
// (16 B), the packings of leankv/turboquant/quantizer.py:38-62.  Narrow rows
// are widened to nibbles in registers as they arrive, so the decode after
// that (v_perm over a centroid table padded with zeros) is the 3-bit one.
template <int CB>
__host__ __device__ constexpr int code_row_bytes() {
  return 16 * CB;
}
// 16 bits of 2-bit codes (dims 0..7 at bits 2d) -> dims at bits 4d.
__device__ __forceinline__ uint32_t nib_from2(uint32_t x) {
  uint32_t t = x & 0xffffu;
  t = (t | (t << 8)) & 0x00ff00ffu;
  t = (t | (t << 4)) & 0x0f0f0f0fu;
  return (t | (t << 2)) & 0x33333333u;
}
// 8 bits of 1-bit codes (dim d at bit d) -> dims at bits 4d.
__device__ __forceinline__ uint32_t nib_from1(uint32_t x) {
  uint32_t t = x & 0xffu;
  t = (t | (t << 12)) & 0x000f000fu;
  t = (t | (t << 6)) & 0x03030303u;
  return (t | (t << 3)) & 0x11111111u;
}
// Dims 32k .. 32k+31 of a code row (voff: the row's byte 4*CB*k) as loaded, and widened to 4 nibble dwords.  The two
// are apart so that a load can stay in flight until its codes are used.
template <int CB>
__device__ __forceinline__ u32x4 load_raw32(__amdgpu_buffer_rsrc_t r, int voff) {
  if constexpr (CB == 4) {
    return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, voff, 0, 0));
  } else if constexpr (CB == 2) {
    const auto v = __builtin_amdgcn_raw_buffer_load_b64(r, voff, 0, 0);
    return u32x4{v[0], v[1], 0u, 0u};
  } else {
    return u32x4{__builtin_amdgcn_raw_buffer_load_b32(r, voff, 0, 0), 0u, 0u, 0u};
  }
}
template <int CB>
__device__ __forceinline__ uint32_t widen32(const u32x4& v, int k) {
  if constexpr (CB == 4)
    return v[k];
  else if constexpr (CB == 2)
    return nib_from2(v[k >> 1] >> (16 * (k & 1)));
  else
    return nib_from1(v[0] >> (8 * k));
}
// Dims 8k .. 8k+7 of a code row (row byte CB*k), the same way: one nibble dword.
template <int CB>
__device__ __forceinline__ uint32_t load_raw8(__amdgpu_buffer_rsrc_t r, int voff) {
  if constexpr (CB == 4)
    return __builtin_amdgcn_raw_buffer_load_b32(r, voff, 0, 0);
  else if constexpr (CB == 2)
    return __builtin_amdgcn_raw_buffer_load_b16(r, voff, 0, 0);
  else
    return __builtin_amdgcn_raw_buffer_load_b8(r, voff, 0, 0);
}
template <int CB>
__device__ __forceinline__ uint32_t widen8(uint32_t v) {
  if constexpr (CB == 4)
    return v;
  else if constexpr (CB == 2)
    return nib_from2(v);
  else
    return nib_from1(v);
}

// Buffer resource over `bytes` bytes at base (raw addressing, stride 0).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, bytes, 0x00020000);
}

// dims 32k .. 32k + 31 of a row whose code bytes start at p (row byte 4 CB k)
template <int CB>
__device__ __forceinline__ uint4 codes32(const uint8_t* p) {
  if constexpr (CB == 4) {
    return *reinterpret_cast<const uint4*>(p);
  } else if constexpr (CB == 2) {
    const uint2 v = *reinterpret_cast<const uint2*>(p);
    return uint4{nib_from2(v.x), nib_from2(v.x >> 16), nib_from2(v.y), nib_from2(v.y >> 16)};
  } else {
    const uint32_t v = *reinterpret_cast<const uint32_t*>(p);
    return uint4{nib_from1(v), nib_from1(v >> 8), nib_from1(v >> 16), nib_from1(v >> 24)};
  }
}
__device__ __forceinline__ float vmax3(float a, float b, float c) { return fmaxf(fmaxf(a, b), c); }  // v_max3_f32

// Online-softmax offset headroom, log2 units.  When a block's score exceeds
// the running offset m, m moves to that score plus the headroom, so the
// following blocks, whose scores mostly stay below it, skip the rescale of
// the accumulators.  Any offset at or above every score seen gives the same
// softmax (sums and accumulators are relative to it); every weight stays
// exp2(s - m) <= 1, so p * n_v cannot overflow its fp16 operand, and weights
// shrink by at most 2^-headroom, far above the fp16 denormal floor for any
// weight that matters.  0 gives the plain running maximum.
#ifndef LKV_SOFTMAX_HEADROOM
#define LKV_SOFTMAX_HEADROOM 4.0f
#endif
constexpr float kHeadroom = LKV_SOFTMAX_HEADROOM;

// Max / sum over the four lanes l, l^16, l^32, l^48 (the lane groups that
// hold the other tokens of the same head), result in all four.
__device__ __forceinline__ float xgroup_max(float v) {
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float xgroup_sum(float v) {
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

}  // namespace
}  // namespace lkv
