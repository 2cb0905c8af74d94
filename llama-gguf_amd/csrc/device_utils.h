// device_utils.h — small gfx950 device helpers (internal).
#pragma once

#include "common.h"

namespace lgh {

// streamed-once weights: non-temporal 16-byte loads straight to VGPRs (no LDS round trip for GEMV)
__device__ __forceinline__ u32x4 ldg_nt128(const void* p) {
  return __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
}
__device__ __forceinline__ u32x2 ldg_nt64(const void* p) {
  return __builtin_nontemporal_load(reinterpret_cast<const u32x2*>(p));
}
__device__ __forceinline__ uint32_t ldg_nt32(const void* p) {
  return __builtin_nontemporal_load(reinterpret_cast<const uint32_t*>(p));
}
__device__ __forceinline__ uint16_t ldg_nt16(const void* p) {
  return __builtin_nontemporal_load(reinterpret_cast<const uint16_t*>(p));
}

__device__ __forceinline__ float h2f(uint32_t bits16) {
  _Float16 h;
  uint16_t b = (uint16_t)bits16;
  __builtin_memcpy(&h, &b, 2);
  return (float)h;  // v_cvt_f32_f16, subnormals preserved
}

__device__ __forceinline__ float ub0(uint32_t v) { return (float)(v & 0xFFu); }
__device__ __forceinline__ float ub1(uint32_t v) { return (float)((v >> 8) & 0xFFu); }
__device__ __forceinline__ float ub2(uint32_t v) { return (float)((v >> 16) & 0xFFu); }
__device__ __forceinline__ float ub3(uint32_t v) { return (float)(v >> 24); }

// 4 FMAs of the 4 bytes of `v` against x[0..3]
__device__ __forceinline__ float fma4(uint32_t v, const float* x, float acc) {
  acc = __builtin_fmaf(ub0(v), x[0], acc);
  acc = __builtin_fmaf(ub1(v), x[1], acc);
  acc = __builtin_fmaf(ub2(v), x[2], acc);
  acc = __builtin_fmaf(ub3(v), x[3], acc);
  return acc;
}

// Makes `v` opaque to the optimizer at this point (no instruction is emitted).  Used after nibble masks so
// that `(m >> 8) & 0xFF` stays a single v_cvt_f32_ubyte1 instead of being re-folded into v_bfe_u32 + cvt.
__device__ __forceinline__ uint32_t opaque(uint32_t v) {
  asm volatile("" : "+v"(v));
  return v;
}

// the 4 bytes of `v` dotted with x[0..3], as a fresh chain (first term is a plain multiply)
__device__ __forceinline__ float fma4z(uint32_t v, const float* x) {
  float acc = ub0(v) * x[0];
  acc = __builtin_fmaf(ub1(v), x[1], acc);
  acc = __builtin_fmaf(ub2(v), x[2], acc);
  acc = __builtin_fmaf(ub3(v), x[3], acc);
  return acc;
}

// full-wave (64 lanes) sum; every lane gets the result; fixed order -> deterministic
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// DPP lane permutation of a float (gfx9 DPP controls): no LDS crossbar, full-rate VALU
template <int CTRL, int ROW_MASK = 0xF>
__device__ __forceinline__ float dpp_f(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, ROW_MASK, 0xF, false));
}

// 64-lane sum by DPP; the total is valid in LANE 63 only.  Fixed order -> deterministic.
__device__ __forceinline__ float wave_sum_to_lane63(float v) {
  v += dpp_f<0xB1>(v);        // quad_perm [1,0,3,2]
  v += dpp_f<0x4E>(v);        // quad_perm [2,3,0,1]
  v += dpp_f<0x141>(v);       // row_half_mirror
  v += dpp_f<0x140>(v);       // row_mirror  -> every lane of a 16-lane row holds the row sum
  v += dpp_f<0x142, 0xA>(v);  // row_bcast15 into rows 1 and 3
  v += dpp_f<0x143, 0xC>(v);  // row_bcast31 into rows 2 and 3
  return v;
}

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
  return v;
}

// sums and maxima over the rows of 16 lanes of a wave, without LDS
__device__ __forceinline__ float swap16_add(float v) {   // sum of rows 2i and 2i + 1 of 16 lanes, in both
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float swap32_add(float v) {   // sum of lanes l and l + 32, in both
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float swap16_max(float v) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float swap32_max(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// silu for activations that are rounded to 16 bits next: x / (1 + e^-x) as the library's expf and the compiler's division compute it (from -88.7 to 88 the largest relative error, 1.73e-7,
// and the mean square, 2.9e-8, are theirs), in 15 instructions instead of 31.  A clamped exponent spares expf's special cases; it still reaches infinity where e^-x does, so that the division's last step gives -0 there and no
// number for -inf.  Both sides of the division are a sixteenth, so that the reciprocal of its largest divisors is no subnormal (which the hardware's comes out as 0).
__device__ __forceinline__ float silu_act_f(float x) {
  const float c = __builtin_amdgcn_fmed3f(x, -127.0f, 87.0f), n = __builtin_rintf(c * -1.44269504f);
  const float f = __builtin_fmaf(c, -1.92596299e-8f, __builtin_fmaf(c, -1.44269504f, -n));   // log2 e in two parts
  const float y = x * 0.0625f, d = __builtin_fmaf(__builtin_amdgcn_ldexpf(__builtin_amdgcn_exp2f(f), (int)n), 0.0625f, 0.0625f), r = __builtin_amdgcn_rcpf(d), q = y * r;
  return __builtin_amdgcn_div_fixupf(__builtin_fmaf(__builtin_fmaf(-d, q, y), r, q), d, y);
}

// Factors with which NW waves' partial results (their m, l: ml[w * stride], behind it) become one, and the merged m and l.  A quad's four lanes merge the same waves: each lane has one factor (two of eight) and takes the
// others from its neighbours, for expf is a dozen instructions.  Sums in the waves' order.
template <int NW>
__device__ __forceinline__ void merge_factors(const float* ml, uint32_t stride, float (&f)[NW], float& m, float& l) {
  static_assert(NW == 4 || NW == 8, "");
  const uint32_t q = threadIdx.x & 3;
  float mw[NW / 4], lw[NW / 4];
#pragma unroll
  for (int h = 0; h < NW / 4; h++) { mw[h] = ml[(q + 4 * h) * stride]; lw[h] = ml[(q + 4 * h) * stride + 1]; }
  m = NW == 8 ? fmaxf(mw[0], mw[NW / 8]) : mw[0];
  m = fmaxf(m, dpp_f<0xB1>(m));
  m = fmaxf(m, dpp_f<0x4E>(m));
  l = 0.0f;
#pragma unroll
  for (int h = 0; h < NW / 4; h++) {
    const float e = expf(mw[h] - m), p = lw[h] * e;
    f[4 * h] = dpp_f<0x00>(e); f[4 * h + 1] = dpp_f<0x55>(e); f[4 * h + 2] = dpp_f<0xAA>(e); f[4 * h + 3] = dpp_f<0xFF>(e);
    l += dpp_f<0x00>(p); l += dpp_f<0x55>(p); l += dpp_f<0xAA>(p); l += dpp_f<0xFF>(p);
  }
}
// exp(m0 - max) and exp(m1 - max): the larger one's is 1
__device__ __forceinline__ void merge_two(float m0, float m1, float& m, float& a, float& b) {
  m = fmaxf(m0, m1);
  const float e = expf(fminf(m0, m1) - m);
  a = m0 >= m1 ? 1.0f : e;
  b = m1 >= m0 ? 1.0f : e;
}

}  // namespace lgh
