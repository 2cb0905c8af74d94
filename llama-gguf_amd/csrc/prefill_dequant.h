// prefill_dequant.h — tile16 weights to f16 matrix-core operands (prefill.hip, prefill_wide.hip; internal).
// Weights are dequantized as w * 2^8 (kPfScale) to keep small block scales out of the f16 subnormals; |w| < 256 is assumed (f16 overflow
// otherwise) — GGUF weights are O(1).
#pragma once

#include <type_traits>

#include "device_utils.h"
#include "prefill.h"

namespace lgh {

typedef _Float16 h16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 h16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 h16x2 __attribute__((ext_vector_type(2)));

// formats as in matvec_mfma.hip (same tile16 layouts)
enum : int { PF_Q4K = 0, PF_Q6K = 1, PF_Q5K = 2, PF_Q80 = 3, PF_Q40 = 4 };
__host__ __device__ constexpr uint32_t pf_tile_bytes(int f) {
  return f == PF_Q4K ? 2304u : f == PF_Q6K ? 3392u : f == PF_Q5K ? 2816u : f == PF_Q80 ? 4352u : 2304u;
}
static inline int pf_fmt_of(int dev_type) {
  return dev_type == kDevQ4K_T16 ? PF_Q4K : dev_type == kDevQ6K_T16 ? PF_Q6K : dev_type == kDevQ5K_T16 ? PF_Q5K
         : dev_type == kDevQ80_T16 ? PF_Q80 : dev_type == kDevQ40_T16 ? PF_Q40 : -1;
}

constexpr float kPfScale = 256.0f;

struct PfRaw { u32x4 hd; u32x4 q[4]; };

template <int F>
__device__ __forceinline__ void pf_load(PfRaw& r, const uint8_t* tile, uint32_t lane, uint32_t n) {
  if (F == PF_Q6K) {
    r.hd = ldg_nt128(tile + 3072 + n * 16);
#pragma unroll
    for (int i = 0; i < 3; i++) r.q[i] = ldg_nt128(tile + i * 1024 + lane * 16);
    r.q[3].x = ldg_nt32(tile + 3328 + (n >> 1) * 4);
  } else if (F == PF_Q80) {
    r.hd = ldg_nt128(tile + 4096 + n * 16);
#pragma unroll
    for (int i = 0; i < 4; i++) r.q[i] = ldg_nt128(tile + i * 1024 + lane * 16);
  } else {
    r.hd = ldg_nt128(tile + 2048 + n * 16);
    r.q[0] = ldg_nt128(tile + lane * 16);
    r.q[1] = ldg_nt128(tile + 1024 + lane * 16);
    if (F == PF_Q5K) {
      const u32x2 h = ldg_nt64(tile + 2304 + lane * 8);
      r.q[2].x = h.x;
      r.q[2].y = h.y;
    }
  }
}

__device__ __forceinline__ h16x2 pf_bcast(float v) {
  const _Float16 h = (_Float16)v;
  h16x2 r = {h, h};
  return r;
}

// scale S and offset O (both times kPfScale, as f16 pairs) of MFMA step pp of the lane's row n and k-chunk c:
// weight = S * u + O with u the unsigned stored quant
template <int F>
__device__ __forceinline__ void pf_scale(const PfRaw& r, int pp, uint32_t n, uint32_t c, h16x2& S, h16x2& O) {
  if (F == PF_Q6K) {   // y = d * sc * (q' - 32), one int8 scale per 16 elements (dequant.rs:321-356)
    const uint32_t hdw = pp == 0 ? r.hd.x : pp == 1 ? r.hd.y : pp == 2 ? r.hd.z : r.hd.w;
    const float scf = (float)(int)__builtin_amdgcn_sbfe((int)hdw, c * 8, 8);
    const uint32_t dh = (n & 1) ? r.q[3].x >> 16 : r.q[3].x & 0xFFFFu;
    S = pf_bcast(h2f(dh) * kPfScale * scf);
    O = S * pf_bcast(-32.0f);
  } else if (F == PF_Q80 || F == PF_Q40) {   // y = d * q (Q8_0, stored q + 128 after the sign flip) / d * (q - 8) (Q4_0)
    const uint32_t hdw = pp == 0 ? r.hd.x : pp == 1 ? r.hd.y : pp == 2 ? r.hd.z : r.hd.w;
    const float dd = h2f((c >> 1) ? hdw >> 16 : hdw & 0xFFFFu);
    S = pf_bcast(dd * kPfScale);
    O = S * pf_bcast(F == PF_Q80 ? -128.0f : -8.0f);
  } else {   // Q4_K / Q5_K: y = d * sc * q - dmin * m, 6-bit (sc, m) per 32 elements (dequant.rs:210-255)
    const uint32_t s8 = (c >> 1) * 8;
    const uint32_t a = (r.hd.y >> s8) & 0x00FF00FFu, bq = (r.hd.z >> s8) & 0x00FF00FFu, cq = (r.hd.w >> s8) & 0x00FF00FFu;
    uint32_t sc, mn;
    if (pp < 2) {
      const uint32_t sc01 = a & 0x003F003Fu, mn01 = bq & 0x003F003Fu;
      sc = pp == 0 ? sc01 & 0xFFu : sc01 >> 16;
      mn = pp == 0 ? mn01 & 0xFFu : mn01 >> 16;
    } else {
      const uint32_t sc23 = (cq & 0x000F000Fu) | ((a >> 2) & 0x00300030u);
      const uint32_t mn23 = ((cq >> 4) & 0x000F000Fu) | ((bq >> 2) & 0x00300030u);
      sc = pp == 2 ? sc23 & 0xFFu : sc23 >> 16;
      mn = pp == 2 ? mn23 & 0xFFu : mn23 >> 16;
    }
    const float dd = h2f(r.hd.x & 0xFFFFu) * kPfScale, dmin = h2f(r.hd.x >> 16) * -kPfScale;
    S = pf_bcast(dd * (float)sc);
    O = pf_bcast(dmin * (float)mn);
  }
}

__device__ __forceinline__ h16x8 pf_join4(h16x2 w0, h16x2 w1, h16x2 w2, h16x2 w3) {
  const h16x8 r = {w0.x, w0.y, w1.x, w1.y, w2.x, w2.y, w3.x, w3.y};
  return r;
}

// four words of two f16 (0x6400 | u == 1024 + u exactly) -> S * u + O.  Stage by stage over the four words (not word by
// word): a packed-f16 op that consumes the previous instruction's result costs an extra s_nop on gfx950.
__device__ __forceinline__ h16x8 pf_fin4(uint32_t b0, uint32_t b1, uint32_t b2, uint32_t b3, h16x2 S, h16x2 O) {
  const h16x2 k = {(_Float16)1024.0f, (_Float16)1024.0f};
  const h16x2 u0 = __builtin_bit_cast(h16x2, b0) - k, u1 = __builtin_bit_cast(h16x2, b1) - k;
  const h16x2 u2 = __builtin_bit_cast(h16x2, b2) - k, u3 = __builtin_bit_cast(h16x2, b3) - k;
  const h16x2 w0 = __builtin_elementwise_fma(u0, S, O), w1 = __builtin_elementwise_fma(u1, S, O);
  const h16x2 w2 = __builtin_elementwise_fma(u2, S, O), w3 = __builtin_elementwise_fma(u3, S, O);
  return pf_join4(w0, w1, w2, w3);
}

// eight nibbles (word byte t = w[t] | w[t+4] << 4) -> f16.  A byte up to 16 is, as an 8-bit float, 2^-9 of itself: two whole numbers a conversion, 11 instructions for eight weights
// (with masks and an exponent, (x & m) | 0x6400 - 1024, 15).  The products' loops are bound by the sum of their matrix and vector instructions, about two of the latter a 16 x 16 matrix
// instruction hidden: 2047 tokens of 16 layers of an 8B model in Q4_K_M 17.2 -> 16.9 ms, 128 of 32 layers 6.00 -> 5.91
__device__ __forceinline__ h16x8 pf_frag_nib(uint32_t N, h16x2 S, h16x2 O) {
  const uint32_t m = 0x0F0F0F0Fu, lo = N & m, hi = (N >> 4) & m;
  auto two = [](uint32_t b, auto up) { return __builtin_bit_cast(h16x2, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(b, 512.0f, up.value)); };
  const h16x2 u0 = two(lo, std::false_type{}), u1 = two(lo, std::true_type{}), u2 = two(hi, std::false_type{}), u3 = two(hi, std::true_type{});
  return pf_join4(__builtin_elementwise_fma(u0, S, O), __builtin_elementwise_fma(u1, S, O), __builtin_elementwise_fma(u2, S, O), __builtin_elementwise_fma(u3, S, O));
}
// eight bytes (B0 = w0..w3, B1 = w4..w7) -> f16
__device__ __forceinline__ h16x8 pf_frag_bytes(uint32_t B0, uint32_t B1, h16x2 S, h16x2 O) {
  const uint32_t e = 0x64646464u;
  return pf_fin4(__builtin_amdgcn_perm(e, B0, 0x04010400u), __builtin_amdgcn_perm(e, B0, 0x04030402u),
                 __builtin_amdgcn_perm(e, B1, 0x04010400u), __builtin_amdgcn_perm(e, B1, 0x04030402u), S, O);
}

// the A operand of MFMA (pp, h): elements 64pp + 16c + 8h .. +7 of row n, dequantized
template <int F>
__device__ __forceinline__ h16x8 pf_frag(const PfRaw& r, int pp, int h, h16x2 S, h16x2 O) {
  if (F == PF_Q80) {
    const u32x4 b = r.q[pp];
    const uint32_t B0 = (h ? b.z : b.x) ^ 0x80808080u, B1 = (h ? b.w : b.y) ^ 0x80808080u;
    return pf_frag_bytes(B0, B1, S, O);
  }
  const uint32_t N0 = (pp & 1) ? r.q[pp >> 1].z : r.q[pp >> 1].x, N1 = (pp & 1) ? r.q[pp >> 1].w : r.q[pp >> 1].y;
  const uint32_t N = h ? N1 : N0;
  if (F == PF_Q4K || F == PF_Q40) return pf_frag_nib(N, S, O);
  uint32_t B0 = N & 0x0F0F0F0Fu, B1 = (N >> 4) & 0x0F0F0F0Fu;
  if (F == PF_Q6K) {   // H byte t = f[t] | f[t+4] << 2 | f[t+8] << 4 | f[t+12] << 6 (the two high bits of the chunk's 16 weights)
    const uint32_t H = pp == 0 ? r.q[2].x : pp == 1 ? r.q[2].y : pp == 2 ? r.q[2].z : r.q[2].w;
    B0 |= ((H >> (4 * h)) & 0x03030303u) << 4;
    B1 |= ((H >> (4 * h + 2)) & 0x03030303u) << 4;
  } else {             // Q5_K: fifth bits, dword of the step pair, low nibbles = even step, high nibbles = odd step
    const uint32_t H = ((pp >> 1) ? r.q[2].y : r.q[2].x) >> (4 * (pp & 1));
    B0 |= ((H >> (2 * h)) & 0x01010101u) << 4;
    B1 |= ((H >> (2 * h + 1)) & 0x01010101u) << 4;
  }
  return pf_frag_bytes(B0, B1, S, O);
}

}  // namespace lgh
