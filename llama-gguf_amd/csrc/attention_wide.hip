// attention_wide.hip — causal attention of long prompt blocks (prefill_wide.hip) over the f32 cache, on the bf16 matrix cores.
//
// Every f32 operand is taken as three bf16 numbers, x = hi + mid + lo, each the rest of the one before rounded to 8 bits: all 24 bits of x, at f32's own exponents,
// so that what a row, a tile or a later token holds changes nothing for any other.  Six products (hi hi, hi mid, mid hi, mid mid, hi lo, lo hi) of v_mfma_f32_16x16x32_bf16
// with f32 accumulation stand for the f32 product; the three left out are 2^-24 of it together at most, what one f32 rounding may do.  (An infinity becomes a NaN.)
// The output is rounded to f16 (2^-12), as in the 128-token blocks.
//
// attn_wide_split_kernel lays the layer's rows out once, in the order in which a workgroup's LDS wants them (one verbatim copy per half tile); the f32
// kernel (attention.hip) reads and uses them as they are, once per 16 tokens and query head.
// Measured: 2047 tokens, 32 query heads on 8 of 128 dims: 523 us a layer with the f32 kernel, 209 + 11 us for the rows here, bound by the matrix products.  (Two f16 limbs
// under an exponent per tile take 139 + 8: they lose what lies far below its tile's largest value, whole weights where a tile's values do.)  Error against 64 bits, 2-norm, random
// inputs of 129 to 1000 rows: 2.3e-7 to 4.8e-7; an emulation of the f32 kernel's order of sums 4.5e-7 to 7.2e-7 on the same inputs.
#include <algorithm>

#include "device_utils.h"
#include "prefill.h"

namespace lgh {

typedef _Float16 h16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 b16x8 __attribute__((ext_vector_type(8)));

constexpr uint32_t kAwRows = 32;                                  // cached rows of a tile
constexpr float kAwNeg = -1.0e30f;
template <int D> constexpr uint32_t aw_limb() { return kAwRows * D * 2; }
template <int D> constexpr uint32_t aw_half() { return 3 * aw_limb<D>(); }   // a tile's K, or its V: hi | mid | lo
template <int D> constexpr uint32_t aw_tile() { return 2 * aw_half<D>(); }

struct AwLimbs { b16x8 l[3]; };   // of eight values
__device__ __forceinline__ AwLimbs aw_split8(const float* v) {
  AwLimbs o;
#pragma unroll
  for (int j = 0; j < 8; j++) {
    o.l[0][j] = (__bf16)v[j];
    const float r = v[j] - (float)o.l[0][j];
    o.l[1][j] = (__bf16)r;
    o.l[2][j] = (__bf16)(r - (float)o.l[1][j]);
  }
  return o;
}
// acc[t] += a b[t] but for hi hi (small products first, the two tiles' in turn); acc[t] += hi hi
__device__ __forceinline__ void aw_mma_rest(f32x4 (&acc)[2], const AwLimbs& a, const AwLimbs& b0, const AwLimbs& b1) {
  constexpr int la[5] = {2, 1, 0, 1, 0}, lb[5] = {0, 1, 2, 0, 1};
#pragma unroll
  for (int i = 0; i < 5; i++) {
    acc[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.l[la[i]], b0.l[lb[i]], acc[0], 0, 0, 0);
    acc[1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.l[la[i]], b1.l[lb[i]], acc[1], 0, 0, 0);
  }
}
__device__ __forceinline__ void aw_mma_hi(f32x4 (&acc)[2], b16x8 a, const AwLimbs& b0, const AwLimbs& b1) {
  acc[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b0.l[0], acc[0], 0, 0, 0);
  acc[1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b1.l[0], acc[1], 0, 0, 0);
}

// One tile of one kv head.  K: row r, 16-byte chunk q of it at q ^ (r & 7); V transposed: dim d's 32 rows in the order in which a lane of the score
// product holds them (slot 8c + j: row 4c + j, or 16 + 4c + j - 4), chunk c at c ^ (d >> 1 & 3): the reads of a fragment touch every bank once.
template <int D>
__global__ void __launch_bounds__(256) attn_wide_split_kernel(const float* __restrict__ kc, const float* __restrict__ vc, uint32_t max_seq, uint32_t kv_len,
                                                              uint32_t tiles, uint8_t* __restrict__ out) {
  constexpr int U = kAwRows * D / 8 / 256;   // chunks per thread
  const uint32_t t = blockIdx.x, h = blockIdx.y, r0 = t * kAwRows;
  const float* kp = kc + (size_t)h * max_seq * D;
  const float* vp = vc + (size_t)h * max_seq * D;
  float k[U][8], v[U][8];
#pragma unroll
  for (int u = 0; u < U; u++) {
    const uint32_t i = u * 256 + threadIdx.x, r = r0 + i / (D / 8), q = i % (D / 8);
    const float* p = kp + (size_t)(r < kv_len ? r : kv_len - 1) * D + q * 8;
    const f32x4 a = *reinterpret_cast<const f32x4*>(p), b = *reinterpret_cast<const f32x4*>(p + 4);
    const uint32_t d = i % D, c = i / D;
#pragma unroll
    for (int j = 0; j < 8; j++) {
      k[u][j] = r < kv_len ? (j < 4 ? a[j & 3] : b[j & 3]) : 0.0f;
      const uint32_t vr = r0 + (j < 4 ? 4 * c + j : 12 + 4 * c + j);
      const float x = vp[(size_t)(vr < kv_len ? vr : kv_len - 1) * D + d];
      v[u][j] = vr < kv_len ? x : 0.0f;
    }
  }
  uint8_t* o = out + ((size_t)h * tiles + t) * aw_tile<D>();
#pragma unroll
  for (int u = 0; u < U; u++) {
    const uint32_t i = u * 256 + threadIdx.x, r = i / (D / 8), q = i % (D / 8), d = i % D, c = i / D;
    const AwLimbs kl = aw_split8(k[u]), vl = aw_split8(v[u]);
#pragma unroll
    for (int l = 0; l < 3; l++) {
      *reinterpret_cast<b16x8*>(o + l * aw_limb<D>() + r * D * 2 + ((q ^ (r & 7)) << 4)) = kl.l[l];
      *reinterpret_cast<b16x8*>(o + aw_half<D>() + l * aw_limb<D>() + d * 64 + ((c ^ (d >> 1 & 3)) << 4)) = vl.l[l];
    }
  }
}

// A workgroup: one kv head, up to four of its query heads, 128 (token, head) rows: a wave has two tiles of 16 tokens of one head.  S^T = K Q^T leaves a
// lane with the scores of one token and eight of a tile's rows, which is the operand of O^T += V^T P^T: weights never leave their registers.  K and V of a tile of
// 32 rows arrive by DMA in turn, through a ring of three buffers, each requested while the one two before it is used up.  Two workgroups share a CU (72 KB of LDS each at 128 dims).
// Few tokens behind many rows leave the chip idle: grid y = splits of the tiles, each leaving its sums, maximum and weight of every (token, head) to attn_wide_merge_kernel.
// OUT: f16 rows to out, f32 rows to part (unrounded sums), or a split's parts to part and ml.
enum : int { AW_F16 = 0, AW_F32 = 1, AW_PART = 2 };
template <int D, int OUT>
__global__ void __launch_bounds__(256, 2) attn_wide_kernel(const float* __restrict__ q, const uint8_t* __restrict__ kv, uint32_t n_heads, uint32_t g, uint32_t tiles,
                                                           float scale, uint32_t pos0, uint32_t m_tokens, uint32_t n_blk, uint32_t paired, uint8_t* __restrict__ out,
                                                           float* __restrict__ part, float* __restrict__ ml) {
  constexpr int KK = D / 32, DT = D / 16;
  constexpr uint32_t LIMB = aw_limb<D>(), HALF = aw_half<D>(), OPS = HALF / 4096;   // DMA operations of a wave per half tile
  extern __shared__ __attribute__((aligned(16))) uint8_t aw_lds[];
  const uint32_t lane = threadIdx.x & 63, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), n = lane & 15, c = lane >> 4;
  const uint32_t gw = g < 4 ? g : 4, per = n_heads / gw;                  // heads of a workgroup; workgroups per token block
  const uint32_t hw = blockIdx.x % per, idx = blockIdx.x / per;           // its heads hw * gw .. + gw - 1
  // token blocks: the longest first; with every workgroup resident at once, the second half in rising order, so that a CU's two add up to the same work
  const uint32_t blk = paired && idx >= n_blk / 2 ? idx - n_blk / 2 : n_blk - 1 - idx;
  const uint32_t head = hw * gw + wave % gw, kvh = head / g;
  const uint32_t tok0 = blk * (128 / gw) + wave / gw * 32;                // the wave's first token
  const uint32_t last_blk = min(blk * (128 / gw) + 128 / gw, m_tokens) - 1, n_tiles = (pos0 + last_blk) / kAwRows + 1;
  const uint32_t sp = blockIdx.y, first = n_tiles * sp / gridDim.y * 2, last = n_tiles * (sp + 1) / gridDim.y * 2;   // its half tiles (no split is empty: attn_wide_splits)
  const uint32_t last_wave = min(tok0 + 31, m_tokens - 1);
  const uint8_t* src = kv + (size_t)kvh * tiles * aw_tile<D>() + lane * 16;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)aw_lds;
  auto dma = [&](uint32_t h, uint32_t buf) {                              // half tile h
#pragma unroll
    for (uint32_t i = 0; i < OPS; i++) {
      const uint32_t at = (i * 4 + wave) * 1024;
      uint32_t keep;
      asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off\n\ts_mov_b32 m0, %0"
                   : "=&s"(keep) : "v"(src + (size_t)h * HALF + at), "s"(lds0 + buf * HALF + at) : "memory");
    }
  };
  AwLimbs ql[2][KK];
#pragma unroll
  for (int t = 0; t < 2; t++) {
    const uint32_t tok = min(tok0 + t * 16 + n, m_tokens - 1);
    const float* p = q + ((size_t)tok * n_heads + head) * D + c * 8;
#pragma unroll
    for (int k = 0; k < KK; k++) {
      const f32x4 a = *reinterpret_cast<const f32x4*>(p + k * 32), b = *reinterpret_cast<const f32x4*>(p + k * 32 + 4);
      const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
      ql[t][k] = aw_split8(v);
    }
  }
  dma(first, 0);
  dma(first + 1, 1);
  const float f = scale * 1.44269504088896f;                              // scores in units of log2
  f32x4 acc[DT][2];
  float m_run[2] = {kAwNeg, kAwNeg}, l_run[2] = {0.0f, 0.0f};
#pragma unroll
  for (int x = 0; x < DT; x++) acc[x][0] = acc[x][1] = (f32x4)(0.0f);

  // half tile h is there (its wave's operations; only those of the next one may be under way), every wave is done with the one before: its buffer takes the one after the next
  auto arrive = [&](uint32_t h, uint32_t free_buf) {
    if (h + 1 < last) __builtin_amdgcn_s_waitcnt(0x0070 | OPS);         // vmcnt(OPS) lgkmcnt(0)
    else __builtin_amdgcn_s_waitcnt(0x0070);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (h + 2 < last) dma(h + 2, free_buf);
  };
  const uint32_t k_off = n * D * 2, v_off = n * 64 + ((c ^ (n >> 1 & 3)) << 4);
  uint32_t kb = 0, vb = 1, fb = 2;                                        // buffers of this tile's K and V, and the third
  for (uint32_t h = first; h < last; h += 2) {
    const uint32_t kv0 = h / 2 * kAwRows;
    const bool seen = kv0 <= pos0 + last_wave;                            // something of the tile is visible to this wave
    arrive(h, fb);
    AwLimbs pl[2];
    if (seen) {
      const uint8_t* kt = aw_lds + kb * HALF;
      f32x4 st[2][2];   // [rows 16 * i ..][token tile]
#pragma unroll
      for (int i = 0; i < 2; i++) {
        st[i][0] = st[i][1] = (f32x4)(0.0f);
#pragma unroll
        for (int k = 0; k < KK; k++) {
          const uint8_t* p = kt + i * 16 * D * 2 + k_off + (((uint32_t)(k * 4 + c) ^ (n & 7)) << 4);
          AwLimbs a;
#pragma unroll
          for (int l = 0; l < 3; l++) a.l[l] = *reinterpret_cast<const b16x8*>(p + l * LIMB);
          aw_mma_rest(st[i], a, ql[0][k], ql[1][k]);
        }
        // the large products last: a sum as large as the score is rounded D / 32 times
#pragma unroll
        for (int k = 0; k < KK; k++)
          aw_mma_hi(st[i], *reinterpret_cast<const b16x8*>(kt + i * 16 * D * 2 + k_off + (((uint32_t)(k * 4 + c) ^ (n & 7)) << 4)), ql[0][k], ql[1][k]);
      }
#pragma unroll
      for (int t = 0; t < 2; t++) {
        float s[8], mx = kAwNeg;
#pragma unroll
        for (int j = 0; j < 8; j++) s[j] = st[j >> 2][t][j & 3] * f;
        if (kv0 + kAwRows - 1 > pos0 + tok0 + t * 16) {                    // the diagonal: row 4c + j (16 + ...) against the token
          const uint32_t tok = tok0 + t * 16 + n;
#pragma unroll
          for (int j = 0; j < 8; j++) s[j] = kv0 + (j >> 2) * 16 + 4 * c + (j & 3) <= pos0 + tok ? s[j] : kAwNeg;
        }
#pragma unroll
        for (int j = 0; j < 8; j++) mx = fmaxf(mx, s[j]);
        mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        if (__any(mx > m_run[t])) {                                        // (rare after the first tiles)
          const float mn = fmaxf(m_run[t], mx), alpha = __builtin_amdgcn_exp2f(m_run[t] - mn);
          m_run[t] = mn;
          l_run[t] *= alpha;
#pragma unroll
          for (int x = 0; x < DT; x++) acc[x][t] = acc[x][t] * alpha;
        }
        float ps = 0.0f;
#pragma unroll
        for (int j = 0; j < 8; j++) { s[j] = __builtin_amdgcn_exp2f(s[j] - m_run[t]); ps += s[j]; }
        l_run[t] += ps;                                                    // (this lane's rows: the lanes of a token meet at the end)
        pl[t] = aw_split8(s);
      }
    }
    arrive(h + 1, kb);
    if (seen) {
      const uint8_t* vt = aw_lds + vb * HALF;
#pragma unroll
      for (int x = 0; x < DT; x++) {
        const uint8_t* p = vt + v_off + x * 1024;
        AwLimbs a;
#pragma unroll
        for (int l = 0; l < 3; l++) a.l[l] = *reinterpret_cast<const b16x8*>(p + l * LIMB);
        aw_mma_rest(acc[x], a, pl[0], pl[1]);
        aw_mma_hi(acc[x], a.l[0], pl[0], pl[1]);
      }
    }
    const uint32_t k0 = kb;
    kb = fb;
    fb = vb;
    vb = k0;
  }
#pragma unroll
  for (int t = 0; t < 2; t++) {
    float l = l_run[t];
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    const uint32_t tok = tok0 + t * 16 + n;
    if (tok >= m_tokens) continue;
    const size_t row = ((size_t)(OUT == AW_PART ? sp * m_tokens : 0) + tok) * n_heads + head, at = row * D + c * 4;
    const float inv = OUT == AW_PART ? 1.0f : 1.0f / l;
    if (OUT == AW_PART && c == 0) { ml[row * 2] = m_run[t]; ml[row * 2 + 1] = l; }
#pragma unroll
    for (int x = 0; x < DT; x++) {                                         // dims 16 x + 4c .. + 3
      const f32x4 v = acc[x][t] * inv;
      if constexpr (OUT != AW_F16) {
        *reinterpret_cast<f32x4*>(part + at + x * 16) = v;
      } else {
        const h16x4 w = {(_Float16)v.x, (_Float16)v.y, (_Float16)v.z, (_Float16)v.w};
        *reinterpret_cast<h16x4*>(out + (at + x * 16) * 2) = w;
      }
    }
  }
}

// splits of a (token, head) -> its row.  A split that the token sees nothing of has the maximum kAwNeg: its parts count for nothing.
template <int D>
__global__ void __launch_bounds__(256) attn_wide_merge_kernel(const float* __restrict__ part, const float* __restrict__ ml, uint32_t n_rows, uint32_t n_splits,
                                                              uint8_t* __restrict__ out, float* __restrict__ out32) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x, row = i / (D / 4), q = i % (D / 4);
  if (row >= n_rows) return;
  float mn = kAwNeg, l = 0.0f;
  for (uint32_t s = 0; s < n_splits; s++) mn = fmaxf(mn, ml[((size_t)s * n_rows + row) * 2]);
  f32x4 v = (f32x4)(0.0f);
  for (uint32_t s = 0; s < n_splits; s++) {
    const size_t r = (size_t)s * n_rows + row;
    const float f = __builtin_amdgcn_exp2f(ml[r * 2] - mn);
    l += ml[r * 2 + 1] * f;
    v += *reinterpret_cast<const f32x4*>(part + r * D + q * 4) * f;
  }
  v *= 1.0f / l;
  if (out32) {
    *reinterpret_cast<f32x4*>(out32 + (size_t)row * D + q * 4) = v;
  } else {
    const h16x4 w = {(_Float16)v.x, (_Float16)v.y, (_Float16)v.z, (_Float16)v.w};
    *reinterpret_cast<h16x4*>(out + ((size_t)row * D + q * 4) * 2) = w;
  }
}

uint32_t attn_wide_tiles(uint32_t rows) { return (rows + kAwRows - 1) / kAwRows; }
size_t attn_wide_bytes(uint32_t n_kv, uint32_t head_dim, uint32_t rows) {
  return (size_t)n_kv * attn_wide_tiles(rows) * (head_dim == 128 ? aw_tile<128>() : aw_tile<64>());
}

// Splits of a launch of `wgs` workgroups: until two a CU are there, none of fewer than 8 tiles nor without one (the first token block's tiles end behind pos0).  256 tokens of an 8B
// model are 64 workgroups, and behind many rows each walked them all: 256 tokens behind 1000 / 4000 / 16000 rows, 4 layers, 1059 / 1805 / 4741 us, with splits 948 / 1140 / 1911
// (blocks of 128 with the f32 kernel 1120 / 1497 / 3142); of 16 tiles or more each 1109 behind 1000.
static uint32_t attn_wide_splits(uint32_t wgs, uint32_t pos0, uint32_t m_tokens, uint32_t n_heads, uint32_t head_dim, size_t part_floats) {
  const size_t room = part_floats / ((size_t)m_tokens * n_heads * (head_dim + 2));
  const uint32_t s = std::min({2u * kNumCU / wgs, pos0 / kAwRows / 8, (uint32_t)std::min<size_t>(room, 16)});
  return s > 1 ? s : 1;
}

template <int D, int OUT>
static hipError_t attn_wide_run(const float* q, const uint8_t* kv, uint32_t n_heads, uint32_t g, uint32_t tiles, float scale, uint32_t pos0, uint32_t m_tokens, uint32_t n_blk,
                                uint32_t wgs, uint32_t splits, uint8_t* out, float* part, float* ml, hipStream_t st) {
  static bool attr_set[64] = {};
  constexpr uint32_t lds = 3 * aw_half<D>();
  if (hipError_t e = lds_opt_in(reinterpret_cast<const void*>(&attn_wide_kernel<D, OUT>), (int)lds, attr_set); e != hipSuccess) return e;
  hipLaunchKernelGGL((attn_wide_kernel<D, OUT>), dim3(wgs, splits), dim3(256), lds, st, q, kv, n_heads, g, tiles, scale, pos0, m_tokens, n_blk,
                     (uint32_t)(wgs <= 2u * kNumCU), out, part, ml);
  return hipGetLastError();
}

template <int D>
static hipError_t attn_wide_go(const float* q, const float* kc, const float* vc, uint32_t n_heads, uint32_t n_kv, uint32_t max_seq, float scale, uint32_t pos0,
                               uint32_t m_tokens, uint8_t* scratch, float* part, size_t part_floats, uint8_t* out, hipStream_t st, float* out32) {
  const uint32_t kv_len = pos0 + m_tokens, tiles = attn_wide_tiles(kv_len), g = n_heads / n_kv, gw = g < 4 ? g : 4;
  hipLaunchKernelGGL((attn_wide_split_kernel<D>), dim3(tiles, n_kv), dim3(256), 0, st, kc, vc, max_seq, kv_len, tiles, scratch);
  const uint32_t n_blk = (m_tokens + 128 / gw - 1) / (128 / gw), wgs = n_blk * (n_heads / gw);
  const uint32_t splits = attn_wide_splits(wgs, pos0, m_tokens, n_heads, D, part_floats), rows = m_tokens * n_heads;
  if (splits == 1)
    return out32 ? attn_wide_run<D, AW_F32>(q, scratch, n_heads, g, tiles, scale, pos0, m_tokens, n_blk, wgs, 1, nullptr, out32, nullptr, st)
                 : attn_wide_run<D, AW_F16>(q, scratch, n_heads, g, tiles, scale, pos0, m_tokens, n_blk, wgs, 1, out, nullptr, nullptr, st);
  float* ml = part + (size_t)splits * rows * D;
  if (hipError_t e = attn_wide_run<D, AW_PART>(q, scratch, n_heads, g, tiles, scale, pos0, m_tokens, n_blk, wgs, splits, nullptr, part, ml, st); e != hipSuccess) return e;
  hipLaunchKernelGGL((attn_wide_merge_kernel<D>), dim3((rows * (D / 4) + 255) / 256), dim3(256), 0, st, part, ml, rows, splits, out, out32);
  return hipGetLastError();
}

// scratch: attn_wide_bytes(n_kv, head_dim, pos0 + m_tokens); part: memory for splits (a launch without it has one).  out: row-major f16 [token][head][dim] in XH's element
// order; or out32, f32 in plain order
hipError_t attn_wide_launch(const float* q, const float* kcache, const float* vcache, uint32_t n_heads, uint32_t n_kv, uint32_t head_dim, uint32_t max_seq, float scale,
                            uint32_t pos0, uint32_t m_tokens, uint8_t* scratch, float* part, size_t part_bytes, uint8_t* out, hipStream_t st, float* out32) {
  if (n_kv == 0 || n_heads % n_kv || m_tokens == 0 || (head_dim != 64 && head_dim != 128) || pos0 + m_tokens > max_seq || n_kv > 65535 || (!out && !out32)) return hipErrorInvalidValue;
  const uint32_t g = n_heads / n_kv;
  if (g != 1 && g != 2 && g != 4 && g != 8) return hipErrorInvalidValue;
  if ((size_t)m_tokens * n_heads * 32 > 0xFFFFFFFFull) return hipErrorInvalidValue;   // (the merge's threads)
  return head_dim == 128 ? attn_wide_go<128>(q, kcache, vcache, n_heads, n_kv, max_seq, scale, pos0, m_tokens, scratch, part, part ? part_bytes / 4 : 0, out, st, out32)
                         : attn_wide_go<64>(q, kcache, vcache, n_heads, n_kv, max_seq, scale, pos0, m_tokens, scratch, part, part ? part_bytes / 4 : 0, out, st, out32);
}

}  // namespace lgh
