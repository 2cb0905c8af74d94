// attention_wide.hip — causal attention of long prompt blocks (prefill_wide.hip) over the f32 cache, on the f16 matrix cores.
//
// Every f32 operand is taken as two f16 numbers, x = 2^e (hi + lo): 22 bits, against the 24 of f32.  e is one exponent per tile of 32 cached rows (K and V
// each), per row of q, and a constant for the softmax weights, so that a tile's largest value lies just under 2^14: values down to 2^-16 of it keep
// all 22 bits, smaller ones an absolute error of 2^-38 of it.  Three products (hi hi, hi lo, lo hi) of v_mfma_f32_16x16x32_f16 with f32 accumulation stand for one of
// v_mfma_f32_16x16x4_f32, at a fifth of its time.  Against 64 bits the emulated attention of 2047 random positions is 3.1e-7 off with these sums and 4.6e-7 with the f32
// form (a product of 32 terms is rounded once, not eight times); the output is rounded to f16 (2e-4) either way.
//
// attn_wide_split_kernel lays the layer's rows out once, in the order in which a workgroup's LDS wants them (one verbatim copy per tile); the f32
// kernel (attention.hip) read and used them as they are, once per 16 tokens and query head.
// Measured: 2047 tokens, 32 query heads on 8 of 128 dims: 523 -> 127 us a layer + 8 us for the rows (bound by matrix and vector issue in turn); 2047 tokens
// of Llama-3-8B widths, 16 layers, 23.8 -> 18.0 ms.
#include "device_utils.h"
#include "prefill.h"

namespace lgh {

typedef _Float16 h16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 h16x4 __attribute__((ext_vector_type(4)));

constexpr uint32_t kAwRows = 32;                                  // cached rows of a tile
constexpr float kAwNeg = -1.0e30f;
template <int D> constexpr uint32_t aw_limb() { return kAwRows * D * 2; }
template <int D> constexpr uint32_t aw_tile() { return 4 * aw_limb<D>(); }   // K hi | K lo | V hi | V lo

// hi and lo of eight values
__device__ __forceinline__ void aw_split8(const float* v, float scale, h16x8& hi, h16x8& lo) {
#pragma unroll
  for (int j = 0; j < 8; j++) {
    const float x = v[j] * scale;
    hi[j] = (_Float16)x;
    lo[j] = (_Float16)(x - (float)hi[j]);
  }
}
// exponent e with m < 2^e; nothing but zeros: far below any other
__device__ __forceinline__ int aw_exponent(float m) { return m > 0.0f ? max(__builtin_amdgcn_frexp_expf(m), -100) : -100; }
__device__ __forceinline__ float aw_pow2(int e) { return __builtin_ldexpf(1.0f, e); }

// One tile of one kv head.  K: row r, 16-byte chunk q of it at q ^ (r & 7); V transposed: dim d's 32 rows in the order in which a lane of the score
// product holds them (slot 8c + j: row 4c + j, or 16 + 4c + j - 4), chunk c at c ^ (d >> 1 & 3): the reads of a fragment touch every bank once.
template <int D>
__global__ void __launch_bounds__(256) attn_wide_split_kernel(const float* __restrict__ kc, const float* __restrict__ vc, uint32_t max_seq, uint32_t kv_len,
                                                              uint32_t tiles, uint8_t* __restrict__ out, int* __restrict__ exps) {
  constexpr int U = kAwRows * D / 8 / 256;   // chunks per thread
  __shared__ float red[8];
  const uint32_t t = blockIdx.x, h = blockIdx.y, r0 = t * kAwRows;
  const float* kp = kc + (size_t)h * max_seq * D;
  const float* vp = vc + (size_t)h * max_seq * D;
  float k[U][8], v[U][8], km = 0.0f, vm = 0.0f;
#pragma unroll
  for (int u = 0; u < U; u++) {
    const uint32_t i = u * 256 + threadIdx.x, r = r0 + i / (D / 8), q = i % (D / 8);
    const float* p = kp + (size_t)(r < kv_len ? r : kv_len - 1) * D + q * 8;
    const f32x4 a = *reinterpret_cast<const f32x4*>(p), b = *reinterpret_cast<const f32x4*>(p + 4);
    const uint32_t d = i % D, c = i / D;
#pragma unroll
    for (int j = 0; j < 8; j++) {
      k[u][j] = r < kv_len ? (j < 4 ? a[j & 3] : b[j & 3]) : 0.0f;
      km = fmaxf(km, fabsf(k[u][j]));
      const uint32_t vr = r0 + (j < 4 ? 4 * c + j : 12 + 4 * c + j);
      const float x = vp[(size_t)(vr < kv_len ? vr : kv_len - 1) * D + d];
      v[u][j] = vr < kv_len ? x : 0.0f;
      vm = fmaxf(vm, fabsf(v[u][j]));
    }
  }
  km = wave_max(km);
  vm = wave_max(vm);
  if ((threadIdx.x & 63) == 0) { red[threadIdx.x >> 6] = km; red[4 + (threadIdx.x >> 6)] = vm; }
  __syncthreads();
  const int ek = aw_exponent(fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]))), ev = aw_exponent(fmaxf(fmaxf(red[4], red[5]), fmaxf(red[6], red[7])));
  if (threadIdx.x == 0) { exps[((size_t)h * tiles + t) * 2] = ek; exps[((size_t)h * tiles + t) * 2 + 1] = ev; }
  uint8_t* o = out + ((size_t)h * tiles + t) * aw_tile<D>();
#pragma unroll
  for (int u = 0; u < U; u++) {
    const uint32_t i = u * 256 + threadIdx.x, r = i / (D / 8), q = i % (D / 8), d = i % D, c = i / D;
    h16x8 hi, lo;
    aw_split8(k[u], aw_pow2(14 - ek), hi, lo);
    *reinterpret_cast<h16x8*>(o + r * D * 2 + ((q ^ (r & 7)) << 4)) = hi;
    *reinterpret_cast<h16x8*>(o + aw_limb<D>() + r * D * 2 + ((q ^ (r & 7)) << 4)) = lo;
    aw_split8(v[u], aw_pow2(14 - ev), hi, lo);
    *reinterpret_cast<h16x8*>(o + 2 * aw_limb<D>() + d * 64 + ((c ^ (d >> 1 & 3)) << 4)) = hi;
    *reinterpret_cast<h16x8*>(o + 3 * aw_limb<D>() + d * 64 + ((c ^ (d >> 1 & 3)) << 4)) = lo;
  }
}

// A workgroup: one kv head, up to four of its query heads, 128 (token, head) rows: a wave has two tiles of 16 tokens of one head.  S^T = K Q^T leaves a
// lane with the scores of one token and eight of a tile's rows, which is the operand of O^T += V^T P^T: weights never leave their registers.  Tiles of
// 32 rows arrive by DMA in two buffers, the next one during a tile's products.  Two workgroups share a CU (64 KB of LDS each at 128 dims).
template <int D>
__global__ void __launch_bounds__(256, 2) attn_wide_kernel(const float* __restrict__ q, const uint8_t* __restrict__ kv, const int* __restrict__ exps, uint32_t n_heads,
                                                           uint32_t g, uint32_t tiles, float scale, uint32_t pos0, uint32_t m_tokens, uint32_t n_blk, uint32_t paired,
                                                           uint8_t* __restrict__ out) {
  constexpr int KK = D / 32, DT = D / 16;
  constexpr uint32_t LIMB = aw_limb<D>(), TB = aw_tile<D>(), OPS = TB / 4096;   // DMA operations of a wave per tile
  extern __shared__ __attribute__((aligned(16))) uint8_t aw_lds[];
  const uint32_t lane = threadIdx.x & 63, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), n = lane & 15, c = lane >> 4;
  const uint32_t gw = g < 4 ? g : 4, per = n_heads / gw;                  // heads of a workgroup; workgroups per token block
  const uint32_t hw = blockIdx.x % per, idx = blockIdx.x / per;           // its heads hw * gw .. + gw - 1
  // token blocks: the longest first; with every workgroup resident at once, the second half in rising order, so that a CU's two add up to the same work
  const uint32_t blk = paired && idx >= n_blk / 2 ? idx - n_blk / 2 : n_blk - 1 - idx;
  const uint32_t head = hw * gw + wave % gw, kvh = head / g;
  const uint32_t tok0 = blk * (128 / gw) + wave / gw * 32;                // the wave's first token
  const uint32_t last_blk = min(blk * (128 / gw) + 128 / gw, m_tokens) - 1, n_tiles = (pos0 + last_blk) / kAwRows + 1;
  const uint32_t last_wave = min(tok0 + 31, m_tokens - 1);
  const uint8_t* src = kv + (size_t)kvh * tiles * TB + lane * 16;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)aw_lds;
  auto dma = [&](uint32_t t, uint32_t buf) {
#pragma unroll
    for (uint32_t i = 0; i < OPS; i++) {
      const uint32_t at = (i * 4 + wave) * 1024;
      uint32_t keep;
      asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off\n\ts_mov_b32 m0, %0"
                   : "=&s"(keep) : "v"(src + (size_t)t * TB + at), "s"(lds0 + buf * TB + at) : "memory");
    }
  };
  dma(0, 0);
  const int* ex = exps + (size_t)kvh * tiles * 2;
  int vmax = -100;                                                        // the largest V exponent in sight: the sums' common one
  for (uint32_t t = lane; t < n_tiles; t += 64) vmax = max(vmax, ex[t * 2 + 1]);
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) vmax = max(vmax, __shfl_xor(vmax, o, 64));
  vmax = __builtin_amdgcn_readfirstlane(vmax);

  h16x8 qh[2][KK], ql[2][KK];
  float qf[2];                                                            // what a raw score times 2^ek is multiplied by
#pragma unroll
  for (int t = 0; t < 2; t++) {
    const uint32_t tok = min(tok0 + t * 16 + n, m_tokens - 1);
    const float* p = q + ((size_t)tok * n_heads + head) * D + c * 8;
    float v[KK][8], mx = 0.0f;
#pragma unroll
    for (int k = 0; k < KK; k++) {
      const f32x4 a = *reinterpret_cast<const f32x4*>(p + k * 32), b = *reinterpret_cast<const f32x4*>(p + k * 32 + 4);
#pragma unroll
      for (int j = 0; j < 8; j++) { v[k][j] = j < 4 ? a[j & 3] : b[j & 3]; mx = fmaxf(mx, fabsf(v[k][j])); }
    }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const int e = aw_exponent(mx);
#pragma unroll
    for (int k = 0; k < KK; k++) aw_split8(v[k], aw_pow2(14 - e), qh[t][k], ql[t][k]);
    qf[t] = aw_pow2(e - 28) * (scale * 1.44269504088896f);                // scores in units of log2
  }
  f32x4 acc[2][DT];
  float m_run[2] = {kAwNeg, kAwNeg}, l_run[2] = {0.0f, 0.0f};
#pragma unroll
  for (int t = 0; t < 2; t++)
#pragma unroll
    for (int x = 0; x < DT; x++) acc[t][x] = (f32x4)(0.0f);

  const uint32_t k_off = n * D * 2, v_off = 2 * LIMB + n * 64 + ((c ^ (n >> 1 & 3)) << 4);
  for (uint32_t tile = 0; tile < n_tiles; tile++) {
    __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0): this tile (requested a tile ago)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (tile + 1 < n_tiles) dma(tile + 1, (tile + 1) & 1);
    const uint32_t kv0 = tile * kAwRows;
    if (kv0 > pos0 + last_wave) continue;                                 // nothing of it is visible to this wave
    const uint8_t* kb = aw_lds + (tile & 1) * TB;
    const int ek = ex[tile * 2], ev = ex[tile * 2 + 1];
    f32x4 st[2][2];   // [rows 16 * i ..][token tile]
#pragma unroll
    for (int i = 0; i < 2; i++) {
      st[i][0] = st[i][1] = (f32x4)(0.0f);
#pragma unroll
      for (int k = 0; k < KK; k++) {
        const uint8_t* p = kb + i * 16 * D * 2 + k_off + (((uint32_t)(k * 4 + c) ^ (n & 7)) << 4);
        const h16x8 kh = *reinterpret_cast<const h16x8*>(p), kl = *reinterpret_cast<const h16x8*>(p + LIMB);
#pragma unroll
        for (int t = 0; t < 2; t++) {
          st[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kl, qh[t][k], st[i][t], 0, 0, 0);
          st[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kh, ql[t][k], st[i][t], 0, 0, 0);
          st[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kh, qh[t][k], st[i][t], 0, 0, 0);
        }
      }
    }
    const float fk = aw_pow2(ek), up = aw_pow2(14 + ev - vmax);           // softmax weights as operands: the tile's own exponent against the common one
    h16x8 ph[2], pl[2];
#pragma unroll
    for (int t = 0; t < 2; t++) {
      const float f = qf[t] * fk;
      float s[8], mx = kAwNeg;
#pragma unroll
      for (int j = 0; j < 8; j++) s[j] = st[j >> 2][t][j & 3] * f;
      if (kv0 + kAwRows - 1 > pos0 + tok0 + t * 16) {                      // the diagonal: row 4c + j (16 + ...) against the token
        const uint32_t tok = tok0 + t * 16 + n;
#pragma unroll
        for (int j = 0; j < 8; j++) s[j] = kv0 + (j >> 2) * 16 + 4 * c + (j & 3) <= pos0 + tok ? s[j] : kAwNeg;
      }
#pragma unroll
      for (int j = 0; j < 8; j++) mx = fmaxf(mx, s[j]);
      mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
      mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
      if (__any(mx > m_run[t])) {                                          // (rare after the first tiles)
        const float mn = fmaxf(m_run[t], mx), alpha = __builtin_amdgcn_exp2f(m_run[t] - mn);
        m_run[t] = mn;
        l_run[t] *= alpha;
#pragma unroll
        for (int x = 0; x < DT; x++) acc[t][x] = acc[t][x] * alpha;
      }
      float ps = 0.0f;
#pragma unroll
      for (int j = 0; j < 8; j++) { s[j] = __builtin_amdgcn_exp2f(s[j] - m_run[t]); ps += s[j]; }
      l_run[t] += ps;                                                      // (this lane's rows: the lanes of a token meet at the end)
      aw_split8(s, up, ph[t], pl[t]);
    }
#pragma unroll
    for (int x = 0; x < DT; x++) {
      const uint8_t* p = kb + v_off + x * 1024;
      const h16x8 vh = *reinterpret_cast<const h16x8*>(p), vl = *reinterpret_cast<const h16x8*>(p + LIMB);
#pragma unroll
      for (int t = 0; t < 2; t++) {
        acc[t][x] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vl, ph[t], acc[t][x], 0, 0, 0);
        acc[t][x] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vh, pl[t], acc[t][x], 0, 0, 0);
        acc[t][x] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vh, ph[t], acc[t][x], 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int t = 0; t < 2; t++) {
    float l = l_run[t];
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    const float f = aw_pow2(vmax - 28) / l;
    const uint32_t tok = tok0 + t * 16 + n;
    if (tok >= m_tokens) continue;
    uint8_t* o = out + ((size_t)tok * n_heads + head) * D * 2 + c * 8;
#pragma unroll
    for (int x = 0; x < DT; x++) {                                         // dims 16 x + 4c .. + 3, in the chunk's element order
      const f32x4 v = acc[t][x] * f;
      const h16x4 w = {(_Float16)v.x, (_Float16)v.z, (_Float16)v.y, (_Float16)v.w};
      *reinterpret_cast<h16x4*>(o + x * 32) = w;
    }
  }
}

uint32_t attn_wide_tiles(uint32_t rows) { return (rows + kAwRows - 1) / kAwRows; }
size_t attn_wide_bytes(uint32_t n_kv, uint32_t head_dim, uint32_t rows) {
  return (size_t)n_kv * attn_wide_tiles(rows) * ((head_dim == 128 ? aw_tile<128>() : aw_tile<64>()) + 2 * sizeof(int));
}

template <int D>
static hipError_t attn_wide_go(const float* q, const float* kc, const float* vc, uint32_t n_heads, uint32_t n_kv, uint32_t max_seq, float scale, uint32_t pos0,
                               uint32_t m_tokens, uint8_t* scratch, uint8_t* out, hipStream_t st) {
  static bool attr_set[64] = {};
  constexpr uint32_t lds = 2 * aw_tile<D>();
  if (hipError_t e = lds_opt_in(reinterpret_cast<const void*>(&attn_wide_kernel<D>), (int)lds, attr_set); e != hipSuccess) return e;
  const uint32_t kv_len = pos0 + m_tokens, tiles = attn_wide_tiles(kv_len), g = n_heads / n_kv, gw = g < 4 ? g : 4;
  int* exps = reinterpret_cast<int*>(scratch + (size_t)n_kv * tiles * aw_tile<D>());
  hipLaunchKernelGGL((attn_wide_split_kernel<D>), dim3(tiles, n_kv), dim3(256), 0, st, kc, vc, max_seq, kv_len, tiles, scratch, exps);
  const uint32_t n_blk = (m_tokens + 128 / gw - 1) / (128 / gw), wgs = n_blk * (n_heads / gw);
  hipLaunchKernelGGL((attn_wide_kernel<D>), dim3(wgs), dim3(256), lds, st, q, scratch, exps, n_heads, g, tiles, scale, pos0, m_tokens, n_blk,
                     (uint32_t)(wgs <= 2u * kNumCU), out);
  return hipGetLastError();
}

// scratch: attn_wide_bytes(n_kv, head_dim, pos0 + m_tokens).  out: row-major f16 [token][head][dim] in XH's element order
hipError_t attn_wide_launch(const float* q, const float* kcache, const float* vcache, uint32_t n_heads, uint32_t n_kv, uint32_t head_dim, uint32_t max_seq, float scale,
                            uint32_t pos0, uint32_t m_tokens, uint8_t* scratch, uint8_t* out, hipStream_t st) {
  if (n_kv == 0 || n_heads % n_kv || m_tokens == 0 || (head_dim != 64 && head_dim != 128) || pos0 + m_tokens > max_seq || n_kv > 65535) return hipErrorInvalidValue;
  const uint32_t g = n_heads / n_kv;
  if (g != 1 && g != 2 && g != 4 && g != 8) return hipErrorInvalidValue;
  return head_dim == 128 ? attn_wide_go<128>(q, kcache, vcache, n_heads, n_kv, max_seq, scale, pos0, m_tokens, scratch, out, st)
                         : attn_wide_go<64>(q, kcache, vcache, n_heads, n_kv, max_seq, scale, pos0, m_tokens, scratch, out, st);
}

}  // namespace lgh
