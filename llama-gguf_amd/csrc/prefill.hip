// prefill.hip — batched prompt processing: up to 128 prompt tokens per pass as one GEMM per weight on the f16 matrix
// cores (v_mfma_f32_16x16x32_f16), causal attention over the block, everything else row-wise.
//
// The reference has no counterpart: its prefill is `prefill_token` once per prompt token (src/backend/cuda/gpu_only.rs:
// 776-806; CPU: src/model/llama.rs:327-345), i.e. the whole model is streamed from memory once per token.  Here the
// quantized weights are read ONCE per 128 tokens.  This is the one place where f16 rounding enters the engine: the
// activations and the dequantized weights are rounded to f16 (11 significant bits each) in front of the matrix cores,
// products are accumulated in f32.  The KV cache it leaves must equal the one left by the same tokens fed one by one
// within the stated tolerance (tests/test_gpu_prefill.py); the exact token-by-token path stays available
// (LGH_FLAG_EXACT_PREFILL).
//
// Data flow per layer (all launches on the context's stream, nothing is captured in a graph):
//   XH(h * attn_norm) --GEMM wq|wk|wv--> partial sums --pf_qkv_epi (x 1/rms, bias, RoPE)--> q [M][QD] f32, K/V cache rows
//   q, cache --attention (attention.hip, PF variant; causal: token t sees pos0 + t + 1 rows)--> XH(attn)
//   XH(attn) --GEMM wo--> partials --pf_resid (+bias, +residual)--> h, XH(h * ffn_norm), sums of squares per token
//   XH --GEMM gate|up--> partials --pf_swiglu (x 1/rms)--> XH(act), or both in pf_pair_kernel; --GEMM down--> partials --pf_resid--> h, XH(h * attn_norm')
// MoE layers (moe.rs:321-413): the f32 decode router runs once per token of the block, the (token, slot) pairs are grouped
// by expert into one row space (prefill.h), and every expert runs ONCE over its rows: one gather launch, one gate|up GEMM
// of all experts, one SwiGLU launch, one down GEMM, one combine launch (routing weight * expert output in selection order,
// then the residual).
// The RMSNorm's 1/rms is a per-token scalar and the GEMM is linear: XH holds h * norm_weight and the kernel that adds
// up the GEMM's partial sums multiplies by 1/rms (from the sums of squares the producer of h left) — as in the decode path.
//
// "XH": an activation matrix [128 tokens][K] in f16, laid out for the GEMM's B operand: one 64 KB slab per 256
// elements of K (copied verbatim into LDS by LDS-DMA), inside a slab token t owns 512 B = 32 chunks of 8 elements, chunk
// q stored at position q ^ (t & 15) (so that the 16 tokens of an MFMA operand read 16 different LDS banks groups).
//
// GEMM: weights go HBM -> registers -> f16 (never through LDS: the dequantized lane layout IS the A operand), activations by LDS-DMA.  Dense layers: a workgroup = 8 waves = 128 weight
// rows x one k-range x all tokens in tiles of 32, in two teams that halve every block of k (pf_team).  A mixture's experts: 4 waves = 256 weight rows, a wave 4 row tiles (64 rows), an
// activation fragment feeds 4 MFMAs (pf_body).  K is split over gridDim.y workgroups to fill the chip; the f32 partial sums [split][token][column] are added up by the row-wise kernel that
// consumes them (together with bias, RoPE, residual, RMSNorm, SwiGLU).
#include <type_traits>

#include "device_utils.h"
#include "dispatch_rules.h"
#include "mv_epilogue.h"
#include "prefill.h"
#include "prefill_dequant.h"

namespace lgh {

// waves per workgroup: 4 (one per SIMD, 4 row tiles each).  8 waves of 2 tiles (-DPF_WAVES=8: two per SIMD, twice the LDS
// reads per MFMA) measured the same 4.68 ms per 128-token Llama-3-8B prompt: the loop is not latency-bound.
#ifndef PF_EXP
#define PF_EXP 0
#endif
#ifndef PF_WAVES
#define PF_WAVES 4
#endif
constexpr int kPfWaves = PF_WAVES;
constexpr int kPfRT = 16 / kPfWaves;     // row tiles per wave (a workgroup covers 256 rows)
constexpr int kPfMT = kPfTokens / 16;    // token tiles of a full block

#ifdef LGH_STAMPS
// diagnostic build: per-workgroup phase stamps (100 MHz s_memrealtime) of the GEMM launches whose output is LGH_PF_STAMP_COLS wide
#ifndef LGH_PF_STAMP_COLS
#define LGH_PF_STAMP_COLS 28672
#endif
__device__ unsigned long long g_pf_stamps[1024 * 16];
#define LGH_PF_STAMP(i)                                                                                         \
  do {                                                                                                          \
    if (G.ncols == LGH_PF_STAMP_COLS && threadIdx.x == 0 && (i) < 16) {                                         \
      const uint32_t wgid = blockIdx.y * gridDim.x + blockIdx.x;                                                \
      if (wgid < 1024) g_pf_stamps[wgid * 16 + (i)] = __builtin_amdgcn_s_memrealtime();                         \
    }                                                                                                           \
  } while (0)
hipError_t pf_read_stamps(unsigned long long* host, size_t n) {
  return hipMemcpyFromSymbol(host, HIP_SYMBOL(g_pf_stamps), std::min(n, (size_t)1024 * 16) * 8);
}
#else
#define LGH_PF_STAMP(i)
#endif

// A mixture's experts.  MT = token tiles computed: 8 for a full block, 4 / 2 when at most 64 / 32 rows are routed to the expert
// (about 32 of 128 with 2-of-8 routing): the MFMAs, the LDS reads and the activation DMA shrink with it.
template <int F, int MT>
__device__ __forceinline__ void pf_body(const PfGemm& G, const PfSeg& sg, uint32_t z, uint32_t rg, uint32_t ks, uint32_t m_tiles, uint8_t* smem) {
  constexpr uint32_t kBuf = (uint32_t)MT * 16 * 512;                // a slab's rows that are copied
  constexpr uint32_t kDma = kBuf / kPfWaves;   // a wave's share of the MT * 16 rows of a slab that are copied
  const uint32_t lane = threadIdx.x & 63, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const uint32_t n = lane & 15, c = lane >> 4;
  constexpr uint32_t tb = pf_tile_bytes(F);
  // this split's k-blocks
  const uint32_t per = (G.nblk + G.S - 1) / G.S;
  const uint32_t b0 = ks * per, b1 = b0 + per < G.nblk ? b0 + per : G.nblk;
  const uint32_t tile0 = (rg * kPfWaves + wave) * kPfRT;
  const uint8_t* wt[kPfRT];
#pragma unroll
  for (int r = 0; r < kPfRT; r++) {
    const uint32_t tl = tile0 + r < sg.ntiles ? tile0 + r : sg.ntiles - 1;   // clamped: loads are unconditional
    wt[r] = sg.w + (size_t)z * sg.w_z + (size_t)tl * G.nblk * tb;
  }
  const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem;

  f32x4 acc[kPfRT][MT];
#pragma unroll
  for (int r = 0; r < kPfRT; r++)
#pragma unroll
    for (int t = 0; t < MT; t++) acc[r][t] = (f32x4)(0.0f);

  // one 64 KB slab -> LDS buffer `buf`: this wave's quarter, 16 x 1 KB by LDS-DMA (no registers)
  auto x_dma = [&](uint32_t b, uint32_t buf) {
    const uint8_t* src = G.xh + (size_t)z * G.xh_z + (size_t)b * kPfSlabBytes + wave * kDma + lane * 16;
    const uint32_t dst = lds_base + buf * kBuf + wave * kDma;
#pragma unroll
    for (int i = 0; i < (int)(kDma / 1024); i++) {
      uint32_t keep;
      asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off\n\ts_mov_b32 m0, %0"
                   : "=&s"(keep) : "v"(src + i * 1024), "s"(dst + i * 1024) : "memory");
    }
  };

  LGH_PF_STAMP(0);
  PfRaw nxt[kPfRT];
  if (b0 < b1) {
    x_dma(b0, 0);
#pragma unroll
    for (int r = 0; r < kPfRT; r++) pf_load<F>(nxt[r], wt[r] + (size_t)b0 * tb, lane, n);
  }
  // (the BUILTIN, not inline asm: hipcc's wait-count pass must see that nothing is outstanding past this point.  With an
  // asm wait it still counted the previous block's weight loads as pending and protected their first uses with
  // `s_waitcnt vmcnt(21..12)` — in the hardware's count those are the NEXT slab's 16 LDS-DMA loads, issued just before, so
  // every block began by waiting for part of the next slab.  They come from L2: 4.86 -> 4.80 ms per prompt pass.)
  __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0)
  __syncthreads();
  LGH_PF_STAMP(1);
  auto block = [&](auto more, uint32_t b) {   // more: another block comes.  (The last one has a body without requests: re-requesting its own weights, for one body, cost 1 to 3 % of a prompt)
    const uint32_t cur = (b - b0) & 1;
    PfRaw w[kPfRT];
#pragma unroll
    for (int r = 0; r < kPfRT; r++) w[r] = nxt[r];
    if constexpr (more.value) {
#if PF_EXP != 4 && PF_EXP != 6   /* experiment 4 / 6: no activation slabs after the first */
      x_dma(b + 1, cur ^ 1);
#endif
#if PF_EXP != 5 && PF_EXP != 6   /* experiment 5 / 6: no weight loads after the first block's */
#pragma unroll
      for (int r = 0; r < kPfRT; r++) pf_load<F>(nxt[r], wt[r] + (size_t)(b + 1) * tb, lane, n);
#endif
    }
    // The block's 32 units (MFMA step pp, half h, row tile r) as a software pipeline, one scheduling region per unit:
    // the unit's 8 MFMAs, the dequantization of the NEXT unit's A fragment, and — in the first unit of a (pp, h) phase —
    // the LDS reads of the next phase's activation fragments.  Measured on Llama-3-8B Q4_K_M (128 tokens, 4.9 ms): with
    // the LDS reads removed 4.89 ms, with the dequantization removed 4.19 ms; forcing an MFMA / VALU interleave with
    // sched_group_barrier changed nothing (4.94 vs 4.88 ms).  Phase stamps of the gate|up GEMM (tools/pf_phases.py, the PF_EXP
    // switches below; 224 workgroups, 256 MFMAs + ~720 VALU ops per wave and block): 4.3 us per block as written, 3.3 us with
    // MFMAs only (no dequantization, no LDS reads: 1.3 PFLOP/s chip-wide, what f16 MFMAs sustain here with every CU issuing
    // them; PF_EXP 4 / 5 / 6 — no activation slabs / no weight loads / neither after the first block — 4.35 / 4.19 / 4.12 ms per pass
    // against 4.63: the loads are not what bounds the loop), 3.7 us with the dequantization and LDS reads only — the two overlap to within 30 %, the wait + barrier at the end
    // of a block is 0.2 us.  The loop runs at 77 % of its MFMA-only rate.
    const uint8_t* xb = smem + cur * kBuf + n * 512;
    h16x8 bf[2][MT];
    h16x2 S[kPfRT], O[kPfRT];
    auto read_bf = [&](int ph, h16x8* dst) {
      const uint32_t q = (uint32_t)((ph >> 1) * 8 + (ph & 1)) + c * 2;
#pragma unroll
      for (int t = 0; t < MT; t++) dst[t] = *reinterpret_cast<const h16x8*>(xb + t * 8192 + ((q ^ n) << 4));
    };
    read_bf(0, bf[0]);
    pf_scale<F>(w[0], 0, n, c, S[0], O[0]);
    h16x8 af[2];
    af[0] = pf_frag<F>(w[0], 0, 0, S[0], O[0]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < 8 * kPfRT; u++) {
      const int ph = u / kPfRT, r = u % kPfRT;
      if (u + 1 < 8 * kPfRT) {
        const int ph2 = (u + 1) / kPfRT, r2 = (u + 1) % kPfRT, pp2 = ph2 >> 1, h2 = ph2 & 1;
#if PF_EXP == 1 || PF_EXP == 3   /* experiment: no dequantization */
        af[(u + 1) & 1] = __builtin_bit_cast(h16x8, w[r2].q[pp2 & 1]);
#else
        if (h2 == 0) pf_scale<F>(w[r2], pp2, n, c, S[r2], O[r2]);
        af[(u + 1) & 1] = pf_frag<F>(w[r2], pp2, h2, S[r2], O[r2]);
#endif
      }
#if PF_EXP == 2   /* experiment: no MFMAs (the fragment is folded into one accumulator so that it stays live) */
      acc[r][0] += __builtin_bit_cast(f32x4, af[u & 1]) * __builtin_bit_cast(f32x4, bf[ph & 1][u & 7]);
#else
#pragma unroll
      for (int t = 0; t < MT; t++) acc[r][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[u & 1], bf[ph & 1][t], acc[r][t], 0, 0, 0);
#endif
      const bool rd = r == 0 && ph + 1 < 8;
#if PF_EXP == 3   /* experiment: no LDS reads either */
      if (rd) { for (int t = 0; t < MT; t++) bf[(ph + 1) & 1][t] = bf[ph & 1][t] + af[u & 1]; }
#else
      if (rd) read_bf(ph + 1, bf[(ph + 1) & 1]);
#endif
      __builtin_amdgcn_sched_barrier(0);
    }
    LGH_PF_STAMP(2 + 2 * (b - b0 < 5 ? b - b0 : 5));
    if constexpr (more.value) {
      __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0)
      __syncthreads();
    }
    LGH_PF_STAMP(3 + 2 * (b - b0 < 5 ? b - b0 : 5));
  };
  uint32_t b = b0;
  for (; b + 1 < b1; b++) block(std::true_type{}, b);
  if (b < b1) block(std::false_type{}, b);
  // partial sums: lane holds, per (row tile, token tile), rows 4c .. 4c+3 of token n
  uint32_t row0 = 0;
  if (G.row_base) asm volatile("s_load_dword %0, %1, 0x0\n\ts_waitcnt lgkmcnt(0)" : "=s"(row0) : "s"(G.row_base + z) : "memory");
  float* part = G.part + ((size_t)ks * G.part_rows + row0) * G.ncols;
#pragma unroll
  for (int r = 0; r < kPfRT; r++) {
    if (tile0 + r >= sg.ntiles) continue;
    const uint32_t col = sg.col0 + (tile0 + r) * 16 + c * 4;
#pragma unroll
    for (int t = 0; t < MT; t++) {
      if ((uint32_t)t >= m_tiles) continue;
      const f32x4 v = acc[r][t] * (1.0f / kPfScale);
      *reinterpret_cast<f32x4*>(part + (size_t)(t * 16 + n) * G.ncols + col) = v;
    }
  }
#ifdef LGH_STAMPS
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#endif
  LGH_PF_STAMP(14);
}

// All experts of a layer in one launch (blockIdx.z; a launch each, gate | up and down, was 16 launches of a third of the chip's rate: 8 experts of 14336 x 4096 in Q5_K, 64 tokens, 370 -> 288 us with the sums' fold; one block
// of weights under way a wave, 3.5 TB/s).  The token tiles are chosen here: experts of full blocks alone, a kernel with eight tiles fixed and this one, two of two, two layers, 97 / 112 / 128 tokens: 4096 x 14336 in
// Q4_K 254 / 253 / 263 and 253 / 254 / 264 us, in Q8_0 273 / 273 / 284 and 273 / 274 / 284.
template <uint32_t MASK>
__global__ void __launch_bounds__(kPfWaves * 64) pf_gemm_kernel(const PfGemm G) {
  extern __shared__ __attribute__((aligned(16))) uint8_t pf_smem[];
  const uint32_t rgid = blockIdx.x, z = blockIdx.z;
  int si = 0;
  if (G.nseg > 1 && rgid >= G.seg[1].rg_begin) si = 1;
  if (G.nseg > 2 && rgid >= G.seg[2].rg_begin) si = 2;
  const PfSeg& sg = G.seg[si];
  const uint32_t rg = rgid - sg.rg_begin;
  auto is = [&](int f) { return (MASK & (1u << f)) && (MASK == (1u << f) || sg.fmt == f); };
  uint32_t cnt;   // this expert's row count lives on the device (no host round trip per layer)
  asm volatile("s_load_dword %0, %1, 0x0\n\ts_waitcnt lgkmcnt(0)" : "=s"(cnt) : "s"(G.m_count + z) : "memory");
  if (cnt == 0) return;
  const uint32_t m_tiles = (cnt + 15) / 16;
#define LGH_PF_RUN(F)                                                                    \
  do {                                                                                   \
    if (m_tiles <= 2) pf_body<F, 2>(G, sg, z, rg, blockIdx.y, m_tiles, pf_smem);         \
    else if (m_tiles <= 4) pf_body<F, 4>(G, sg, z, rg, blockIdx.y, m_tiles, pf_smem);    \
    else pf_body<F, kPfMT>(G, sg, z, rg, blockIdx.y, m_tiles, pf_smem);                  \
  } while (0)
  if (is(PF_Q4K)) LGH_PF_RUN(PF_Q4K);
  else if (is(PF_Q6K)) LGH_PF_RUN(PF_Q6K);
  else if (is(PF_Q5K)) LGH_PF_RUN(PF_Q5K);
  else if (is(PF_Q80)) LGH_PF_RUN(PF_Q80);
  else if (is(PF_Q40)) LGH_PF_RUN(PF_Q40);
#undef LGH_PF_RUN
}

// 1 / rms of token t from the per-chunk sums of squares its producer left (simd.rs:847-878); 1 when there is no norm
__device__ __forceinline__ float pf_inv_rms(const float* ssq, uint32_t n_ssq, uint32_t t, uint32_t H, float eps) {
  if (!ssq) return 1.0f;
  // all that a token may have at once: a loop over those there are waits for each (64 tokens of gate | up: 4.5 us of the launch)
  const f32x4 a = *reinterpret_cast<const f32x4*>(ssq + t * kPfSsqChunks), b = *reinterpret_cast<const f32x4*>(ssq + t * kPfSsqChunks + 4);
  float tot = 0.0f;
#pragma unroll
  for (uint32_t j = 0; j < (uint32_t)kPfSsqChunks; j++) {
    const float v = j < 4 ? a[j & 3] : b[j & 3];
    tot = j < n_ssq ? tot + v : tot;
  }
  return 1.0f / __builtin_sqrtf(tot / (float)H + eps);
}

// Blocks of a dense model: a wave has 32 weight rows and up to 32 TT tokens on v_mfma_f32_32x32x16_f16 (less power per product than the 16 x 16 shape, and power is what bounds these loops).  Lane
// 32g + 16s + n holds row n of 16-row tile s, and of every 64 elements the two 16-element chunks 2g + j that the tile16 layout keeps for lanes 16(2g + j) + n; 256 elements have 16 phases (pp, j, h), each
// the contraction of elements 64pp + 16(2g + j) + 8h .. + 7 of both g.
//   PAIR   the tiles are the 16 gate rows and the 16 up rows of the same columns, over all of k: SwiGLU in registers, no partial sums
//   else   32 rows of one matrix over the blocks of a k-range (blockIdx.y), partial sums as pf_body
// Eight waves in two teams: both walk all blocks, team 0 with the first 128 elements of each and their weights, team 1 with the others; their sums meet through LDS.  So two waves a SIMD hide what one waits for (with
// one, 42 % of the cycles issued, 29 % waited for memory or the barrier and 29 % for the matrix cores), and a wave needs half of a block's raw weights, which leaves registers to ask for them two blocks ahead.
// 128 weight rows a workgroup instead of 256: half as many k-ranges fill the chip, and half the partial sums.  8B model, Q4_K_M, us a layer, four waves of 64 rows (gate | up: of 32) and here:
//   127 tokens  gate | up 44 and 38, SwiGLU included; wo, QKV, down 16.5, 18.7, 26.5 and 14.8, 18.2, 25.2; the residual's fold 7.1 and 5.2
//    96 tokens  (three tiles; four before) gate | up 43.7 and 30.7; wo, QKV, down 15.0, 18.3, 25.6 and 12.1, 15.0, 21.6; fold 6.2 and 5.4
//    49 tokens  gate | up 25.5 and 26.5; wo, QKV, down 11.6, 14.1, 18.1 and 10.3, 10.4, 17.6; fold 5.0 and 4.8
//    19 tokens  (gate | up: pf_pair_few_kernel) wo, QKV, down 7.9, 11.2, 14.0 and 7.3, 8.9, 13.5; fold 4.9 and 4.7
constexpr uint32_t pf_half_lds(int tt) { return (uint32_t)tt * 2 * 32 * 512; }
template <int F> constexpr uint32_t pf_half_loads() { return F == PF_Q6K ? 6 : F == PF_Q5K || F == PF_Q80 ? 5 : 3; }   // vector-memory operations of a load below
// the raw weights of 128 elements (TEAM) of one block: chunks 2g and 2g + 1 of row n.  pf_scale and pf_frag read what belongs to their step only
template <int F, int TEAM>
__device__ __forceinline__ void pf_half_load(PfRaw (&to)[2], const uint8_t* tile, uint32_t g, uint32_t n) {
  const u32x4 hd = ldg_nt128(tile + (F == PF_Q6K ? 3072 : F == PF_Q80 ? 4096 : 2048) + n * 16);
  uint32_t dh = 0;
  if (F == PF_Q6K) dh = ldg_nt32(tile + 3328 + (n >> 1) * 4);
#pragma unroll
  for (int j = 0; j < 2; j++) {
    const uint32_t l16 = 16 * (2 * g + j) + n;
    to[j].hd = hd;
    if (F == PF_Q80) {
      to[j].q[2 * TEAM] = ldg_nt128(tile + 2 * TEAM * 1024 + l16 * 16);
      to[j].q[2 * TEAM + 1] = ldg_nt128(tile + (2 * TEAM + 1) * 1024 + l16 * 16);
    } else {
      to[j].q[TEAM] = ldg_nt128(tile + TEAM * 1024 + l16 * 16);
      if (F == PF_Q6K) {
        const u32x2 h = ldg_nt64(tile + 2048 + l16 * 16 + TEAM * 8);
        if (TEAM == 0) { to[j].q[2].x = h.x; to[j].q[2].y = h.y; }
        else { to[j].q[2].z = h.x; to[j].q[2].w = h.y; }
        to[j].q[3].x = dh;
      }
      if (F == PF_Q5K) {
        const uint32_t h = ldg_nt32(tile + 2304 + l16 * 8 + TEAM * 4);
        if (TEAM == 0) to[j].q[2].x = h;
        else to[j].q[2].y = h;
      }
    }
  }
}

// one team's sums over the blocks [b0, b1); wrow: its lanes' 16-row tiles
template <int F, int TT, int TEAM, typename M>
__device__ __forceinline__ void pf_team(const PfGemm& G, const uint8_t* wrow, uint32_t b0, uint32_t b1, uint8_t* smem, f32x16 (&acc)[TT], M meanwhile) {
  constexpr uint32_t kBuf = (uint32_t)TT * 32 * 512, kDma = kBuf / (2 * kPfWaves), tb = pf_tile_bytes(F), LOADS = pf_half_loads<F>();
  constexpr int AHEAD = 2;                                            // phases the activations are read ahead
  const uint32_t lane = threadIdx.x & 63, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const uint32_t n = lane & 15, g = lane >> 5, tk = lane & 31;
  const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem;
  auto x_dma = [&](uint32_t b) {   // an eighth of a block's activations
    const uint8_t* src = G.xh + (size_t)b * kPfSlabBytes + wave * kDma;
    const uint32_t dst = lds_base + (b & 1) * kBuf + wave * kDma;
#pragma unroll
    for (int i = 0; i < (int)(kDma / 1024); i++)
      asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(lane * 16), "s"(src + i * 1024), "s"(dst + i * 1024) : "memory", "m0");
  };
  PfRaw w[3][2];   // [block in turn][j]
  x_dma(b0);
  if (b0 + 1 < b1) x_dma(b0 + 1);
  const uint8_t* from = wrow + (size_t)b0 * tb;
  auto load = [&](uint32_t b, PfRaw (&to)[2]) {   // (past the end the last ones again: the waits below count them)
    pf_half_load<F, TEAM>(to, from, g, n);
    from += b + 1 < b1 ? tb : 0u;
  };
  load(b0, w[0]);
  load(b0 + 1, w[1]);
#pragma unroll
  for (int t = 0; t < TT; t++) acc[t] = (f32x16)(0.0f);
  meanwhile();
  // all but the newest weights (asked for behind everything that is awaited) have arrived, and every wave has read what it will of the buffer in turn
  auto landed = [&](auto more) {
    __builtin_amdgcn_s_waitcnt(more.value ? 0x0070 | LOADS : 0x0070);   // vmcnt(LOADS or 0) lgkmcnt(0); the builtin: see pf_body
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  landed(std::true_type{});
  h16x8 af[2], bf[4][TT];
  h16x2 S, O;
  auto read_bf = [&](uint32_t b, int p) {   // p = 4 (pp - 2 TEAM) + 2 j + h
    const uint32_t q = (uint32_t)(16 * TEAM + 8 * (p >> 2) + (p & 3)) + 4 * g;
#pragma unroll
    for (int t = 0; t < TT; t++) bf[p & 3][t] = *reinterpret_cast<const h16x8*>(smem + (b & 1) * kBuf + (t * 32 + tk) * 512 + ((q ^ n) << 4));
  };
  auto frag = [&](const PfRaw (&cw)[2], int p) {
    const int pp = 2 * TEAM + (p >> 2), j = p >> 1 & 1;
    if ((p & 3) == 0 || (F == PF_Q6K && (p & 1) == 0)) pf_scale<F>(cw[j], pp, n, 2 * g + j, S, O);
    af[p & 1] = pf_frag<F>(cw[j], pp, p & 1, S, O);
  };
  // more: it asks for weights.  (What the last one reads of the buffer and the registers beyond the end is not used)
  auto block = [&](auto more, uint32_t b, PfRaw (&cw)[2], PfRaw (&nw)[2], PfRaw (&ow)[2]) {
    if constexpr (more.value) load(b + 2, ow);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int p = 0; p < 8; p++) {
      if (p == 8 - AHEAD) {
        landed(more);
        if (more.value && b + 2 < b1) x_dma(b + 2);
      }
      if (p + AHEAD < 8) read_bf(b, p + AHEAD);
      else read_bf(b + 1, p + AHEAD - 8);
      if (p < 7) frag(cw, p + 1);
      else frag(nw, 0);
#pragma unroll
      for (int t = 0; t < TT; t++) acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[p & 1], bf[p & 3][t], acc[t], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
#pragma unroll
  for (int p = 0; p < AHEAD; p++) read_bf(b0, p);
  frag(w[0], 0);
  uint32_t b = b0;   // (whole turns, then what is left: with a test inside the loop the compiler sees a way round on which a block's weights are still under way, and waits for them)
  for (; b + 3 <= b1; b += 3) {
    block(std::true_type{}, b, w[0], w[1], w[2]);
    block(std::true_type{}, b + 1, w[1], w[2], w[0]);
    block(std::true_type{}, b + 2, w[2], w[0], w[1]);
  }
  if (b < b1) block(std::false_type{}, b, w[0], w[1], w[2]);
  if (b + 1 < b1) block(std::false_type{}, b + 1, w[1], w[2], w[0]);
}

template <int F, int TT, bool PAIR>
__device__ __forceinline__ void pf_half_device(const PfGemm& G, const PfSeg& sg, uint32_t rg, uint32_t ks, uint8_t* smem) {
  constexpr int OWN = (TT + 1) / 2;   // token tiles whose sums team 0 puts together; team 1 has the others
  const uint32_t lane = threadIdx.x & 63, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6 & 3)), team = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 8));
  const uint32_t s = lane >> 4 & 1, g = lane >> 5, tk = lane & 31;
  const uint32_t unit = rg * kPfWaves + wave;                                   // PAIR: a tile of each matrix, else two tiles
  const uint32_t want = PAIR ? unit : 2 * unit + s, tl = want < sg.ntiles ? want : sg.ntiles - 1;   // clamped: loads are unconditional
  const uint8_t* const wrow = (PAIR && s ? G.seg[1].w : sg.w) + (size_t)tl * G.nblk * pf_tile_bytes(F);
  const uint32_t per = (G.nblk + G.S - 1) / G.S, b0 = ks * per, b1 = b0 + per < G.nblk ? b0 + per : G.nblk;
  f32x16 acc[TT];
  float inv[TT];   // 1 / rms of this lane's tokens
  auto norms = [&] {
    if (PAIR) {
#pragma unroll
      for (int t = 0; t < TT; t++) inv[t] = pf_inv_rms(G.ssq, G.n_ssq, t * 32 + tk, G.norm_cols, G.eps) * (1.0f / kPfScale);
    }
  };
  if (team == 0) pf_team<F, TT, 0>(G, wrow, b0, b1, smem, acc, norms);
  else pf_team<F, TT, 1>(G, wrow, b0, b1, smem, acc, norms);
  // lane (tk, g) has of token 32 t + tk rows 8i + 4g .. + 3, i = 0 .. 3.  A team leaves the tiles that the other one owns in LDS (36 floats a token: banks) and adds what it finds there to its own
  float* const place = reinterpret_cast<float*>(smem) + wave * (TT * 32 * 36) + tk * 36 + 4 * g;
  __syncthreads();   // (every read of the slabs has returned)
#pragma unroll
  for (int t = 0; t < TT; t++)
    if ((t < OWN) != (team == 0)) {
#pragma unroll
      for (int i = 0; i < 4; i++) *reinterpret_cast<f32x4*>(place + t * 32 * 36 + 8 * i) = f32x4{acc[t][4 * i], acc[t][4 * i + 1], acc[t][4 * i + 2], acc[t][4 * i + 3]};
    }
  __syncthreads();
  if (PAIR && unit >= sg.ntiles) return;
#pragma unroll
  for (int t = 0; t < TT; t++) {
    if ((t < OWN) != (team == 0)) continue;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const f32x4 v = *reinterpret_cast<const f32x4*>(place + t * 32 * 36 + 8 * i);
#pragma unroll
      for (int e = 0; e < 4; e++) acc[t][4 * i + e] += v[e];
    }
    if constexpr (PAIR) {   // gate with i = 0, 1, up with i + 2
      const uint32_t tok = t * 32 + tk;
      if (tok >= G.m_tokens) continue;
#pragma unroll
      for (int i = 0; i < 2; i++) {
        h16x4 o;
#pragma unroll
        for (int e = 0; e < 4; e++) o[e] = (_Float16)(silu_act_f(acc[t][4 * i + e] * inv[t]) * (acc[t][4 * i + 8 + e] * inv[t]));
        *reinterpret_cast<h16x4*>(G.act + xh_offset(tok, unit * 16 + 8 * i + 4 * g)) = o;
      }
    } else {   // turned round in the same place, so that a token's 32 sums leave side by side
#pragma unroll
      for (int i = 0; i < 4; i++) *reinterpret_cast<f32x4*>(place + t * 32 * 36 + 8 * i) = f32x4{acc[t][4 * i], acc[t][4 * i + 1], acc[t][4 * i + 2], acc[t][4 * i + 3]} * (1.0f / kPfScale);
      const uint32_t row = unit * 32 + (lane & 7) * 4;
      float* const part = G.part + (size_t)ks * G.part_rows * G.ncols + sg.col0 + row;
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const uint32_t tok = i * 8 + (lane >> 3);
        const f32x4 v = *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(smem) + wave * (TT * 32 * 36) + (t * 32 + tok) * 36 + (lane & 7) * 4);
        if (t * 32 + tok < G.m_tokens && row < sg.ntiles * 16) *reinterpret_cast<f32x4*>(part + (size_t)(t * 32 + tok) * G.ncols) = v;
      }
    }
  }
}

template <int F, int TT>
__global__ void __launch_bounds__(2 * kPfWaves * 64) pf_pair_kernel(const PfGemm G) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  pf_half_device<F, TT, true>(G, G.seg[0], blockIdx.x, 0, smem);
}

// gate | up for up to 32 tokens and whole pairs of blocks a team: each team has half of k, a block between two barriers is twice as long and the weights' addresses and scales are made once for two phases' more products.
// 28672 rows of 4096 in Q4_K: 20.5 us against 23.4 in halves of blocks, where a block is over before what was asked for has come.
template <int F>
__global__ void __launch_bounds__(2 * kPfWaves * 64) pf_pair_few_kernel(const PfGemm G) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  constexpr uint32_t kBuf = 32 * 512, kDma = kBuf / kPfWaves, tb = pf_tile_bytes(F);
  constexpr int AHEAD = 2;                                            // phases the activations are read ahead
  const uint32_t lane = threadIdx.x & 63, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6 & 3)), team = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 8));
  const uint32_t n = lane & 15, s = lane >> 4 & 1, g = lane >> 5, tk = lane & 31, nblk = G.nblk / 2;   // this team's blocks
  const uint32_t tile = blockIdx.x * kPfWaves + wave, tl = tile < G.seg[0].ntiles ? tile : G.seg[0].ntiles - 1;   // clamped: loads are unconditional
  const uint8_t* const wrow = (s ? G.seg[1].w : G.seg[0].w) + ((size_t)tl * G.nblk + team * nblk) * tb;
  uint8_t* const slab = smem + team * 2 * kBuf;
  const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)slab;
  auto x_dma = [&](uint32_t b) {
    const uint8_t* src = G.xh + (size_t)(team * nblk + b) * kPfSlabBytes + wave * kDma;
    const uint32_t dst = lds_base + (b & 1) * kBuf + wave * kDma;
#pragma unroll
    for (int i = 0; i < (int)(kDma / 1024); i++)
      asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(lane * 16), "s"(src + i * 1024), "s"(dst + i * 1024) : "memory", "m0");
  };
  auto load = [&](uint32_t b, PfRaw (&to)[2]) {
#pragma unroll
    for (int j = 0; j < 2; j++) pf_load<F>(to[j], wrow + (size_t)b * tb, 16 * (2 * g + j) + n, n);   // (the row's scales once: the compiler sees that they are the same)
  };
  f32x16 acc = (f32x16)(0.0f);
  PfRaw w[2][2];   // [block parity][j]
  x_dma(0);
  load(0, w[0]);
  const float inv = pf_inv_rms(G.ssq, G.n_ssq, tk, G.norm_cols, G.eps) * (1.0f / kPfScale);   // of this lane's token
  auto landed = [&] {
    __builtin_amdgcn_s_waitcnt(0x0070);   // vmcnt(0) lgkmcnt(0): see pf_body
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  landed();
  h16x8 af[2], bf[4];
  h16x2 S, O;
  auto read_bf = [&](uint32_t b, int p) {   // p = 4 pp + 2 j + h
    const uint32_t q = (uint32_t)(8 * (p >> 2) + (p & 3)) + 4 * g;
    bf[p & 3] = *reinterpret_cast<const h16x8*>(slab + (b & 1) * kBuf + tk * 512 + ((q ^ n) << 4));
  };
  auto frag = [&](const PfRaw (&cw)[2], int p) {
    const int pp = p >> 2, j = p >> 1 & 1;
    if ((p & 3) == 0 || (F == PF_Q6K && (p & 1) == 0)) pf_scale<F>(cw[j], pp, n, 2 * g + j, S, O);
    af[p & 1] = pf_frag<F>(cw[j], pp, p & 1, S, O);
  };
  auto block = [&](uint32_t b, PfRaw (&cw)[2], PfRaw (&nw)[2]) {   // (the last one requests nothing; what it reads of the buffer and the registers beyond the end is not used)
    if (b + 1 < nblk) {
      x_dma(b + 1);
      load(b + 1, nw);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int p = 0; p < 16; p++) {
      if (p == 16 - AHEAD) landed();
      if (p + AHEAD < 16) read_bf(b, p + AHEAD);
      else read_bf(b + 1, p + AHEAD - 16);
      if (p < 15) frag(cw, p + 1);
      else frag(nw, 0);
      acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[p & 1], bf[p & 3], acc, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
#pragma unroll
  for (int p = 0; p < AHEAD; p++) read_bf(0, p);
  frag(w[0], 0);
  for (uint32_t b = 0; b < nblk; b += 2) {
    block(b, w[0], w[1]);
    block(b + 1, w[1], w[0]);
  }
  f32x4* const sums = reinterpret_cast<f32x4*>(smem) + wave * (4 * 64) + lane;
  __syncthreads();   // (every read of the slabs has returned)
  if (team == 1) {
#pragma unroll
    for (int i = 0; i < 4; i++) sums[i * 64] = f32x4{acc[4 * i], acc[4 * i + 1], acc[4 * i + 2], acc[4 * i + 3]};
  }
  __syncthreads();
  if (team == 1 || tile >= G.seg[0].ntiles || tk >= G.m_tokens) return;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const f32x4 v = sums[i * 64];
#pragma unroll
    for (int e = 0; e < 4; e++) acc[4 * i + e] += v[e];
  }
  // a lane has rows 8i + 4g .. + 3: gate with i = 0, 1, up with i + 2
#pragma unroll
  for (int i = 0; i < 2; i++) {
    h16x4 o;
#pragma unroll
    for (int e = 0; e < 4; e++) o[e] = (_Float16)(silu_act_f(acc[4 * i + e] * inv) * (acc[4 * i + 8 + e] * inv));
    *reinterpret_cast<h16x4*>(G.act + xh_offset(tk, tile * 16 + 8 * i + 4 * g)) = o;
  }
}

template <uint32_t MASK, int TT>
__global__ void __launch_bounds__(2 * kPfWaves * 64) pf_rows_kernel(const PfGemm G) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  int si = 0;
  if (G.nseg > 1 && blockIdx.x >= G.seg[1].rg_begin) si = 1;
  if (G.nseg > 2 && blockIdx.x >= G.seg[2].rg_begin) si = 2;
  const PfSeg& sg = G.seg[si];
  auto is = [&](int f) { return (MASK & (1u << f)) && (MASK == (1u << f) || sg.fmt == f); };
  const uint32_t rg = blockIdx.x - sg.rg_begin;
  if (is(PF_Q4K)) pf_half_device<PF_Q4K, TT, false>(G, sg, rg, blockIdx.y, smem);
  else if (is(PF_Q6K)) pf_half_device<PF_Q6K, TT, false>(G, sg, rg, blockIdx.y, smem);
  else if (is(PF_Q5K)) pf_half_device<PF_Q5K, TT, false>(G, sg, rg, blockIdx.y, smem);
  else if (is(PF_Q80)) pf_half_device<PF_Q80, TT, false>(G, sg, rg, blockIdx.y, smem);
  else if (is(PF_Q40)) pf_half_device<PF_Q40, TT, false>(G, sg, rg, blockIdx.y, smem);
}

template <auto* Kernel, size_t LDS, int WAVES>
static hipError_t pf_gemm_run(const PfGemm& G, uint32_t n_rg, hipStream_t st) {
  static bool attr_set[64] = {};
  if (hipError_t e = lds_opt_in(reinterpret_cast<const void*>(Kernel), (int)LDS, attr_set); e != hipSuccess) return e;
  hipLaunchKernelGGL(Kernel, dim3(n_rg, G.S, G.n_experts ? G.n_experts : 1), dim3(WAVES * 64), LDS, st, G);
  return hipGetLastError();
}
template <uint32_t MASK>
static hipError_t pf_gemm_go(const PfGemm& G, uint32_t n_rg, hipStream_t st) {
  if (G.m_count) return pf_gemm_run<&pf_gemm_kernel<MASK>, 2 * (size_t)kPfSlabBytes, kPfWaves>(G, n_rg, st);
  switch ((G.m_tokens + 31) / 32) {
    case 1: return pf_gemm_run<&pf_rows_kernel<MASK, 1>, pf_half_lds(1), 2 * kPfWaves>(G, n_rg, st);
    case 2: return pf_gemm_run<&pf_rows_kernel<MASK, 2>, pf_half_lds(2), 2 * kPfWaves>(G, n_rg, st);
    case 3: return pf_gemm_run<&pf_rows_kernel<MASK, 3>, pf_half_lds(3), 2 * kPfWaves>(G, n_rg, st);
    default: return pf_gemm_run<&pf_rows_kernel<MASK, 4>, pf_half_lds(4), 2 * kPfWaves>(G, n_rg, st);
  }
}

bool pf_supported_type(int dev_type) { return pf_fmt_of(dev_type) >= 0; }

// 16-row tiles of a workgroup
static uint32_t pf_wg_tiles(bool experts) { return experts ? kPfWaves * kPfRT : kPfWaves * 2; }

// k-splits of a GEMM over matrices with n_rows[i] rows and k columns: as many as keep the launch within one workgroup per CU;  of a layer's experts, whose workgroups have unequal work, as many as make two per CU
// (a layer of 8 experts of 14336 x 4096 in Q5_K, us, products and fold, 16 / 64 / 128 tokens: gate | up unsplit 148 / 198 / 231, in two 156 / 196 / 229; down, 128 workgroups unsplit, in two 88 / 106 / 140, in four 89 / 102 / 122)
static void pf_plan(const uint32_t* n_rows, int nw, uint32_t k, uint32_t n_experts, uint32_t* S_out) {
  const uint32_t nblk = k / 256, wt = pf_wg_tiles(n_experts != 0), fill = n_experts ? 2 * kNumCU : kNumCU;
  uint32_t wgs = 0;
  for (int i = 0; i < nw; i++) wgs += (n_rows[i] / 16 + wt - 1) / wt;
  if (n_experts) wgs *= n_experts;
  *S_out = pf_ranges(wgs, fill, nblk);
}

// bytes of partial sums such a GEMM writes
size_t pf_part_bytes(const uint32_t* n_rows, int nw, uint32_t k, uint32_t n_experts) {
  uint32_t S, cols = 0;
  pf_plan(n_rows, nw, k, n_experts, &S);
  for (int i = 0; i < nw; i++) cols += n_rows[i];
  return (size_t)S * (n_experts ? kPfMoeRows : kPfTokens) * cols * 4;
}

// Plans and launches one GEMM: up to 3 weight matrices that share the input XH (k elements per token), outputs side by
// side in the partial-sum buffer.  Returns the split count through *S_out (the consumer adds that many partials).
hipError_t pf_gemm_launch(const DevWeight* const* W, int nw, const uint8_t* xh, float* part, size_t part_bytes, uint32_t m_tokens,
                          uint32_t* S_out, uint32_t* ncols_out, hipStream_t st, uint32_t n_experts, size_t xh_z, const int* m_count, uint32_t part_rows,
                          const int* row_base) {
  if (nw < 1 || nw > 3 || m_tokens == 0 || m_tokens > (uint32_t)kPfTokens || (n_experts != 0) != (m_count != nullptr)) return hipErrorInvalidValue;
  PfGemm G{};
  const uint32_t k = W[0]->k;
  if (k % 256) return hipErrorInvalidValue;
  G.nseg = nw;
  G.nblk = k / 256;
  const uint32_t wt = pf_wg_tiles(m_count != nullptr);
  uint32_t rg = 0, col = 0, mask = 0, n_rows[3] = {0, 0, 0};
  for (int i = 0; i < nw; i++) {
    const int f = pf_fmt_of(W[i]->type);
    if (f < 0 || W[i]->k != k || W[i]->n % 16 || std::max(n_experts, 1u) > W[i]->n_stack) return hipErrorInvalidValue;
    G.seg[i].w = W[i]->plane[0];
    G.seg[i].w_z = W[i]->stack_stride[0];   // expert stacks: [expert][tiles]
    G.seg[i].ntiles = W[i]->n / 16;
    G.seg[i].col0 = col;
    G.seg[i].rg_begin = rg;
    G.seg[i].fmt = f;
    mask |= 1u << f;
    rg += (G.seg[i].ntiles + wt - 1) / wt;
    col += W[i]->n;
    n_rows[i] = W[i]->n;
  }
  pf_plan(n_rows, nw, k, n_experts, &G.S);
  G.ncols = col;
  G.xh = xh;
  G.xh_z = xh_z;
  G.n_experts = n_experts;
  G.part = part;
  G.m_tokens = m_tokens;
  G.m_count = m_count;
  G.part_rows = part_rows;
  G.row_base = row_base;
  if (part_rows < (uint32_t)kPfTokens || (size_t)G.S * part_rows * col * 4 > part_bytes) return hipErrorInvalidValue;
  *S_out = G.S;
  *ncols_out = col;
  switch (mask) {
    case 1u << PF_Q4K: return pf_gemm_go<1u << PF_Q4K>(G, rg, st);
    case 1u << PF_Q6K: return pf_gemm_go<1u << PF_Q6K>(G, rg, st);
    case (1u << PF_Q4K) | (1u << PF_Q6K): return pf_gemm_go<(1u << PF_Q4K) | (1u << PF_Q6K)>(G, rg, st);
    case 1u << PF_Q5K: return pf_gemm_go<1u << PF_Q5K>(G, rg, st);
    case (1u << PF_Q5K) | (1u << PF_Q6K): return pf_gemm_go<(1u << PF_Q5K) | (1u << PF_Q6K)>(G, rg, st);
    case 1u << PF_Q80: return pf_gemm_go<1u << PF_Q80>(G, rg, st);
    case 1u << PF_Q40: return pf_gemm_go<1u << PF_Q40>(G, rg, st);
    default: return pf_gemm_go<31u>(G, rg, st);   // any other mix of the five formats
  }
}

// chunks of per-token sums of squares a row of H elements is reduced to (pf_inv_rms adds them up)
uint32_t pf_ssq_chunks(uint32_t H) { return (H + 2047) / 2048; }

// gate | up as one product without partial sums (pf_pair_pays)
bool pf_pairs(const DevWeight* gate, const DevWeight* up, uint32_t m_tokens) {
  if (!pf_supported_type(gate->type) || gate->type != up->type || gate->k != up->k || gate->n != up->n || gate->k % 256 || gate->n % 256) return false;
  const uint32_t n_rows[2] = {gate->n, up->n};
  uint32_t S;
  pf_plan(n_rows, 2, gate->k, 0, &S);
  return pf_pair_pays(gate->k / 256, S, m_tokens);
}

template <int F>
static hipError_t pf_pair_go(const PfGemm& G, hipStream_t st) {
  const uint32_t wgs = (G.seg[0].ntiles + kPfWaves - 1) / kPfWaves;
  switch ((G.m_tokens + 31) / 32) {
    case 1: if (G.nblk % 4 == 0) return pf_gemm_run<&pf_pair_few_kernel<F>, 2 * pf_half_lds(1), 2 * kPfWaves>(G, wgs, st);
            return pf_gemm_run<&pf_pair_kernel<F, 1>, pf_half_lds(1), 2 * kPfWaves>(G, wgs, st);
    case 2: return pf_gemm_run<&pf_pair_kernel<F, 2>, pf_half_lds(2), 2 * kPfWaves>(G, wgs, st);
    case 3: return pf_gemm_run<&pf_pair_kernel<F, 3>, pf_half_lds(3), 2 * kPfWaves>(G, wgs, st);
    default: return pf_gemm_run<&pf_pair_kernel<F, 4>, pf_half_lds(4), 2 * kPfWaves>(G, wgs, st);
  }
}

hipError_t pf_pair_launch(const DevWeight* gate, const DevWeight* up, const uint8_t* xh, uint8_t* act, const float* ssq, uint32_t norm_cols, float eps, uint32_t m_tokens, hipStream_t st) {
  if (m_tokens == 0 || !pf_pairs(gate, up, m_tokens) || m_tokens > (uint32_t)kPfTokens || !act || !ssq) return hipErrorInvalidValue;
  PfGemm G{};
  for (int i = 0; i < 2; i++) {
    const DevWeight* W = i ? up : gate;
    G.seg[i].w = W->plane[0];
    G.seg[i].ntiles = W->n / 16;
  }
  G.nseg = 1;
  G.nblk = gate->k / 256;
  G.S = 1;
  G.xh = xh;
  G.act = act;
  G.ssq = ssq;
  G.n_ssq = pf_ssq_chunks(norm_cols);
  G.norm_cols = norm_cols;
  G.eps = eps;
  G.m_tokens = m_tokens;
  switch (pf_fmt_of(gate->type)) {
    case PF_Q4K: return pf_pair_go<PF_Q4K>(G, st);
    case PF_Q6K: return pf_pair_go<PF_Q6K>(G, st);
    case PF_Q5K: return pf_pair_go<PF_Q5K>(G, st);
    case PF_Q80: return pf_pair_go<PF_Q80>(G, st);
    case PF_Q40: return pf_pair_go<PF_Q40>(G, st);
  }
  return hipErrorInvalidValue;
}

// ------------------------------------------------------------------------------------------------
// XH writers and the row-wise kernels between the GEMMs
// ------------------------------------------------------------------------------------------------
// chunk `ch` (8 consecutive elements starting at 8*ch) of token t
__device__ __forceinline__ void xh_store_chunk(uint8_t* xh, uint32_t t, uint32_t ch, const float v[8]) {
  const uint32_t b = ch >> 5, q = ch & 31;
  h16x8 o = {(_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)v[3], (_Float16)v[4], (_Float16)v[5], (_Float16)v[6], (_Float16)v[7]};
  *reinterpret_cast<h16x8*>(xh + (size_t)b * kPfSlabBytes + t * 512 + ((q ^ (t & 15)) << 4)) = o;
}

// The residual's partial sums are requested eight splits at a time and added in order: 16 tokens and 16 splits 6.5 -> 4.8 us (128 tokens 7.2 -> 7.1).  QKV's eight splits of two values
// a thread are no faster that way (4.4 -> 4.9).
constexpr uint32_t kPfAtOnce = 8;

// Row epilogue, (2048-column chunks) x (tokens) workgroups:
//   v[i] = sum_s part[s][t][col0 + i] (+ bias[i]) + hidden[t][i]  (the residual, layers.rs:1201-1208, 1235-1241);
//   hidden[t][i] = v[i];  XH[t][i] = f16(v[i] * nw[i]);  ssq[t][chunk] = sum of v^2 over the chunk.
// The RMSNorm's 1/rms is a per-token scalar and the GEMM is linear, so it is applied by the kernel that consumes the
// GEMM's partial sums (pf_inv_rms) — no second pass over the row.  S == 0: v = hidden[t][i] as it is (embedding rows).
__global__ void __launch_bounds__(256) pf_resid_kernel(const float* __restrict__ part, uint32_t S, uint32_t ncols, uint32_t col0,
                                                       const float* __restrict__ bias, float* __restrict__ hidden, uint32_t H,
                                                       const float* __restrict__ nw, uint8_t* __restrict__ xh, float* __restrict__ ssq,
                                                       const float* __restrict__ moe_w) {
  __shared__ float s_ss[4];
  const uint32_t t = blockIdx.y, ch = blockIdx.x * 256 + threadIdx.x, i = ch * 8;
  float ss = 0.0f;
  if (i < H) {
    f32x4 v0 = *reinterpret_cast<const f32x4*>(hidden + (size_t)t * H + i), v1 = *reinterpret_cast<const f32x4*>(hidden + (size_t)t * H + i + 4);
    if (S) {
      f32x4 a0 = (f32x4)(0.0f), a1 = (f32x4)(0.0f);
      for (uint32_t s0 = 0; s0 < S; s0 += kPfAtOnce) {
        f32x4 r0[kPfAtOnce], r1[kPfAtOnce];
#pragma unroll
        for (uint32_t k = 0; k < kPfAtOnce; k++) {
          const float* row = part + ((size_t)(s0 + k < S ? s0 + k : s0) * kPfTokens + t) * ncols + col0 + i;
          r0[k] = *reinterpret_cast<const f32x4*>(row);
          r1[k] = *reinterpret_cast<const f32x4*>(row + 4);
        }
#pragma unroll
        for (uint32_t k = 0; k < kPfAtOnce; k++) {
          if (s0 + k >= S) break;
          if (moe_w) {   // MoeLayer::forward (moe.rs:363-368): zero-initialised, += routing weight * expert output in selection order
            const float w = moe_w[t * S + s0 + k];
            a0 += r0[k] * w;
            a1 += r1[k] * w;
          } else {
            a0 += r0[k];
            a1 += r1[k];
          }
        }
      }
      if (bias) { a0 += *reinterpret_cast<const f32x4*>(bias + i); a1 += *reinterpret_cast<const f32x4*>(bias + i + 4); }
      v0 += a0;
      v1 += a1;
      *reinterpret_cast<f32x4*>(hidden + (size_t)t * H + i) = v0;
      *reinterpret_cast<f32x4*>(hidden + (size_t)t * H + i + 4) = v1;
    }
    const f32x4 q = v0 * v0 + v1 * v1;
    ss = (q.x + q.y) + (q.z + q.w);
    if (xh) {
      const f32x4 w0 = *reinterpret_cast<const f32x4*>(nw + i), w1 = *reinterpret_cast<const f32x4*>(nw + i + 4);
      float v[8];
#pragma unroll
      for (int j = 0; j < 4; j++) { v[j] = v0[j] * w0[j]; v[4 + j] = v1[j] * w1[j]; }
      xh_store_chunk(xh, t, ch, v);
    }
  }
  ss = wave_sum(ss);
  if ((threadIdx.x & 63) == 0) s_ss[threadIdx.x >> 6] = ss;
  __syncthreads();
  if (threadIdx.x == 0 && ssq) ssq[t * kPfSsqChunks + blockIdx.x] = (s_ss[0] + s_ss[1]) + (s_ss[2] + s_ss[3]);
}

hipError_t pf_row_epi_launch(const float* part, uint32_t S, uint32_t ncols, uint32_t col0, const float* bias, float* hidden, uint32_t H,
                             const float* nw, uint8_t* xh, float* ssq, uint32_t m_tokens, hipStream_t st, const float* moe_w) {
  if (H % 8 || (xh && (!nw || !ssq)) || (S && (ncols % 4 || col0 % 4)) || pf_ssq_chunks(H) > (uint32_t)kPfSsqChunks) return hipErrorInvalidValue;
  hipLaunchKernelGGL(pf_resid_kernel, dim3(pf_ssq_chunks(H), m_tokens), dim3(256), 0, st, part, S, ncols, col0, bias, hidden, H, nw, xh, ssq, moe_w);
  return hipGetLastError();
}

// q, k, v of token t: partial sums (+bias), RoPE on the (2i, 2i+1) — NeoX: (i, i + d/2) — pairs of q and k at position
// pos0 + t (ops.rs:1285-1337), q -> qbuf[t][QD], k / v -> cache rows pos0 + t (layers.rs:577-600)
__global__ void __launch_bounds__(256) pf_qkv_epi_kernel(const float* __restrict__ part, uint32_t S, uint32_t ncols, uint32_t QD, uint32_t KD,
                                                         uint32_t head_dim, const float* __restrict__ bq, const float* __restrict__ bk,
                                                         const float* __restrict__ bv, const float* __restrict__ rope_cs, uint32_t pos0,
                                                         uint32_t max_seq, float* __restrict__ qbuf, float* __restrict__ kcache,
                                                         float* __restrict__ vcache, const float* __restrict__ ssq, uint32_t n_ssq,
                                                         uint32_t H, float eps, int neox) {
  const uint32_t t = blockIdx.y, pos = pos0 + t, half = head_dim / 2;
  const float inv = pf_inv_rms(ssq, n_ssq, t, H, eps);
  const uint32_t npairs = (QD + 2 * KD) / 2, nq = QD / 2, nk = KD / 2;
  for (uint32_t p = blockIdx.x * 256 + threadIdx.x; p < npairs; p += gridDim.x * 256) {
    // the two columns of pair p: (2i, 2i+1) of a head for RopeType::Normal, (i, i + d/2) for NeoX (ops.rs:1316-1331); V: plain pairs
    const bool isq = p < nq, isk = !isq && p < nq + nk;
    const uint32_t pr = isq ? p : isk ? p - nq : p - nq - nk;           // pair index inside its region
    const uint32_t base = isq ? 0 : isk ? QD : QD + KD;                 // first column of the region
    const bool rot = isq || isk;
    const uint32_t i = rot ? (neox ? pr % half : (2 * pr % head_dim) / 2) : 0;
    const uint32_t r0 = rot && neox ? (pr / half) * head_dim + i : 2 * pr, r1 = rot && neox ? r0 + half : r0 + 1;   // rows of the matrix
    float x0 = 0.0f, x1 = 0.0f;
    for (uint32_t s = 0; s < S; s++) {
      const float* row = part + ((size_t)s * kPfTokens + t) * ncols + base;
      x0 += row[r0];
      x1 += row[r1];
    }
    x0 *= inv;
    x1 *= inv;
    const float* b = isq ? bq : isk ? bk : bv;
    if (b) { x0 += b[r0]; x1 += b[r1]; }
    float y0 = x0, y1 = x1;
    if (rot) {
      const float cs = rope_cs[((size_t)pos * half + i) * 2], sn = rope_cs[((size_t)pos * half + i) * 2 + 1];
      y0 = x0 * cs - x1 * sn;
      y1 = x0 * sn + x1 * cs;
    }
    if (isq) {
      qbuf[(size_t)t * QD + r0] = y0;
      qbuf[(size_t)t * QD + r1] = y1;
    } else {
      float* cache = isk ? kcache : vcache;
      cache[((size_t)(r0 / head_dim) * max_seq + pos) * head_dim + (r0 % head_dim)] = y0;
      cache[((size_t)(r1 / head_dim) * max_seq + pos) * head_dim + (r1 % head_dim)] = y1;
    }
  }
}

hipError_t pf_qkv_epi_launch(const float* part, uint32_t S, uint32_t ncols, uint32_t QD, uint32_t KD, uint32_t head_dim, const float* bq,
                             const float* bk, const float* bv, const float* rope_cs, uint32_t pos0, uint32_t max_seq, float* qbuf,
                             float* kcache, float* vcache, const float* ssq, uint32_t H, float eps, int neox, uint32_t m_tokens, hipStream_t st) {
  if (head_dim % 2 || ncols != QD + 2 * KD) return hipErrorInvalidValue;
  hipLaunchKernelGGL(pf_qkv_epi_kernel, dim3(((QD + 2 * KD) / 2 + 255) / 256, m_tokens), dim3(256), 0, st, part, S, ncols, QD, KD, head_dim, bq, bk, bv, rope_cs, pos0, max_seq,
                     qbuf, kcache, vcache, ssq, pf_ssq_chunks(H), H, eps, neox);
  return hipGetLastError();
}

// act = silu(gate) * up (simd.rs:598-649) from the partial sums (gate in columns [0, F), up in [F, 2F)) -> XH[t][F]
__global__ void __launch_bounds__(256) pf_swiglu_kernel(const float* __restrict__ part, uint32_t S, uint32_t F, uint8_t* __restrict__ xh,
                                                        const float* __restrict__ ssq, uint32_t n_ssq, uint32_t H, float eps,
                                                        const int* __restrict__ row_tok, const int* __restrict__ m_count) {
  const uint32_t t = blockIdx.y, ch = blockIdx.x * 256 + threadIdx.x;
  if (ch >= F / 8 || (m_count && t >= (uint32_t)*m_count)) return;
  // MoE: row t of this expert's batch is token row_tok[t] & 0xFF (its 1/rms), dense: row t is token t
  const float inv = pf_inv_rms(ssq, n_ssq, row_tok ? (uint32_t)row_tok[t] & 0xFFu : t, H, eps);
  float g[8] = {0, 0, 0, 0, 0, 0, 0, 0}, u[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  for (uint32_t s = 0; s < S; s++) {
    const float* row = part + ((size_t)s * kPfTokens + t) * (2 * (size_t)F);
    const f32x4 g0 = *reinterpret_cast<const f32x4*>(row + ch * 8), g1 = *reinterpret_cast<const f32x4*>(row + ch * 8 + 4);
    const f32x4 u0 = *reinterpret_cast<const f32x4*>(row + F + ch * 8), u1 = *reinterpret_cast<const f32x4*>(row + F + ch * 8 + 4);
#pragma unroll
    for (int j = 0; j < 4; j++) { g[j] += g0[j]; g[4 + j] += g1[j]; u[j] += u0[j]; u[4 + j] += u1[j]; }
  }
  float v[8];
#pragma unroll
  for (int j = 0; j < 8; j++) v[j] = silu_act_f(g[j] * inv) * (u[j] * inv);
  xh_store_chunk(xh, t, ch, v);
}

hipError_t pf_swiglu_launch(const float* part, uint32_t S, uint32_t F, uint8_t* xh, const float* ssq, uint32_t H, float eps, uint32_t m_tokens,
                            hipStream_t st, const int* row_tok, const int* m_count) {
  if (F % 8) return hipErrorInvalidValue;
  hipLaunchKernelGGL(pf_swiglu_kernel, dim3((F / 8 + 255) / 256, m_tokens), dim3(256), 0, st, part, S, F, xh, ssq, pf_ssq_chunks(H), H, eps, row_tok, m_count);
  return hipGetLastError();
}

// ------------------------------------------------------------------------------------------------
// MoE layers: tokens grouped by expert so that every expert's matrices are read once per block of tokens
// ------------------------------------------------------------------------------------------------
// Routing table -> per-expert row lists in ONE row space (prefill.h).  One wave per expert (round-robin): 64 routing entries per
// step, positions by ballot + popcount, entry order (token-major) kept.  (A thread per expert walking the table entry by entry
// took 30 us: 256 dependent LDS reads.)  Pass 0 counts, thread 0 lays out the bases (padded to 16 rows), pass 1 writes.
__global__ void __launch_bounds__(256) pf_moe_group_kernel(const int* __restrict__ sel, uint32_t m_tokens, uint32_t top_k, uint32_t n_experts,
                                                           int* __restrict__ counts, int* __restrict__ bases, int* __restrict__ lists,
                                                           int* __restrict__ rowmap, int* __restrict__ tokmap) {
  __shared__ int s_sel[kPfTokens * kPfMaxTopK];
  __shared__ int s_cnt[kPfMaxExperts], s_base[kPfMaxExperts];
  const uint32_t n = m_tokens * top_k;
  for (uint32_t i = threadIdx.x; i < n; i += 256) s_sel[i] = sel[i];
  for (uint32_t r = threadIdx.x; r < (uint32_t)kPfMoeRows; r += 256) rowmap[r] = -1;
  __syncthreads();
  const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int pass = 0; pass < 2; pass++) {
    for (uint32_t e = wave; e < n_experts; e += 4) {
      uint32_t pos0 = 0;
      const uint32_t base = pass ? (uint32_t)s_base[e] : 0u;
      for (uint32_t j0 = 0; j0 < n; j0 += 64) {
        const uint32_t i = j0 + lane;
        const bool hit = i < n && (uint32_t)s_sel[i] == e;
        const unsigned long long mask = __ballot(hit);
        const uint32_t pos = pos0 + (uint32_t)__popcll(mask & ((1ull << lane) - 1ull));
        if (pass && hit && pos < (uint32_t)kPfTokens) {
          lists[e * kPfTokens + pos] = (int)((i / top_k) | (i % top_k) << 8);
          rowmap[base + pos] = (int)(e | pos << 8);
          tokmap[i] = (int)(base + pos);
        }
        pos0 += (uint32_t)__popcll(mask);
      }
      if (!pass && lane == 0) s_cnt[e] = (int)(pos0 < (uint32_t)kPfTokens ? pos0 : (uint32_t)kPfTokens);
    }
    __syncthreads();
    if (!pass && threadIdx.x == 0) {
      int b = 0;
      for (uint32_t e = 0; e < n_experts; e++) {
        s_base[e] = b;
        counts[e] = s_cnt[e];
        bases[e] = b;
        b += (s_cnt[e] + 15) & ~15;
      }
    }
    __syncthreads();
  }
}

hipError_t pf_moe_group_launch(const int* sel, uint32_t m_tokens, uint32_t top_k, uint32_t n_experts, int* counts, int* bases, int* lists,
                               int* rowmap, int* tokmap, hipStream_t st) {
  // rows: m * top_k real ones + up to 15 of padding per expert
  if (n_experts > (uint32_t)kPfMaxExperts || top_k == 0 || top_k > (uint32_t)kPfMaxTopK || m_tokens > (uint32_t)kPfTokens ||
      m_tokens * top_k + 15 * n_experts > (uint32_t)kPfMoeRows)
    return hipErrorInvalidValue;
  hipLaunchKernelGGL(pf_moe_group_kernel, dim3(1), dim3(256), 0, st, sel, m_tokens, top_k, n_experts, counts, bases, lists, rowmap, tokmap);
  return hipGetLastError();
}

// row i of the expert's XH batch = the XH row of token list[i] (the chunk swizzle depends on the row index: re-swizzled)
// (all experts in one launch: blockIdx.z = expert, its list / count / output at stride kPfTokens / 1 / out_stride)
__global__ void __launch_bounds__(256) pf_moe_gather_kernel(const uint8_t* __restrict__ xh, const int* __restrict__ list, const int* __restrict__ count,
                                                            uint8_t* __restrict__ xh_out, size_t out_stride) {
  const uint32_t slab = blockIdx.x, i = blockIdx.y * 8 + (threadIdx.x >> 5), q = threadIdx.x & 31;
  list += blockIdx.z * kPfTokens;
  count += blockIdx.z;
  xh_out += blockIdx.z * out_stride;
  if (i >= (uint32_t)*count) return;
  const uint32_t ts = (uint32_t)list[i] & 0xFFu;
  const u32x4 v = *reinterpret_cast<const u32x4*>(xh + (size_t)slab * kPfSlabBytes + ts * 512 + ((q ^ (ts & 15)) << 4));
  *reinterpret_cast<u32x4*>(xh_out + (size_t)slab * kPfSlabBytes + i * 512 + ((q ^ (i & 15)) << 4)) = v;
}

hipError_t pf_moe_gather_launch(const uint8_t* xh, uint32_t K, const int* lists, const int* counts, uint8_t* xh_out, uint32_t n_experts,
                                hipStream_t st) {
  if (K % 256 || n_experts == 0 || n_experts > (uint32_t)kPfMaxExperts) return hipErrorInvalidValue;
  hipLaunchKernelGGL(pf_moe_gather_kernel, dim3(K / 256, kPfTokens / 8, n_experts), dim3(256), 0, st, xh, lists, counts, xh_out, xh_bytes(K));
  return hipGetLastError();
}

// act = silu(gate) * up (simd.rs:598-649) for the rows of ALL experts: row r of the shared row space belongs to expert
// rowmap[r] & 0xFF, is its row rowmap[r] >> 8, and carries the 1/rms of token lists[e][i] & 0xFF
__global__ void __launch_bounds__(256) pf_moe_swiglu_kernel(const float* __restrict__ part, uint32_t S, uint32_t F, uint8_t* __restrict__ xh_out,
                                                            size_t out_stride, const int* __restrict__ rowmap, const int* __restrict__ lists,
                                                            const float* __restrict__ ssq, uint32_t n_ssq, uint32_t H, float eps) {
  const uint32_t r = blockIdx.y, ch = blockIdx.x * 256 + threadIdx.x;
  const int rm = rowmap[r];
  if (rm < 0 || ch >= F / 8) return;
  const uint32_t e = (uint32_t)rm & 0xFFu, i = (uint32_t)rm >> 8;
  const float inv = pf_inv_rms(ssq, n_ssq, (uint32_t)lists[e * kPfTokens + i] & 0xFFu, H, eps);
  float g[8] = {0, 0, 0, 0, 0, 0, 0, 0}, u[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  for (uint32_t s = 0; s < S; s++) {
    const float* row = part + ((size_t)s * kPfMoeRows + r) * (2 * (size_t)F);
    const f32x4 g0 = *reinterpret_cast<const f32x4*>(row + ch * 8), g1 = *reinterpret_cast<const f32x4*>(row + ch * 8 + 4);
    const f32x4 u0 = *reinterpret_cast<const f32x4*>(row + F + ch * 8), u1 = *reinterpret_cast<const f32x4*>(row + F + ch * 8 + 4);
#pragma unroll
    for (int j = 0; j < 4; j++) { g[j] += g0[j]; g[4 + j] += g1[j]; u[j] += u0[j]; u[4 + j] += u1[j]; }
  }
  float v[8];
#pragma unroll
  for (int j = 0; j < 8; j++) v[j] = silu_act_f(g[j] * inv) * (u[j] * inv);
  xh_store_chunk(xh_out + e * out_stride, i, ch, v);
}

hipError_t pf_moe_swiglu_launch(const float* part, uint32_t S, uint32_t F, uint8_t* xh_out, const int* rowmap, const int* lists,
                                const float* ssq, uint32_t H, float eps, hipStream_t st) {
  if (F % 256) return hipErrorInvalidValue;
  hipLaunchKernelGGL(pf_moe_swiglu_kernel, dim3((F / 8 + 255) / 256, kPfMoeRows), dim3(256), 0, st, part, S, F, xh_out, xh_bytes(F), rowmap, lists, ssq,
                     pf_ssq_chunks(H), H, eps);
  return hipGetLastError();
}

// MoeLayer::forward's tail (moe.rs:363-368) + the layer's residual for every token of the block: out = 0; out += w[s] * expert
// output of slot s, in selection order; h += out; then the next layer's XH and sums of squares (as pf_resid_kernel).
__global__ void __launch_bounds__(256) pf_moe_combine_kernel(const float* __restrict__ part, uint32_t S, const int* __restrict__ tokmap,
                                                             const float* __restrict__ moe_w, uint32_t top_k, float* __restrict__ hidden, uint32_t H,
                                                             const float* __restrict__ nw, uint8_t* __restrict__ xh, float* __restrict__ ssq) {
  __shared__ float s_ss[4];
  const uint32_t t = blockIdx.y, ch = blockIdx.x * 256 + threadIdx.x, i = ch * 8;
  float ss = 0.0f;
  if (i < H) {
    f32x4 a0 = (f32x4)(0.0f), a1 = (f32x4)(0.0f);
    for (uint32_t s = 0; s < top_k; s++) {
      const uint32_t row = (uint32_t)tokmap[t * top_k + s];
      f32x4 y0 = (f32x4)(0.0f), y1 = (f32x4)(0.0f);
      for (uint32_t sp = 0; sp < S; sp++) {
        const float* p = part + ((size_t)sp * kPfMoeRows + row) * H + i;
        y0 += *reinterpret_cast<const f32x4*>(p);
        y1 += *reinterpret_cast<const f32x4*>(p + 4);
      }
      const float w = moe_w[t * top_k + s];
      a0 += y0 * w;
      a1 += y1 * w;
    }
    const f32x4 v0 = *reinterpret_cast<const f32x4*>(hidden + (size_t)t * H + i) + a0;
    const f32x4 v1 = *reinterpret_cast<const f32x4*>(hidden + (size_t)t * H + i + 4) + a1;
    *reinterpret_cast<f32x4*>(hidden + (size_t)t * H + i) = v0;
    *reinterpret_cast<f32x4*>(hidden + (size_t)t * H + i + 4) = v1;
    const f32x4 q = v0 * v0 + v1 * v1;
    ss = (q.x + q.y) + (q.z + q.w);
    if (xh) {
      const f32x4 w0 = *reinterpret_cast<const f32x4*>(nw + i), w1 = *reinterpret_cast<const f32x4*>(nw + i + 4);
      float v[8];
#pragma unroll
      for (int j = 0; j < 4; j++) { v[j] = v0[j] * w0[j]; v[4 + j] = v1[j] * w1[j]; }
      xh_store_chunk(xh, t, ch, v);
    }
  }
  ss = wave_sum(ss);
  if ((threadIdx.x & 63) == 0) s_ss[threadIdx.x >> 6] = ss;
  __syncthreads();
  if (threadIdx.x == 0 && ssq) ssq[t * kPfSsqChunks + blockIdx.x] = (s_ss[0] + s_ss[1]) + (s_ss[2] + s_ss[3]);
}

hipError_t pf_moe_combine_launch(const float* part, uint32_t S, const int* tokmap, const float* moe_w, uint32_t top_k, float* hidden, uint32_t H,
                                 const float* nw, uint8_t* xh, float* ssq, uint32_t m_tokens, hipStream_t st) {
  if (H % 8 || (xh && (!nw || !ssq)) || pf_ssq_chunks(H) > (uint32_t)kPfSsqChunks) return hipErrorInvalidValue;
  hipLaunchKernelGGL(pf_moe_combine_kernel, dim3(pf_ssq_chunks(H), m_tokens), dim3(256), 0, st, part, S, tokmap, moe_w, top_k, hidden, H, nw, xh, ssq);
  return hipGetLastError();
}

// plain f32 [M][K] -> XH (no scaling): the attention output in front of wo
__global__ void __launch_bounds__(256) pf_to_xh_kernel(const float* __restrict__ x, uint32_t K, uint8_t* __restrict__ xh) {
  const uint32_t t = blockIdx.y, ch = blockIdx.x * 256 + threadIdx.x;
  if (ch >= K / 8) return;
  float v[8];
#pragma unroll
  for (int j = 0; j < 8; j++) v[j] = x[(size_t)t * K + ch * 8 + j];
  xh_store_chunk(xh, t, ch, v);
}

hipError_t pf_to_xh_launch(const float* x, uint32_t K, uint8_t* xh, uint32_t m_tokens, hipStream_t st) {
  if (K % 8) return hipErrorInvalidValue;
  hipLaunchKernelGGL(pf_to_xh_kernel, dim3((K / 8 + 255) / 256, m_tokens), dim3(256), 0, st, x, K, xh);
  return hipGetLastError();
}

}  // namespace lgh
