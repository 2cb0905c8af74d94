// prefill_wide.hip — long prompts: products of quantized weights with up to kPfwTokens prompt tokens at once on the f16 matrix cores
// (v_mfma_f32_32x32x16_f16), and the row kernels around them.
//
// prefill.hip takes 128 tokens per weight read; its loop is bound by the vector issue port, because every weight is dequantized for 128
// tokens only, and a product of 128 tokens must be split over k to fill the chip, which costs partial sums and a row kernel to fold them.
// Here a workgroup keeps 256 weight rows x 256 tokens (256 f32 accumulators per lane): a dequantized weight feeds twice as many products, the loop is
// bound by the matrix pipe, and from about 512 tokens on the widest matrices need no split at all, so that SwiGLU runs in the epilogue.
//
// Activations: row-major f16, [token][K].  Same operands, same rounding points and f32 accumulation as prefill.hip.
//
// Measured: 2047 tokens of Llama-3-8B Q4_K_M widths, 16 layers: 44.4 ms in blocks of 128, 18.4 ms here with attention_wide.hip (gate | up 0.44 to 0.47 ms a layer from box
// to box = 1.02 to 1.09 PFLOP/s; torch's f16 product of 8192^3 reaches 1.14); 600 tokens of Mixtral widths, 2 layers: 2.99 and 1.31 ms.  What bounds it: the chip's power
// before any single unit (the same loop without the dequantization takes 26 % less time, without the activations' DMA 22 %, without the stores 11 %).
// Eight waves of half the tokens each (two per SIMD, weights dequantized twice) took the same time.
#include "mv_epilogue.h"
#include "prefill_dequant.h"

namespace lgh {

typedef float f32x2 __attribute__((ext_vector_type(2)));

constexpr int kWWaves = 4, kWRT = 4;                      // waves of a workgroup, 16-row weight tiles of a wave
constexpr uint32_t kWStepBytes = kPfwTile * 128;          // 64 elements of 256 tokens

template <int F> constexpr uint32_t pw_full() { return pf_tile_bytes(F) / 1024; }                         // whole 1 KB pieces of a tile
template <int F> constexpr uint32_t pw_tail() { return (pf_tile_bytes(F) - pw_full<F>() * 1024) / 16; }   // 16-byte units behind them
template <int F> constexpr uint32_t pw_tail_ops() { return (kWRT * pw_tail<F>() + 63) / 64; }
template <int F> constexpr uint32_t pw_raw_ops() { return kWRT * pw_full<F>() + pw_tail_ops<F>(); }       // DMA operations per wave and 256 elements
template <int F> constexpr uint32_t pw_raw_bytes() { return pw_raw_ops<F>() * 1024; }                     // a wave's LDS for them
// three activation buffers where they fit beside the raw weights (Q8_0: two)
template <int F> constexpr uint32_t pw_bufs() { return 3 * kWStepBytes + kWWaves * pw_raw_bytes<F>() <= 160 * 1024 ? 3 : 2; }
constexpr uint32_t pw_lds(int f) {
  return f == PF_Q4K ? pw_bufs<PF_Q4K>() * kWStepBytes + kWWaves * pw_raw_bytes<PF_Q4K>()
         : f == PF_Q6K ? pw_bufs<PF_Q6K>() * kWStepBytes + kWWaves * pw_raw_bytes<PF_Q6K>()
         : f == PF_Q5K ? pw_bufs<PF_Q5K>() * kWStepBytes + kWWaves * pw_raw_bytes<PF_Q5K>()
         : f == PF_Q80 ? pw_bufs<PF_Q80>() * kWStepBytes + kWWaves * pw_raw_bytes<PF_Q80>()
                       : pw_bufs<PF_Q40>() * kWStepBytes + kWWaves * pw_raw_bytes<PF_Q40>();
}

// 16 bytes per lane from global memory into LDS at lds + 16 * lane.  Inline assembly: the compiler's wait-count pass does not see these loads (it would wait
// for all of them before any LDS read); the loop below waits by hand.
__device__ __forceinline__ void pw_dma(const uint8_t* base, uint32_t off, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(off), "s"(base), "s"(lds) : "memory", "m0");
}
// all but the last N vector-memory operations of this wave have completed
template <uint32_t N> __device__ __forceinline__ void pw_wait_vm() { __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14)); }

// The 32 x 32 shape: with one wave per SIMD the 16 x 16 x 32 one sustains 1.25 PFLOP/s on this chip, this one 1.66 (random operands, nothing but MFMAs).
__device__ __forceinline__ void pw_mma(f32x16& acc, h16x8 a, h16x8 b) { acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, acc, 0, 0, 0); }
// keeps a token tile's sums in their accumulation registers until the stores of the one before are under way (read all at once they spill)
__device__ __forceinline__ void pw_settle(f32x16& a, f32x16& b) { asm volatile("" : "+a"(a), "+a"(b) : : "memory"); }

// raw weights of row n of tile r as lane `l16` of the 16-row scheme holds them (chunk l16 >> 4 of every 64 elements)
template <int F> __device__ __forceinline__ void pw_raw_read(PfRaw& w, const uint8_t* raw, uint32_t r, uint32_t l16, uint32_t n) {
  constexpr uint32_t nf = pw_full<F>();
  const uint8_t* full = raw + r * (nf * 1024) + l16 * 16;
  const uint8_t* tail = raw + kWRT * nf * 1024 + r * (pw_tail<F>() * 16);
  w.hd = *reinterpret_cast<const u32x4*>(tail + n * 16);
#pragma unroll
  for (int i = 0; i < (int)nf; i++) w.q[i] = *reinterpret_cast<const u32x4*>(full + i * 1024);
  if (F == PF_Q6K) w.q[3].x = *reinterpret_cast<const uint32_t*>(tail + 256 + (n >> 1) * 4);
  if (F == PF_Q5K) {
    const u32x2 h = *reinterpret_cast<const u32x2*>(tail + 256 + l16 * 8);
    w.q[2].x = h.x;
    w.q[2].y = h.y;
  }
}

// One workgroup: 16 row tiles x up to TT token tiles of 32 over the k-blocks [b0, b1).  A wave's four 16-row tiles are two of 32 rows: lane 32g + 16s + n
// holds row n of tile 2v + s, and of every 64 elements the two 16-element chunks 2g + j that the tile16 layout keeps for lanes 16(2g + j) + n.  A step of
// 64 elements has four phases (j, h), each the contraction of elements 16(2g + j) + 8h .. + 7 of both g, 2 * TT MFMAs.  A operands are dequantized in
// registers one phase ahead, B operands (all tokens) are read from LDS three units ahead.
// What arrives by DMA: the activations of the step after next (256 tokens x 128 bytes, shared by the waves), and per 256 elements the wave's own raw
// weights.  The barrier stands three units before a step's end, where every read of the step's buffer has returned, so that the next step's first
// operands are under way when its first MFMA issues.
template <int F, int TT, bool GRP, int EPI>
__device__ __forceinline__ void pw_body(const PfWide& G, const PfwSeg& sg, uint32_t rg, uint32_t ks, uint32_t m0, uint32_t m_end, uint32_t expert, uint8_t* smem) {
  constexpr uint32_t tb = pf_tile_bytes(F), NB = pw_bufs<F>(), DIST = NB - 1;
  constexpr int NX = TT;   // NX: activation DMA operations per wave and step
  constexpr int UN = 4 * TT, AHEAD = 3;                                                     // units (phase, token tile) of a step
  constexpr int RPP = TT > 4 && TT % 2 == 0 ? 2 : 1, RU = TT / RPP;                         // regions of a phase, units of a region
  const uint32_t lane = threadIdx.x & 63, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const uint32_t n = lane & 15, g = lane >> 5, tk = lane & 31, sub = lane >> 4 & 1;
  const uint32_t per = (G.nblk + G.S - 1) / G.S, b0 = ks * per, b1 = b0 + per < G.nblk ? b0 + per : G.nblk;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem;
  const uint32_t raw_at = NB * kWStepBytes + wave * pw_raw_bytes<F>();
  uint8_t* raw = smem + raw_at;

  // this wave's row tiles; SwiGLU: two gate tiles and the two up tiles of the same columns
  uint32_t tl[kWRT];
#pragma unroll
  for (int r = 0; r < kWRT; r++) {
    const uint32_t t = EPI == PW_SWIGLU ? (rg * kWWaves + wave) * 2 + (r & 1) : (rg * kWWaves + wave) * kWRT + r;
    tl[r] = t < sg.ntiles ? t : sg.ntiles - 1;   // clamped: loads are unconditional
  }
  const uint8_t* wbase[kWRT];
#pragma unroll
  for (int r = 0; r < kWRT; r++) {
    const uint8_t* w = EPI == PW_SWIGLU && r >= 2 ? G.seg[1].w + expert * G.seg[1].expert_stride : sg.w + expert * sg.expert_stride;
    wbase[r] = w + (size_t)tl[r] * G.nblk * tb;
  }
  // tails of the four tiles side by side: this lane's unit of each operation
  uint64_t tail_src[pw_tail_ops<F>()];
#pragma unroll
  for (int i = 0; i < (int)pw_tail_ops<F>(); i++) {
    uint32_t u = i * 64 + lane;
    if (u >= kWRT * pw_tail<F>()) u = kWRT * pw_tail<F>() - 1;
    const uint32_t r = u / pw_tail<F>(), j = u % pw_tail<F>();
    const uint8_t* w = r == 0 ? wbase[0] : r == 1 ? wbase[1] : r == 2 ? wbase[2] : wbase[3];
    tail_src[i] = (uint64_t)(uintptr_t)(w + pw_full<F>() * 1024 + j * 16);
  }
  constexpr int R = (int)pw_raw_ops<F>(), NF = (int)pw_full<F>();
  auto raw_dma = [&](int k, uint32_t b) {   // operation k of a block's raw weights
    const uint32_t at = lds0 + raw_at + k * 1024;
    const size_t bo = (size_t)b * tb;
    if (k < kWRT * NF) {
      pw_dma(wbase[k / NF] + bo + k % NF * 1024, lane * 16, at);
    } else {
      const uint8_t* src = reinterpret_cast<const uint8_t*>(tail_src[k - kWRT * NF]) + bo;
      asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(src), "s"(at) : "memory", "m0");
    }
  };
  // activations: an operation covers 8 tokens x 128 bytes; chunk q of token t lies at position q ^ (t >> 1 & 7): 16 tokens' places
  // differ in their banks, two of a parity included (with t & 7 every second read waited for another: half of the LDS' cycles, 62.8 -> 33.4 M a launch of gate | up of 2047 tokens; the launch 435.8 and 435.7 us, experts' of 600 tokens 464 -> 460)
  uint32_t xoff[NX];
#pragma unroll
  for (int i = 0; i < (int)NX; i++) {
    const uint32_t row = (wave * NX + i) * 8 + (lane >> 3);
    uint32_t m = m0 + row < m_end ? m0 + row : m_end - 1;
    if (GRP && G.src) m = (uint32_t)G.src[m];
    xoff[i] = m * (G.nblk * 512u) + (((lane & 7) ^ (row >> 1 & 7)) << 4);
  }
  const uint32_t s0 = b0 * 4, s1 = b1 * 4;   // steps of 64 elements
  // regions of a step; raw operations per region, spread over a block's first two steps, and how many of them each of the two makes
  constexpr int RS = 4 * RPP, RP = (R + 2 * RS - 1) / (2 * RS), R0 = R < RS * RP ? R : RS * RP, R1 = R - R0;
  constexpr int XP = (NX + RS - 1) / RS;   // activation operations per region
  static_assert(TT % RPP == 0 && RU >= AHEAD, "the last region holds what is awaited");
  auto x_dma = [&](int i, uint32_t s, uint32_t buf) {   // operation i of a step's activations
    const uint8_t* base = G.x + (size_t)(s < s1 ? s : s1 - 1) * 128;   // past the end: requested again, never read
    pw_dma(base, xoff[i], lds0 + buf * kWStepBytes + (wave * NX + i) * 1024);
  };

  f32x16 acc[2][TT];
#pragma unroll
  for (int v = 0; v < 2; v++)
#pragma unroll
    for (int t = 0; t < TT; t++) acc[v][t] = (f32x16)(0.0f);

#pragma unroll
  for (int k = 0; k < R; k++) raw_dma(k, b0);
#pragma unroll
  for (int i = 0; i < NX; i++) x_dma(i, s0, 0);
  if (NB == 3) {
#pragma unroll
    for (int i = 0; i < NX; i++) x_dma(i, s0 + 1, 1);
  }
  pw_wait_vm<NB == 3 ? NX : 0>();
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");

  uint32_t bo[4];   // this lane's place in a token tile, per phase
#pragma unroll
  for (int p = 0; p < 4; p++) bo[p] = tk * 128 + (((4 * g + p) ^ (tk >> 1 & 7)) << 4);
  PfRaw w[2][2];    // [v][j]
  h16x2 S[2], O[2];
  h16x8 af[2][2], bf[4];
  auto raw_read = [&]() {
#pragma unroll
    for (int v = 0; v < 2; v++)
#pragma unroll
      for (int j = 0; j < 2; j++) pw_raw_read<F>(w[v][j], raw, 2 * v + sub, 16 * (2 * g + j) + n, n);
  };
  auto operand = [&](int v, int pp, int p, h16x8& out) {   // phase p = (j, h)
    if (p == 0 || (F == PF_Q6K && p == 2)) pf_scale<F>(w[v][p >> 1], pp, n, 2 * g + (p >> 1), S[v], O[v]);
    out = pf_frag<F>(w[v][p >> 1], pp, p & 1, S[v], O[v]);
  };
  raw_read();
#pragma unroll
  for (int v = 0; v < 2; v++) operand(v, 0, 0, af[0][v]);
  uint32_t cur = 0, nxt = 1, far = NB - 1;   // buffers of this step, the next one, and the one to request
  auto rd = [&](uint32_t buf, int u) { return *reinterpret_cast<const h16x8*>(smem + buf * kWStepBytes + bo[u / TT] + (u % TT) * 4096); };
#pragma unroll
  for (int u = 0; u < AHEAD; u++) bf[u] = rd(0, u);

  for (uint32_t b = b0; b < b1; b++) {
#pragma unroll
    for (int pp = 0; pp < 4; pp++) {
      const uint32_t s = b * 4 + pp;
      if (pp == 0) __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0): the raw weights of this block are in registers
      if (NB == 2) {
#pragma unroll
        for (int i = 0; i < NX; i++) x_dma(i, s + DIST, far);
      }
#pragma unroll
      for (int r = 0; r < RS; r++) {   // regions of 3 to 7 units: two MFMAs and an operand read each, one or both of the next phase's A operands, and the DMA piece by piece
        if (NB == 3) {
#pragma unroll
          for (int i = r * XP; i < (r + 1) * XP; i++)
            if (i < NX) x_dma(i, s + DIST, far);
        }
        if (pp < 2) {
#pragma unroll
          for (int k = (pp * RS + r) * RP; k < (pp * RS + r + 1) * RP; k++)
            if (k < R) raw_dma(k, b + 1 < b1 ? b + 1 : b);
        }
        const int p = r / RPP;
#pragma unroll
        for (int ru = 0; ru < RU; ru++) {
          const int u = r * RU + ru;
          if (u == UN - AHEAD) {   // the last reads of this buffer were issued by the unit before
            __builtin_amdgcn_sched_barrier(0);
            constexpr uint32_t XW = NB == 3 ? NX : 0;   // what this step has requested for later ones may be under way
            if (pp == 0) pw_wait_vm<XW + R0>(); else if (pp == 1) pw_wait_vm<XW + R1>(); else pw_wait_vm<XW>();
            __builtin_amdgcn_s_waitcnt(0xC07F);
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
          }
          bf[(u + AHEAD) & 3] = u + AHEAD < UN ? rd(cur, u + AHEAD) : rd(nxt, u + AHEAD - UN);
#pragma unroll
          for (int v = 0; v < 2; v++) pw_mma(acc[v][u % TT], af[p & 1][v], bf[u & 3]);
        }
        const int p2 = (p + 1) & 3, pp2 = p == 3 ? (pp + 1) & 3 : pp, ri = r % RPP;
        if (RPP == 2) {
          operand(ri, pp2, p2, af[p2 & 1][ri]);
        } else {
          operand(0, pp2, p2, af[p2 & 1][0]);
          operand(1, pp2, p2, af[p2 & 1][1]);
        }
        if (pp == 3 && p == 2 && ri == RPP - 1) raw_read();   // the block's last operands are made: the next block's weights
        // one MFMA keeps the matrix pipe busy for 32 cycles, in which this wave can issue a few other instructions: a quarter of the region's between any two
#pragma unroll
        for (int i = 0; i < 2 * RU; i++) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                    // MFMA
          if (i % 2 == 0) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);    // LDS read
          __builtin_amdgcn_sched_group_barrier(0x002, 24 * (3 - RPP) / (2 * RU), 0);   // vector
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      cur = nxt;
      nxt = nxt + 1 == NB ? 0 : nxt + 1;
      far = far + 1 == NB ? 0 : far + 1;
    }
  }
  pw_wait_vm<0>();   // what was requested past the end has landed before the LDS is given back

  // A lane holds, per (32 rows, 32 tokens), rows 8i + 4g .. + 3 (i = 0 .. 3) of token tk.  A wave turns each token tile round in LDS (the activation buffers
  // are free), so that a token's 64 sums (32 activations) leave in one piece: stored as they lie, every token's 32 bytes of an instruction are a piece
  // of their own, and this phase took a seventh of the kernel.
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  uint8_t* turn = smem + wave * (32 * 68 * 4);
#pragma unroll
  for (int t = 0; t < TT; t++) {
    pw_settle(acc[0][t], acc[1][t]);
    if constexpr (EPI == PW_SWIGLU) {
      const uint32_t m = min(m0 + t * 32 + tk, m_end - 1);
      const float inv = G.inv_rms[GRP ? (uint32_t)G.src[m] : m] * (1.0f / kPfScale);
#pragma unroll
      for (int i = 0; i < 4; i++) {
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = silu_act_f(acc[0][t][4 * i + e] * inv) * (acc[1][t][4 * i + e] * inv);
        const h16x4 o = {(_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)v[3]};
        *reinterpret_cast<h16x4*>(turn + tk * 80 + i * 16 + g * 8) = o;
      }
#pragma unroll
      for (int j = 0; j < 2; j++) {
        const uint32_t tok = j * 16 + (lane >> 2), q = lane & 3, mo = m0 + t * 32 + tok, tile = (rg * kWWaves + wave) * 2 + (q >> 1);
        const h16x8 o = *reinterpret_cast<const h16x8*>(turn + tok * 80 + q * 16);
        if (mo < m_end && tile < sg.ntiles) *reinterpret_cast<h16x8*>(G.act + ((size_t)mo * G.act_cols + tile * 16 + (q & 1) * 8) * 2) = o;
      }
    } else {
#pragma unroll
      for (int v = 0; v < 2; v++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const f32x4 o = {acc[v][t][4 * i], acc[v][t][4 * i + 1], acc[v][t][4 * i + 2], acc[v][t][4 * i + 3]};
          *reinterpret_cast<f32x4*>(turn + tk * 272 + (32 * v + 8 * i + 4 * g) * 4) = o * (1.0f / kPfScale);
        }
      float* part = G.part + (size_t)ks * G.part_rows * G.ncols + sg.col0;
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const uint32_t tok = j * 4 + (lane >> 4), mo = m0 + t * 32 + tok, row = (rg * kWWaves + wave) * (kWRT * 16) + n * 4;
        const f32x4 o = *reinterpret_cast<const f32x4*>(turn + tok * 272 + n * 16);
        if (mo < m_end && row < sg.ntiles * 16) *reinterpret_cast<f32x4*>(part + (size_t)mo * G.ncols + row) = o;
      }
    }
  }
}

template <uint32_t MASK, bool GRP, int EPI>
__global__ void __launch_bounds__(kWWaves * 64) pw_gemm_kernel(const PfWide G, uint32_t n_rg, uint32_t tiles_m) {
  extern __shared__ __attribute__((aligned(16))) uint8_t pw_smem[];
  // token tiles of one weight panel side by side on one XCD (workgroups go round-robin over the 8 XCDs): the panel comes from HBM once per XCD.  A last
  // token tile that is at most three quarters or half full takes so much of the time: its workgroups are the last ones, to fill up the last round.
  uint32_t t = blockIdx.x, total = gridDim.x, wide = tiles_m, tm0 = 0;
  if (!GRP && tiles_m > 1 && (G.m - 1) % kPfwTile < kPfwTile * 3 / 4) {
    const uint32_t first = n_rg * G.S * (tiles_m - 1);
    wide = t < first ? tiles_m - 1 : 1;
    tm0 = t < first ? 0 : tiles_m - 1;
    total = t < first ? first : total - first;
    t -= t < first ? 0 : first;
  }
  {
    const uint32_t q = total / 8, r = total % 8, xcd = t % 8, i = t / 8;
    t = xcd * q + (xcd < r ? xcd : r) + i;
  }
  const uint32_t tm = tm0 + t % wide, ks = t / wide % G.S, rgid = t / (wide * G.S);
  uint32_t m0, m_end, expert = 0;
  if constexpr (GRP) {
    const int e = G.tile_e[tm];
    if (e < 0) return;
    expert = (uint32_t)e;
    m0 = (uint32_t)G.tile_row[tm];
    m_end = (uint32_t)G.row_seg[e + 1];
  } else {   // (G.m as a value the branch above replaces ended up in scratch, to be read through a flat address)
    m0 = tm * kPfwTile;
    m_end = G.m;
  }
  if (m_end - m0 > (uint32_t)kPfwTile) m_end = m0 + kPfwTile;
  int si = 0;
  if (EPI != PW_SWIGLU) {
    if (G.nseg > 1 && rgid >= G.seg[1].rg_begin) si = 1;
    if (G.nseg > 2 && rgid >= G.seg[2].rg_begin) si = 2;
  }
  const PfwSeg& sg = G.seg[si];
  const uint32_t rg = rgid - sg.rg_begin;
  auto is = [&](int f) { return (MASK & (1u << f)) && (MASK == (1u << f) || sg.fmt == f); };
  // Tiles of 256 tokens down to 96 in steps of 32: a product takes time with the tokens computed, and below 96 with the weights' dequantization.  256, 192 and 128 alone, then these: two layers of Mixtral Q5_K_M, 200 / 330 /
  // 600 tokens (experts of some 50, 80, 150 rows) 816 / 830 / 1196 -> 767 / 786 / 1167 us; 4 layers of an 8B model, last tiles of 148, 217 and 160 tokens (660, 729, 416): 1610 / 1706 / 1187 -> 1590 / 1685 / 1181.
  // (Before, 256 and 128 alone: experts of some 100 to 190 rows, 401 tokens of Mixtral widths: gate | up 364 -> 323 us with 192.)
#define LGH_PW_RUN(F)                                                                                       \
  do {                                                                                                      \
    switch ((m_end - m0 + 31) / 32) {                                                                       \
      case 8: pw_body<F, 8, GRP, EPI>(G, sg, rg, ks, m0, m_end, expert, pw_smem); break;                    \
      case 7: pw_body<F, 7, GRP, EPI>(G, sg, rg, ks, m0, m_end, expert, pw_smem); break;                    \
      case 6: pw_body<F, 6, GRP, EPI>(G, sg, rg, ks, m0, m_end, expert, pw_smem); break;                    \
      case 5: pw_body<F, 5, GRP, EPI>(G, sg, rg, ks, m0, m_end, expert, pw_smem); break;                    \
      case 4: pw_body<F, 4, GRP, EPI>(G, sg, rg, ks, m0, m_end, expert, pw_smem); break;                    \
      default: pw_body<F, 3, GRP, EPI>(G, sg, rg, ks, m0, m_end, expert, pw_smem); break;   /* (up to 96) */  \
    }                                                                                                       \
  } while (0)
  if (is(PF_Q4K)) LGH_PW_RUN(PF_Q4K);
  else if (is(PF_Q6K)) LGH_PW_RUN(PF_Q6K);
  else if (is(PF_Q5K)) LGH_PW_RUN(PF_Q5K);
  else if (is(PF_Q80)) LGH_PW_RUN(PF_Q80);
  else if (is(PF_Q40)) LGH_PW_RUN(PF_Q40);
#undef LGH_PW_RUN
}

template <uint32_t MASK, bool GRP, int EPI>
static hipError_t pw_go(const PfWide& G, uint32_t n_rg, uint32_t tiles_m, hipStream_t st) {
  static bool attr_set[64] = {};
  uint32_t lds = 0;
  for (int f = 0; f < 5; f++)
    if (MASK & (1u << f)) lds = std::max(lds, pw_lds(f));
  if (hipError_t e = lds_opt_in(reinterpret_cast<const void*>(&pw_gemm_kernel<MASK, GRP, EPI>), (int)lds, attr_set); e != hipSuccess) return e;
  hipLaunchKernelGGL((pw_gemm_kernel<MASK, GRP, EPI>), dim3(n_rg * tiles_m * G.S), dim3(kWWaves * 64), lds, st, G, n_rg, tiles_m);
  return hipGetLastError();
}
template <bool GRP, int EPI>
static hipError_t pw_pick(const PfWide& G, uint32_t mask, uint32_t n_rg, uint32_t tiles_m, hipStream_t st) {
  switch (mask) {
    case 1u << PF_Q4K: return pw_go<1u << PF_Q4K, GRP, EPI>(G, n_rg, tiles_m, st);
    case 1u << PF_Q6K: return pw_go<1u << PF_Q6K, GRP, EPI>(G, n_rg, tiles_m, st);
    case 1u << PF_Q5K: return pw_go<1u << PF_Q5K, GRP, EPI>(G, n_rg, tiles_m, st);
    case 1u << PF_Q80: return pw_go<1u << PF_Q80, GRP, EPI>(G, n_rg, tiles_m, st);
    case 1u << PF_Q40: return pw_go<1u << PF_Q40, GRP, EPI>(G, n_rg, tiles_m, st);
  }
  if constexpr (EPI == PW_PART && !GRP) {   // matrices of different formats in one launch (q, k, v)
    if (mask == ((1u << PF_Q4K) | (1u << PF_Q6K))) return pw_go<(1u << PF_Q4K) | (1u << PF_Q6K), GRP, EPI>(G, n_rg, tiles_m, st);
    if (mask == ((1u << PF_Q5K) | (1u << PF_Q6K))) return pw_go<(1u << PF_Q5K) | (1u << PF_Q6K), GRP, EPI>(G, n_rg, tiles_m, st);
  }
  if constexpr (EPI == PW_PART) {           // any other mix: one launch per matrix
    for (int i = 0; i < G.nseg; i++) {
      PfWide g = G;
      g.nseg = 1;
      g.seg[0] = G.seg[i];
      g.seg[0].rg_begin = 0;
      const uint32_t rg = (G.seg[i].ntiles + kWWaves * kWRT - 1) / (kWWaves * kWRT);
      if (hipError_t e = pw_pick<GRP, EPI>(g, 1u << G.seg[i].fmt, rg, tiles_m, st); e != hipSuccess) return e;
    }
    return hipSuccess;
  }
  return hipErrorInvalidValue;
}

static uint32_t pw_row_groups(uint32_t rows) { return (rows / 16 + kWWaves * kWRT - 1) / (kWWaves * kWRT); }

// k-splits: as many as fill the last round of workgroups (one per CU) without more than kPfwPartRows rows of partial sums
static uint32_t pw_splits(uint32_t n_rg, uint32_t tiles_m, uint32_t rows, uint32_t nblk) {
  uint32_t best = 1;
  float cost = 1e30f;
  for (uint32_t S = 1; S <= nblk && (S == 1 || S * rows <= (uint32_t)kPfwPartRows); S++) {
    const uint32_t per = (nblk + S - 1) / S;
    if ((nblk + per - 1) / per != S) continue;
    // rounds x (k-blocks of a workgroup + about one block's time for its prologue and epilogue), and the partial sums' fold
    const float rounds = (float)((n_rg * tiles_m * S + kNumCU - 1) / kNumCU);
    const float now = rounds * ((float)per + 1.0f) + (float)S * 0.4f;
    if (now < cost) { cost = now; best = S; }
  }
  return best;
}

bool pfw_pairs(const DevWeight* gate, const DevWeight* up) { return gate->type == up->type && gate->n == up->n && gate->k == up->k; }

hipError_t pfw_gemm_launch(const DevWeight* const* W, int nw, PfWide& G, int epi, uint32_t rows, const PfwGroups* grp, hipStream_t st) {
  if (nw < 1 || nw > 3 || rows == 0 || rows > (uint32_t)kPfwMaxRows || !G.x) return hipErrorInvalidValue;
  const uint32_t k = W[0]->k;
  if (k % 256 || (size_t)rows * k * 2 > 0xFFFFF000ull) return hipErrorInvalidValue;   // (32-bit row offsets)
  G.nseg = nw;
  G.nblk = k / 256;
  uint32_t rg = 0, col = 0, mask = 0;
  for (int i = 0; i < nw; i++) {
    const int f = pf_fmt_of(W[i]->type);
    if (f < 0 || W[i]->k != k || W[i]->n % 16 || (grp && W[i]->n_stack < grp->experts)) return hipErrorInvalidValue;
    G.seg[i] = PfwSeg{W[i]->plane[0], grp ? (uint64_t)W[i]->stack_stride[0] : 0, W[i]->n / 16, col, rg, f};
    mask |= 1u << f;
    rg += pw_row_groups(W[i]->n);
    col += W[i]->n;
  }
  G.ncols = col;
  G.m = rows;
  uint32_t tiles_m = (rows + kPfwTile - 1) / kPfwTile;
  if (grp) {
    if (!grp->seg || !grp->tile_e || !grp->tile_row) return hipErrorInvalidValue;
    G.src = grp->src;
    G.tile_e = grp->tile_e;
    G.tile_row = grp->tile_row;
    G.row_seg = grp->seg;
    tiles_m = grp->tiles;
  }
  if (epi == PW_SWIGLU) {
    if (nw != 2 || !pfw_pairs(W[0], W[1]) || !G.act || !G.inv_rms || G.act_cols != W[0]->n || (grp && !G.src)) return hipErrorInvalidValue;
    G.S = 1;
    const uint32_t n_rg = (W[0]->n / 16 + 2 * kWWaves - 1) / (2 * kWWaves);
    return grp ? pw_pick<true, PW_SWIGLU>(G, mask, n_rg, tiles_m, st) : pw_pick<false, PW_SWIGLU>(G, mask, n_rg, tiles_m, st);
  }
  G.S = pw_splits(rg, grp ? grp->likely : tiles_m, rows, G.nblk);
  G.part_rows = rows;
  if (!G.part || (size_t)G.S * rows * col * 4 > G.part_bytes) return hipErrorInvalidValue;
  return grp ? pw_pick<true, PW_PART>(G, mask, rg, tiles_m, st) : pw_pick<false, PW_PART>(G, mask, rg, tiles_m, st);
}

size_t pfw_part_bytes(uint32_t max_rows, uint32_t cols) { return (size_t)std::max(max_rows, (uint32_t)kPfwPartRows) * cols * 4; }

// ------------------------------------------------------------------------------------------------
// row kernels
// ------------------------------------------------------------------------------------------------
__device__ __forceinline__ void pw_store_chunk(uint8_t* x, uint32_t K, uint32_t t, uint32_t ch, const float v[8]) {
  const h16x8 o = {(_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)v[3], (_Float16)v[4], (_Float16)v[5], (_Float16)v[6], (_Float16)v[7]};
  *reinterpret_cast<h16x8*>(x + (size_t)t * K * 2 + ch * 16) = o;
}

// One workgroup per token: v = hidden (+ bias + sum of the partial sums, or of the token's expert rows times their routing weights); hidden = v;
// x = f16(v * nw); inv_rms = 1 / rms(v) (simd.rs:847-878).  Bound by memory: partial sums and hidden in, hidden and f16 row out.
__global__ void __launch_bounds__(256) pw_resid_kernel(const PfwResid a) {
  __shared__ float s_ss[4];
  const uint32_t t = blockIdx.x;
  float ss = 0.0f;
  for (uint32_t ch = threadIdx.x; ch < a.H / 8; ch += 256) {
    const uint32_t i = ch * 8;
    float* h = a.hidden + (size_t)t * a.H + i;
    f32x4 v0 = *reinterpret_cast<const f32x4*>(h), v1 = *reinterpret_cast<const f32x4*>(h + 4);
    if (a.part) {
      f32x4 a0 = (f32x4)(0.0f), a1 = (f32x4)(0.0f);
      if (a.row_of) {   // MoeLayer::forward (moe.rs:363-368): zero-initialised, += routing weight * expert output in selection order
        for (uint32_t s = 0; s < a.top; s++) {
          const uint32_t row = (uint32_t)a.row_of[t * a.top + s];
          f32x4 y0 = (f32x4)(0.0f), y1 = (f32x4)(0.0f);
          for (uint32_t sp = 0; sp < a.S; sp++) {
            const float* p = a.part + ((size_t)sp * a.part_rows + row) * a.H + i;
            y0 += *reinterpret_cast<const f32x4*>(p);
            y1 += *reinterpret_cast<const f32x4*>(p + 4);
          }
          const float w = a.weight[t * a.top + s];
          a0 += y0 * w;
          a1 += y1 * w;
        }
      } else {
        for (uint32_t s = 0; s < a.S; s++) {
          const float* p = a.part + ((size_t)s * a.part_rows + t) * a.H + i;
          a0 += *reinterpret_cast<const f32x4*>(p);
          a1 += *reinterpret_cast<const f32x4*>(p + 4);
        }
      }
      if (a.bias) { a0 += *reinterpret_cast<const f32x4*>(a.bias + i); a1 += *reinterpret_cast<const f32x4*>(a.bias + i + 4); }
      v0 += a0;
      v1 += a1;
      *reinterpret_cast<f32x4*>(h) = v0;
      *reinterpret_cast<f32x4*>(h + 4) = v1;
    }
    const f32x4 q = v0 * v0 + v1 * v1;
    ss += (q.x + q.y) + (q.z + q.w);
    if (a.x) {
      const f32x4 w0 = *reinterpret_cast<const f32x4*>(a.nw + i), w1 = *reinterpret_cast<const f32x4*>(a.nw + i + 4);
      float v[8];
#pragma unroll
      for (int j = 0; j < 4; j++) { v[j] = v0[j] * w0[j]; v[4 + j] = v1[j] * w1[j]; }
      pw_store_chunk(a.x, a.H, t, ch, v);
    }
  }
  if (!a.inv_rms) return;
  ss = wave_sum(ss);
  if ((threadIdx.x & 63) == 0) s_ss[threadIdx.x >> 6] = ss;
  __syncthreads();
  if (threadIdx.x == 0) a.inv_rms[t] = 1.0f / __builtin_sqrtf(((s_ss[0] + s_ss[1]) + (s_ss[2] + s_ss[3])) / (float)a.H + a.eps);
}

hipError_t pfw_resid_launch(const PfwResid& a, uint32_t m_tokens, hipStream_t st) {
  if (a.H % 8 || !a.hidden || m_tokens == 0 || (a.x && !a.nw) || (a.part && !a.S) || (a.row_of && (!a.weight || !a.top))) return hipErrorInvalidValue;
  hipLaunchKernelGGL(pw_resid_kernel, dim3(m_tokens), dim3(256), 0, st, a);
  return hipGetLastError();
}

// q, k, v of a token: partial sums x 1/rms (+ bias), RoPE at position pos0 + t (ops.rs:1285-1337), q -> q[t][QD], k / v -> cache rows (layers.rs:577-600).
// A thread takes four columns: two neighbouring pairs, or (NeoX) the same two columns of both halves of a head.
__global__ void __launch_bounds__(256) pw_qkv_kernel(const PfwQkv a) {
  const uint32_t t = blockIdx.y, pos = a.pos0 + t, half = a.head_dim / 2, quads = (a.QD + 2 * a.KD) / 4;
  const uint32_t p = blockIdx.x * 256 + threadIdx.x;
  if (p >= quads) return;
  const float inv = a.inv_rms[t];
  const uint32_t nq = a.QD / 4, nk = a.KD / 4;
  const bool isq = p < nq, isk = !isq && p < nq + nk, rot = isq || isk;
  const uint32_t pr = isq ? p : isk ? p - nq : p - nq - nk, base = isq ? 0 : isk ? a.QD : a.QD + a.KD;
  const bool split = rot && a.neox;
  // columns c0, c0 + 1 and c1, c1 + 1; pairs (c0, c0 + 1), (c1, c1 + 1) or, split, (c0, c1), (c0 + 1, c1 + 1)
  const uint32_t hd = split ? pr / (half / 2) : 0, c0 = split ? hd * a.head_dim + pr % (half / 2) * 2 : pr * 4, c1 = split ? c0 + half : c0 + 2;
  f32x2 x0 = (f32x2)(0.0f), x1 = (f32x2)(0.0f);
  const uint32_t ncols = a.QD + 2 * a.KD;
  for (uint32_t s = 0; s < a.S; s++) {
    const float* row = a.part + ((size_t)s * a.part_rows + t) * ncols + base;
    x0 += *reinterpret_cast<const f32x2*>(row + c0);
    x1 += *reinterpret_cast<const f32x2*>(row + c1);
  }
  x0 *= inv;
  x1 *= inv;
  const float* b = isq ? a.bq : isk ? a.bk : a.bv;
  if (b) { x0.x += b[c0]; x0.y += b[c0 + 1]; x1.x += b[c1]; x1.y += b[c1 + 1]; }
  if (rot) {
    const uint32_t i = split ? c0 % a.head_dim : c0 % a.head_dim / 2;   // first of the two frequencies
    const float* cs = a.rope_cs + ((size_t)pos * half + i) * 2;
    const float c_0 = cs[0], s_0 = cs[1], c_1 = cs[2], s_1 = cs[3];
    if (split) {
      const float u0 = x0.x, u1 = x0.y;
      x0.x = u0 * c_0 - x1.x * s_0;
      x0.y = u1 * c_1 - x1.y * s_1;
      x1.x = u0 * s_0 + x1.x * c_0;
      x1.y = u1 * s_1 + x1.y * c_1;
    } else {
      const float u0 = x0.x, u1 = x1.x;
      x0.x = u0 * c_0 - x0.y * s_0;
      x0.y = u0 * s_0 + x0.y * c_0;
      x1.x = u1 * c_1 - x1.y * s_1;
      x1.y = u1 * s_1 + x1.y * c_1;
    }
  }
  float* out = isq ? a.q + (size_t)t * a.QD + c0 : (isk ? a.kcache : a.vcache) + ((size_t)(c0 / a.head_dim) * a.max_seq + pos) * a.head_dim + c0 % a.head_dim;
  *reinterpret_cast<f32x2*>(out) = x0;
  *reinterpret_cast<f32x2*>(out + (c1 - c0)) = x1;
}

hipError_t pfw_qkv_launch(const PfwQkv& a, uint32_t m_tokens, hipStream_t st) {
  if (a.head_dim % 8 || a.QD % a.head_dim || a.KD % a.head_dim || m_tokens == 0 || m_tokens > 65535 || !a.S) return hipErrorInvalidValue;
  hipLaunchKernelGGL(pw_qkv_kernel, dim3(((a.QD + 2 * a.KD) / 4 + 255) / 256, m_tokens), dim3(256), 0, st, a);
  return hipGetLastError();
}

}  // namespace lgh
