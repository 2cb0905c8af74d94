// matvec_batch.hip — the int8 matrix-core mat-vec for SEVERAL sequences at once (multi-sequence decode, engine_batch.hip:
// lgh_forward_multi; the reference's BatchedEngine steps its active sequences one after the other, src/engine_batched.rs:
// 236-290, 355-400 — every sequence with its own InferenceContext / KV cache).  One launch reads every weight tile ONCE and
// multiplies it with the XQ records of all n_seq input vectors.
//
// Arithmetic.  A sequence's result is bit-identical to the single-sequence kernel (matvec_mfma.hip) on the same input: the
// same k-slices (T, blocks per slice), per slice the blocks in ascending order through the same fused operations
// (mvq_core.h: mvq_mac_tile(unpack, load) == mvq_consume_tile), the same two shuffles, the same sum over the slices and the same
// epilogue (mv_epilogue.h) per sequence.  Only WHO computes differs.
//
// Two structures.  mvqb2 (below, the default from 2 sequences on): a workgroup = 8 (row tile, pass) units x one range of blocks,
// the sequences' records staged ONCE per workgroup in LDS and shared by its 8 waves, sequences two at a time (the pair's 8 MFMAs,
// then the vector work while the next pair's operands load), the epilogue as a second small launch — what bounded the first
// structure and what each change bought: profiles/r03e_batched_decode.md.  From three sequences on its products take the sequences in
// groups of four (mvqb4) or, from five on and for weights of up to 6 bits, of eight (mvqb8).  mvqb (first): the single-sequence decomposition (a
// workgroup = the 8 k-slices of a few row tiles) with a loop over the sequences inside it and their records from L2 into a
// register ring; kept for one sequence and for launches whose segments do not share their input vector.
// Epilogues: store, +residual, SwiGLU pair, RoPE (every sequence at its own position) and the K / V rows into the sequence's
// own cache slot; optional XQ image of the output for the next launch.  MoE layers: an expert launch works on an INDIRECT
// entry list (MvBatch::ind_*: the (sequence, top-k slot) pairs that chose the expert, their number read from device memory), so
// that an expert's matrices are read once per step: gate | up of few entries an expert by mvqb_few, the others by mvqb2.
#include <algorithm>
#include <cstdlib>
#include <type_traits>

#include "dispatch_rules.h"
#include "device_utils.h"
#include "xq.h"
#include "mvq_core.h"
#include "mv_epilogue.h"

namespace lgh {

constexpr int kBWaves = 8;

// ---- the tail of a multi-sequence launch: per sequence the RMSNorm's sum of squares (exactly the single-sequence kernel's
// order: mvqb_norms), then the single-sequence epilogue on that sequence's vectors (mvqb_tail).  red: [n_seq][red_floats], ssq: [n_seq][8] (LDS)
// wave w: sequences w, w + waves, ... - per sequence what wave 0 of the single-sequence kernel does; slots 1..7 stay zero
__device__ __forceinline__ void mvqb_norms(const MvLaunch& L, const MvBatch& B, uint32_t n_seq, float* ssq, const int* ind_idx) {
  const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t L_n_ssq = L.n_ssq_part, nw = blockDim.x >> 6;
  for (uint32_t s = wave; s < n_seq; s += nw) {
    const float* part = L.ssq_part + (size_t)(ind_idx ? (uint32_t)ind_idx[s] / B.ind_div : s) * B.ssq_stride;
    float ssp[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int j = 0; j < 4; j++)
      if (lane + 64 * j < L_n_ssq) ssp[j] = part[lane + 64 * j];
    float ss = (ssp[0] + ssp[1]) + (ssp[2] + ssp[3]);
    for (uint32_t i = 256 + lane; i < L_n_ssq; i += 64) ss += part[i];
    ss = wave_sum_to_lane63(ss);
    if (lane == 63) ssq[s * 8] = ss;
    if (lane >= 1 && lane < 8) ssq[s * 8 + lane] = 0.0f;
  }
}

__device__ __forceinline__ void mvqb_tail(const MvLaunch& L, const MvSeg& S, const MvBatch& B, int sg, uint32_t wg, uint32_t rows_per_wg, uint32_t n_seq,
                                          uint32_t red_floats, float* red, float* ssq, uint32_t nslots, const int* ind_idx = nullptr) {
  const uint32_t tid = threadIdx.x;
  __syncthreads();
  // the sequences side by side: a sequence's epilogue needs one thread per row (pair) — groups of `tpr` threads take sequences
  // s, s + n_par, ...; each runs the single-sequence epilogue
  const uint32_t tpr = (rows_per_wg + 15u) & ~15u;   // (16-lane rows: what the XQ image's cross-lane steps work on)
  const uint32_t n_par = max(1u, blockDim.x / tpr);
  const uint32_t grp = tid / tpr, tl = tid - grp * tpr;
  if (grp >= n_par) return;
  for (uint32_t s = grp; s < n_seq; s += n_par) {
    const bool cache = S.epi == EPI_ROPE_K || S.epi == EPI_V_CACHE;
    const uint32_t so = ind_idx ? (uint32_t)ind_idx[s] : s;   // whose output vectors (an indirect entry's (sequence, slot) pair)
    MvEpiView V;
    V.out = cache ? S.out + (size_t)B.slot[s] * B.cache_stride : S.out + (size_t)so * B.out_stride[sg];
    V.resid = S.resid ? S.resid + (size_t)so * B.resid_stride[sg] : nullptr;
    V.xq_out = S.xq_out ? S.xq_out + (size_t)so * B.xq_out_stride[sg] : nullptr;
    V.xq_ssq = S.xq_ssq ? S.xq_ssq + (size_t)so * B.ssq_out_stride[sg] : nullptr;
    V.pos = B.pos + s;
    V.xw_out = B.xw_out[sg] ? B.xw_out[sg] + (size_t)so * kXwRecord : nullptr;
    V.xw_block = B.xw_block;
    mv_epilogue_view(L, S, V, wg, rows_per_wg, red + (size_t)s * red_floats, ssq + s * 8, nslots, tl);
  }
}

template <uint32_t MASK, int NB>
__global__ void __launch_bounds__(kBWaves * 64) mvqb_kernel(uint32_t wbpack, uint32_t geom, uint32_t geom2, uint32_t red_floats, const MvLaunch L,
                                                            const MvBatch B) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem8[];
  const uint32_t bid = blockIdx.x;
  const int sg = (int)(bid >= (wbpack & 0xFFFFu)) + (int)(bid >= (wbpack >> 16));
  const MvSeg& S = L.seg[sg];
  constexpr bool kSingle = (MASK & (MASK - 1)) == 0;
  const int fmt = kSingle ? __builtin_ctz(MASK) : fmt_of_dev_type(S.type);
  auto is = [&](int f) { return ((MASK >> f) & 1u) != 0 && (kSingle || fmt == f); };
  const uint32_t tb = is(F_Q4K) ? fmt_tile_bytes(F_Q4K) : is(F_Q6K) ? fmt_tile_bytes(F_Q6K) : is(F_Q5K) ? fmt_tile_bytes(F_Q5K)
                      : is(F_Q80) ? fmt_tile_bytes(F_Q80) : fmt_tile_bytes(F_Q40);
  const uint32_t S_T = geom & 0xFFu, S_G = (geom >> 8) & 0xFFu, nbw = (geom >> 16) & 0x3FFFu;
  const bool nrm = (geom >> 31) != 0;
  const uint32_t S_nblk = geom2 & 0xFFFFu;
  const uint32_t Rg = L.nseg > 1 ? S.rows_per_wg >> (4 + __builtin_ctz(S_G)) : geom2 >> 16;
  const uint32_t S_rpw = 16u * Rg * S_G;
  const uint32_t wg = bid - S.wg_begin;
  const uint32_t n_seq = B.n_seq;
  const int npass = S.npass;   // 1 or 2 (gate | up); both passes share the input vector

  const uint32_t tid = threadIdx.x, lane = tid & 63;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  uint32_t ks = wave, rg = 0;
  while (ks >= S_T) { ks -= S_T; rg++; }
  const bool active = rg < S_G;
  const uint32_t blk0 = ks * nbw;
  const uint32_t nblk_w = active && blk0 < S_nblk ? min(nbw, S_nblk - blk0) : 0;
  const uint32_t ntiles = (S.n_rows + 15) >> 4;
  const uint32_t tile0 = (wg * S_G + rg) * Rg;
  const uint32_t ntile_w = active && tile0 < ntiles ? min(Rg, ntiles - tile0) : 0;
  float* red = reinterpret_cast<float*>(smem8);           // [n_seq][red_floats]
  float* ssq = red + (size_t)n_seq * red_floats;          // [n_seq][8]
  const uint32_t n = lane & 15, mq = lane >> 4;

  const uint64_t woff = ((uint64_t)tile0 * S_nblk + blk0) * tb;
  const uint8_t* pb0 = S.pass[0].plane[0] + woff;
  const uint8_t* pb1 = npass > 1 ? S.pass[1].plane[0] + woff : pb0;
  const uint8_t* xg = S.pass[0].xq + (size_t)blk0 * kXqRecord;   // sequence 0's records of this wave's k-slice

  // a slice beyond the last block, or a row group beyond the last tile, still owns partial-sum slots: they must read as zero
  const uint32_t npairs = (uint32_t)npass * ntile_w;
  if (nblk_w == 0 && ntile_w > 0) {
    for (uint32_t s = 0; s < n_seq; s++)
      for (uint32_t pr = 0; pr < npairs; pr++) {
        const uint32_t p = pr / ntile_w, tl = pr - p * ntile_w;
        if (mq == 0) red[(size_t)s * red_floats + (size_t)(p * S_T + ks) * S_rpw + (rg * Rg + tl) * 16 + n] = 0.0f;
      }
  }
  const uint32_t ngroups = (npairs + 1) / 2;
  const uint32_t nsteps = nblk_w ? ngroups * nblk_w : 0;

  // ---- the weight stream: step (g, b) = tiles (pair 2g, block b) and (pair 2g + 1, block b); a missing second pair re-reads
  // the first one's tile (an L1 / L2 hit: the issue pattern stays the same for every step, which keeps the waits exact)
  auto tile_ptr = [&](uint32_t pr, uint32_t b) -> const uint8_t* {
    const uint32_t p = pr / ntile_w, tl = pr - p * ntile_w;
    return (p == 0 ? pb0 : pb1) + ((size_t)tl * S_nblk + b) * tb;
  };
  auto issue_step = [&](uint32_t g, uint32_t b, RawT16 (&dst)[2]) {
    const uint32_t p0 = 2 * g, p1 = 2 * g + 1 < npairs ? 2 * g + 1 : 2 * g;
    mvq_issue_tile<MASK>(fmt, tile_ptr(p0, b), lane, dst[0]);
    mvq_issue_tile<MASK>(fmt, tile_ptr(p1, b), lane, dst[1]);
  };
  float acc[NB][2];
  // The sequences' XQ operands come from L2 (~0.7 us away): a ring of kXd operand sets in registers; sequence s + kXd of the step
  // is requested when sequence s has been used, and the first kXd sequences of the NEXT step at the end of a step — i.e. before
  // that step requests its weight prefetch (a wave's loads return in order: a load issued behind the prefetch waits for HBM).
  constexpr int kXd = NB >= 8 && !(NB == 16 && !kSingle) ? 3 : 2;   // (the mixed-format instantiations have no registers to spare at 16 sequences)
  XqOps xr[kXd];
  auto x_issue = [&](uint32_t b, int s, XqOps& o) { xq_load_ops(xg + (size_t)s * B.xq_stride + (size_t)b * kXqRecord, lane, o); };
  auto x_prime = [&](uint32_t b) {
#pragma unroll
    for (int s = 0; s < kXd; s++)
      if ((uint32_t)s < n_seq) x_issue(b, s, xr[s]);
  };
  auto process = [&](uint32_t g, uint32_t b, const RawT16 (&w)[2], bool more, uint32_t b_next) {
    const bool two = 2 * g + 1 < npairs;
    if (b == 0) {
#pragma unroll
      for (int s = 0; s < NB; s++) acc[s][0] = acc[s][1] = 0.0f;
    }
    TileOps t0, t1;
    mvq_unpack_tile<MASK>(fmt, w[0], lane, t0);
    mvq_unpack_tile<MASK>(fmt, w[1], lane, t1);
#pragma unroll
    for (int s = 0; s < NB; s++) {
      if ((uint32_t)s < n_seq) {
        mvq_mac_tile<MASK>(fmt, t0, xr[s % kXd], acc[s][0]);
        if (two) mvq_mac_tile<MASK>(fmt, t1, xr[s % kXd], acc[s][1]);
        if ((uint32_t)(s + kXd) < n_seq) x_issue(b, s + kXd, xr[s % kXd]);
      }
    }
    if (more) x_prime(b_next);   // the next step's first sequences, ahead of its weight prefetch
    if (b + 1 == nblk_w) {   // last block of the group's pairs: the four lane groups -> one partial sum per row and sequence
#pragma unroll
      for (int s = 0; s < NB; s++) {
        if ((uint32_t)s < n_seq) {
#pragma unroll
          for (int j = 0; j < 2; j++) {
            if (j == 0 || two) {
              const uint32_t pr = 2 * g + j, p = pr / ntile_w, tl = pr - p * ntile_w;
              float t = acc[s][j] + __shfl_xor(acc[s][j], 16, 64);
              t += __shfl_xor(t, 32, 64);
              if (mq == 0) red[(size_t)s * red_floats + (size_t)(p * S_T + ks) * S_rpw + (rg * Rg + tl) * 16 + n] = t;
            }
          }
        }
      }
    }
  };

  if (nsteps) {
    RawT16 wa[2], wb[2];
    uint32_t g = 0, b = 0;                                  // the step being processed
    auto next = [&](uint32_t& gg, uint32_t& bb) { if (++bb == nblk_w) { bb = 0; ++gg; } };
    x_prime(0);
    issue_step(0, 0, wa);
    for (uint32_t st = 0; st < nsteps; st += 2) {
      uint32_t g1 = g, b1 = b;
      next(g1, b1);
      const bool has1 = st + 1 < nsteps;
      if (has1) issue_step(g1, b1, wb); else issue_step(g, b, wb);
      process(g, b, wa, has1, b1);
      uint32_t g2 = g1, b2 = b1;
      next(g2, b2);
      const bool has2 = st + 2 < nsteps;
      if (has2) issue_step(g2, b2, wa); else issue_step(g, b, wa);
      if (has1) process(g1, b1, wb, has2, b2);
      g = g2; b = b2;
    }
  }

  if (nrm) mvqb_norms(L, B, n_seq, ssq, nullptr);
  mvqb_tail(L, S, B, sg, wg, S.rows_per_wg, n_seq, red_floats, red, ssq, S_T);
}

// ================================================================================================
// Second structure (mvqb2): the sequences' XQ records through LDS, shared by the eight waves of a workgroup.
//
// Why.  With the k-slices of a row tile spread over the waves of ONE workgroup (above, as in the single-sequence kernel) every wave
// walks its own blocks: an XQ record fetched for a (sequence, block) serves one or two tiles, and a step of 16 sequences moves
// ~2 GB of records per layer from L2 into registers — measured: the memory side alone (arithmetic compiled out) 7.8 ms of the
// 9.9 ms step at 16 sequences, the arithmetic alone 7.6 (profiles/r03e_batched_decode.md).  Here a workgroup is 8 "units" (a unit =
// one row tile of one pass) x ONE range of blocks: all eight waves need the same records, which are staged ONCE per workgroup in
// LDS (cb blocks x n_seq records, <= 40 KB) and read from there — 8x less L2 traffic, no operand ring in registers, half the
// vector registers, two to three workgroups per CU.
//
// Arithmetic.  Unchanged: a unit's blocks in ascending order through mvq_mac_tile; at the end of every k-slice of the
// single-sequence kernel (blocks [ks * nbw, (ks + 1) * nbw)) the four lane groups are folded with the same two shuffles, giving
// the slice's partial sum p_ks.  The single-sequence epilogue adds the slices up as ((0 + p_0) + p_1) + ...:
//   SEQ  = true   a workgroup walks ALL slices of its units and keeps that running sum in registers (same additions, same order);
//                 one value per (sequence, row) goes to the epilogue (nslots = 1: it computes 0 + sum = sum), in the same launch where the launch has one segment
//                 (Mvqb2Geom::fuse), else through the partial buffer;
//   SEQ  = false  (matrices with too few units to fill the chip that way: wo, down, QKV) blockIdx.y = the slice; p_ks goes to
//                 the partial buffer (nslots = T) and the epilogue adds them in slice order.
// Otherwise a second, small launch (mvqb_rows_kernel) adds the partial sums up in that order and does what the single-sequence
// epilogue does — every sequence's result is bit-identical to matvec_mfma.hip's.
// ================================================================================================
struct Mvqb2Geom {
  uint32_t T, nbw, nblk;      // the single-sequence kernel's k-slices
  uint32_t n_units;           // sum over segments of npass * row tiles
  uint32_t ub1, ub2;          // first unit of segment 1 / 2 (n_units when absent)
  uint32_t cb;                // blocks staged per chunk
  uint32_t nslots;            // partial sums per (sequence, row) in the buffer: 1 (SEQ) or T
  // SEQ, one segment (gate | up, the output head): a workgroup has all there is of its rows and runs the epilogue itself, its eight units being 8 tiles, or 4 tiles of both passes.  fuse = passes, 0: no.
  // 16 sequences, 8 layers of an 8B model: gate | up 40.3 -> 43.3 us and the head 58 -> 63, their epilogue launches (7.3 and 7.5 us and a gap each) gone; a batch with its prompts 43.2 -> 42.4 ms
  uint32_t fuse;
  uint32_t ssq_at;            // fuse: LDS byte of the sequences' sums of squares, behind all else
};

// unit of wave w of workgroup wg
__device__ __forceinline__ void mvqb_unit(const Mvqb2Geom& Gm, uint32_t wg, uint32_t w, uint32_t ntiles, uint32_t ul, bool& active, uint32_t& pass, uint32_t& tl) {
  if (Gm.fuse) {
    pass = Gm.fuse == 2 ? w & 1 : 0;
    tl = Gm.fuse == 2 ? wg * (kBWaves / 2) + (w >> 1) : wg * kBWaves + w;
    active = tl < ntiles;
    if (!active) pass = tl = 0;
  } else {
    pass = active ? ul / ntiles : 0;
    tl = active ? ul - pass * ntiles : 0;
  }
}
constexpr uint32_t kFuseRed = kBWaves * 16;   // floats a sequence: [pass][row of the workgroup]
// place of row n of this wave's unit
__device__ __forceinline__ uint32_t mvqb_red_at(const Mvqb2Geom& Gm, uint32_t w, uint32_t n) { return Gm.fuse == 2 ? ((w & 1) * 4 + (w >> 1)) * 16 + n : w * 16 + n; }
__host__ __device__ constexpr uint32_t mvqb_fuse_lds(uint32_t n_seq) { return n_seq * 8 * 4; }

#ifndef LGH_XSTAGE_KB
#define LGH_XSTAGE_KB 40   /* (experiment builds vary it: the cost of a chunk boundary, profiles/r03e_batched_decode.md) */
#endif
constexpr uint32_t kXStageBytes = LGH_XSTAGE_KB * 1024;
// (the two-format instantiations at 16 sequences have no registers to spare: smaller chunks, fewer staging registers)
__host__ __device__ constexpr uint32_t mvqb2_stage_bytes(bool single_format, int nb) { return !single_format && nb == 16 ? 24u * 1024u : kXStageBytes; }
constexpr uint32_t kXZeroBytes = 2 * 1280 + 256;   // the zero block; also what an odd last sequence's partner may read past the records
constexpr uint32_t kXSelBytes = 64;                // behind it: whose input vector entry s reads (s itself, or an indirect entry's sequence)

template <uint32_t MASK, int NB, bool SEQ>
__global__ void __launch_bounds__(kBWaves * 64) mvqb2_kernel(const Mvqb2Geom Gm, const MvLaunch L, const MvBatch B, float* __restrict__ part) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem8[];
  const uint32_t tid = threadIdx.x, lane = tid & 63;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  uint32_t n_seq = B.n_seq;
  const uint32_t ez = blockIdx.z;                                 // expert (indirect launches over a layer's experts; else 0)
  const int* ind_idx = nullptr;
  if (B.ind_cnt) {   // indirect entries (MoE expert launch): how many (sequence, slot) pairs chose this expert — possibly none
    uint32_t cw;
    asm volatile("s_load_dword %0, %1, 0x0\n\ts_waitcnt lgkmcnt(0)" : "=s"(cw) : "s"(B.ind_cnt + ez) : "memory");
    n_seq = min(cw, n_seq);
    if (n_seq == 0) return;
    ind_idx = B.ind_idx + (size_t)ez * B.ind_stride;
    part += (size_t)ez * B.part_z_floats;
  }
  const uint32_t u = blockIdx.x * kBWaves + wave;                 // this wave's unit
  bool active = u < Gm.n_units;
  const int sg = SEQ && Gm.fuse ? 0 : (int)(u >= Gm.ub1) + (int)(u >= Gm.ub2);
  const MvSeg& S = L.seg[active ? sg : 0];
  constexpr bool kSingle = (MASK & (MASK - 1)) == 0;
  const int fmt = kSingle ? __builtin_ctz(MASK) : fmt_of_dev_type(S.type);
  auto is = [&](int f) { return ((MASK >> f) & 1u) != 0 && (kSingle || fmt == f); };
  const uint32_t tb = is(F_Q4K) ? fmt_tile_bytes(F_Q4K) : is(F_Q6K) ? fmt_tile_bytes(F_Q6K) : is(F_Q5K) ? fmt_tile_bytes(F_Q5K)
                      : is(F_Q80) ? fmt_tile_bytes(F_Q80) : fmt_tile_bytes(F_Q40);
  const uint32_t ntiles = (S.n_rows + 15) >> 4;
  const uint32_t ul = u - (sg == 0 ? 0u : sg == 1 ? Gm.ub1 : Gm.ub2);
  uint32_t pass, tl;
  mvqb_unit(Gm, blockIdx.x, wave, ntiles, ul, active, pass, tl);
  const uint8_t* wbase = (pass == 0 ? S.pass[0].plane[0] + (uint64_t)ez * S.pass[0].sel_stride[0] : S.pass[1].plane[0] + (uint64_t)ez * S.pass[1].sel_stride[0]) +
                         (size_t)tl * Gm.nblk * tb;
  const uint8_t* xg = L.seg[0].pass[0].xq;                        // sequence 0's records (all segments and passes share the input)
  const uint32_t n = lane & 15, mq = lane >> 4;

  // this workgroup's slices
  const uint32_t ks0 = SEQ ? 0u : blockIdx.y, ks1 = SEQ ? Gm.T : blockIdx.y + 1;
  float acc[NB], tot[NB];
#pragma unroll
  for (int s = 0; s < NB; s++) acc[s] = tot[s] = 0.0f;

  // LDS: [2][cb * n_seq records][a block of zeros].  A lane outside its own k-chunk must feed zeros to the MFMA's A operand: instead of
  // a masked load + a register clear per sequence, such a lane reads the zero block (one unmasked ds_read_b128 per operand).
  const uint32_t zero_off = 2 * Gm.cb * n_seq * (uint32_t)kXqRecord;   // (behind the two halves of the record buffer)
  for (uint32_t i = tid; i < kXZeroBytes / 16; i += kBWaves * 64) *reinterpret_cast<u32x4*>(smem8 + zero_off + i * 16) = u32x4{0u, 0u, 0u, 0u};
  uint32_t* xsel = reinterpret_cast<uint32_t*>(smem8 + zero_off + kXZeroBytes);
  if (tid < n_seq) xsel[tid] = ind_idx ? (uint32_t)ind_idx[tid] / B.ind_div : tid;
  float* const ssq = reinterpret_cast<float*>(smem8 + Gm.ssq_at);
  if (SEQ && Gm.fuse && L.do_norm) mvqb_norms(L, B, n_seq, ssq, ind_idx);
  __syncthreads();
  const bool a_valid = (n >> 2) == mq;
  const uint32_t a_off = (mq >> 1) * 128 + (n & 3) * 32 + (mq & 1) * 16;
  const uint32_t a_step = a_valid ? (uint32_t)kXqRecord : 0u;   // per sequence
  struct XqA { i32x4 a[4]; };
  struct XqS { f32x4 xs, sx; };
  auto load_a = [&](uint32_t pa, XqA& o) {
#pragma unroll
    for (int pp = 0; pp < 4; pp++) o.a[pp] = *reinterpret_cast<const i32x4*>(smem8 + pa + pp * 256);
  };
  auto load_s = [&](uint32_t px, XqS& o) {
    o.xs = *reinterpret_cast<const f32x4*>(smem8 + px);
    o.sx = *reinterpret_cast<const f32x4*>(smem8 + px + (kXqSx16 - kXqXs16));
  };

  RawT16 nxt;
  {
    const uint32_t bfirst = ks0 * Gm.nbw;
    if (active && bfirst < Gm.nblk) mvq_issue_tile<MASK>(fmt, wbase + (size_t)bfirst * tb, lane, nxt);
  }
  // ---- chunks of <= cb blocks, never across a slice boundary.  The records of chunk i + 1 are fetched into registers while chunk i
  // is computed, and stored into the other half of a two-deep LDS buffer at the next barrier: one barrier per chunk, no load exposed.
  constexpr uint32_t kPieces = (mvqb2_stage_bytes(kSingle, NB) / 16 + kBWaves * 64 - 1) / (kBWaves * 64);   // 16-byte pieces per thread and chunk
  const uint32_t buf_bytes = Gm.cb * n_seq * (uint32_t)kXqRecord;
  u32x4 stg[kPieces];
  auto chunk_len = [&](uint32_t ks, uint32_t b0) { return min(Gm.cb, min(ks * Gm.nbw + Gm.nbw, Gm.nblk) - b0); };
  auto fetch = [&](uint32_t b0, uint32_t cn) {
    const uint32_t pieces = cn * n_seq * (kXqRecord / 16);
#pragma unroll
    for (uint32_t j = 0; j < kPieces; j++) {
      const uint32_t i = tid + j * kBWaves * 64;
      if (i < pieces) {
        const uint32_t rec = i / (kXqRecord / 16), off = i - rec * (kXqRecord / 16);
        const uint32_t bi = rec / n_seq, s = rec - bi * n_seq;
        const uint32_t sx = xsel[s];                                          // whose input vector
        stg[j] = *reinterpret_cast<const u32x4*>(xg + (size_t)sx * B.xq_stride + (size_t)(b0 + bi) * kXqRecord + off * 16);
      }
    }
  };
  auto stash = [&](uint32_t cn, uint32_t buf) {
    const uint32_t pieces = cn * n_seq * (kXqRecord / 16);
#pragma unroll
    for (uint32_t j = 0; j < kPieces; j++) {
      const uint32_t i = tid + j * kBWaves * 64;
      if (i < pieces) *reinterpret_cast<u32x4*>(smem8 + buf * buf_bytes + (size_t)i * 16) = stg[j];
    }
  };
  // the first non-empty chunk of this workgroup's slices
  uint32_t ks = ks0, b0 = ks0 * Gm.nbw;
  while (ks < ks1 && b0 >= min(ks * Gm.nbw + Gm.nbw, Gm.nblk)) { ks++; b0 = ks * Gm.nbw; }
  uint32_t buf = 0;
  if (ks < ks1) fetch(b0, chunk_len(ks, b0));
  while (ks < ks1) {
    const uint32_t sb1 = min(ks * Gm.nbw + Gm.nbw, Gm.nblk);
    const uint32_t cn = chunk_len(ks, b0);
    stash(cn, buf);
    __syncthreads();
    // the chunk after this one
    uint32_t nks = ks, nb0 = b0 + cn;
    if (nb0 >= sb1) {
      nks = ks + 1; nb0 = nks * Gm.nbw;
      while (nks < ks1 && nb0 >= min(nks * Gm.nbw + Gm.nbw, Gm.nblk)) { nks++; nb0 = nks * Gm.nbw; }
    }
    if (nks < ks1) fetch(nb0, chunk_len(nks, nb0));
    if (active) {
      for (uint32_t bi = 0; bi < cn; bi++) {
        const uint32_t b = b0 + bi;
        const RawT16 cur = nxt;
        {   // the unit's next tile (its next block — of this slice, or of the next one this workgroup walks)
          uint32_t bn = b + 1;
          if (bn == sb1) bn = nks < ks1 ? nb0 : Gm.nblk;
          if (bn < Gm.nblk) mvq_issue_tile<MASK>(fmt, wbase + (size_t)bn * tb, lane, nxt);
        }
        TileOps t;
        mvq_unpack_tile<MASK>(fmt, cur, lane, t);
        const uint32_t xb = buf * buf_bytes + bi * n_seq * (uint32_t)kXqRecord;
        const uint32_t pa0 = a_valid ? xb + a_off : zero_off, px0 = xb + (uint32_t)kXqXs16 + mq * 16;
        // The sequences two at a time: the pair's eight matrix-core products first, then — while the vector ALU turns them into the
        // pair's sums — the NEXT pair's A operands are re-read into the registers the products have just released, and its x sums /
        // scales into the other half of a two-deep buffer.  An odd last sequence is paired with whatever follows it in LDS (the next
        // record or the zero block): computed, never stored.
        XqA xa[2];
        XqS xs2[2][2];
        load_a(pa0, xa[0]);
        load_a(pa0 + a_step, xa[1]);
        load_s(px0, xs2[0][0]);
        load_s(px0 + (uint32_t)kXqRecord, xs2[0][1]);
#ifdef LGH_MVQB2_NOMATH   /* experiment: the weight stream, the unpacking and the record staging only (one sequence's arithmetic) */
        const uint32_t n_seq_math = min(n_seq, 1u);
#else
        const uint32_t n_seq_math = n_seq;
#endif
#pragma unroll
        for (int g = 0; g < NB / 2; g++) {
          if ((uint32_t)(2 * g) < n_seq_math) {
            MacD m0, m1;
            mvq_mac_mfma(t, xa[0].a, m0);
            mvq_mac_mfma(t, xa[1].a, m1);
            if ((uint32_t)(2 * g + 2) < n_seq) {
              load_a(pa0 + (2 * g + 2) * a_step, xa[0]);
              load_a(pa0 + (2 * g + 3) * a_step, xa[1]);
              load_s(px0 + (2 * g + 2) * (uint32_t)kXqRecord, xs2[(g + 1) & 1][0]);
              load_s(px0 + (2 * g + 3) * (uint32_t)kXqRecord, xs2[(g + 1) & 1][1]);
            }
            mvq_mac_finish<MASK>(fmt, t, m0, xs2[g & 1][0].xs, xs2[g & 1][0].sx, acc[2 * g]);
            mvq_mac_finish<MASK>(fmt, t, m1, xs2[g & 1][1].xs, xs2[g & 1][1].sx, acc[2 * g + 1]);
          }
        }
      }
      // ---- end of the k-slice: the four lane groups -> the slice's partial sum (lane group 0), as in the single-sequence kernel
      if (b0 + cn >= sb1) {
#pragma unroll
        for (int s = 0; s < NB; s++) {
          if ((uint32_t)s < n_seq) {
            float t = acc[s] + __shfl_xor(acc[s], 16, 64);
            t += __shfl_xor(t, 32, 64);
            if (SEQ) tot[s] += t;
            else tot[s] = t;
            acc[s] = 0.0f;
          }
        }
      }
    }
    ks = nks; b0 = nb0; buf ^= 1u;
  }
  if (SEQ && Gm.fuse) {
    float* red = reinterpret_cast<float*>(smem8);
    __syncthreads();   // every record has been read
    if (mq == 0) {
#pragma unroll
      for (int s = 0; s < NB; s++)
        if ((uint32_t)s < n_seq) red[s * kFuseRed + mvqb_red_at(Gm, wave, n)] = tot[s];
    }
    mvqb_tail(L, S, B, 0, blockIdx.x, Gm.fuse == 2 ? kFuseRed / 2 : kFuseRed, n_seq, kFuseRed, red, ssq, 1, ind_idx);
    return;
  }
  if (active && mq == 0) {
    const uint32_t slot = SEQ ? 0u : blockIdx.y;
    const size_t rows16 = (size_t)Gm.n_units * 16;
#pragma unroll
    for (int s = 0; s < NB; s++)
      if ((uint32_t)s < n_seq) part[((size_t)slot * B.n_seq + s) * rows16 + (size_t)u * 16 + n] = tot[s];
  }
}

// ------------------------------------------------------------------------------------------------
// From three sequences on: the sequences four at a time.  mvqb2 gives every MFMA one sequence: its A operand, the four digits of four chunks, is three
// quarters zeros, and every lane reads 16 bytes for it all the same: six LDS reads of 1 KB per (tile, sequence) and wave, 96 % of what LDS can deliver in the time of
// the vector work.  Here the A operand is the four digits of FOUR sequences, all lanes full, and the weights are masked instead: B operand c keeps chunk c of
// every 64 elements and zeros for the other lane groups (masked once per tile).  A lane then has, per MFMA, the four digit sums of one sequence (4 * group + its lane
// group) for chunk c of weight row n: three LDS reads per (tile, sequence).  Per (row, sequence, chunk class) the floating-point operations and their order are
// mvqb2's (mvq_mac_finish); the classes, there in four lanes, lie in one: (class 0 + 1) + (2 + 3) is what the two exchanges add up.
// Records lie 1296 bytes apart in LDS, so that the four sequences' digits of a read fall into different banks.
// gate | up of an 8B model (28672 rows of 4096, Q4_K), 16 sequences: 72 us with mvqb2, 58 here, of which about 42 are vector instructions (8 a product of 16 elements).
// ------------------------------------------------------------------------------------------------
constexpr uint32_t kXLdsRecord = kXqRecord + 16;
__host__ __device__ constexpr uint32_t mvqb4_buf_bytes(uint32_t records) { return (records * kXLdsRecord + 1023u) & ~1023u; }

// scales of row n for all four chunk classes: f[pp][class], class pairs (a 32-element sub-block) sharing one where the format has it so
struct TileScales { float f[4][4], g[4][2], gq[2], dd, dmin; };   // gq: g[lane group]
template <uint32_t MASK>
__device__ __forceinline__ void mvq_row_scales(int fmt, const RawT16& r, uint32_t lane, TileScales& t) {
  const uint32_t n = lane & 15;
  auto is = [&](int f) { return mvq_is<MASK>(fmt, f); };
  const uint32_t hdw[4] = {r.hd.x, r.hd.y, r.hd.z, r.hd.w};
  if (is(F_Q6K)) {
#pragma unroll
    for (int pp = 0; pp < 4; pp++)
#pragma unroll
      for (int c = 0; c < 4; c++) t.f[pp][c] = (float)(int)__builtin_amdgcn_sbfe((int)hdw[pp], c * 8, 8);
    t.dd = h2f((n & 1) ? r.q[3].x >> 16 : r.q[3].x & 0xFFFFu);
    t.dmin = 0.0f;
  } else if (is(F_Q80) || is(F_Q40)) {
#pragma unroll
    for (int pp = 0; pp < 4; pp++) {
      t.f[pp][0] = t.f[pp][1] = h2f(hdw[pp] & 0xFFFFu);
      t.f[pp][2] = t.f[pp][3] = h2f(hdw[pp] >> 16);
    }
    t.dd = t.dmin = 0.0f;
  } else {
#pragma unroll
    for (int h = 0; h < 2; h++) {   // sub-blocks h, h + 2, h + 4, h + 6 (as mvq_unpack_tile)
      const uint32_t a = (r.hd.y >> (h * 8)) & 0x00FF00FFu, bq = (r.hd.z >> (h * 8)) & 0x00FF00FFu, cq = (r.hd.w >> (h * 8)) & 0x00FF00FFu;
      const uint32_t sc01 = a & 0x003F003Fu, mn01 = bq & 0x003F003Fu;
      const uint32_t sc23 = (cq & 0x000F000Fu) | ((a >> 2) & 0x00300030u);
      const uint32_t mn23 = ((cq >> 4) & 0x000F000Fu) | ((bq >> 2) & 0x00300030u);
      const float f[4] = {ub0(sc01), ub2(sc01), ub0(sc23), ub2(sc23)}, g[4] = {ub0(mn01), ub2(mn01), ub0(mn23), ub2(mn23)};
#pragma unroll
      for (int pp = 0; pp < 4; pp++) { t.f[pp][2 * h] = t.f[pp][2 * h + 1] = f[pp]; t.g[pp][h] = g[pp]; }
      t.gq[h] = ub0(((lane & 32) ? mn23 : mn01) >> (lane & 16));
    }
    t.dd = h2f(r.hd.x & 0xFFFFu);
    t.dmin = h2f(r.hd.x >> 16);
  }
}

template <uint32_t MASK, int NB, bool SEQ>
__global__ void __launch_bounds__(kBWaves * 64) mvqb4_kernel(const Mvqb2Geom Gm, const MvLaunch L, const MvBatch B, float* __restrict__ part) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem8[];
  constexpr int NG = NB / 4;
  const uint32_t tid = threadIdx.x, lane = tid & 63, n_seq = B.n_seq;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t u = blockIdx.x * kBWaves + wave;                 // this wave's unit
  bool active = u < Gm.n_units;
  const int sg = SEQ && Gm.fuse ? 0 : (int)(u >= Gm.ub1) + (int)(u >= Gm.ub2);
  const MvSeg& S = L.seg[active ? sg : 0];
  constexpr bool kSingle = (MASK & (MASK - 1)) == 0;
  const int fmt = kSingle ? __builtin_ctz(MASK) : fmt_of_dev_type(S.type);
  auto is = [&](int f) { return ((MASK >> f) & 1u) != 0 && (kSingle || fmt == f); };
  const uint32_t tb = is(F_Q4K) ? fmt_tile_bytes(F_Q4K) : is(F_Q6K) ? fmt_tile_bytes(F_Q6K) : is(F_Q5K) ? fmt_tile_bytes(F_Q5K)
                      : is(F_Q80) ? fmt_tile_bytes(F_Q80) : fmt_tile_bytes(F_Q40);
  const uint32_t ntiles = (S.n_rows + 15) >> 4;
  const uint32_t ul = u - (sg == 0 ? 0u : sg == 1 ? Gm.ub1 : Gm.ub2);
  uint32_t pass, tl;
  mvqb_unit(Gm, blockIdx.x, wave, ntiles, ul, active, pass, tl);
  float* const ssq = reinterpret_cast<float*>(smem8 + Gm.ssq_at);
  if (SEQ && Gm.fuse && L.do_norm) mvqb_norms(L, B, n_seq, ssq, nullptr);
  const uint8_t* wbase = (pass == 0 ? S.pass[0].plane[0] : S.pass[1].plane[0]) + (size_t)tl * Gm.nblk * tb;
  const uint8_t* xg = L.seg[0].pass[0].xq;                        // sequence 0's records (all segments and passes share the input)
  const uint32_t n = lane & 15, mq = lane >> 4;
  const uint32_t ks0 = SEQ ? 0u : blockIdx.y, ks1 = SEQ ? Gm.T : blockIdx.y + 1;   // this workgroup's slices
  float acc[NG][4], tot[NG];                                      // per group: the lane's sequence, chunk classes
#pragma unroll
  for (int g = 0; g < NG; g++) {
    tot[g] = 0.0f;
#pragma unroll
    for (int c = 0; c < 4; c++) acc[g][c] = 0.0f;
  }
  const uint32_t a_off = (mq >> 1) * 128 + (n & 3) * 32 + (mq & 1) * 16;

  RawT16 nxt;
  {
    const uint32_t bfirst = ks0 * Gm.nbw;
    if (active && bfirst < Gm.nblk) mvq_issue_tile<MASK>(fmt, wbase + (size_t)bfirst * tb, lane, nxt);
  }
  // chunks of records through a two-deep LDS buffer, as mvqb2, but by DMA: no staging registers
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem8;
  const uint32_t buf_bytes = mvqb4_buf_bytes(Gm.cb * n_seq);
  auto chunk_len = [&](uint32_t ks, uint32_t b0) { return min(Gm.cb, min(ks * Gm.nbw + Gm.nbw, Gm.nblk) - b0); };
  auto fetch = [&](uint32_t b0, uint32_t cn, uint32_t buf) {
    constexpr uint32_t kP = kXLdsRecord / 16;
    const uint32_t recs = cn * n_seq, kb = (recs * kP + 63) / 64;
    for (uint32_t k = wave; k < kb; k += kBWaves) {
      const uint32_t i = k * 64 + lane, rec = min(i / kP, recs - 1), off = min(i - rec * kP, kP - 2);   // a record's pad and the tail: any of its bytes
      const uint32_t bi = rec / n_seq, s = rec - bi * n_seq;
      const uint8_t* src = xg + (size_t)s * B.xq_stride + (size_t)(b0 + bi) * kXqRecord + off * 16;
      asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(src), "s"(lds0 + buf * buf_bytes + k * 1024) : "memory", "m0");
    }
  };
  uint32_t ks = ks0, b0 = ks0 * Gm.nbw;
  while (ks < ks1 && b0 >= min(ks * Gm.nbw + Gm.nbw, Gm.nblk)) { ks++; b0 = ks * Gm.nbw; }
  uint32_t buf = 0;
  if (ks < ks1) fetch(b0, chunk_len(ks, b0), 0);
  while (ks < ks1) {
    const uint32_t sb1 = min(ks * Gm.nbw + Gm.nbw, Gm.nblk);
    const uint32_t cn = chunk_len(ks, b0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    uint32_t nks = ks, nb0 = b0 + cn;   // the chunk after this one
    if (nb0 >= sb1) {
      nks = ks + 1; nb0 = nks * Gm.nbw;
      while (nks < ks1 && nb0 >= min(nks * Gm.nbw + Gm.nbw, Gm.nblk)) { nks++; nb0 = nks * Gm.nbw; }
    }
    if (nks < ks1) fetch(nb0, chunk_len(nks, nb0), buf ^ 1u);
    if (active) {
      for (uint32_t bi = 0; bi < cn; bi++) {
        const uint32_t b = b0 + bi;
        TileScales ts;
        i32x4 bm[4][4];   // [class][step]
        {
          TileOps t;
          mvq_unpack_tile<MASK>(fmt, nxt, lane, t);
          mvq_row_scales<MASK>(fmt, nxt, lane, ts);
#pragma unroll
          for (int c = 0; c < 4; c++)
#pragma unroll
            for (int pp = 0; pp < 4; pp++)
#pragma unroll
              for (int e = 0; e < 4; e++) bm[c][pp][e] = mq == (uint32_t)c ? t.bw[pp][e] : 0;
        }
        {   // the unit's next tile (its next block — of this slice, or of the next one this workgroup walks)
          uint32_t bn = b + 1;
          if (bn == sb1) bn = nks < ks1 ? nb0 : Gm.nblk;
          if (bn < Gm.nblk) mvq_issue_tile<MASK>(fmt, wbase + (size_t)bn * tb, lane, nxt);
        }
        const uint32_t xb = buf * buf_bytes + bi * n_seq * kXLdsRecord;
        // sequences past the last one repeat it: computed, never stored
        i32x4 a[4];
        auto load_a = [&](uint32_t g) {
          const uint8_t* p = smem8 + xb + min(4 * g + (n >> 2), n_seq - 1) * kXLdsRecord + a_off;
#pragma unroll
          for (int pp = 0; pp < 4; pp++) a[pp] = *reinterpret_cast<const i32x4*>(p + pp * 256);
        };
        f32x4 xs[2], sx[2];   // by step (group, class) parity
        auto load_x = [&](uint32_t step) {
          const uint8_t* p = smem8 + xb + min((step & ~3u) + mq, n_seq - 1) * kXLdsRecord + kXqXs16 + (step & 3) * 16;
          xs[step & 1] = *reinterpret_cast<const f32x4*>(p);
          sx[step & 1] = *reinterpret_cast<const f32x4*>(p + (kXqSx16 - kXqXs16));
        };
        MacD m[2];
        const i32x4 zero = {0, 0, 0, 0};
        auto mfma = [&](uint32_t step) {
#pragma unroll
          for (int pp = 0; pp < 4; pp++) m[step & 1].d[pp] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[pp], bm[step & 3][pp], zero, 0, 0, 0);
        };
        load_a(0);
        load_x(0);
        mfma(0);
#pragma unroll
        for (int step = 0; step < 4 * NG; step++) {   // a step's products and factors ahead of the vector work of the one before
          if ((step & 3) == 0 && (uint32_t)step >= n_seq) break;
          if ((step & 3) == 3 && step + 1 < 4 * NG) load_a(step / 4 + 1);
          if (step + 1 < 4 * NG) { load_x(step + 1); mfma(step + 1); }
          const int c = step & 3;
          TileOps t;
#pragma unroll
          for (int pp = 0; pp < 4; pp++) { t.f[pp] = ts.f[pp][c]; t.g[pp] = ts.g[pp][c >> 1]; }
          t.dd = ts.dd;
          t.dmin = ts.dmin;
          mvq_mac_finish<MASK>(fmt, t, m[c & 1], xs[c & 1], sx[c & 1], acc[step / 4][c]);
          asm volatile("" : "+v"(acc[step / 4][c]));   // here, not sunk past the later groups' products
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      if (b0 + cn >= sb1) {   // end of the k-slice: the slice's partial sum, in the single-sequence kernel's order
#pragma unroll
        for (int g = 0; g < NG; g++) {
          const float t = (acc[g][0] + acc[g][1]) + (acc[g][2] + acc[g][3]);
          if (SEQ) tot[g] += t;
          else tot[g] = t;
#pragma unroll
          for (int c = 0; c < 4; c++) acc[g][c] = 0.0f;
        }
      }
    }
    ks = nks; b0 = nb0; buf ^= 1u;
  }
  if (SEQ && Gm.fuse) {
    float* red = reinterpret_cast<float*>(smem8);
    const uint32_t at = mvqb_red_at(Gm, wave, n);
    __syncthreads();   // every record has been read
#pragma unroll
    for (int g = 0; g < NG; g++)
      if (4 * g + mq < n_seq) red[(4 * g + mq) * kFuseRed + at] = tot[g];
    mvqb_tail(L, S, B, 0, blockIdx.x, Gm.fuse == 2 ? kFuseRed / 2 : kFuseRed, n_seq, kFuseRed, red, ssq, 1);
    return;
  }
  if (active) {
    const uint32_t slot = SEQ ? 0u : blockIdx.y;
    const size_t rows16 = (size_t)Gm.n_units * 16;
#pragma unroll
    for (int g = 0; g < NG; g++)
      if (4 * g + mq < n_seq) part[((size_t)slot * n_seq + 4 * g + mq) * rows16 + (size_t)u * 16 + n] = tot[g];
  }
}

// ------------------------------------------------------------------------------------------------
// The same for formats whose weights are whole numbers below 32 (Q6_K: below), on the bf16 matrix cores: what a digit needs beside its product moves into the
// operands.  mvqb4 spends eight vector instructions per (row, sequence, 16 elements): two shifts and additions of digit sums, two conversions, a fused
// multiply-add, and the scales.  Here a digit is a bf16 number, the digit times its power of 256 times the chunk's scale, itself a power of two (both exact),
// and the high two and the low two digits of 16 elements lie along one K of 32: the product IS the scaled high or low half, in f32.  Every partial sum is a whole
// multiple of the scale below 2^24 of it (16 elements, weights <= 31; high half |I| >> 16 <= 2^14: 31 * 2^18; low half, two balanced digits, up to 128 * 256 + 128: 16 * 31 * 32896 = 16 316 416),
// so nothing rounds in it.  What is left is one
// addition (the halves: the rounding that the fused multiply-add of the other kernels does, shifted by a power of two) and the fused multiply-add with the weights' scale: the same
// bits.  The sum over the minima, a chain of four fused multiply-adds, is a 16x16x4 f32 matrix instruction, which rounds as that chain does.
//   A: row 4 m + 2 q + half of sequence m + 4 q of eight (a lane of group m gets both halves of sequences m and m + 4), K = lane group's four elements of the half's first digit, then of its second
//   B: the lane group's four weights twice; a lane unpacks one chunk of 64 elements, so the chunks' words are exchanged between the lane groups (4 x 4, four swaps, of packed words three)
// (Inputs beyond 2^117 in magnitude may overflow a half where a zero scale would have hidden it.)
// Q6_K: 0 .. 63 would reach 33 158 336 in the low half, and of sums beyond 2^24 the matrix instruction rounds some (0.07 % of those made so on purpose) otherwise than to the nearest.  So a row of A is ONE digit of one of four
// sequences, K the chunk's 16 elements: a digit's sum is exact whatever its weights, the high half's addition is exact (63 * 2^18), the low half's rounds as the integer's conversion does, and the third is the one above:
// twice the matrix instructions (which have the time) and two additions more a sum.  Against the integer cores (mvqb4: 843 vector instructions a tile and block of 16 sequences), 16 sequences of an 8B model: down
// 29.5 -> 24.2 us, Q, K and V with one Q6_K matrix 21.0 -> 16.0, the head (32000 rows) 65 -> 51; a step of 4 layers, us, 5 / 8 / 16 sequences: Q4_K_M 382 / 410 / 588 -> 371 / 403 / 556, Q6_K 440 / 472 / 709 -> 405 / 447 / 628,
// Q5_K_M 411 / 440 / 614 -> 398 / 430 / 578; Mixtral Q5_K_M, one layer, 297 / 374 / 554 -> 288 / 365 / 530.
// (Signed weights, -32 .. 31, and halves cut at 15 bits need no second product, 20.3, 15.0 and 38 us for the three.  But they are another rounding than ql | qh << 4 less 32 times the sum of x, in the single-sequence kernel
// as well then, and a compressed cache's codes turn on such a rounding.)
// Who writes the input leaves it in this form (xq.h: the wide image), and a chunk's records of all sequences come as they lie in memory, a chunk ahead, by LDS-DMA.  Rewritten from the digits by every workgroup as they
// were staged, they took a quarter of the vector instructions.  gate | up of an 8B model (28672 rows of 4096, Q4_K): 16 sequences 47.4 -> 42.7 us (58 with mvqb4), 8 33.7 -> 30.5; wo 13.6 -> 12.4; a step of 4 layers, 16
// sequences, Q4_K_M 639 -> 617 us, Q4_0 599 -> 554.  Bound by the vector instructions: 339 a tile and block of 16 sequences, 192 of them the sums' own, 65 % of the SIMDs' cycles (the matrix cores 23 %; two waves a SIMD).
// (Matrix and vector instructions dealt out one to six by the scheduler instead of a step's products in front of the sums of the one before: 40.2 -> 41.8 us; without the priorities 41.1.  Two workgroups a CU with half the
// records a chunk, where registers allow, 5 to 8 sequences: no difference.  In 128 registers 16 sequences spill.)
// ------------------------------------------------------------------------------------------------
constexpr uint32_t kX8Records = 32;                  // records of a chunk at most
constexpr uint32_t mvqb8_block_bytes(uint32_t n_seq) { return (n_seq * kXwRecord + 1023) & ~1023u; }   // a block's records in LDS: whole transfers of a wave
typedef __bf16 b16x8 __attribute__((ext_vector_type(8)));
typedef short s16x4 __attribute__((ext_vector_type(4)));

template <int F, int NB, bool SEQ>
__device__ __forceinline__ void mvqb8_body(const Mvqb2Geom& Gm, const MvLaunch& L, const MvBatch& B, float* __restrict__ part, const MvSeg& S, int sg, bool active, uint8_t* smem8) {
  static_assert(F != F_Q80, "weights of eight bits do not fit the exact range");
  constexpr uint32_t MASK = 1u << F;
  constexpr int NG = (NB + 7) / 8, fmt = F;
  auto nq = [](int g) { return NB - 8 * g > 4 ? 2 : 1; };          // a last group of up to four sequences: one per lane
  const uint32_t tid = threadIdx.x, lane = tid & 63, n_seq = B.n_seq;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t u = blockIdx.x * kBWaves + wave;                 // this wave's unit
  auto is = [](int f) { return f == fmt; };
  constexpr uint32_t tb = fmt_tile_bytes(fmt);
  const uint32_t ntiles = (S.n_rows + 15) >> 4;
  const uint32_t ul = u - (sg == 0 ? 0u : sg == 1 ? Gm.ub1 : Gm.ub2);
  uint32_t pass, tl;
  mvqb_unit(Gm, blockIdx.x, wave, ntiles, ul, active, pass, tl);
  float* const ssq = reinterpret_cast<float*>(smem8 + Gm.ssq_at);
  if (SEQ && Gm.fuse && L.do_norm) mvqb_norms(L, B, n_seq, ssq, nullptr);
  const uint8_t* wbase = (pass == 0 ? S.pass[0].plane[0] : S.pass[1].plane[0]) + (size_t)tl * Gm.nblk * tb;
  const uint32_t n = lane & 15, mq = lane >> 4;
  const uint32_t ks0 = SEQ ? 0u : blockIdx.y, ks1 = SEQ ? Gm.T : blockIdx.y + 1;   // this workgroup's slices
  float acc[NG][4][2], tot[NG][2];                                // per group: chunk classes, the lane's sequences 8 g + mq + 4 q
#pragma unroll
  for (int g = 0; g < NG; g++)
#pragma unroll
    for (int q = 0; q < 2; q++) {
      tot[g][q] = 0.0f;
#pragma unroll
      for (int c = 0; c < 4; c++) acc[g][c][q] = 0.0f;
    }

  // a chunk of records (cb blocks x sequences), requested a chunk ahead into a two-deep LDS buffer
  const uint32_t blk_bytes = mvqb8_block_bytes(n_seq), buf_bytes = Gm.cb * blk_bytes;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem8;
  auto chunk_len = [&](uint32_t ks, uint32_t b0) { return min(Gm.cb, min(ks * Gm.nbw + Gm.nbw, Gm.nblk) - b0); };
  auto fetch = [&](uint32_t b0, uint32_t cn, uint32_t buf) {
    const uint32_t np = blk_bytes >> 10;
    for (uint32_t i = 0; i < cn; i++) {
      const uint8_t* src = B.xw + (size_t)(b0 + i) * B.xw_block + lane * 16;
      for (uint32_t p = wave; p < np; p += kBWaves)
        asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
                     : : "v"(src + p * 1024), "s"(__builtin_amdgcn_readfirstlane((int)(lds0 + buf * buf_bytes + i * blk_bytes + p * 1024))) : "memory", "m0");
    }
  };
  uint32_t ks = ks0, b0 = ks0 * Gm.nbw;
  while (ks < ks1 && b0 >= min(ks * Gm.nbw + Gm.nbw, Gm.nblk)) { ks++; b0 = ks * Gm.nbw; }
  uint32_t buf = 0;
  if (ks < ks1) fetch(b0, chunk_len(ks, b0), 0);
  RawT16 nxt;
  if (active && ks < ks1) mvq_issue_tile<MASK>(fmt, wbase + (size_t)b0 * tb, lane, nxt);
  while (ks < ks1) {
    const uint32_t sb1 = min(ks * Gm.nbw + Gm.nbw, Gm.nblk);
    const uint32_t cn = chunk_len(ks, b0);
    // this wave's transfers have arrived: behind them only the next tile's loads
    if (active) asm volatile("s_waitcnt vmcnt(%0)" : : "n"(fmt_loads_per_tile(fmt)) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
    __syncthreads();
    uint32_t nks = ks, nb0 = b0 + cn;   // the chunk after this one
    if (nb0 >= sb1) {
      nks = ks + 1; nb0 = nks * Gm.nbw;
      while (nks < ks1 && nb0 >= min(nks * Gm.nbw + Gm.nbw, Gm.nblk)) { nks++; nb0 = nks * Gm.nbw; }
    }
    if (!active && nks < ks1) fetch(nb0, chunk_len(nks, nb0), buf ^ 1u);   // (every wave has read the chunk that lay there)
    if (active) {
      for (uint32_t bi = 0; bi < cn; bi++) {
        const uint32_t b = b0 + bi;
        // sequences past the last one repeat it: computed, never stored
        const uint8_t* rec0 = smem8 + buf * buf_bytes + bi * blk_bytes;
        if constexpr (F == F_Q6K) {   // one digit of one sequence a row: sequence 4 g + mq is the (g & 1)-th of group g >> 1
          constexpr int N4 = NB / 4, kSteps = 4 * N4;
          const uint8_t *pa[N4], *px[N4];
#pragma unroll
          for (int g = 0; g < N4; g++) {
            pa[g] = rec0 + min(4 * g + (n >> 2), n_seq - 1) * kXwRecord + mq * 512 + (n & 3) * 8;
            px[g] = rec0 + min(4 * g + mq, n_seq - 1) * kXwRecord + kXwSums;
          }
          s16x4 a[2][4], w[4];
          f32x4 d[2][4], xs[2];
          auto load_a = [&](int st) {
#pragma unroll
            for (int pp = 0; pp < 4; pp++) a[st & 1][pp] = *reinterpret_cast<const s16x4*>(pa[st % N4] + (pp * 4 + st / N4) * 32);
          };
          load_a(0);
          load_a(1);
          TileScales ts;
          uint32_t tw[4][4];
          {
            TileOps t;
            mvq_unpack_tile<MASK>(fmt, nxt, lane, t);
            mvq_row_scales<MASK>(fmt, nxt, lane, ts);
#pragma unroll
            for (int pp = 0; pp < 4; pp++) {
              const auto r01 = __builtin_amdgcn_permlane16_swap((uint32_t)t.bw[pp][0], (uint32_t)t.bw[pp][1], false, false);
              const auto r23 = __builtin_amdgcn_permlane16_swap((uint32_t)t.bw[pp][2], (uint32_t)t.bw[pp][3], false, false);
              const auto r02 = __builtin_amdgcn_permlane32_swap(r01[0], r23[0], false, false);
              const auto r13 = __builtin_amdgcn_permlane32_swap(r01[1], r23[1], false, false);
              tw[pp][0] = r02[0]; tw[pp][1] = r13[0]; tw[pp][2] = r02[1]; tw[pp][3] = r13[1];
            }
          }
          asm volatile("" : : "v"(tw[3][0]), "v"(ts.dd));   // (of the tile's last loads)
          if (bi == 0 && nks < ks1) fetch(nb0, chunk_len(nks, nb0), buf ^ 1u);
          {
            uint32_t bn = b + 1;
            if (bn == sb1) bn = nks < ks1 ? nb0 : Gm.nblk;
            if (bn < Gm.nblk) mvq_issue_tile<MASK>(fmt, wbase + (size_t)bn * tb, lane, nxt);
          }
          const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
          auto products = [&](int st) {
            const int c = st / N4, g = st % N4;
            if (g == 0) {
#pragma unroll
              for (int pp = 0; pp < 4; pp++) {
                const uint32_t v = tw[pp][c];
                w[pp] = __builtin_bit_cast(s16x4, make_uint2(__builtin_amdgcn_perm(__float_as_uint(ub1(v)), __float_as_uint(ub0(v)), 0x07060302u),
                                                             __builtin_amdgcn_perm(__float_as_uint(ub3(v)), __float_as_uint(ub2(v)), 0x07060302u)));
              }
            }
#pragma unroll
            for (int pp = 0; pp < 4; pp++) d[st & 1][pp] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[st & 1][pp], w[pp], zero, 0, 0, 0);
            xs[st & 1] = *reinterpret_cast<const f32x4*>(px[g] + c * 16);
          };
          products(0);
#pragma unroll
          for (int st = 0; st < kSteps; st++) {
            const int c = st / N4, g = st % N4;
            if (st + 1 < kSteps) {
              __builtin_amdgcn_s_setprio(1);
              products(st + 1);
              __builtin_amdgcn_s_setprio(0);
            }
            if (st + 2 < kSteps) load_a(st + 2);
            float s1 = 0.0f, V[4];
#pragma unroll
            for (int pp = 0; pp < 4; pp++) {   // high half exact; low half, where it passes 2^24, rounded as the integer's conversion rounds it
              const f32x4 e = d[st & 1][pp];
              V[pp] = (e[0] + e[1]) + (e[2] + e[3]);
            }
#pragma unroll
            for (int pp = 0; pp < 4; pp++) s1 = __builtin_fmaf(ts.f[pp][c], __builtin_fmaf(-32.0f, xs[st & 1][pp], V[pp]), s1);
            acc[g >> 1][c][g & 1] = __builtin_fmaf(ts.dd, s1, acc[g >> 1][c][g & 1]);
            asm volatile("" : "+v"(acc[g >> 1][c][g & 1]));
            __builtin_amdgcn_sched_barrier(0);
          }
          continue;
        }
        const uint8_t *pa[NG], *px[NG][2];
#pragma unroll
        for (int g = 0; g < NG; g++) {
          pa[g] = rec0 + min(8 * g + (n >> 2) + (n & 2) * 2, n_seq - 1) * kXwRecord + mq * 512 + (n & 1) * 16;
#pragma unroll
          for (int q = 0; q < 2; q++) px[g][q] = rec0 + min(8 * g + mq + 4 * q, n_seq - 1) * kXwRecord + kXwSums;
        }
        const bool mins = is(F_Q4K) || is(F_Q5K);
        float xm[4];   // the minima's operand: row 4 m + 2 g + q = sequence 8 g + m + 4 q, K = step
        if (mins) {
          const uint8_t* p = rec0 + min((n & 2) * 4 + (n >> 2) + (n & 1) * 4, n_seq - 1) * kXwRecord + kXwSums + mq * 4;
#pragma unroll
          for (int c = 0; c < 4; c++) xm[c] = *reinterpret_cast<const float*>(p + c * 16);
        }
        // steps (class, group), a step's products ahead of the vector work of the one before, its operands a step ahead of those
        constexpr int kSteps = 4 * NG;
        b16x8 a[2][4], w[4];
        f32x4 d[2][4], xs[2][2], s2[2];
        auto load_a = [&](int st) {
#pragma unroll
          for (int pp = 0; pp < 4; pp++) a[st & 1][pp] = *reinterpret_cast<const b16x8*>(pa[st % NG] + (pp * 4 + st / NG) * 32);
        };
        load_a(0);
        load_a(1);
        TileScales ts;
        uint32_t tw[4][4];   // [step pp][class c]: the lane group's four weights of chunk 4 pp + c
        {
          mvq_row_scales<MASK>(fmt, nxt, lane, ts);
          if constexpr (F == F_Q4K || F == F_Q40) {
            // a word holds the nibbles of two elements' fours: whole words change halves first, then the unpacked ones rows (three swaps a step instead of four:
            // 16 sequences, gate | up 39.7 -> 39.4 us, the products split over k 12.45 -> 12.2)
#pragma unroll
            for (int pp = 0; pp < 4; pp++) {
              const uint32_t N0 = (pp & 1) ? nxt.q[pp >> 1].z : nxt.q[pp >> 1].x, N1 = (pp & 1) ? nxt.q[pp >> 1].w : nxt.q[pp >> 1].y;
              const auto h = __builtin_amdgcn_permlane32_swap(N0, N1, false, false);
              const auto r01 = __builtin_amdgcn_permlane16_swap(h[0] & 0x0F0F0F0Fu, (h[0] >> 4) & 0x0F0F0F0Fu, false, false);
              const auto r23 = __builtin_amdgcn_permlane16_swap(h[1] & 0x0F0F0F0Fu, (h[1] >> 4) & 0x0F0F0F0Fu, false, false);
              tw[pp][0] = r01[0]; tw[pp][1] = r01[1]; tw[pp][2] = r23[0]; tw[pp][3] = r23[1];
            }
          } else {
            TileOps t;
            mvq_unpack_tile<MASK>(fmt, nxt, lane, t);
#pragma unroll
            for (int pp = 0; pp < 4; pp++) {
              const auto r01 = __builtin_amdgcn_permlane16_swap((uint32_t)t.bw[pp][0], (uint32_t)t.bw[pp][1], false, false);
              const auto r23 = __builtin_amdgcn_permlane16_swap((uint32_t)t.bw[pp][2], (uint32_t)t.bw[pp][3], false, false);
              const auto r02 = __builtin_amdgcn_permlane32_swap(r01[0], r23[0], false, false);
              const auto r13 = __builtin_amdgcn_permlane32_swap(r01[1], r23[1], false, false);
              tw[pp][0] = r02[0]; tw[pp][1] = r13[0]; tw[pp][2] = r02[1]; tw[pp][3] = r13[1];
            }
          }
        }
        asm volatile("" : : "v"(tw[3][0]), "v"(ts.dd));   // (of the tile's last load)
        if (bi == 0 && nks < ks1) fetch(nb0, chunk_len(nks, nb0), buf ^ 1u);   // the chunk after this one: behind this tile's wait, which would wait for it too, and in front of the next tile's loads
        {   // the unit's next tile (its next block — of this slice, or of the next one this workgroup walks)
          uint32_t bn = b + 1;
          if (bn == sb1) bn = nks < ks1 ? nb0 : Gm.nblk;
          if (bn < Gm.nblk) mvq_issue_tile<MASK>(fmt, wbase + (size_t)bn * tb, lane, nxt);
        }
        const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
        auto products = [&](int st) {
          const int c = st / NG, g = st % NG;
          if (g == 0) {
#pragma unroll
            for (int pp = 0; pp < 4; pp++) {
              const uint32_t v = tw[pp][c];
              uint32_t lo, hi;
              if (is(F_Q5K)) {
                lo = __builtin_amdgcn_perm(__float_as_uint(ub1(v)), __float_as_uint(ub0(v)), 0x07060302u);
                hi = __builtin_amdgcn_perm(__float_as_uint(ub3(v)), __float_as_uint(ub2(v)), 0x07060302u);
              } else {   // a byte up to 16 is, as an 8-bit float, 2^-9 of itself: two a conversion (gate | up as above 42.7 -> 40.3 us)
                lo = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(v, 512.0f, false));
                hi = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(v, 512.0f, true));
              }
              w[pp] = __builtin_bit_cast(b16x8, u32x4{lo, hi, lo, hi});
            }
            if (mins) s2[c & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(xm[c], ts.gq[c >> 1], zero, 0, 0, 0);
          }
#pragma unroll
          for (int pp = 0; pp < 4; pp++) d[st & 1][pp] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[st & 1][pp], w[pp], zero, 0, 0, 0);
          if (!mins) {
#pragma unroll
            for (int q = 0; q < nq(g); q++) xs[st & 1][q] = *reinterpret_cast<const f32x4*>(px[g][q] + c * 16);
          }
        };
        products(0);
#pragma unroll
        for (int st = 0; st < kSteps; st++) {
          const int c = st / NG, g = st % NG;
          if (st + 1 < kSteps) {   // (ahead of the other wave's vector work)
            __builtin_amdgcn_s_setprio(1);
            products(st + 1);
            __builtin_amdgcn_s_setprio(0);
          }
          if (st + 2 < kSteps) load_a(st + 2);
#pragma unroll
          for (int q = 0; q < nq(g); q++) {
            float s1 = 0.0f, V[4];
#pragma unroll
            for (int pp = 0; pp < 4; pp++) V[pp] = d[st & 1][pp][2 * q] + d[st & 1][pp][2 * q + 1];
            if (mins) {
#pragma unroll
              for (int pp = 0; pp < 4; pp++) s1 = __builtin_fmaf(ts.f[pp][c], V[pp], s1);
              acc[g][c][q] += ts.dd * s1 - ts.dmin * s2[c & 1][2 * g + q];
            } else {
#pragma unroll
              for (int pp = 0; pp < 4; pp++) s1 = __builtin_fmaf(ts.f[pp][c], __builtin_fmaf(-8.0f, xs[st & 1][q][pp], V[pp]), s1);
              acc[g][c][q] += s1;
            }
            asm volatile("" : "+v"(acc[g][c][q]));   // here, not sunk past the later steps' products
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      if (b0 + cn >= sb1) {   // end of the k-slice: the slice's partial sum, in the single-sequence kernel's order
#pragma unroll
        for (int g = 0; g < NG; g++)
#pragma unroll
          for (int q = 0; q < 2; q++) {
            const float t = (acc[g][0][q] + acc[g][1][q]) + (acc[g][2][q] + acc[g][3][q]);
            if (SEQ) tot[g][q] += t;
            else tot[g][q] = t;
#pragma unroll
            for (int c = 0; c < 4; c++) acc[g][c][q] = 0.0f;
          }
      }
    }
    ks = nks; b0 = nb0; buf ^= 1u;
  }
  if (SEQ && Gm.fuse) {
    float* red = reinterpret_cast<float*>(smem8);
    const uint32_t at = mvqb_red_at(Gm, wave, n);
    __syncthreads();   // every record has been read
#pragma unroll
    for (int g = 0; g < NG; g++)
#pragma unroll
      for (int q = 0; q < 2; q++) {
        const uint32_t s = 8 * g + mq + 4 * q;
        if (q < nq(g) && s < n_seq) red[s * kFuseRed + at] = tot[g][q];
      }
    mvqb_tail(L, S, B, 0, blockIdx.x, Gm.fuse == 2 ? kFuseRed / 2 : kFuseRed, n_seq, kFuseRed, red, ssq, 1);
    return;
  }
  if (active) {
    const uint32_t slot = SEQ ? 0u : blockIdx.y;
    const size_t rows16 = (size_t)Gm.n_units * 16;
#pragma unroll
    for (int g = 0; g < NG; g++)
#pragma unroll
      for (int q = 0; q < 2; q++) {
        const uint32_t s = 8 * g + mq + 4 * q;
        if (q < nq(g) && s < n_seq) part[((size_t)slot * n_seq + s) * rows16 + (size_t)u * 16 + n] = tot[g][q];
      }
  }
}

// (a launch of two formats: a wave takes its unit's path; both meet at the same barriers, which the launch's geometry alone decides)
template <uint32_t MASK, int NB, bool SEQ>
__global__ void __launch_bounds__(kBWaves * 64) mvqb8_kernel(const Mvqb2Geom Gm, const MvLaunch L, const MvBatch B, float* __restrict__ part) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem8[];
  const uint32_t u = blockIdx.x * kBWaves + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const bool active = u < Gm.n_units;
  const int sg = SEQ && Gm.fuse ? 0 : (int)(u >= Gm.ub1) + (int)(u >= Gm.ub2);
  const MvSeg& S = L.seg[active ? sg : 0];
  if constexpr ((MASK & (MASK - 1)) == 0) {
    mvqb8_body<__builtin_ctz(MASK), NB, SEQ>(Gm, L, B, part, S, sg, active, smem8);
  } else {
    if (fmt_of_dev_type(S.type) == F_Q6K) mvqb8_body<F_Q6K, NB, SEQ>(Gm, L, B, part, S, sg, active, smem8);
    else mvqb8_body<__builtin_ctz(MASK & ~(1u << F_Q6K)), NB, SEQ>(Gm, L, B, part, S, sg, active, smem8);
  }
}

// ------------------------------------------------------------------------------------------------
// The epilogue of a launch whose partial sums went through memory: per row and sequence the sum over the slices, then what mv_epilogue_view does with it.  Workgroups are the single-sequence geometry's.
// A launch of this size is nothing but latency, so it is one chain: a thread has one (sequence, row), everything it will need (partial sums, residual, the next norm's weight, position and slot, the rotation) is
// requested at once, the sum is made in registers, and what a launch does with its rows is compiled in.  No LDS, and no barrier but for the norm's factors.  (Before, the partial sums went through LDS and everything
// else was asked for behind their barrier: 5.7 to 6.2 us a launch at 16 sequences of an 8B model, now 5.0, of which an empty launch is 1.5 to 2; prompts and 24 steps of 8 layers 37.9 -> 36.8 ms, five sequences of
// Mixtral, two layers, 24 steps 12.30 -> 12.15.)
// ------------------------------------------------------------------------------------------------
enum : int { ER_OUT = 0, ER_PAIR = 1, ER_QKV = 2 };   // store / + residual; SwiGLU; RoPE, caches and what is stored beside them
struct MvqbRowsSeg {
  float* out;
  const float *resid, *nw, *bias;
  uint8_t* xq;
  float* ssq;
  uint8_t* xw;
  uint32_t n_rows, wg_begin, rows, unit_begin;   // rows: of a workgroup
  uint32_t out_stride, resid_stride, xq_stride, ssq_stride;
  uint32_t epi, head_dim, max_seq, pad;
};
struct MvqbRows {
  const float *part, *ssq_part, *rope_cs;
  const int *pos, *slot, *ind_cnt, *ind_idx;
  uint64_t cache_stride, part_z_floats;
  uint32_t n_seq, nslots, rows16, wb1, wb2;      // rows16: of all units; wb: first workgroups of segments 1 and 2
  uint32_t n_ssq, ssq_stride, k;
  uint32_t ind_div, ind_stride, xw_block;
  float eps;
  MvqbRowsSeg seg[3];
};

template <int KIND, bool NORM>
__global__ void __launch_bounds__(kBWaves * 64) mvqb_rows_kernel(const MvqbRows A) {
  constexpr int NP = KIND == ER_PAIR ? 2 : 1, kSlots = 8;
  __shared__ float s_inv[kMaxBatch];
  const uint32_t tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), bid = blockIdx.x;
  const int sg = KIND == ER_QKV ? (int)(bid >= A.wb1) + (int)(bid >= A.wb2) : 0;
  const MvqbRowsSeg& S = A.seg[sg];
  const float* part = A.part;
  uint32_t n_seq = A.n_seq;
  const uint32_t n_part = n_seq;
  const int* ind_idx = nullptr;
  if (KIND != ER_QKV && A.ind_cnt) {
    uint32_t cw;
    asm volatile("s_load_dword %0, %1, 0x0\n\ts_waitcnt lgkmcnt(0)" : "=s"(cw) : "s"(A.ind_cnt + blockIdx.z) : "memory");
    n_seq = min(cw, n_seq);
    if (n_seq == 0) return;
    ind_idx = A.ind_idx + (size_t)blockIdx.z * A.ind_stride;
    part += (size_t)blockIdx.z * A.part_z_floats;
  }
  const uint32_t rows = S.rows, chunks = rows >> 4, items = n_seq * rows, row0 = (bid - S.wg_begin) * rows;
  const uint32_t n_rows = S.n_rows, padded = (n_rows + 15) & ~15u, nslots = A.nslots;
  const bool rope = KIND == ER_QKV && (S.epi == EPI_ROPE_Q || S.epi == EPI_ROPE_K), cache = KIND == ER_QKV && (S.epi == EPI_ROPE_K || S.epi == EPI_V_CACHE);
  // the norm's partial sums: wave w has sequences w and w + 8 (as wave 0 of the single-sequence kernel has its own)
  float nsum[2][4];
  auto norm_part = [&](uint32_t s) { return A.ssq_part + (size_t)(ind_idx ? (uint32_t)ind_idx[s] / A.ind_div : s) * A.ssq_stride; };
  if (NORM) {
#pragma unroll
    for (uint32_t h = 0; h < 2; h++) {
      const uint32_t s = wave + h * kBWaves;
#pragma unroll
      for (uint32_t j = 0; j < 4; j++) {
        nsum[h][j] = 0.0f;
        if (s < n_seq && lane + 64 * j < A.n_ssq) nsum[h][j] = norm_part(s)[lane + 64 * j];
      }
    }
  }
  for (uint32_t i0 = 0; i0 < items; i0 += kBWaves * 64) {
    const uint32_t c = (i0 + tid) >> 4, sc = c / chunks;
    const bool in = sc < n_seq;
    const uint32_t s = in ? sc : 0, rl = in ? (c - sc * chunks) * 16 + (tid & 15) : tid & 15, row = row0 + rl;
    const bool live = in && row < n_rows;
    const uint32_t rc = row < padded ? row : 0, rl_ = row < n_rows ? row : 0;   // (loads are unconditional)
    uint32_t so = s;                                   // whose output vectors (an indirect entry's (sequence, slot) pair)
    if (KIND != ER_QKV && ind_idx) so = (uint32_t)ind_idx[s];
    uint32_t pos = 0, slot = 0;
    if (KIND == ER_QKV) { pos = (uint32_t)A.pos[s]; slot = (uint32_t)A.slot[s]; }
    float v[NP][kSlots];
#pragma unroll
    for (int p = 0; p < NP; p++)
#pragma unroll
      for (uint32_t j = 0; j < kSlots; j++)
        v[p][j] = part[((size_t)(j < nslots ? j : 0) * n_part + s) * A.rows16 + (size_t)S.unit_begin * 16 + p * padded + rc];
    const float res = KIND == ER_OUT && S.resid ? S.resid[(size_t)so * S.resid_stride + rl_] : 0.0f;
    const float nw = KIND != ER_QKV && S.nw ? S.nw[rl_] : 1.0f;
    const float bias = S.bias ? S.bias[rl_] : 0.0f;
    const uint32_t d = KIND == ER_QKV ? S.head_dim : 0, head = d == 0 ? 0 : (d & (d - 1)) == 0 ? row >> __builtin_ctz(d) : row / d, e = row - head * d;
    float cs = 0.0f, sn = 0.0f;
    if (rope) {
      const float* at = A.rope_cs + ((size_t)pos * (d / 2) + e / 2) * 2;
      cs = at[0];
      sn = at[1];
    }
    if (NORM && i0 == 0) {
#pragma unroll
      for (uint32_t h = 0; h < 2; h++) {
        const uint32_t q = wave + h * kBWaves;
        if (q < n_seq) {
          float ss = (nsum[h][0] + nsum[h][1]) + (nsum[h][2] + nsum[h][3]);
          const float* np = norm_part(q);
          for (uint32_t i = 256 + lane; i < A.n_ssq; i += 64) ss += np[i];
          ss = wave_sum_to_lane63(ss);
          if (lane == 63) s_inv[q] = mv_inv_rms(ss, A.k, A.eps);
        }
      }
      __syncthreads();
    }
    const float inv = NORM ? s_inv[s] : 1.0f;
    float t[NP];
#pragma unroll
    for (int p = 0; p < NP; p++) {
      t[p] = 0.0f;
#pragma unroll
      for (uint32_t j = 0; j < kSlots; j++)
        if (j < nslots) t[p] += v[p][j];
      t[p] *= inv;
    }
    if (S.bias) t[0] += bias;
    if (KIND == ER_QKV) {
      const float other = dpp_f<0xB1>(t[0]);           // the pair's other element
      if (rope) {
        const float x0 = (tid & 1) ? other : t[0], x1 = (tid & 1) ? t[0] : other;
        const float y0 = x0 * cs - x1 * sn, y1 = x0 * sn + x1 * cs;  // ops.rs:1326-1331
        t[0] = (tid & 1) ? y1 : y0;
      }
      if (live) {
        float* dst = cache ? S.out + (size_t)slot * A.cache_stride + ((size_t)head * S.max_seq + pos) * d + e : S.out + (size_t)s * S.out_stride + row;
        *dst = t[0];
      }
    } else if (live) {
      const float outv = KIND == ER_PAIR ? silu_f(t[0]) * t[1] : S.resid ? t[0] + res : t[0];
      S.out[(size_t)so * S.out_stride + row] = outv;
      if (S.xq)                                        // (n_rows is a multiple of 16 here: a chunk's 16 threads are all live)
        xq_store_chunk(S.xq + (size_t)so * S.xq_stride, row >> 4, outv * nw, S.ssq ? S.ssq + (size_t)so * S.ssq_stride : nullptr, outv, tid, S.xw ? S.xw + (size_t)so * kXwRecord : nullptr, A.xw_block);
    }
  }
}

// ------------------------------------------------------------------------------------------------
// gate | up of a mixture's experts in a step of few sequences: an expert has one entry or two, so the launch is a stream of weights.  mvqb2 keeps one tile a wave under way behind a barrier per chunk (22 KB a CU);
// here a workgroup is the single-sequence kernel's (mvq_body): four waves = k-slices x unit groups, every wave with its slices' records of up to two entries in LDS of its own and a few tiles under way, no barrier
// before the sums meet, and SwiGLU in place; three workgroups a CU.  More entries than two: another turn over the same weights.  Slices, operations and sums are the single-sequence kernel's.
// Bound by the weights' stream; one layer of 8 experts of 14336 x 4096, two a sequence, mvqb2 -> this: Q5_K 5 sequences 137 -> 104 us (3.6 -> 4.8 TB/s), Q6_K 4: 122 -> 96, 8: 176 -> 165, Q8_0 4: 128 -> 112, 8: 176 -> 194
// (an expert's third entry reads the weights again).  Q4_0 stays with mvqb2 (60 us of 4 sequences against 69: nothing to convert, and a tile is too small a request).
// down stays with mvqb2 too: its slices are a grid dimension, so that it has bytes enough under way (Q6_K 51 us as the same stream 50, Q8_0 57 and 58).
// ------------------------------------------------------------------------------------------------
constexpr int few_depth(int f) { return f == F_Q4K ? 4 : f == F_Q6K ? 2 : 3; }   // tiles a wave has under way: what the registers of three waves a SIMD hold
struct MvqbFew { uint32_t T, nbw, nblk; };

template <int F, int SQ>
__device__ __forceinline__ void mvqb_few_turn(const MvqbFew& Gm, const MvLaunch& L, const MvBatch& B, uint8_t* smem8, uint32_t ez, const int* ind_idx, uint32_t s0, uint32_t n_seq) {
  constexpr uint32_t tb = fmt_tile_bytes(F), MASK = 1u << F, W = kFewWaves;
  constexpr int LPT = fmt_loads_per_tile(F), D = few_depth(F);
  const MvSeg& S = L.seg[0];
  const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), n = lane & 15, mq = lane >> 4;
  // T is 1, 2, 4 or 8.  The waves share the slices, SL consecutive ones from ks0 on, and with fewer slices than waves the units
  const uint32_t SL = Gm.T > W ? Gm.T / W : 1, tw = Gm.T > W ? W : Gm.T, ks0 = (wave & (tw - 1)) * SL;
  const uint32_t units_w = kBWaves * tw / W, unit0 = Gm.T < W ? (wave >> __builtin_ctz(Gm.T)) * units_w : 0;   // units of this wave
  const uint32_t blk0 = ks0 * Gm.nbw, blk1 = min(Gm.nblk, blk0 + SL * Gm.nbw);
  const uint32_t nblk_w = blk0 < blk1 ? blk1 - blk0 : 0;
  const uint32_t ntiles = (S.n_rows + 15) >> 4, rows = kFuseRed / 2;
  const uint8_t* const plane0 = S.pass[0].plane[0] + (uint64_t)ez * S.pass[0].sel_stride[0];
  const uint8_t* const plane1 = S.pass[1].plane[0] + (uint64_t)ez * S.pass[1].sel_stride[0];
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem8;
  const uint32_t wrecs = SL * Gm.nbw, wreg = wave * wrecs * SQ * (uint32_t)kXqRecord;
  float* const red = reinterpret_cast<float*>(smem8 + few_red_at(Gm.T, Gm.nbw));
  const uint32_t red_floats = kFuseRed * Gm.T;             // a sequence's, [pass][slice][row]
  auto store = [&](uint32_t i, uint32_t ks, int s, float t) __attribute__((always_inline)) {
    const uint32_t w = unit0 + i;
    if (mq == 0 && (uint32_t)s < n_seq) red[(size_t)s * red_floats + ((w & 1) * Gm.T + ks) * rows + (w >> 1) * 16 + n] = t;
  };
  const uint32_t nitems = units_w * nblk_w;
  // slices beyond the last block: their sums read as zero
  for (uint32_t ks = ks0 + (nblk_w + Gm.nbw - 1) / Gm.nbw; ks < ks0 + SL; ks++)
    for (uint32_t i = 0; i < units_w; i++)
#pragma unroll
      for (int s = 0; s < SQ; s++) store(i, ks, s, 0.0f);
  if (nitems == 0) return;
  // the records of the slices, first of all that is asked for
#pragma unroll
  for (int s = 0; s < SQ; s++) {
    uint32_t v;
    const uint32_t at = (uint32_t)__builtin_amdgcn_readfirstlane((int)min(s0 + s, s0 + n_seq - 1));
    asm volatile("s_load_dword %0, %1, 0x0\n\ts_waitcnt lgkmcnt(0)" : "=s"(v) : "s"(ind_idx + at) : "memory");
    const uint8_t* src = S.pass[0].xq + (size_t)(v / B.ind_div) * B.xq_stride + (size_t)blk0 * kXqRecord;
    for (uint32_t b = 0; b < nblk_w; b++, src += kXqRecord)
      asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off\n\ts_add_u32 m0, m0, 0x400\n\ts_nop 0\n\tglobal_load_lds_dword %1, off"
                   : : "v"(src + lane * 16), "v"(src + 1024 + lane * 4), "s"(__builtin_amdgcn_readfirstlane((int)(lds0 + wreg + (s * wrecs + b) * (uint32_t)kXqRecord))) : "memory", "m0", "scc");
  }
  // items in order: unit, then block
  uint32_t ni = 0, nb = 0;   // the next to request
  const uint8_t* src = nullptr;
  auto locate = [&]() __attribute__((always_inline)) {   // a unit is a tile of gate, or of up; beyond the last tile its rows again, never stored
    const uint32_t w = unit0 + ni, tl = min(blockIdx.x * (kBWaves / 2) + (w >> 1), ntiles - 1);
    src = (w & 1 ? plane1 : plane0) + ((size_t)tl * Gm.nblk + blk0) * tb;
  };
  locate();
  auto issue = [&](RawT16& r) __attribute__((always_inline)) {
    mvq_issue_tile<MASK>(F, src, lane, r);
    src += tb;
    if (++nb == nblk_w) {
      nb = 0;
      if (++ni < units_w) locate();
    }
  };
  uint32_t ci = 0, cb = 0, cs = 0, ck = ks0;   // the item at hand: unit, block, block of the slice, slice
  float acc[SQ];
#pragma unroll
  for (int s = 0; s < SQ; s++) acc[s] = 0.0f;
  auto consume = [&](const RawT16& r) __attribute__((always_inline)) {
    const uint8_t* rec = smem8 + wreg + cb * (uint32_t)kXqRecord;
    if constexpr (SQ == 1) {
      mvq_consume_tile<MASK>(F, r, rec, lane, acc[0]);
    } else {
      TileOps t;
      mvq_unpack_tile<MASK>(F, r, lane, t);
#pragma unroll
      for (int s = 0; s < SQ; s++) {
        XqOps o;
        xq_load_ops(rec + s * wrecs * (uint32_t)kXqRecord, lane, o);
        mvq_mac_tile<MASK>(F, t, o, acc[s]);
      }
    }
    cb++;
    if (++cs == Gm.nbw || cb == nblk_w) {   // the four lane groups: the slice's sum
#pragma unroll
      for (int s = 0; s < SQ; s++) {
        float t = acc[s] + __shfl_xor(acc[s], 16, 64);
        t += __shfl_xor(t, 32, 64);
        store(ci, ck, s, t);
        acc[s] = 0.0f;
      }
      cs = 0;
      ck++;
      if (cb == nblk_w) {
        cb = 0;
        ck = ks0;
        ci++;
      }
    }
  };
  RawT16 buf[D];
  auto run = [&](auto first) __attribute__((always_inline)) {
    constexpr int NF = decltype(first)::value;
#pragma unroll
    for (int j = 0; j < NF; j++) issue(buf[j]);
    asm volatile("s_waitcnt vmcnt(%0)" : : "n"(NF * LPT) : "memory");   // the records alone
    if constexpr (NF < D) {
#pragma unroll
      for (int j = 0; j < NF; j++) consume(buf[j]);
    } else {
      uint32_t rem = nitems;   // not yet consumed, D of them under way
      while (rem >= 2 * D) {
#pragma unroll
        for (int j = 0; j < D; j++) { consume(buf[j]); issue(buf[j]); }
        rem -= D;
      }
      const uint32_t more = rem - D;
#pragma unroll
      for (int j = 0; j < D; j++) {
        consume(buf[j]);
        if ((uint32_t)j < more) issue(buf[j]);
      }
#pragma unroll
      for (int j = 0; j < D - 1; j++)
        if ((uint32_t)j < more) consume(buf[j]);
    }
  };
  if (nitems == 1) run(std::integral_constant<int, 1>{});
  else if (nitems == 2) run(std::integral_constant<int, 2>{});
  else if (nitems == 3 && D > 3) run(std::integral_constant<int, 3>{});
  else run(std::integral_constant<int, D>{});
}

template <int F>
__global__ void __launch_bounds__(kFewWaves * 64, 3) mvqb_few_kernel(const MvqbFew Gm, const MvLaunch L, const MvBatch B) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem8[];
  const uint32_t ez = blockIdx.z;
  uint32_t n_seq;
  asm volatile("s_load_dword %0, %1, 0x0\n\ts_waitcnt lgkmcnt(0)" : "=s"(n_seq) : "s"(B.ind_cnt + ez) : "memory");
  n_seq = (uint32_t)__builtin_amdgcn_readfirstlane((int)min(n_seq, B.n_seq));
  if (n_seq == 0) return;
  const int* ind_idx = B.ind_idx + (size_t)ez * B.ind_stride;
  float* const ssq = reinterpret_cast<float*>(smem8 + few_ssq_at(Gm.T, Gm.nbw));
  if (L.do_norm) mvqb_norms(L, B, n_seq, ssq, ind_idx);
  for (uint32_t s0 = 0; s0 < n_seq; s0 += kFewEntries) {
    const uint32_t left = n_seq - s0, now = left < kFewEntries ? left : kFewEntries;
    if (now == 1) mvqb_few_turn<F, 1>(Gm, L, B, smem8, ez, ind_idx, s0, now);
    else mvqb_few_turn<F, 2>(Gm, L, B, smem8, ez, ind_idx, s0, now);
    // SwiGLU as mv_epilogue_view has it: a thread a row and entry
    constexpr uint32_t rows = kFuseRed / 2;
    const MvSeg& S = L.seg[0];
    const float* red = reinterpret_cast<const float*>(smem8 + few_red_at(Gm.T, Gm.nbw));
    const uint32_t s = threadIdx.x / rows, rl = threadIdx.x % rows, row = blockIdx.x * rows + rl;
    __syncthreads();
    if (s < now && row < S.n_rows) {
      float inv = 1.0f;
      if (L.do_norm) {
        float tot = 0.0f;
        for (uint32_t w = 0; w < (uint32_t)kBWaves; w++) tot += ssq[(s0 + s) * 8 + w];
        inv = 1.0f / __builtin_sqrtf(tot / (float)L.k + L.eps);
      }
      float v[2];
#pragma unroll
      for (uint32_t p = 0; p < 2; p++) {
        float t = 0.0f;
        for (uint32_t ks = 0; ks < Gm.T; ks++) t += red[(size_t)s * kFuseRed * Gm.T + (p * Gm.T + ks) * rows + rl];
        v[p] = t * inv;
      }
      const float a = silu_f(v[0]) * v[1];
      const uint32_t so = (uint32_t)ind_idx[s0 + s];
      S.out[(size_t)so * B.out_stride[0] + row] = a;
      if (S.xq_out) {
        const float w = S.xq_nw ? S.xq_nw[row] : 1.0f;
        xq_store_chunk(S.xq_out + (size_t)so * B.xq_out_stride[0], row >> 4, a * w, S.xq_ssq ? S.xq_ssq + (size_t)so * B.ssq_out_stride[0] : nullptr, a, rl);
      }
    }
    __syncthreads();   // (the next turn's sums go where these were)
  }
}

// ------------------------------------------------------------------------------------------------
// host
// ------------------------------------------------------------------------------------------------
static size_t mvqb_lds_bytes(uint32_t n_seq, uint32_t red_floats) { return ((size_t)n_seq * red_floats + (size_t)n_seq * 8) * 4 + 64; }

template <uint32_t MASK, int NB>
static hipError_t mvqb_go(const MvLaunch& L, const MvBatch& B, const MvGeom& g, uint32_t threads, size_t lds, hipStream_t st) {
  static bool attr_set[64] = {};
  if (hipError_t e = lds_opt_in(reinterpret_cast<const void*>(&mvqb_kernel<MASK, NB>), 160 * 1024, attr_set); e != hipSuccess) return e;
  hipLaunchKernelGGL((mvqb_kernel<MASK, NB>), dim3(g.n_wg), dim3(threads), lds, st, g.wbpack, g.geom, g.geom2, L.red_floats, L, B);
  return hipGetLastError();
}

// Sequences from which the groups of four are the faster ones (a step, 4 layers of an 8B model in Q4_K_M / Q8_0, us: 2 sequences 366 / 411 with mvqb2,
// 388 / 398 in groups; 3: 416 / 439 against 390 / 419; 5: 495 / 494 against 504 / 488; 8: 579 / 567 against 529 / 520; 16: 905 / 867 against 786 / 751).
// Indirect launches (a mixture's experts) have one or two sequences per expert: they go to mvqb_few or mvqb2.
constexpr uint32_t kMvqb4MinSeq = 3;

// Sequences from which groups of eight on the bf16 matrix cores are the faster ones (a step, 4 layers, us, groups of four against groups of eight over wide images, 3 / 4 sequences: an 8B model in Q4_K_M 342 / 354 against
// 357 / 370, Q5_K_M 362 / 373 against 389 / 400, Q4_0 323 / 334 against 335 / 347; 2048 x 5632, Q4_K_M, 239 / 249 against 242 / 253; 8192 x 28672 Q4_K_M 775 / 816 against 780 / 808.  Before the wide images, with Q6_K in
// groups of eight as two products, 5: 503 / 484 (Q4_K_M / Q4_0) against 479 / 455, 8: 531 / 512 against 502 / 480, 16: 786 / 761 against 683 / 679)
constexpr uint32_t kMvqb8MinSeq = 5;

bool mvqb_wide_input(int dev_type, uint32_t n_seq) {
  const int f = fmt_of_dev_type(dev_type);
  return n_seq >= kMvqb8MinSeq && f >= 0 && f != F_Q80;
}

// a wide image where the input's writer left none: a workgroup per record, a thread per word of digits
__global__ void __launch_bounds__(256) xw_from_xq_kernel(const uint8_t* __restrict__ xq, uint32_t xq_stride, uint8_t* __restrict__ xw, uint32_t xw_block) {
  const uint8_t* rec = xq + (size_t)blockIdx.y * xq_stride + (size_t)blockIdx.x * kXqRecord;
  uint8_t* wide = xw + (size_t)blockIdx.x * xw_block + (size_t)blockIdx.y * kXwRecord;
  const uint32_t t = threadIdx.x, i = (t >> 3) & 3, j = (t >> 5) * 2 + ((t >> 2) & 1), Q = t & 3, slot = (j & 3) * 4 + (j >> 2);   // digit 3 - i of elements 4 Q .. of chunk j
  const float sx = *reinterpret_cast<const float*>(rec + kXqSx16 + slot * 4) * (float)(1u << (8 * (3 - i)));
  *reinterpret_cast<uint2*>(wide + Q * 512 + j * 32 + (i >> 1) * 16 + (i & 1) * 8) = xw_digits(*reinterpret_cast<const uint32_t*>(rec + t * 4), sx);
  if (t < 16) *reinterpret_cast<float*>(wide + kXwSums + t * 4) = *reinterpret_cast<const float*>(rec + kXqXs16 + t * 4);
}

hipError_t xw_from_xq_launch(const uint8_t* xq, uint32_t xq_stride, uint8_t* xw, uint32_t xw_block, uint32_t k, uint32_t n_seq, hipStream_t st) {
  if (k == 0 || k % 256 || n_seq == 0 || (uint64_t)n_seq * kXwRecord > xw_block) return hipErrorInvalidValue;
  hipLaunchKernelGGL(xw_from_xq_kernel, dim3(k / 256, n_seq), dim3(256), 0, st, xq, xq_stride, xw, xw_block);
  return hipGetLastError();
}

template <uint32_t MASK, int NB>
static hipError_t mvqb8_go(const MvLaunch& L, const MvBatch& B, Mvqb2Geom Gm, bool seq, uint32_t groups, hipStream_t st) {
  static bool attr_set[2][64] = {};
  if (!B.xw || (uint64_t)B.n_seq * kXwRecord > B.xw_block) return hipErrorInvalidValue;
  Gm.cb = std::max(1u, std::min(Gm.nbw, kX8Records / B.n_seq));
  Gm.ssq_at = 2 * Gm.cb * mvqb8_block_bytes(B.n_seq);
  const size_t lds = Gm.ssq_at + mvqb_fuse_lds(B.n_seq);
  if (seq) {
    if (hipError_t e = lds_opt_in(reinterpret_cast<const void*>(&mvqb8_kernel<MASK, NB, true>), 160 * 1024, attr_set[0]); e != hipSuccess) return e;
    hipLaunchKernelGGL((mvqb8_kernel<MASK, NB, true>), dim3(groups), dim3(kBWaves * 64), lds, st, Gm, L, B, B.part);
  } else {
    if (hipError_t e = lds_opt_in(reinterpret_cast<const void*>(&mvqb8_kernel<MASK, NB, false>), 160 * 1024, attr_set[1]); e != hipSuccess) return e;
    hipLaunchKernelGGL((mvqb8_kernel<MASK, NB, false>), dim3(groups, Gm.T), dim3(kBWaves * 64), lds, st, Gm, L, B, B.part);
  }
  return hipGetLastError();
}

template <uint32_t MASK, int NB>
static hipError_t mvqb4_go(const MvLaunch& L, const MvBatch& B, Mvqb2Geom Gm, bool seq, uint32_t groups, hipStream_t st) {
  static bool attr_set[2][64] = {};
  Gm.ssq_at = 2 * mvqb4_buf_bytes(Gm.cb * B.n_seq);
  const size_t lds = Gm.ssq_at + mvqb_fuse_lds(B.n_seq);
  if (seq) {
    if (hipError_t e = lds_opt_in(reinterpret_cast<const void*>(&mvqb4_kernel<MASK, NB, true>), 160 * 1024, attr_set[0]); e != hipSuccess) return e;
    hipLaunchKernelGGL((mvqb4_kernel<MASK, NB, true>), dim3(groups), dim3(kBWaves * 64), lds, st, Gm, L, B, B.part);
  } else {
    if (hipError_t e = lds_opt_in(reinterpret_cast<const void*>(&mvqb4_kernel<MASK, NB, false>), 160 * 1024, attr_set[1]); e != hipSuccess) return e;
    hipLaunchKernelGGL((mvqb4_kernel<MASK, NB, false>), dim3(groups, Gm.T), dim3(kBWaves * 64), lds, st, Gm, L, B, B.part);
  }
  return hipGetLastError();
}

template <int KIND, bool NORM>
static hipError_t mvqb_rows_go(const MvqbRows& A, uint32_t n_wg, uint32_t nz, hipStream_t st) {
  hipLaunchKernelGGL((mvqb_rows_kernel<KIND, NORM>), dim3(n_wg, 1, nz), dim3(kBWaves * 64), 0, st, A);
  return hipGetLastError();
}

// what mvqb_rows_kernel does with the rows of a launch, or -1
static int mvqb_rows_kind(const MvLaunch& L) {
  const MvSeg& S0 = L.seg[0];
  if (L.nseg == 1 && S0.npass == 1 && (S0.epi == EPI_STORE || S0.epi == EPI_RESID)) return ER_OUT;
  if (L.nseg == 1 && S0.npass == 2 && S0.epi == EPI_SWIGLU) return ER_PAIR;
  for (int i = 0; i < L.nseg; i++) {
    const MvSeg& S = L.seg[i];
    const bool turned = S.epi == EPI_ROPE_Q || S.epi == EPI_ROPE_K;
    if (S.npass != 1 || S.xq_out || !(turned || S.epi == EPI_V_CACHE || S.epi == EPI_STORE) || (S.epi != EPI_STORE && S.head_dim == 0) || (turned && S.head_dim % 2)) return -1;
  }
  return ER_QKV;
}

static hipError_t mvqb_rows_launch(const MvLaunch& L, const MvBatch& B, const Mvqb2Geom& Gm, uint32_t n_wg, uint32_t nz, hipStream_t st) {
  const int kind = mvqb_rows_kind(L);
  if (kind < 0 || (kind == ER_QKV && B.ind_cnt) || Gm.nslots > 8) return hipErrorInvalidValue;
  MvqbRows A{};
  A.part = B.part; A.ssq_part = L.ssq_part; A.rope_cs = L.rope_cs;
  A.pos = B.pos; A.slot = B.slot; A.ind_cnt = B.ind_cnt; A.ind_idx = B.ind_idx;
  A.cache_stride = B.cache_stride; A.part_z_floats = B.part_z_floats;
  A.n_seq = B.n_seq; A.nslots = Gm.nslots; A.rows16 = Gm.n_units * 16;
  A.wb1 = L.nseg > 1 ? L.seg[1].wg_begin : 0xFFFFFFFFu; A.wb2 = L.nseg > 2 ? L.seg[2].wg_begin : 0xFFFFFFFFu;
  A.n_ssq = L.n_ssq_part; A.ssq_stride = B.ssq_stride; A.k = L.k; A.eps = L.eps;
  A.ind_div = B.ind_div; A.ind_stride = B.ind_stride; A.xw_block = B.xw_block;
  for (int i = 0; i < L.nseg; i++) {
    const MvSeg& S = L.seg[i];
    MvqbRowsSeg& D = A.seg[i];
    D.out = S.out; D.resid = S.epi == EPI_RESID ? S.resid : nullptr; D.nw = S.xq_out ? S.xq_nw : nullptr; D.bias = S.bias;
    D.xq = S.xq_out; D.ssq = S.xq_ssq; D.xw = B.xw_out[i];
    D.n_rows = S.n_rows; D.wg_begin = S.wg_begin; D.rows = S.rows_per_wg;
    D.unit_begin = i == 0 ? 0u : i == 1 ? Gm.ub1 : Gm.ub2;
    D.out_stride = B.out_stride[i]; D.resid_stride = B.resid_stride[i]; D.xq_stride = B.xq_out_stride[i]; D.ssq_stride = B.ssq_out_stride[i];
    D.epi = (uint32_t)S.epi; D.head_dim = S.head_dim; D.max_seq = S.max_seq;
  }
  switch (kind) {
    case ER_OUT: return L.do_norm ? mvqb_rows_go<ER_OUT, true>(A, n_wg, nz, st) : mvqb_rows_go<ER_OUT, false>(A, n_wg, nz, st);
    case ER_PAIR: return L.do_norm ? mvqb_rows_go<ER_PAIR, true>(A, n_wg, nz, st) : mvqb_rows_go<ER_PAIR, false>(A, n_wg, nz, st);
    default: return L.do_norm ? mvqb_rows_go<ER_QKV, true>(A, n_wg, nz, st) : mvqb_rows_go<ER_QKV, false>(A, n_wg, nz, st);
  }
}

// enough units to fill the chip with whole rows per workgroup; with fewer the k-slices are a grid dimension
static bool mvqb2_whole_rows(uint32_t n_units, uint32_t T) {
  static const uint32_t min_groups = [] { const char* e = std::getenv("LGH_MVQB2_SEQ_GROUPS"); return e ? (uint32_t)std::atoi(e) : 160u; }();
  return (n_units + kBWaves - 1) / kBWaves >= min_groups || T == 1;
}

// partial sums of one expert in a launch over a layer's experts: matrices of n_units row tiles in T k-slices
uint64_t mvqb_expert_part_floats(uint32_t n_units, uint32_t T, uint32_t n_seq) { return (uint64_t)(mvqb2_whole_rows(n_units, T) ? 1 : T) * n_seq * n_units * 16; }

// gate | up of a layer's experts with few entries each (few_quarters).  mvqb2 where the format is Q4_0.
bool mvqb_few_takes(int dev_type, uint32_t T, uint32_t nbw, uint32_t n_units, uint32_t n_seq, uint32_t top_k, uint32_t n_experts) {
  const int f = fmt_of_dev_type(dev_type);
  if (f < 0 || f == F_Q40 || !mvqb2_whole_rows(n_units, T) || n_experts < 2 || T > kBWaves || kBWaves % T) return false;
  return 4 * n_seq * top_k <= few_quarters(f == F_Q6K, f == F_Q80, few_lds(T, nbw, n_seq)) * n_experts;
}
static bool mvqb_few(const MvLaunch& L, const MvBatch& B, const Mvqb2Geom& Gm) {
  return Gm.fuse == 2 && B.ind_cnt && B.ind_nz >= 2 && L.nseg == 1 && L.seg[0].epi == EPI_SWIGLU && !L.seg[0].bias && mvqb_few_takes(L.seg[0].type, Gm.T, Gm.nbw, Gm.n_units, B.n_seq, B.ind_div, B.ind_nz);
}

template <int F>
static hipError_t mvqb_few_go(const MvLaunch& L, const MvBatch& B, const Mvqb2Geom& Gm, uint32_t groups, hipStream_t st) {
  static_assert(kXqRecord == 1280 && kFuseRed == 128 && mvqb_fuse_lds(1) == 32, "as few_lds counts");
  static bool attr_set[64] = {};
  const MvqbFew few{Gm.T, Gm.nbw, Gm.nblk};
  if (hipError_t e = lds_opt_in(reinterpret_cast<const void*>(&mvqb_few_kernel<F>), 160 * 1024, attr_set); e != hipSuccess) return e;
  hipLaunchKernelGGL(mvqb_few_kernel<F>, dim3(groups, 1, B.ind_nz), dim3(kFewWaves * 64), few_lds(Gm.T, Gm.nbw, B.n_seq), st, few, L, B);
  return hipGetLastError();
}

template <uint32_t MASK, int NB>
static hipError_t mvqb2_go(const MvLaunch& L, const MvBatch& B, const MvGeom& g, Mvqb2Geom Gm, bool seq, uint32_t groups, size_t lds_x, hipStream_t st) {
  static bool attr_set[2][64] = {};
  const uint32_t nz = B.ind_cnt && B.ind_nz > 1 ? B.ind_nz : 1;   // a layer's experts as the grid's third dimension
  Gm.ssq_at = (uint32_t)lds_x;
  lds_x += mvqb_fuse_lds(B.n_seq);
  if constexpr ((MASK & (MASK - 1)) == 0 && MASK != 1u << F_Q40) {
    if (mvqb_few(L, B, Gm)) return mvqb_few_go<__builtin_ctz(MASK)>(L, B, Gm, groups, st);
  }
  if (!B.ind_cnt && B.n_seq >= kMvqb4MinSeq) {
    hipError_t e;
    if constexpr ((MASK & (1u << F_Q80)) != 0) e = mvqb4_go<MASK, NB>(L, B, Gm, seq, groups, st);
    else if (B.n_seq < kMvqb8MinSeq) e = mvqb4_go<MASK, 4>(L, B, Gm, seq, groups, st);
    else if (B.n_seq <= 8) e = mvqb8_go<MASK, 8>(L, B, Gm, seq, groups, st);
    else if (B.n_seq <= 12) e = mvqb8_go<MASK, 12>(L, B, Gm, seq, groups, st);
    else e = mvqb8_go<MASK, 16>(L, B, Gm, seq, groups, st);
    if (e != hipSuccess) return e;
  } else if (seq) {
    if (hipError_t e = lds_opt_in(reinterpret_cast<const void*>(&mvqb2_kernel<MASK, NB, true>), 160 * 1024, attr_set[0]); e != hipSuccess) return e;
    hipLaunchKernelGGL((mvqb2_kernel<MASK, NB, true>), dim3(groups, 1, nz), dim3(kBWaves * 64), lds_x, st, Gm, L, B, B.part);
  } else {
    if (hipError_t e = lds_opt_in(reinterpret_cast<const void*>(&mvqb2_kernel<MASK, NB, false>), 160 * 1024, attr_set[1]); e != hipSuccess) return e;
    hipLaunchKernelGGL((mvqb2_kernel<MASK, NB, false>), dim3(groups, Gm.T, nz), dim3(kBWaves * 64), lds_x, st, Gm, L, B, B.part);
  }
  if (hipError_t e = hipGetLastError(); e != hipSuccess || Gm.fuse) return e;
  return mvqb_rows_launch(L, B, Gm, g.n_wg, nz, st);
}

// from how many sequences on the records go through LDS (mvqb2 and the kernels beside it)
uint32_t mvqb2_min_seq() {
  static const uint32_t v = [] {
    const char* e = std::getenv("LGH_MVQB2_MIN");
    return e ? (uint32_t)std::atoi(e) : 2u;
  }();
  return v;
}

// `L` built like a single-sequence launch (engine.hip: build_mv_group, with the batch cap on tiles per workgroup); sequences'
// vectors at the strides in `B`
hipError_t mvqb_launch(const MvLaunch& L, const MvBatch& Bin, uint32_t n_wg, uint32_t threads, hipStream_t st) {
  MvBatch B = Bin;
  if (B.n_seq == 0 || B.n_seq > (uint32_t)kMaxBatch || threads != kBWaves * 64) return hipErrorInvalidValue;
  MvGeom g;
  size_t lds1 = 0;
  const uint32_t mask = mvq_pack(L, n_wg, threads, &g, &lds1);
  if (!mask) return hipErrorInvalidValue;
  for (int i = 0; i < L.nseg; i++)
    if (L.seg[i].npass > 2 || L.seg[i].pass[0].sel || (L.seg[i].npass == 2 && L.seg[i].pass[1].xq != L.seg[i].pass[0].xq)) return hipErrorInvalidValue;
  if (B.ind_cnt && (B.part == nullptr || B.n_seq < mvqb2_min_seq() || !B.ind_idx || B.ind_div == 0)) return hipErrorInvalidValue;   // indirect entries: mvqb2 only
  bool shared_x = B.part != nullptr;
  for (int i = 0; i < L.nseg; i++) shared_x = shared_x && L.seg[i].pass[0].xq == L.seg[0].pass[0].xq;
  if (shared_x && B.n_seq >= mvqb2_min_seq()) {
    const MvSeg& S0 = L.seg[0];
    Mvqb2Geom Gm{};
    Gm.T = S0.T; Gm.nbw = S0.units; Gm.nblk = S0.nblk;
    uint32_t ub[4] = {0, 0, 0, 0};
    for (int i = 0; i < L.nseg; i++) ub[i + 1] = ub[i] + (uint32_t)L.seg[i].npass * ((L.seg[i].n_rows + 15) / 16);
    Gm.n_units = ub[L.nseg];
    Gm.ub1 = L.nseg > 1 ? ub[1] : Gm.n_units;
    Gm.ub2 = L.nseg > 2 ? ub[2] : Gm.n_units;
    uint32_t groups = (Gm.n_units + kBWaves - 1) / kBWaves;
    const bool seq = mvqb2_whole_rows(Gm.n_units, Gm.T);
    Gm.nslots = seq ? 1 : Gm.T;
    if (seq && L.nseg == 1 && (S0.epi == EPI_STORE || S0.epi == EPI_RESID || S0.epi == EPI_SWIGLU)) {
      Gm.fuse = S0.npass == 2 ? 2 : 1;
      const uint32_t a_wg = kBWaves / (uint32_t)S0.npass;
      groups = ((S0.n_rows + 15) / 16 + a_wg - 1) / a_wg;
    }
    const int nb_inst = B.n_seq <= 4 ? 4 : B.n_seq <= 8 ? 8 : 16;
    Gm.cb = std::max(1u, std::min(Gm.nbw, mvqb2_stage_bytes((mask & (mask - 1)) == 0, nb_inst) / (B.n_seq * (uint32_t)kXqRecord)));
    const size_t lds_x = (size_t)2 * Gm.cb * B.n_seq * kXqRecord + kXZeroBytes + kXSelBytes;
    B.part_z_floats = mvqb_expert_part_floats(Gm.n_units, Gm.T, B.n_seq);
    if (B.part_z_floats * (B.ind_cnt && B.ind_nz > 1 ? B.ind_nz : 1) <= B.part_floats) {
#define LGH_MVQB2_CASE(M)                                                                         \
  case M:                                                                                         \
    if (B.n_seq <= 4) return mvqb2_go<M, 4>(L, B, g, Gm, seq, groups, lds_x, st);  \
    if (B.n_seq <= 8) return mvqb2_go<M, 8>(L, B, g, Gm, seq, groups, lds_x, st);  \
    return mvqb2_go<M, 16>(L, B, g, Gm, seq, groups, lds_x, st)
      switch (mask) {
        LGH_MVQB2_CASE(1u << F_Q4K); LGH_MVQB2_CASE(1u << F_Q6K); LGH_MVQB2_CASE(1u << F_Q5K); LGH_MVQB2_CASE(1u << F_Q80); LGH_MVQB2_CASE(1u << F_Q40);
        LGH_MVQB2_CASE((1u << F_Q4K) | (1u << F_Q6K)); LGH_MVQB2_CASE((1u << F_Q5K) | (1u << F_Q6K));
        default: break;
      }
#undef LGH_MVQB2_CASE
    }
  }
  if (B.ind_cnt) return hipErrorInvalidValue;   // (indirect entries exist in the mvqb2 structure only)
  const size_t lds = mvqb_lds_bytes(B.n_seq, L.red_floats);
  if (lds > 160 * 1024) return hipErrorInvalidValue;
#define LGH_MVQB_NB(M, NBV) return mvqb_go<M, NBV>(L, B, g, threads, lds, st)
#define LGH_MVQB_CASE(M)                                         \
  case M:                                                        \
    if (B.n_seq <= 4) LGH_MVQB_NB(M, 4);                         \
    else if (B.n_seq <= 8) LGH_MVQB_NB(M, 8);                    \
    else LGH_MVQB_NB(M, 16)
  switch (mask) {
    LGH_MVQB_CASE(1u << F_Q4K); LGH_MVQB_CASE(1u << F_Q6K); LGH_MVQB_CASE(1u << F_Q5K); LGH_MVQB_CASE(1u << F_Q80); LGH_MVQB_CASE(1u << F_Q40);
    LGH_MVQB_CASE((1u << F_Q4K) | (1u << F_Q6K)); LGH_MVQB_CASE((1u << F_Q5K) | (1u << F_Q6K));
    default: return hipErrorInvalidValue;
  }
#undef LGH_MVQB_CASE
#undef LGH_MVQB_NB
}

}  // namespace lgh
