// prefill.h — batched prompt processing on the f16 matrix cores (prefill.hip; internal).
#pragma once

#include "common.h"

namespace lgh {

constexpr int kPfTokens = 128;                    // tokens per pass = rows of an XH activation matrix
constexpr uint32_t kPfSlabBytes = kPfTokens * 512;   // one 256-element slab of XH: 128 tokens x 256 f16

constexpr int kPfSsqChunks = 8;                   // per-token partial sums of squares (one per 2048 columns): hidden <= 16384

inline size_t xh_bytes(uint32_t k) { return (size_t)(k / 256) * kPfSlabBytes; }

struct PfSeg {
  const uint8_t* w;      // tile16 weights
  uint32_t ntiles;       // 16-row tiles
  uint32_t col0;         // first column in the partial-sum rows
  uint32_t rg_begin;     // first row group (workgroup x index) of this matrix
  int fmt;
  uint64_t w_z = 0;      // bytes between the weights of consecutive experts
};

struct PfGemm {
  PfSeg seg[3];
  int nseg;
  uint32_t nblk;         // 256-element blocks of k
  uint32_t S;            // k-splits (gridDim.y)
  uint32_t ncols;        // floats per partial-sum row
  const uint8_t* xh;     // input activations [128][k] f16, XH layout
  size_t xh_z;           // bytes between the inputs of consecutive experts
  uint32_t n_experts;    // experts of the launch (gridDim.z; MoE), 0: a dense product
  float* part;           // [S][part_rows][ncols]
  uint32_t part_rows;    // rows per split: 128, or kPfMoeRows when the experts of a MoE layer share one buffer
  const int* row_base;   // MoE: device words, the first row of each expert's batch in the buffer
  uint32_t m_tokens;     // (MoE: of the block; an expert's own: m_count)
  const int* m_count;    // MoE: device words, the number of each expert's real rows; 0 rows = nothing to do
  // gate | up with SwiGLU: the activations (XH), the input's sums of squares and the norm they stand for
  uint8_t* act;
  const float* ssq;
  uint32_t n_ssq, norm_cols;
  float eps;
};

bool pf_supported_type(int dev_type);
size_t pf_part_bytes(const uint32_t* n_rows, int nw, uint32_t k, uint32_t n_experts = 0);
hipError_t pf_gemm_launch(const DevWeight* const* W, int nw, const uint8_t* xh, float* part, size_t part_bytes, uint32_t m_tokens,
                          uint32_t* S_out, uint32_t* ncols_out, hipStream_t st, uint32_t n_experts = 0, size_t xh_z = 0, const int* m_count = nullptr,
                          uint32_t part_rows = kPfTokens, const int* row_base = nullptr);
// silu(gate) * up of one launch -> XH
bool pf_pairs(const DevWeight* gate, const DevWeight* up, uint32_t m_tokens);
hipError_t pf_pair_launch(const DevWeight* gate, const DevWeight* up, const uint8_t* xh, uint8_t* act, const float* ssq, uint32_t norm_cols, float eps, uint32_t m_tokens, hipStream_t st);
hipError_t pf_row_epi_launch(const float* part, uint32_t S, uint32_t ncols, uint32_t col0, const float* bias, float* hidden, uint32_t H,
                             const float* nw, uint8_t* xh, float* ssq, uint32_t m_tokens, hipStream_t st, const float* moe_w = nullptr);
hipError_t pf_qkv_epi_launch(const float* part, uint32_t S, uint32_t ncols, uint32_t QD, uint32_t KD, uint32_t head_dim, const float* bq,
                             const float* bk, const float* bv, const float* rope_cs, uint32_t pos0, uint32_t max_seq, float* qbuf,
                             float* kcache, float* vcache, const float* ssq, uint32_t H, float eps, int neox, uint32_t m_tokens, hipStream_t st);
hipError_t pf_swiglu_launch(const float* part, uint32_t S, uint32_t F, uint8_t* xh, const float* ssq, uint32_t H, float eps, uint32_t m_tokens,
                            hipStream_t st, const int* row_tok = nullptr, const int* m_count = nullptr);
// ---- MoE layers (moe.rs:321-413): the block's (token, slot) pairs grouped by expert.  Expert e's rows are
// base[e] .. base[e] + counts[e] - 1 of ONE row space shared by all experts (bases padded to 16: at most kPfMoeRows rows),
// so that the SwiGLU of all experts and the final combine are one launch each.
//   lists[e][i]   token | slot << 8 of the expert's i-th row (token order)
//   rowmap[r]     e | i << 8 of row r, -1 for padding          tokmap[t * top_k + s]   row of (token, slot)
constexpr int kPfMaxExperts = 64;
constexpr int kPfMaxTopK = 8;
constexpr int kPfMoeRows = kPfTokens * 2 + 128;   // 2 experts per token is what the buffers are sized for (checked on the host)
hipError_t pf_moe_group_launch(const int* sel, uint32_t m_tokens, uint32_t top_k, uint32_t n_experts, int* counts, int* bases, int* lists,
                               int* rowmap, int* tokmap, hipStream_t st);
// rows of every expert's batch gathered in one launch: expert e's XH at xh_out + e * xh_bytes(K)
hipError_t pf_moe_gather_launch(const uint8_t* xh, uint32_t K, const int* lists, const int* counts, uint8_t* xh_out, uint32_t n_experts,
                                hipStream_t st);
// silu(gate) * up of every expert's rows in one launch: partial sums [S][kPfMoeRows][2F] -> expert e's XH at xh_out + e * xh_bytes(F)
hipError_t pf_moe_swiglu_launch(const float* part, uint32_t S, uint32_t F, uint8_t* xh_out, const int* rowmap, const int* lists,
                                const float* ssq, uint32_t H, float eps, hipStream_t st);
// h += sum_s w[t][s] * (down-projection row of (t, s)), next XH and sums of squares: pf_row_epi with the rows looked up in tokmap
hipError_t pf_moe_combine_launch(const float* part, uint32_t S, const int* tokmap, const float* moe_w, uint32_t top_k, float* hidden, uint32_t H,
                                 const float* nw, uint8_t* xh, float* ssq, uint32_t m_tokens, hipStream_t st);
hipError_t pf_to_xh_launch(const float* x, uint32_t K, uint8_t* xh, uint32_t m_tokens, hipStream_t st);
// ---- long prompts (prefill_wide.hip): blocks of up to kPfwTokens tokens, row-major f16 activations [token][K] ----
constexpr uint32_t kPfwTile = 256;                // tokens of a workgroup
constexpr uint32_t kPfwTokens = 2048;             // tokens of a block
constexpr uint32_t kPfwMaxRows = kPfwTokens * kPfMaxTopK;   // rows of a product: tokens, or the (token, expert) pairs of a mixture
constexpr uint32_t kPfwPartRows = 4096;           // k-splits x rows whose partial sums the buffer holds beyond one split
constexpr int PW_PART = 0, PW_SWIGLU = 1;         // what becomes of a product: partial sums | silu(gate) * up as f16 rows

struct PfwSeg {
  const uint8_t* w;      // tile16 weights
  uint64_t expert_stride;
  uint32_t ntiles, col0, rg_begin;
  int fmt;
};
struct PfWide {
  PfwSeg seg[3];
  int nseg;
  uint32_t nblk, S, ncols, m;                      // 256-element blocks of k, k-splits, floats per row of partial sums, rows
  const uint8_t* x;      // [row][k] f16
  float* part;           // PW_PART: [S][part_rows][ncols]
  size_t part_bytes;
  uint32_t part_rows;
  uint8_t* act;          // PW_SWIGLU: [row][act_cols] f16
  uint32_t act_cols;
  const float* inv_rms;  // PW_SWIGLU: per token
  const int *src, *tile_e, *tile_row, *row_seg;    // mixtures: token of a row (null: the row itself), expert and first row of a tile, first row of an expert
};
// rows grouped by expert: at most `tiles` tiles of kPfwTile rows, about `likely` of them used
struct PfwGroups { const int *seg, *tile_e, *tile_row, *src; uint32_t experts, tiles, likely; };
struct PfwResid {
  const float* part;     // null: the hidden rows as they are
  uint32_t S, part_rows;
  const int* row_of;     // mixtures: row of (token, slot)
  const float* weight;
  uint32_t top;
  const float* bias;
  float* hidden;
  uint32_t H;
  const float* nw;       // norm weight of the next product's input
  uint8_t* x;            // that input, or null
  float* inv_rms;
  float eps;
};
struct PfwQkv {
  const float* part;
  uint32_t S, part_rows, QD, KD, head_dim;
  const float *bq, *bk, *bv, *rope_cs, *inv_rms;
  uint32_t pos0, max_seq;
  float *q, *kcache, *vcache;
  int neox;
};
bool pfw_pairs(const DevWeight* gate, const DevWeight* up);      // the two can run as one PW_SWIGLU product
size_t pfw_part_bytes(uint32_t max_rows, uint32_t cols);
// up to 3 matrices on the same input; G: x, and part / part_bytes or act / act_cols / inv_rms; S and ncols come back in it
hipError_t pfw_gemm_launch(const DevWeight* const* W, int nw, PfWide& G, int epi, uint32_t rows, const PfwGroups* grp, hipStream_t st);
hipError_t pfw_resid_launch(const PfwResid& a, uint32_t m_tokens, hipStream_t st);
hipError_t pfw_qkv_launch(const PfwQkv& a, uint32_t m_tokens, hipStream_t st);
// dequant.hip: rows tokens[0..m) of the embedding table -> dst[m][hidden]
hipError_t embed_batch_launch(int src_type, const uint8_t* table, const int* tokens, float* dst, uint32_t hidden, uint32_t m_tokens,
                              hipStream_t st);
// the same for a block of up to kPfTokens tokens, ids in host memory that is free again when this returns
hipError_t embed_block_launch(int src_type, const uint8_t* table, const uint32_t* tokens, float* dst, uint32_t hidden, uint32_t m_tokens, hipStream_t st);
// attention.hip: causal attention of a block of m tokens at positions pos0 .. pos0+m-1 (their K/V rows already cached)
hipError_t attn_prefill_launch(const float* q, const float* kcache, const float* vcache, uint32_t n_heads, uint32_t n_kv,
                               uint32_t head_dim, uint32_t max_seq, float scale, uint32_t pos0, uint32_t m_tokens, uint8_t* xh_out,
                               hipStream_t st);
// attention_wide.hip: the same for long blocks; scratch holds the layer's rows as the kernel wants them, out is row-major f16 (or out32, f32)
uint32_t attn_wide_tiles(uint32_t rows);
size_t attn_wide_bytes(uint32_t n_kv, uint32_t head_dim, uint32_t rows);
hipError_t attn_wide_launch(const float* q, const float* kcache, const float* vcache, uint32_t n_heads, uint32_t n_kv, uint32_t head_dim, uint32_t max_seq, float scale,
                            uint32_t pos0, uint32_t m_tokens, uint8_t* scratch, float* part, size_t part_bytes, uint8_t* out, hipStream_t st, float* out32 = nullptr);
// byte offset of element k of token t in an XH matrix
__host__ __device__ inline size_t xh_offset(uint32_t t, uint32_t k) {
  const uint32_t ch = k >> 3;
  return (size_t)(ch >> 5) * kPfSlabBytes + t * 512 + (((ch & 31) ^ (t & 15)) << 4) + (k & 7) * 2;
}

}  // namespace lgh
