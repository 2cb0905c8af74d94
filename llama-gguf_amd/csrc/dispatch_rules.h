// Which kernels take a call: rules on sizes and formats alone, on the host.
#pragma once

#include <cstddef>
#include <cstdint>

namespace lgh {

// ---- prompt blocks of up to 128 tokens (prefill.hip)
// k-ranges of a product of `wgs` workgroups over nblk blocks of 256 columns: as many as keep the launch within `fill` workgroups, none of them empty
constexpr uint32_t pf_ranges(uint32_t wgs, uint32_t fill, uint32_t nblk) {
  uint32_t S = wgs >= fill ? 1 : fill / wgs;
  if (S > nblk) S = nblk;
  const uint32_t per = (nblk + S - 1) / S;
  return (nblk + per - 1) / per;
}
// gate | up of S k-ranges as one product without partial sums: while walking all of k costs its workgroups no more than the fold and its launch.  A block is 0.8 us, the fold about 5.  In ranges and in one, six layers, us:
// 4096 x 4096 (ranges of 4 of 16 blocks), 50 / 90 / 128 tokens 372 / 446 / 539 and 403 / 479 / 548; 2048 x 5632 (4 of 8) 335 / 390 / 445 and 329 / 378 / 431; 1024 x 2816 (1 of 4) 268 / 308 / 344 and 257 / 294 / 328.
// Seven blocks more (2048 columns, up to 2048 x 2048) are even on the device with up to 64 tokens and lose with more (2048 x 768, 20 / 64 / 96 / 128 tokens 253 / 292 / 329 / 364 and 240 / 300 / 342 / 384).  But there
// the host's launches are what a prompt with its last token's step beside it waits for, so one launch a layer less is the faster way up to 64.
constexpr bool pf_pair_pays(uint32_t nblk, uint32_t S, uint32_t m_tokens) { return nblk - (nblk + S - 1) / S <= (m_tokens <= 64 ? 7u : 6u); }

// ---- a mixture's experts in a batched step (matvec_batch.hip, engine_batch.hip)
constexpr uint32_t kFewWaves = 4, kFewEntries = 2;   // mvqb_few's waves, and the entries of a turn over the weights
// its LDS: the records of a turn's entries for T k-slices of nbw blocks (an own copy for each wave that shares a slice), their sums, the norms of n_seq sequences
constexpr uint32_t few_red_at(uint32_t T, uint32_t nbw) { return (T > kFewWaves ? T : kFewWaves) * nbw * kFewEntries * 1280; }
constexpr uint32_t few_ssq_at(uint32_t T, uint32_t nbw) { return few_red_at(T, nbw) + kFewEntries * 128 * T * 4; }
constexpr size_t few_lds(uint32_t T, uint32_t nbw, uint32_t n_seq) { return few_ssq_at(T, nbw) + n_seq * 8 * 4; }

// Quarters of an entry that an expert may have on average for gate | up to go to mvqb_few, by how many of its workgroups a CU holds.  Steps of two layers of 8 experts, two a sequence (so n sequences are n quarters), what mvqb2
// takes over what mvqb_few takes, 4 / 6 / 8 sequences:
//   three (hidden up to 4096; 4096 x 14336)  Q4_K 1.16 1.15 1.08, Q5_K 1.12 1.13 1.06, Q6_K 1.10 1.08 1.02, Q8_0 1.04 1.01 0.94 (2048 x 10240: 1.14 1.09 1.02)
//   two (6144 x 16384)                       Q4_K 1.10 1.08 1.04, Q5_K 1.08 1.05 1.03, Q6_K 1.05 1.03 0.98, Q8_0 0.98 0.95 0.91 (3: 1.04)
//   one (8192 x 14336)                       Q4_K 0.98 0.97 0.91, Q6_K 0.98 0.96 0.90; 6656 x 10240 (26 blocks in slices of four: the last has none): Q4_K 0.94 0.91 0.85, Q6_K 0.93 0.90 0.83, 2 sequences 0.98 0.97
constexpr uint32_t few_quarters(bool q6k, bool q80, size_t lds) {
  const size_t wgs = 160 * 1024 / lds;
  return wgs >= 3 ? (q80 ? 5 : 8) : wgs == 2 ? (q80 ? 3 : q6k ? 6 : 8) : 0;
}

// Two sequences by expert (seven launches a layer, every selected expert read once) or one after the other (three launches each).  A step of two layers, us, one after the other / by expert, Q4_K_M (Q8_0):
//   where mvqb_few takes gate | up  4096 x 14336 324 / 298 (408 / 370), 4096 x 10240 281 / 269, 2048 x 10240 222 / 199, 6144 x 16384 459 / 431
//   in Q4_0                         4096 x 14336 306 / 258, 8192 x 14336 477 / 409, 6656 x 10240 368 / 342, 4096 x 8192 246 / 249
//   small experts                   2048 x 1024 179 / 160 (183 / 163), 1024 x 2048 171 / 152, 512 x 1024 162 / 138, 2048 x 2048 180 / 176 (185 / 184)
//   the others                      2048 x 4096 189 / 204 (199 / 215), 2048 x 5632 200 / 221, 4096 x 4096 222 / 250, 4096 x 8192 262 / 304, 6656 x 10240 395 / 408, 8192 x 14336 509 / 545
constexpr bool two_by_expert(bool few, bool q40, uint32_t hidden, uint32_t ff) { return few || q40 || (uint64_t)hidden * ff <= 2048u * 2048u; }

}  // namespace lgh
