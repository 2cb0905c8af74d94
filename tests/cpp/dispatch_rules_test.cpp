// csrc/dispatch_rules.h on the host
#include <cstdio>

#include "dispatch_rules.h"

static int bad = 0;
#define CHECK(c) do { if (!(c)) { std::printf("%s:%d: %s\n", __FILE__, __LINE__, #c); bad++; } } while (0)

int main() {
  using namespace lgh;
  // k-ranges: all blocks in ranges of one size but the last, none empty
  for (uint32_t wgs = 1; wgs <= 600; wgs++)
    for (uint32_t nblk = 1; nblk <= 112; nblk++) {
      const uint32_t S = pf_ranges(wgs, 256, nblk), per = (nblk + S - 1) / S;
      CHECK(S >= 1 && S <= nblk && S * per >= nblk && (S - 1) * per < nblk && (S == 1 || S * wgs <= 256));
    }
  // gate | up as one product: 2048 columns with up to 64 tokens whatever the ranges (eight of one block), with more up to ranges of two; 4096 in ranges of four or eight not, in one always
  CHECK(pf_pair_pays(8, 8, 1) && pf_pair_pays(8, 8, 64) && !pf_pair_pays(8, 8, 65) && pf_pair_pays(8, 4, 128));
  CHECK(!pf_pair_pays(16, 4, 20) && !pf_pair_pays(16, 2, 20) && pf_pair_pays(16, 1, 128) && pf_pair_pays(12, 2, 128) && pf_pair_pays(56, 1, 9));
  // mvqb_few: as many entries as pay by the workgroups that a CU holds, and never more LDS than there is
  const struct { uint32_t T, nbw, k45, k6, k8; } want[] = {{2, 1, 8, 8, 5}, {8, 1, 8, 8, 5}, {8, 2, 8, 8, 5}, {8, 3, 8, 6, 3}, {8, 4, 0, 0, 0}, {8, 5, 0, 0, 0}, {8, 64, 0, 0, 0}};
  for (const auto& w : want)
    for (uint32_t n = 2; n <= 16; n++) {
      const size_t lds = few_lds(w.T, w.nbw, n);
      CHECK(few_quarters(false, false, lds) == w.k45);
      CHECK(few_quarters(true, false, lds) == w.k6);
      CHECK(few_quarters(false, true, lds) == w.k8);
      CHECK(w.k45 == 0 || lds <= 160 * 1024);
    }
  // two sequences: where mvqb_few takes gate | up, in Q4_0, and small experts; the others one after the other
  CHECK(two_by_expert(true, false, 4096, 14336) && two_by_expert(false, true, 8192, 14336));
  CHECK(two_by_expert(false, false, 2048, 1024) && two_by_expert(false, false, 2048, 2048));
  const struct { uint32_t hidden, ff; } others[] = {{2048, 4096}, {2048, 5632}, {4096, 4096}, {8192, 14336}, {6656, 10240}};
  for (const auto& o : others) CHECK(!two_by_expert(false, false, o.hidden, o.ff));
  return bad != 0;
}
