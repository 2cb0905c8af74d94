// csrc/batch_rules.h on the host
#include <cstdio>

#include "batch_rules.h"

static int bad = 0;
#define CHECK(c) do { if (!(c)) { std::printf("%s:%d: %s\n", __FILE__, __LINE__, #c); bad++; } } while (0)

int main() {
  using namespace lgh;
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
