// Prints how the vector form of the gather would cover a part, for extents no test could allocate (plain host arithmetic).
//   usage: gather_plan_check cover D0 D1 D2 D3 D4 dim aligned16      strides of a packed tensor
//          gather_plan_check pack THREADS...                         the parts of a vector, threads of each
// cover: "refused", or "vec threads first-of-last-thread": the elements a thread owns, the number of threads, and where in its
// slice the last thread's elements begin.  pack: "parts:blocks" of every launch.
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "gather_plan.h"

using namespace gelib_hip;

int main(int argc, char **argv) {
  if (argc == 9 && !std::strcmp(argv[1], "cover")) {
    long long D[5], st[5];
    for (int k = 0; k < 5; k++) D[k] = std::atoll(argv[2 + k]);
    st[4] = 1;
    for (int k = 3; k >= 0; k--) st[k] = st[k + 1] * D[k + 1];
    GatherSlices p;
    if (!gather_slices(st, st, D, std::atoi(argv[7]), std::atoi(argv[8]) != 0, &p)) {
      std::puts("refused");
      return 0;
    }
    std::printf("%d %lld %lld\n", p.vec, p.total, gather_element(p.per_target - 1, p.vec));
    return 0;
  }
  if (argc > 2 && !std::strcmp(argv[1], "pack")) {
    int parts = 0;
    long long blocks = 0;
    for (int k = 2; k <= argc; k++) {
      const long long more = k < argc ? gather_blocks(std::atoll(argv[k])) : 0;
      if (k == argc || !gather_shares_launch(parts, blocks, more)) {
        std::printf("%d:%lld ", parts, blocks);
        parts = 0, blocks = 0;
      }
      parts++, blocks += more;
    }
    std::puts("");
    return 0;
  }
  return 2;
}
