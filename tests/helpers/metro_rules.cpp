// Test helper: the sweep's rules (klft_amd/csrc/metro_rules.hpp, the header the
// library compiles) evaluated on the host, one line per set of arguments.
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "metro_rules.hpp"

int main(int argc, char **argv) {
  if (argc < 2) return 1;
  if (!strcmp(argv[1], "row_redrawn")) {  // n2 ...
    for (int i = 2; i < argc; ++i) printf("%d\n", (int)klft_metro::row_redrawn(strtod(argv[i], nullptr)));
    return 0;
  }
  if (!strcmp(argv[1], "rows_drawn")) {  // delta seed cap: draws until a row is kept, at most cap
    const double delta = strtod(argv[2], nullptr);
    klft_rng::Stream s(strtoull(argv[3], nullptr, 10), klft_rng::TAG_METROPOLIS, 0, 0, 0, 0, 0);
    const int cap = atoi(argv[4]);
    int n = 0;
    bool again = true;
    while (again && n < cap) {
      double n2 = 0.0;
      for (int i = 0; i < 6; ++i) {
        const double v = delta * s.u01();
        n2 += v * v;
      }
      ++n;
      again = klft_metro::row_redrawn(n2);
    }
    printf("%d %d\n", n, (int)again);
    return 0;
  }
  if (!strcmp(argv[1], "rows_kept")) {  // fp64 delta ...
    for (int i = 3; i < argc; ++i)
      printf("%d\n", (int)klft_metro::rows_kept(strtod(argv[i], nullptr), atoi(argv[2]) != 0));
    return 0;
  }
  if (!strcmp(argv[1], "hits_in_parallel")) {  // nd nc Vh cus nhits beta symmetric
    printf("%d\n", (int)klft_metro::hits_in_parallel(atoi(argv[2]), atoi(argv[3]), atoll(argv[4]), atoi(argv[5]),
                                                     atoi(argv[6]), strtod(argv[7], nullptr), atoi(argv[8]) != 0));
    return 0;
  }
  return 1;
}
