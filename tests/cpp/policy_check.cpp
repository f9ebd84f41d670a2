// policy_check.cpp -- asks the launch policy about a batch (test infrastructure): compute
// units and then every m+n on stdin; prints whether Dantzig pricing takes 512 threads.
#include <cstdio>

#include "../../flock_amd/csrc/policy.h"

int main() {
  int units = 0, v = 0;
  if (std::scanf("%d", &units) != 1) return 1;
  flock::BatchShape s;
  while (std::scanf("%d", &v) == 1) s.add(v);
  std::printf("%d\n", s.dantzig_wide(units) ? 1 : 0);
}
