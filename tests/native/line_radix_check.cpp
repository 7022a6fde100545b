// The plans of line_plan.h use a radix above 8 only where no chain of smaller ones
// fits a line's threads: such passes run kernels whose registers spill.  Exits 1 and
// names the length otherwise.
#include <cstdio>

#include "../../tertia_amd/csrc/line_plan.h"

// a chain of radices 2 .. 8 for m, at least two and at most kLinePasses
static bool small_chain(int m, int left, int p) {
  if (left == 1 && p >= 2) return true;
  if (p == kLinePasses) return false;
  for (int r = 2; r <= 8; ++r)
    if (left % r == 0 && m / r <= 2 * kLineT && small_chain(m, left / r, p + 1)) return true;
  return false;
}

int main() {
  int with = 0, big = 0;
  for (int n = 4; n <= 512; n += 2) {
    LineAxis ax;
    if (!line_chain(n, &ax)) continue;
    ++with;
    if (!line_big(ax)) continue;
    ++big;
    if (small_chain(n / 2, n / 2, 0)) {
      printf("n = %d has a chain of radices up to 8\n", n);
      return 1;
    }
  }
  printf("%d lengths with a chain, %d with a radix above 8\n", with, big);
  return 0;
}
