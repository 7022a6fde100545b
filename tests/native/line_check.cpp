// Every plan of line_plan.h (n = 2 .. 514) run on the CPU with the register DFTs of
// line_dft.h, against the direct sums in long double; prints the worst error over
// the largest result and the lengths without a chain, exits 1 above the bound.
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <utility>
#include <vector>

#include "../../tertia_amd/csrc/line_dft.h"
#include "../../tertia_amd/csrc/line_plan.h"

using namespace qss_line;

template <int R>
void pass(const LineAxis &ax, int p, long ns, const std::vector<cplx> &src, std::vector<cplx> &dst,
          const double *tw) {
  const int mr = ax.m / R;
  for (int b = 0; b < mr; ++b) {
    cplx v[R];
    for (int r = 0; r < R; ++r) {
      const int i = b + r * mr;
      v[r] = p ? mul(src[i], {tw[2 * i], tw[2 * i + 1]}) : turn<R>(src[i], r);
    }
    dft<R>(v);
    for (int k = 0; k < R; ++k) {
      if (p == ax.np - 1) v[k] = turn<R>(v[k], k);
      dst[b / ns * ns * R + b % ns + k * ns] = v[k];
    }
  }
}

int main() {
  double worst = 0;
  int none = 0;
  for (int n = 2; n <= 514; ++n) {
    LineAxis ax;
    int left = n / 2;
    for (int q : {2, 3, 5, 7, 11, 13})
      while (left > 1 && left % q == 0) left /= q;
    // with factors of at most 5 always; with 7, 11 and 13 where no pass is longer
    // than two butterflies per thread (2 x 7 x 11 and 3^5 have no such chain)
    const bool may = n >= 4 && n % 2 == 0 && n <= 512 && left == 1;
    const bool must = may && (n / 2) % 7 && (n / 2) % 11 && (n / 2) % 13 && n != 486;
    const bool has = line_chain(n, &ax);
    if ((has && !may) || (!has && must)) {
      printf("n = %d: chain %d\n", n, has);
      return 1;
    }
    if (!has) {
      ++none;
      continue;
    }
    int prod = 1;
    for (int p = 0; p < ax.np; ++p) {
      prod *= ax.radix(p);
      if (ax.radix(p) < 1 || ax.radix(p) > 13 || ax.m / ax.radix(p) > 2 * kLineT) return 1;
    }
    if (prod != ax.m || ax.np < 2 || ax.np > kLinePasses) return 1;
    std::vector<double> tw, x(n);
    line_table(ax, tw);
    for (auto &v : x) v = drand48() - 0.5;
    for (int kind = 0; kind < 2; ++kind) {
      std::vector<cplx> a(ax.m), b(ax.m);
      for (int i = 0; i < ax.m; ++i) {
        a[i] = {x[2 * i], x[n - 1 - 2 * i]};
        if (kind) std::swap(a[i].x, a[i].y);
      }
      long ns = 1;
      for (int p = 0; p < ax.np; ++p) {
        const double *t = p ? tw.data() + 2L * ax.m * (p - 1) : nullptr;
        switch (ax.radix(p)) {
#define X(R) case R: pass<R>(ax, p, ns, a, b, t); break;
          X(1) X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(11) X(12) X(13)
#undef X
        }
        ns *= ax.radix(p);
        std::swap(a, b);
      }
      double err = 0, big = 0;
      for (int k = 0; k < n; ++k) {
        const double got = k % 2 == 0 ? a[k / 2].x : (kind ? 1 : -1) * a[(n - 1 - k) / 2].y;
        long double s = 0;
        for (int i = 0; i < n; ++i) {
          const long double th = M_PIl * ((2L * i + 1) * (2 * k + 1) % (8L * n)) / (4.0L * n);
          s += 2 * x[i] * (kind ? sinl(th) : cosl(th));
        }
        err = std::max(err, (double)fabsl(s - got));
        big = std::max(big, (double)fabsl(s));
      }
      worst = std::max(worst, err / big);
    }
  }
  printf("worst %.2e, %d lengths without a chain\n", worst, none);
  return worst <= 5e-15 ? 0 : 1;
}
