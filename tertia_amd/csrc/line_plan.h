// line_plan.h — the plan of a fast half-integer line transform (line.hip): the
// chain of radices for a length and the tables of its passes.  Host code only, so
// that the CPU tests run the same plans.
#pragma once

#include <cmath>
#include <functional>
#include <vector>

#ifdef __HIPCC__
#define QSS_LP __host__ __device__
#else
#define QSS_LP
#endif

constexpr int kLinePasses = 4;   // at most
constexpr int kLineT = 32;       // threads per line at most; a pass has at most two
                                 // butterflies per thread

struct LineAxis {
  int n = 0, m = 0, np = 0;   // length, n / 2, passes (0: no chain, the dense table)
  unsigned R = 0;             // radices, 4 bits each: m is their product
  const double *tw = nullptr;                  // tables of passes 1, 2, ... (pairs re, im)
  const double *Tc = nullptr, *Ts = nullptr;   // dense tables
  QSS_LP int radix(int p) const { return R >> 4 * p & 15; }
};

// Chains compiled for their length, X(m, threads per line, radices): small first
// radices fill the threads, radix 8 keeps the passes at three
#define QSS_FIXED_CHAINS(X)                                                            \
  X(16, 8, 4, 4, 1) X(32, 8, 8, 4, 1) X(64, 8, 8, 8, 1) X(128, 32, 8, 4, 4)            \
  X(256, 32, 8, 8, 4) X(24, 8, 6, 4, 1) X(48, 8, 8, 6, 1) X(96, 32, 8, 4, 3)           \
  X(192, 32, 8, 8, 3) X(20, 8, 5, 4, 1) X(40, 8, 8, 5, 1) X(80, 32, 5, 4, 4)           \
  X(160, 32, 8, 5, 4)

inline bool line_fixed(const LineAxis &ax) {
#define X(m_, t_, a_, b_, c_) if (ax.np && ax.m == m_) return true;
  QSS_FIXED_CHAINS(X)
#undef X
  return false;
}

// a radix above 8
inline bool line_big(const LineAxis &ax) {
  for (int p = 0; p < ax.np; ++p)
    if (ax.radix(p) > 8) return true;
  return false;
}

// Fills n, m, np and R; false (np = 0) where n has no chain: odd, a prime factor of
// n / 2 above 13, or beyond 512.  Other lengths than the fixed ones take the
// cheapest chain (cycles of one wave, fitted by hand): per pass an exchange
// through LDS, per butterfly of a thread its loads, products and DFT; primes from 5
// on cost their square.  Radices above 8 only where m has no chain without: the row
// kernels that hold them spill, which costs more than a pass more does (layers of
// 288 x 288 as 12 12 321 us, as 3 6 8 218; 480 x 480 459, 327; 162 x 162 as 9 9 269, as
// 3 3 3 3 228; planes of 216 x 216 29.3, 24.3).
inline bool line_chain(int n, LineAxis *ax) {
  ax->n = n;
  ax->np = 0;
  if (n < 4 || n % 2 || n > 512) return false;
  const int m = n / 2;
  ax->m = m;
#define X(m_, t_, a_, b_, c_)                        \
  if (m == m_) {                                     \
    ax->np = c_ > 1 ? 3 : 2;                         \
    ax->R = a_ | b_ << 4 | (c_ > 1 ? c_ << 8 : 0);   \
    return true;                                     \
  }
  QSS_FIXED_CHAINS(X)
#undef X
  double best = 1e30;
  unsigned R = 0;
  const auto cost = [&](int r) {
    const bool prime = r == 5 || r == 7 || r == 11 || r == 13;
    return 300.0 +
           ((m / r + kLineT - 1) / kLineT) * (40.0 * r + (prime ? 4.0 * r * r : 0.0));
  };
  int most = 8;   // the largest radix to try
  const std::function<void(int, int, double)> search = [&](int p, int left, double c) {
    if (c >= best) return;
    if (left == 1 && p >= 2) {
      best = c;
      ax->np = p;
      ax->R = R;
      return;
    }
    if (p == kLinePasses) return;
    for (int r = left == 1 ? 1 : 2; r <= (left == 1 ? 1 : most); ++r) {
      // radix 1: the second pass of a prime m
      if (left % r || m / r > 2 * kLineT || (r == 1 && m > 13)) continue;
      R = (R & ~(15u << 4 * p)) | (unsigned)r << 4 * p;
      search(p + 1, left / r, c + cost(r));
      R &= ~(15u << 4 * p);
    }
  };
  search(0, m, 0.0);
  if (!ax->np) {
    most = 13;
    search(0, m, 0.0);
  }
  return ax->np > 0;
}

// T_1, T_2, ... of the passes after the first (see line.hip): entry i of pass p is
// the Stockham twiddle e^{-2 pi i (b % ns) r / (ns R)}, i = b + r m/R; pass 1 also
// carries the pre-twiddle's factor e^{-i pi (4 b0 + 1)/4n} of the first pass's
// butterfly b0 = i / R_0, the last the post-twiddle's 2 e^{-i pi b/n}
inline void line_table(const LineAxis &ax, std::vector<double> &tw) {
  const long n = ax.n, m = ax.m;
  tw.clear();
  long ns = ax.radix(0);
  for (int p = 1; p < ax.np; ++p) {
    const long R = ax.radix(p), mr = m / R;
    for (long i = 0; i < m; ++i) {
      const long b = i % mr, r = i / mr;
      // the phase as an exact multiple of pi / 4n (a turn is 8n)
      long q = (b % ns) * r % (ns * R) * (8 * n / (ns * R));
      double scale = 1.0;
      if (p == 1) q += 4 * (i / ax.radix(0)) + 1;
      if (p == ax.np - 1) {
        q += 4 * b;
        scale = 2.0;
      }
      const long double th = 3.14159265358979323846264338327950288L * (q % (8 * n)) / (4.0L * n);
      tw.push_back((double)(scale * std::cos(th)));
      tw.push_back((double)(-scale * std::sin(th)));
    }
    ns *= R;
  }
}
