// line.hip — fast half-integer line transforms and the spectral updates fused
// with them (the FP64 default wherever both axes have a line form).
//
// A length-N DCT-IV, N = 2m, is an m-point complex DFT between twiddles:
//   v_n = (x_2n + i x_{N-1-2n}) e^{-i pi (4n+1)/4N},  V = DFT_m(v),
//   w_k = 2 V_k e^{-i pi k/N},  y_2k = Re w_k,  y_{N-1-2k} = -Im w_k
// (a DST-IV is the DCT-IV of the reversed line with its odd outputs negated:
// swap the two inputs, flip the sign of Im).  The DFT is a Stockham chain of
// two to four passes of radix R_0, R_1, ... (1 to 13, at most 8 where m allows): pass p
// takes elements b + r m/R_p, multiplies them by a table T_p, transforms R_p
// points in registers and leaves them in the order of the next pass, so there is
// no bit reversal.  The outer twiddles cost nothing of their own: with
// n = b + r m/R the pre-twiddle is a constant turn per register times a factor
// of b, which moves through the DFT into T_1; the post-twiddle splits the same
// way into T_last and a turn after the last DFT.  An axis with no such chain
// (odd, or a prime factor above 13) takes the dense N x N table, sum_n T[n][k] x[n],
// 16 lines of 16 results at a time on the FP64 matrix cores.
//
// Small radices on purpose: two register DFTs of 16 points (one exchange) were
// measured first.  A thread then holds 16 elements and a 512^2 launch is one
// wave per SIMD, which runs every instruction at its latency and fetches twice
// the straight-line code: 6,150 cycles per line transform at 256 points (9,700
// with cold instructions).
//
// Why not the matrix cores: O(N log N) work leaves nothing to multiply.  The
// factored GEMMs do 2 N^3 flops per plane (9.4 GFLOP per 512^2 layer step, half
// of the 78 TF peak at best); this form does 1/25 of them and is bound by the
// planes it moves and by the latency of a launch.
//
// Kernels:
//   k_line_cols   transforms along z: strips of L columns, line index fastest
//                 in lanes and LDS, so global rows are read L doubles at a time
//                 and every LDS access is contiguous; optional epilogue (scale,
//                 accumulate, corrector residual, push field)
//   k_line_rows   transforms along y, 8 lines per work-group
//   k_line_plane  both transforms of a plane of at most 64 x 64
//   k_line_modes  one row kz of every field at once: forward along y, the
//                 per-mode Guess or Iterate map (spectral_mode.h), inverse
//                 along y of the six to eight results.  The spectra between
//                 the transforms never leave the CU, and only what the next
//                 pass reads is written.
// The map's arithmetic is compiled without contraction, as in spectral.hip.

#include "line_dft.h"
#include "qss_internal.h"
#include "spectral_mode.h"

#include <hip/hip_ext.h>

#include <cmath>
#include <type_traits>

namespace {

using namespace qss_line;

constexpr int kXcd = 8;
constexpr int kLines = 8;     // lines per work-group (columns of a strip, rows of a row kernel)
constexpr int kMaxT = kLineT;
constexpr int NTL = kLines * kMaxT;
constexpr int kDenseModesNT = 1024;   // threads of k_line_modes with the dense table
static_assert(kLineDenseY <= kDenseModesNT, "a mode per thread");
constexpr int kPer = 2;       // elements of a line per thread of the work-group at most
constexpr int kPre = 8;       // result pairs whose epilogue operands a thread loads ahead

// consecutive work items on one XCD (they share lines of the planes in its
// L2); work-groups are dealt to the XCDs round robin
__device__ inline int xcd_item(int b, int n) {
  const int x = b % kXcd, i = b / kXcd, q = n / kXcd, r = n % kXcd;
  return x * q + (x < r ? x : r) + i;
}

// ---- shapes ------------------------------------------------------------------
// A kernel's line length is fixed at compile time for N = 32 .. 512 of the form
// 2^a, 3 2^a, 5 2^a (every address of a pass is then one base and immediates, and a
// pass is half the instructions: 11.9 -> 7.2 us for the corrector's row kernel at
// 256^2), or read from the axis.  A loose chain with a radix above 8 runs kernels
// of its own (BIG), whose registers cost the others nothing.
template <int M_, int T_, int R0, int R1, int R2>
struct Fixed {
  static constexpr bool fixed = true, small = M_ <= 32 && R2 == 1;   // small: k_line_plane
  static constexpr int M = M_, T = T_, NP = R2 > 1 ? 3 : 2;
  static constexpr int R[3] = {R0, R1, R2};
  static_assert(R0 * R1 * R2 == M && M * 2 <= T * kLines * kPer, "chain");
  static __device__ constexpr int n(const LineAxis &) { return 2 * M; }
  static __device__ constexpr int m(const LineAxis &) { return M; }
  static __device__ constexpr int np(const LineAxis &) { return NP; }
  static __device__ constexpr int radix(const LineAxis &, int p) { return R[p]; }
  static __device__ constexpr int threads() { return T; }
};
template <bool BIG_>
struct Loose {
  static constexpr bool fixed = false, small = false, BIG = BIG_;
  static __device__ int n(const LineAxis &ax) { return ax.n; }
  static __device__ int m(const LineAxis &ax) { return ax.m; }
  static __device__ int np(const LineAxis &ax) { return ax.np; }
  static __device__ int radix(const LineAxis &ax, int p) { return ax.radix(p); }
  static __device__ int threads() { return blockDim.x / kLines; }
};
#define QSS_RADIX_SMALL(X) X(1) X(2) X(3) X(4) X(5) X(6) X(7) X(8)
#define QSS_RADIX_BIG(X) X(9) X(10) X(11) X(12) X(13)
#define QSS_RADIX_SWITCH(r, X)                                          \
  if (!BIG || r <= 8) {                                                 \
    switch (r) { QSS_RADIX_SMALL(X) }                                   \
  } else if constexpr (BIG) {                                           \
    switch (r) { QSS_RADIX_BIG(X) }                                     \
  }

// pass tables T_1, T_2, ...: fetched early with the other loads, put into LDS
// once the first pass has its inputs.  m is at most the work-group's threads, so a
// thread holds an entry per table.
template <class C>
struct Tables {
  double x0, y0, x1, y1, x2, y2;
  __device__ explicit Tables(const LineAxis &ax) {
    fetch(ax, 0, x0, y0);
    fetch(ax, 1, x1, y1);
    fetch(ax, 2, x2, y2);
  }
  static __device__ void fetch(const LineAxis &ax, int q, double &x, double &y) {
    const int i = threadIdx.x + q * blockDim.x;
    double2 z = make_double2(0.0, 0.0);
    if (i < C::m(ax) * (C::np(ax) - 1)) z = reinterpret_cast<const double2 *>(ax.tw)[i];
    x = z.x;
    y = z.y;
  }
  static __device__ void put(const LineAxis &ax, cplx *tw, int q, double x, double y) {
    const int i = threadIdx.x + q * blockDim.x;
    if (i < C::m(ax) * (C::np(ax) - 1)) tw[i] = {x, y};
  }
  __device__ void put(const LineAxis &ax, cplx *tw) const {
    put(ax, tw, 0, x0, y0);
    put(ax, tw, 1, x1, y1);
    put(ax, tw, 2, x2, y2);
  }
};
static_assert(kLinePasses == 4 && kPer == 2, "Tables holds three entries per thread");

// exchange slot of element i of a line: columns lie side by side; a row has a
// free slot after every eight, which keeps the first pass's writes (R consecutive
// elements per lane) off each other's banks
__host__ __device__ constexpr int padded(int i) { return i + (i >> 3); }
template <bool COLS>
__device__ inline int slot_of(int i) {
  return COLS ? i * kLines : padded(i);
}
// slot of b + step, step a compile-time constant: an immediate where it can be
template <bool COLS>
__device__ inline int slot_at(int b, int step) {
  if (COLS) return b * kLines + step * kLines;
  return step % 8 == 0 ? padded(b) + step / 8 * 9 : padded(b + step);
}

// One pass of every line, butterflies b = t, t + T of the line's m / R, from src
// to dst (the line's exchange sides).
//   first: ld(n, x, y) gives the pair (x_2n, x_{N-1-2n}) in kind order
//   last: st(slot, k, w) takes the result pair of frequency k; slot counts the
//   thread's pairs (a constant after unrolling)
template <int R, bool COLS, class Ld>
__device__ inline void pass_first_r(const LineAxis &ax, cplx *dst, int t, int T, Ld ld) {
  const int mr = ax.m / R;
#pragma unroll 1
  for (int b = t; b < mr; b += T) {
    cplx v[R];
#pragma unroll
    for (int r = 0; r < R; ++r) ld(b + r * mr, v[r].x, v[r].y);
#pragma unroll
    for (int r = 1; r < R; ++r) v[r] = turn<R>(v[r], r);
    dft<R>(v);
#pragma unroll
    for (int k = 0; k < R; ++k) dst[slot_of<COLS>(b * R + k)] = v[k];
  }
}
template <int R, bool COLS>
__device__ inline void pass_mid_r(const LineAxis &ax, int ns, const cplx *src, cplx *dst,
                                  const cplx *tw, int t, int T) {
  const int mr = ax.m / R;
  const int inv = 65536 / ns + 1;   // b / ns for b < 256: exact
#pragma unroll 1
  for (int b = t; b < mr; b += T) {
    cplx v[R];
#pragma unroll
    for (int r = 0; r < R; ++r) v[r] = mul(src[slot_of<COLS>(b + r * mr)], tw[b + r * mr]);
    dft<R>(v);
    const int g = (b * inv) >> 16, o = g * ns * R + (b - g * ns);
#pragma unroll
    for (int k = 0; k < R; ++k) dst[slot_of<COLS>(o + k * ns)] = v[k];
  }
}
template <int R, bool COLS, class St>
__device__ inline void pass_last_r(const LineAxis &ax, const cplx *src, const cplx *tw, int t,
                                   int T, St st) {
  const int mr = ax.m / R;
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int b = t + q * T;
    if (b >= mr) break;
    cplx v[R];
#pragma unroll
    for (int r = 0; r < R; ++r) v[r] = mul(src[slot_of<COLS>(b + r * mr)], tw[b + r * mr]);
    dft<R>(v);
#pragma unroll
    for (int k = 1; k < R; ++k) v[k] = turn<R>(v[k], k);
#pragma unroll
    for (int k = 0; k < R; ++k) st(q * R + k, b + k * mr, v[k]);
  }
}

// the same with the sizes known: butterflies b = t + T q
template <class C, int P, bool COLS, class Ld>
__device__ inline void fixed_first(cplx *dst, int t, Ld ld) {
  constexpr int R = C::R[0], mr = C::M / R;
#pragma unroll
  for (int q = 0; q < (mr + C::T - 1) / C::T; ++q) {
    const int b = t + q * C::T;
    if (mr % C::T && b >= mr) break;
    cplx v[R];
#pragma unroll
    for (int r = 0; r < R; ++r) ld(b + r * mr, v[r].x, v[r].y);
#pragma unroll
    for (int r = 1; r < R; ++r) v[r] = turn<R>(v[r], r);
    dft<R>(v);
    const int o = R % 8 == 0 ? slot_at<COLS>(b * R, 0) : 0;
#pragma unroll
    for (int k = 0; k < R; ++k)
      dst[R % 8 == 0 ? o + (COLS ? k * kLines : k) : slot_of<COLS>(b * R + k)] = v[k];
  }
}
template <class C, int NS, bool COLS>
__device__ inline void fixed_mid(const cplx *src, cplx *dst, const cplx *tw, int t) {
  constexpr int R = C::R[1], mr = C::M / R;
#pragma unroll
  for (int q = 0; q < (mr + C::T - 1) / C::T; ++q) {
    const int b = t + q * C::T;
    if (mr % C::T && b >= mr) break;
    cplx v[R];
#pragma unroll
    for (int r = 0; r < R; ++r) v[r] = mul(src[slot_at<COLS>(b, r * mr)], tw[b + r * mr]);
    dft<R>(v);
    const int o = b / NS * (NS * R) + b % NS;
#pragma unroll
    for (int k = 0; k < R; ++k) dst[slot_at<COLS>(o, k * NS)] = v[k];
  }
}
template <class C, bool COLS, class St>
__device__ inline void fixed_last(const cplx *src, const cplx *tw, int t, St st) {
  constexpr int R = C::R[C::NP - 1], mr = C::M / R;
#pragma unroll
  for (int q = 0; q < (mr + C::T - 1) / C::T; ++q) {
    const int b = t + q * C::T;
    if (mr % C::T && b >= mr) break;
    cplx v[R];
#pragma unroll
    for (int r = 0; r < R; ++r) v[r] = mul(src[slot_at<COLS>(b, r * mr)], tw[b + r * mr]);
    dft<R>(v);
#pragma unroll
    for (int k = 1; k < R; ++k) v[k] = turn<R>(v[k], k);
#pragma unroll
    for (int k = 0; k < R; ++k) st(q * R + k, b + k * mr, v[k]);
  }
}

// All passes of the work-group's lines; on: this thread has a line.  The first
// pass writes side0, then the sides alternate (the first pass's loads may come
// from side1's memory).  put(): what has to be in LDS for the passes after it.
template <class C, bool COLS, class Ld, class St, class Put>
__device__ inline void line_passes(const LineAxis &ax, bool on, int t, int T, const cplx *tw,
                                   cplx *side0, cplx *side1, Ld ld, St st, Put put) {
  if constexpr (C::fixed) {
    if (on) fixed_first<C, 0, COLS>(side0, t, ld);
    put();
    __syncthreads();
    if constexpr (C::NP == 3) {
      if (on) fixed_mid<C, C::R[0], COLS>(side0, side1, tw, t);
      __syncthreads();
      if (on) fixed_last<C, COLS>(side1, tw + C::M, t, st);
    } else {
      if (on) fixed_last<C, COLS>(side0, tw, t, st);
    }
    return;
  } else {
    constexpr bool BIG = C::BIG;
    if (on) {
#define X(R) case R: pass_first_r<R, COLS>(ax, side0, t, T, ld); break;
      QSS_RADIX_SWITCH(ax.radix(0), X)
#undef X
    }
    put();
    __syncthreads();
    int ns = ax.radix(0);
#pragma unroll 1
    for (int p = 1; p < ax.np - 1; ++p) {
      if (on) {
#define X(R) case R: pass_mid_r<R, COLS>(ax, ns, side0, side1, tw, t, T); break;
        QSS_RADIX_SWITCH(ax.radix(p), X)
#undef X
      }
      __syncthreads();
      ns *= ax.radix(p);
      tw += ax.m;
      cplx *const s = side0;
      side0 = side1;
      side1 = s;
    }
    if (on) {
#define X(R) case R: pass_last_r<R, COLS>(ax, side0, tw, t, T, st); break;
      QSS_RADIX_SWITCH(ax.radix(ax.np - 1), X)
#undef X
    }
  }
}

// ---- columns ---------------------------------------------------------------
__device__ inline double wave_max(double v) {
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
  return v;
}

// one column's results: scale, accumulate, residual maxima, push field.  What
// they are combined with (the old C, the P plane) is loaded by the caller
// ahead of the results, all of it at once: a load between two stores waits
// for its full latency.
struct ColEnd {
  const ColArgs &a;
  double *C, *F;
  const double *P;
  bool resid, push, store;
  double dmax = 0.0, vmax = 0.0;
  __device__ ColEnd(const ColArgs &a_, int f, int w) : a(a_) {
    C = a.out[f] + w * a.nc;
    P = a.P[f] ? a.P[f] + w * a.nc : nullptr;
    push = a.push[f] >= 0;
    F = push ? a.F + w * a.w_f + a.push[f] * a.nc : nullptr;
    resid = a.resid[f] >= 0;
    store = a.store[f] != 0;
  }
  // residual maxima: NaN -> +inf so the non-finite guard sees it (fmax drops NaN)
  __device__ void see(double v, double o) {
    const double d = fabs(o - v), m = fabs(v);
    dmax = fmax(dmax, d == d ? d : INFINITY);
    vmax = fmax(vmax, m == m ? m : INFINITY);
  }
  // result y at n; o: the operand that EPI loads ahead
  template <int EPI>
  __device__ void put(long n, double y, double o) {
    if constexpr (EPI == 0) {
      C[n] = y;
    } else if constexpr (EPI == 3) {
      C[n] = y + a.beta * o;
    } else {
      if (EPI != 1) see(y, o);
      if (EPI == 2 || store) C[n] = y;
      if (EPI == 1 && push) F[n] = 0.5 * (o + y);
      if (EPI == 4 && push) F[n] = 0.5 * (P[n] + y);
    }
  }
  // every thread of the work-group
  __device__ void finish(int f, int w) {
    if (!resid) return;
    dmax = wave_max(dmax);
    vmax = wave_max(vmax);
    if ((threadIdx.x & 63) == 0) {
      unsigned long long *r =
          a.rslots + w * (long)kResidPerWake + (blockIdx.x % kResidSlots) * 8;
      atomicMax(&r[a.resid[f]], (unsigned long long)__double_as_longlong(dmax));
      atomicMax(&r[3 + a.resid[f]], (unsigned long long)__double_as_longlong(vmax));
    }
  }
};

// strip of L columns of one field of one wake
struct Strip {
  int f, w, j0;
  __device__ Strip(const ColArgs &a, int L) {
    const int per = (a.ny + L - 1) / L;
    const int id = xcd_item(blockIdx.x, gridDim.x);
    const int fw = id / per;
    j0 = (id - fw * per) * L;
    w = fw / a.nbatch;
    f = fw - w * a.nbatch;
  }
};

// EPI: 0 scaled stores; 1 push field (its P plane loaded ahead); 2 residual of
// the fields that ask for it (the old C loaded ahead); 3 C += (the old C loaded
// ahead); 4 residual and push field (the P plane is read late; made by an Iterate
// called by itself, not in sweeps)
template <int EPI, class C>
__global__ __launch_bounds__(NTL) void k_line_cols(ColArgs a) {
  constexpr int L = kLines;
  extern __shared__ cplx lds[];   // two sides of m * L, then the tables
  const Strip s(a, L);
  const LineAxis &ax = a.ax;
  const int line = threadIdx.x % L, t = threadIdx.x / L, T = C::threads();
  const int j = s.j0 + line, ny = a.ny, N = C::n(ax), m = C::m(ax);
  const bool on = j < ny;
  const double *in = a.in[s.f] + s.w * a.nc + j;
  const bool sine = a.kz[s.f] != QSS_KIND_C;
  cplx *const tw = lds + 2 * m * L;
  const Tables<C> tables(ax);
  ColEnd e(a, s.f, s.w);
  const auto row = [&](int k, int h) { return (long)(h ? N - 1 - 2 * k : 2 * k) * ny + j; };
  // epilogue operands of this thread's results, in the order of the last pass
  double pre[EPI ? 2 * kPre : 1];
  bool late = false;
  const double *from = EPI == 1 ? e.P : e.C;
  const bool want = EPI == 1 ? e.push : EPI == 3 || (EPI && e.resid);
  if constexpr (EPI) {
    const int R = C::radix(ax, C::np(ax) - 1), mr = m / R;
    late = want && (mr + T - 1) / T * R > kPre;   // uniform
    int b = t, k = 0;
#pragma unroll
    for (int i = 0; i < kPre; ++i) {
      pre[2 * i] = pre[2 * i + 1] = 0.0;
      if (want && on && b < mr) {
        pre[2 * i] = from[row(b + k * mr, 0)];
        pre[2 * i + 1] = from[row(b + k * mr, 1)];
      }
      if (++k == R) {
        k = 0;
        b += T;
      }
    }
  }
  const double alpha = a.alpha;
  line_passes<C, true>(
      ax, on, t, T, tw, lds + line, lds + m * L + line,
      [&](int n, double &x, double &y) {
        const double q0 = in[row(n, 0) - j], q1 = in[row(n, 1) - j];
        x = sine ? q1 : q0;
        y = sine ? q0 : q1;
      },
      [&](int slot, int k, cplx v) {
        const double y[2] = {alpha * v.x, alpha * (sine ? v.y : -v.y)};
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const long n = row(k, h);
          double o = 0.0;
          if constexpr (EPI != 0) {
            o = slot < kPre ? pre[2 * slot + h] : 0.0;
            if (late) o = from[n];
          }
          e.template put<EPI>(n, y[h], o);
        }
      },
      [&]() { tables.put(ax, tw); });
  if constexpr (EPI == 2 || EPI == 4) e.finish(s.f, s.w);
}

// ---- the dense table ---------------------------------------------------------
// v_mfma_f64_16x16x4f64: lane l holds A[l % 16][l / 16] and B[l / 16][l % 16];
// register r of lane l holds D[l / 16 + 4 r][l % 16]
typedef double double4v __attribute__((ext_vector_type(4)));
constexpr int kDenseL = 16;     // columns per strip
constexpr int kDenseNT = 512;   // one 16-row tile of results per wave up to N = 128

// D[k][j] = sum_n T[n][k] X[n][j]: the table's rows stream from L2 (every strip
// reads the same), the strip sits in LDS
template <int EPI>
__global__ __launch_bounds__(kDenseNT) void k_line_cols_dense(ColArgs a) {
  extern __shared__ double xs[];   // N * kDenseL
  const Strip s(a, kDenseL);
  const int N = a.ax.n, ny = a.ny;
  const double *in = a.in[s.f] + s.w * a.nc + s.j0;
  const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
  const int j = s.j0 + li;
  ColEnd e(a, s.f, s.w);
  // the whole strip and the first steps of the table are asked for before anything
  // is waited for: one latency, where a loop that stores each value pays one for
  // every 32 rows (97 rows: 8.1 us a launch, 7.3 like this)
  constexpr int PER = kLineDenseZ * kDenseL / kDenseNT;
  static_assert(PER * kDenseNT == kLineDenseZ * kDenseL, "a strip in registers");
  double v[PER];
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    const int i = threadIdx.x + kDenseNT * q, n = i / kDenseL, l = i % kDenseL;
    v[q] = n < N && s.j0 + l < ny ? in[(long)n * ny + l] : 0.0;
  }
  const double *T = a.kz[s.f] == QSS_KIND_C ? a.ax.Tc : a.ax.Ts;
  constexpr int S = 8;   // steps of 4 n fetched ahead
  double t[S], next[S];
  const auto fetch = [&](int n0, int kk, double(&v)[S]) {
#pragma unroll
    for (int q = 0; q < S; ++q) {
      const int n = n0 + 4 * q + lk < N ? n0 + 4 * q + lk : N - 1;
      v[q] = T[n * N + kk];
    }
  };
  // the table is symmetric: T[n][k]
  const auto column = [&](int k0) { return k0 + li < N ? k0 + li : N - 1; };
  const int first = (threadIdx.x >> 6) * 16;
  fetch(0, column(first), t);
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    const int i = threadIdx.x + kDenseNT * q;
    if (i < N * kDenseL) xs[i] = v[q];
  }
  __syncthreads();
  for (int k0 = first; k0 < N; k0 += kDenseNT / 4) {
    double o[4] = {0, 0, 0, 0};
    const bool want = EPI == 1 ? e.push : EPI == 3 || (EPI && e.resid);
    const double *from = EPI == 1 ? e.P : e.C;
    if (EPI && want && j < ny) {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (k0 + lk + 4 * r < N) o[r] = from[(long)(k0 + lk + 4 * r) * ny + j];
    }
    double4v d = {0, 0, 0, 0};
    const int kk = column(k0);
    if (k0 != first) fetch(0, kk, t);
#pragma unroll 1
    for (int n0 = 0; n0 < N; n0 += 4 * S) {
      fetch(n0 + 4 * S, kk, next);   // past the end: the last row again, not used
#pragma unroll
      for (int q = 0; q < S; ++q) {
        // past the strip's end: zero
        const int n = n0 + 4 * q + lk;
        const double v = xs[(n < N ? n : 0) * kDenseL + li];
        d = __builtin_amdgcn_mfma_f64_16x16x4f64(t[q], n < N ? v : 0.0, d, 0, 0, 0);
      }
#pragma unroll
      for (int q = 0; q < S; ++q) t[q] = next[q];
    }
    if (j < ny) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int k = k0 + lk + 4 * r;
        if (k < N) e.template put<EPI>((long)k * ny + j, a.alpha * d[r], o[r]);
      }
    }
  }
  if constexpr (EPI == 2 || EPI == 4) e.finish(s.f, s.w);
}

// ---- rows ------------------------------------------------------------------
// complex slots per line and side in LDS
__host__ __device__ inline int line_pitch(const LineAxis &ax) {
  return ax.np ? padded(ax.m - 1) + 1 : (ax.n + 1) / 2;
}

template <class C>
__device__ inline int pitch_of(const LineAxis &ax) {
  if constexpr (C::fixed) return padded(C::M - 1) + 1;
  else return line_pitch(ax);
}

// transform of the work-group's lines in LDS, lines l < count, from the real
// line l at src + l * pitch (doubles) to dst + l * pitch; sine: bit l set = DST.
// src and dst are the two sides of the exchange and trade contents.
// Returns the side that holds the results.
template <class C>
__device__ inline cplx *lines_fft(const LineAxis &ax, cplx *src, cplx *dst, const cplx *tw,
                                  int count, unsigned sine_mask) {
  const int T = C::threads(), line = threadIdx.x / T, t = threadIdx.x % T;
  const int pitch = pitch_of<C>(ax), N = C::n(ax);
  const double *const x = reinterpret_cast<const double *>(src + line * pitch);
  // the side that the last pass does not read
  cplx *const out = C::np(ax) % 2 ? dst : src;
  double *const y = reinterpret_cast<double *>(out + line * pitch);
  const bool on = line < count, sine = sine_mask >> line & 1u;
  line_passes<C, false>(
      ax, on, t, T, tw, dst + line * pitch, src + line * pitch,
      [&](int n, double &a, double &b) {
        const double p = x[2 * n], q = x[N - 1 - 2 * n];
        a = sine ? q : p;
        b = sine ? p : q;
      },
      [&](int, int k, cplx v) {
        y[2 * k] = v.x;
        y[N - 1 - 2 * k] = sine ? v.y : -v.y;
      },
      []() {});
  __syncthreads();
  return out;
}

// Lines of one kind by fours, for v_mfma_f64_4x4x4_4b: group g's line i in the low 4
// bits of nibble 4 g + i (15: none); the first nc groups are cosine lines.
struct LineGroups {
  unsigned long long lines;
  int n, nc;
};
constexpr LineGroups line_groups(int nl, unsigned sine) {
  LineGroups r{~0ull, 0, 0};
  for (int kind = 0; kind < 2; ++kind) {
    int used = 0;
    for (int l = 0; l < nl; ++l) {
      if ((int)(sine >> l & 1u) != kind) continue;
      const int at = 4 * (4 * (r.n + used / 4) + used % 4);
      r.lines = (r.lines & ~(15ull << at)) | (unsigned long long)l << at;
      ++used;
    }
    r.n += (used + 3) / 4;
    if (kind == 0) r.nc = r.n;
  }
  return r;
}

// the same with the dense table, NL lines (SINE: which take the sine table), from x
// to y (pitch in doubles): D[line][k] = sum_n X[line][n] T[n][k].  A wave makes 16
// columns of up to four lines of one kind at a time with v_mfma_f64_4x4x4_4b (lane
// l: A[l % 4][l / 16] in each block, B[l / 16][l % 16], D[l / 16][l % 16] over the four
// blocks' columns), and asks for 64 rows of its columns of the table before the
// first product: the table comes from beyond L2, and its latency, once per 16 rows
// of it, was most of the time when 16-line tiles were made by four waves (121
// columns: 23.0 us a launch for 3 in and 6 out, 15.1 like this).
template <int NL, unsigned SINE>
__device__ inline void lines_dense(const LineAxis &ax, const double *x, double *y, int pitch) {
  constexpr LineGroups G = line_groups(NL, SINE);
  constexpr int S = 16;   // steps of 4 n whose table entries are asked for at once
  const int N = ax.n, lane = threadIdx.x & 63, lk = lane >> 4;
  const int tiles = (N + 15) / 16;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  for (int task = wave; task < tiles * G.n; task += kDenseModesNT / 64) {
    const int g = task / tiles, col = (task - g * tiles) * 16 + (lane & 15);
    const char *const T = reinterpret_cast<const char *>(g < G.nc ? ax.Tc : ax.Ts);
    const int in = (int)(G.lines >> (16 * g + 4 * (lane & 3))) & 15;
    const double *const xl = x + (in < NL ? in : 0) * pitch;
    double d[2] = {};
#pragma unroll 1
    for (int n0 = 0; n0 < N; n0 += 4 * S) {
      double t[S];
#pragma unroll
      for (int q = 0; q < S; ++q) {
        const int n = n0 + 4 * q + lk;   // 32-bit byte offsets: a table is below 2 MB
        const unsigned at = 8u * ((n < N ? n : N - 1) * N + (col < N ? col : N - 1));
        t[q] = *reinterpret_cast<const double *>(T + at);
      }
#pragma unroll
      for (int q = 0; q < S; ++q) {
        const int n = n0 + 4 * q + lk;
        const double v = xl[n < N ? n : N - 1];
        d[q & 1] = __builtin_amdgcn_mfma_f64_4x4x4f64(in < NL && n < N ? v : 0.0, t[q], d[q & 1],
                                                      0, 0, 0);
      }
    }
    const int to = (int)(G.lines >> (16 * g + 4 * lk)) & 15;
    if (to < NL && col < N) y[to * pitch + col] = d[0] + d[1];
  }
  __syncthreads();
}

template <class C>
__global__ __launch_bounds__(NTL) void k_line_rows(RowArgs a) {
  extern __shared__ cplx lds[];   // two sides of kLines * pitch, then the tables
  const LineAxis &ax = a.ax;
  const int N = C::n(ax), pitch = 2 * pitch_of<C>(ax), NT = kLines * C::threads();
  cplx *const side = lds + kLines * pitch / 2, *const tw = side + kLines * pitch / 2;
  double *x = reinterpret_cast<double *>(lds);
  // rows in the order wake, field, k (fewer than 2^31 in all): the first one's
  // place by division, the next ones' by counting
  const unsigned rows = (unsigned)a.nz * a.nbatch * a.nw;
  const unsigned first = (unsigned)xcd_item(blockIdx.x, gridDim.x) * kLines;
  const int count = rows - first < (unsigned)kLines ? (int)(rows - first) : kLines;
  const unsigned fw0 = first / (unsigned)a.nz, w0 = fw0 / (unsigned)a.nbatch;
  const int k0 = first - fw0 * a.nz, f0 = fw0 - w0 * a.nbatch;
  const auto row = [&](int l, int &f, long &off) {
    int k = k0 + l, w = w0;
    f = f0;
    while (k >= a.nz) {
      k -= a.nz;
      if (++f == a.nbatch) {
        f = 0;
        ++w;
      }
    }
    off = w * a.nc + (long)k * N;
  };
  unsigned sine = 0;
  double v[kLines][kPer];
#pragma unroll
  for (int l = 0; l < kLines; ++l) {
    int f = 0;
    long off = 0;
    if (l < count) row(l, f, off);
    if (a.ky[f] != QSS_KIND_C) sine |= 1u << l;
    const double *in = a.in[f] + off;
#pragma unroll
    for (int q = 0; q < kPer; ++q) {
      const int i = threadIdx.x + NT * q;
      v[l][q] = l < count && i < N ? in[i] : 0.0;
    }
  }
  const Tables<C> tables(ax);
#pragma unroll
  for (int l = 0; l < kLines; ++l)
#pragma unroll
    for (int q = 0; q < kPer; ++q) {
      const int i = threadIdx.x + NT * q;
      if (i < N) x[l * pitch + i] = v[l][q];
    }
  tables.put(ax, tw);
  __syncthreads();
  x = reinterpret_cast<double *>(lines_fft<C>(ax, lds, side, tw, count, sine));
  for (int l = 0; l < count; ++l) {
    int f;
    long off;
    row(l, f, off);
    double *out = a.out[f] + off;
    for (int i = threadIdx.x; i < N; i += NT) out[i] = x[l * pitch + i];
  }
}

// ---- a small plane in one work-group -------------------------------------------
// Both transforms of a plane of at most 64 x 64 without leaving LDS: such a call
// is launches and waits, so one launch instead of two (20.4 -> 17.1 us for a
// 64^2 plane, its wait included).  Every line of the plane at once, 8 threads
// each; rows with their threads side by side, columns with the lines side by
// side, as in the kernels above.
constexpr int kSmallN = 64;
template <class CY, class CZ>
__global__ __launch_bounds__(kSmallN * 8) void k_line_plane(SmallPlaneArgs a) {
  constexpr int NY = 2 * CY::M, NZ = 2 * CZ::M, T = 8, NT = kSmallN * T;
  static_assert(CY::T == T && CZ::T == T && CY::NP == 2 && CZ::NP == 2 && NY <= kSmallN &&
                    NZ <= kSmallN, "small plane");
  constexpr int PY = padded(CY::M - 1) + 1;   // exchange slots of a row
  constexpr int P = NY + 1;                   // doubles from row to row of the real plane
  constexpr int X = NZ * PY > NY * CZ::M ? NZ * PY : NY * CZ::M;
  __shared__ cplx ex[X], tw[CY::M + CZ::M];
  __shared__ double x[NZ * P];
  const int tid = threadIdx.x, b = blockIdx.x % a.nbatch;
  const long off = (long)(blockIdx.x / a.nbatch) * a.nc;
  const double *in = a.in[b] + off;
  double *out = a.out[b] + off;
  constexpr int PER = (NY * NZ + NT - 1) / NT;
  double v[PER];
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    const int i = tid + NT * q;
    v[q] = i < NY * NZ ? in[i] : 0.0;
  }
  if (tid < CY::M) tw[tid] = reinterpret_cast<const cplx *>(a.y.tw)[tid];
  else if (tid < CY::M + CZ::M) tw[tid] = reinterpret_cast<const cplx *>(a.z.tw)[tid - CY::M];
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    const int i = tid + NT * q;
    if (i < NY * NZ) x[i / NY * P + i % NY] = v[q];
  }
  __syncthreads();
  {
    const int line = tid / T, t = tid % T;
    const bool on = line < NZ, sine = a.ky[b] != QSS_KIND_C;
    double *const r = x + line * P;
    line_passes<CY, false>(
        a.y, on, t, T, tw, ex + line * PY, ex + line * PY,
        [&](int n, double &p, double &q) {
          const double u = r[2 * n], w = r[NY - 1 - 2 * n];
          p = sine ? w : u;
          q = sine ? u : w;
        },
        [&](int, int k, cplx z) {
          r[2 * k] = z.x;
          r[NY - 1 - 2 * k] = sine ? z.y : -z.y;
        },
        []() {});
  }
  __syncthreads();
  {
    const int j = tid % NY, t = tid / NY;
    const bool on = t < T, sine = a.kz[b] != QSS_KIND_C;
    const auto at = [&](int i) -> cplx & { return ex[i * NY + j]; };
    if (on) {
      constexpr int R = CZ::R[0], mr = CZ::M / R;
      if (t < mr) {
        cplx v[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const int n = t + r * mr;
          const double u = x[2 * n * P + j], w = x[(NZ - 1 - 2 * n) * P + j];
          v[r] = sine ? cplx{w, u} : cplx{u, w};
        }
#pragma unroll
        for (int r = 1; r < R; ++r) v[r] = turn<R>(v[r], r);
        dft<R>(v);
#pragma unroll
        for (int k = 0; k < R; ++k) at(t * R + k) = v[k];
      }
    }
    __syncthreads();
    if (on) {
      constexpr int R = CZ::R[1], mr = CZ::M / R;
      if (t < mr) {
        cplx v[R];
#pragma unroll
        for (int r = 0; r < R; ++r) v[r] = mul(at(t + r * mr), tw[CY::M + t + r * mr]);
        dft<R>(v);
#pragma unroll
        for (int k = 1; k < R; ++k) v[k] = turn<R>(v[k], k);
#pragma unroll
        for (int k = 0; k < R; ++k) {
          const int f = t + k * mr;
          out[2 * f * NY + j] = a.alpha * v[k].x;
          out[(NZ - 1 - 2 * f) * NY + j] = a.alpha * (sine ? v[k].y : -v[k].y);
        }
      }
    }
  }
}

// ---- rows with the per-mode map between forward and inverse -----------------
// kinds along y (bit set: sine) of the fields in the order the maps use them
constexpr unsigned kSineJ = 0b010;        // Jx Jy Jz
constexpr unsigned kSineEB = 0b00101010;  // Ex Ey Ez Bx By Bz rho psi

// The spectra that a mode's map reads beside the sources.  They are loaded before
// the forward transform, so that their latency hides behind it.
constexpr int kGuessIn[8] = {SP_RHOBP, SP_RHOP, SP_JXP, SP_JYP, SP_JZP, SP_EXP, SP_EYP, SP_EZP};
constexpr int kIterIn[10] = {SP_RHOP, SP_JXP, SP_JYP, SP_JZP, SP_RHOB,
                             SP_RHOBP, SP_EYP, SP_EZP, SP_RHO, SP_JXB};

template <bool GUESS, int NOUT, bool DENSE, class C>
__global__ __launch_bounds__(DENSE ? kDenseModesNT : NTL) void k_line_modes(ModeArgs a) {
  using namespace qss_spec;
  extern __shared__ cplx lds[];   // two sides of NOUT * pitch, then the tables
  constexpr int NIN = GUESS ? 2 : 3, NS = GUESS ? 8 : 10;
  const LineAxis &ax = a.ax;
  const int N = C::n(ax), pitch = 2 * pitch_of<C>(ax);
  const int NT = DENSE ? kDenseModesNT : kLines * C::threads();
  constexpr int PER = DENSE ? 1 : kPer;   // a dense axis has at most kLineDenseY modes
  cplx *const side = lds + NOUT * pitch / 2, *const tw = side + NOUT * pitch / 2;
  double *x = reinterpret_cast<double *>(lds);
  const int item = xcd_item(blockIdx.x, gridDim.x);
  const int w = item / a.nz, kz = item - w * a.nz;
  const long row = (long)w * a.nc + (long)kz * N;
  double *const *S = a.S;
  double v[PER][NIN], sp[PER][NS];
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    const int i = threadIdx.x + NT * q;
    if (i < N) {
#pragma unroll
      for (int l = 0; l < NIN; ++l) v[q][l] = a.in[l][row + i];
    }
  }
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    const int i = threadIdx.x + NT * q;
    if (i < N) {
#pragma unroll
      for (int r = 0; r < NS; ++r) sp[q][r] = S[GUESS ? kGuessIn[r % 8] : kIterIn[r]][row + i];
    }
  }
  const Tables<C> tables(ax);
  // the residual slots of the inverse passes that follow on the stream
  if (!GUESS && a.rslots)
    for (long i = (long)blockIdx.x * NT + threadIdx.x; i < (long)kResidPerWake * a.nw;
         i += (long)gridDim.x * NT)
      a.rslots[i] = 0ull;
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    const int i = threadIdx.x + NT * q;
    if (i < N) {
#pragma unroll
      for (int l = 0; l < NIN; ++l) x[l * pitch + i] = v[q][l];
    }
  }
  if (!DENSE) tables.put(ax, tw);
  __syncthreads();
  if constexpr (DENSE) {
    double *y = reinterpret_cast<double *>(side);
    lines_dense<NIN, GUESS ? 0u : kSineJ>(ax, x, y, pitch);
    x = y;
  } else {
    x = reinterpret_cast<double *>(
        lines_fft<C>(ax, lds, side, tw, NIN, GUESS ? 0u : kSineJ));
  }
  Mode m;
  m.dens = a.dens;
  m.hx = a.hx;
  m.akz = M_PI / a.lz * (kz + 0.5);
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    const int i = threadIdx.x + NT * q;
    if (i >= N) continue;
    const long n1 = row + i;
    m.aky = M_PI / a.ly * (i + 0.5);
    m.ak2 = m.aky * m.aky + m.akz * m.akz;
    double *xi = x + i;   // this mode's slots: only this thread touches them
    if constexpr (GUESS) {
      double in[GI_N], out[GO_N];
      in[GI_RB] = xi[0];
      in[GI_JXB] = xi[pitch];
      in[GI_RBP] = sp[q][0];
      in[GI_RP] = sp[q][1];
      in[GI_JXP] = sp[q][2];
      in[GI_JYP] = sp[q][3];
      in[GI_JZP] = sp[q][4];
      in[GI_EXP] = sp[q][5];
      in[GI_EYP] = sp[q][6];
      in[GI_EZP] = sp[q][7];
      guess(m, in, out);
      S[SP_RHOB][n1] = in[GI_RB];
      S[SP_JXB][n1] = in[GI_JXB];
      S[SP_RHO][n1] = out[GO_RHO];
      if (a.all) {
        S[SP_EX][n1] = out[GO_EX];
        S[SP_EY][n1] = out[GO_EY];
        S[SP_EZ][n1] = out[GO_EZ];
        S[SP_BX][n1] = out[GO_BX];
        S[SP_BY][n1] = out[GO_BY];
        S[SP_BZ][n1] = out[GO_BZ];
        S[SP_JX][n1] = out[GO_JX];
        S[SP_JY][n1] = out[GO_JY];
        S[SP_JZ][n1] = out[GO_JZ];
      }
      xi[0] = out[GO_EX];
      xi[pitch] = out[GO_EY];
      xi[2 * pitch] = out[GO_EZ];
      xi[3 * pitch] = out[GO_BX];
      xi[4 * pitch] = out[GO_BY];
      xi[5 * pitch] = out[GO_BZ];
    } else {
      double in[II_N], out[IO_N];
      in[II_JX] = xi[0];
      in[II_JY] = xi[pitch];
      in[II_JZ] = xi[2 * pitch];
      in[II_RP] = sp[q][0];
      in[II_JXP] = sp[q][1];
      in[II_JYP] = sp[q][2];
      in[II_JZP] = sp[q][3];
      in[II_RB] = sp[q][4];
      in[II_RBP] = sp[q][5];
      in[II_EYP] = sp[q][6];
      in[II_EZP] = sp[q][7];
      in[II_RHO_OLD] = sp[q][8];
      in[II_JXB] = sp[q][9];
      iterate(m, in, out);
      S[SP_RHO][n1] = out[IO_RHO];
      if (a.all) {
        S[SP_JX][n1] = in[II_JX];
        S[SP_JY][n1] = in[II_JY];
        S[SP_JZ][n1] = in[II_JZ];
        S[SP_EX][n1] = out[IO_EX];
        S[SP_EY][n1] = out[IO_EY];
        S[SP_EZ][n1] = out[IO_EZ];
        S[SP_BX][n1] = out[IO_BX];
        S[SP_BY][n1] = out[IO_BY];
        S[SP_BZ][n1] = out[IO_BZ];
        if (a.fin) S[SP_PSI][n1] = out[IO_PSI];
      }
      xi[0] = out[IO_EX];
      xi[pitch] = out[IO_EY];
      xi[2 * pitch] = out[IO_EZ];
      xi[3 * pitch] = out[IO_BX];
      xi[4 * pitch] = out[IO_BY];
      xi[5 * pitch] = out[IO_BZ];
      if constexpr (NOUT == 8) {
        xi[6 * pitch] = out[IO_RHO];
        xi[7 * pitch] = out[IO_PSI];
      }
    }
  }
  __syncthreads();
  {
    cplx *const from = reinterpret_cast<cplx *>(x), *const to = from == lds ? side : lds;
    if constexpr (DENSE) {
      double *y = reinterpret_cast<double *>(to);
      lines_dense<NOUT, kSineEB>(ax, x, y, pitch);
      x = y;
    } else {
      x = reinterpret_cast<double *>(lines_fft<C>(ax, from, to, tw, NOUT, kSineEB));
    }
  }
#pragma unroll
  for (int l = 0; l < NOUT; ++l)
    for (int i = threadIdx.x; i < N; i += NT) a.out[l][row + i] = x[l * pitch + i];
}

// events: the dispatch stamps its own start and end (not under capture)
template <class Fn, class Args>
hipError_t launch(Fn fn, unsigned grid, unsigned threads, size_t lds, hipStream_t s,
                  hipEvent_t ev0, hipEvent_t ev1, const Args &a) {
  if (ev0 || ev1)
    hipExtLaunchKernelGGL(fn, dim3(grid), dim3(threads), lds, s, ev0, ev1, 0, a);
  else
    hipLaunchKernelGGL(fn, dim3(grid), dim3(threads), lds, s, a);
  return hipGetLastError();
}

// threads of a work-group: a fixed chain's own, otherwise a butterfly of the
// longest pass each (two at 32 threads per line), and at most kPer elements of a
// line
inline unsigned line_threads(const LineAxis &ax) {
  if (!ax.np) return NTL;
#define X(m_, t_, a_, b_, c_) if (ax.m == m_) return t_ * kLines;
  QSS_FIXED_CHAINS(X)
#undef X
  int T = 8;
  for (int p = 0; p < ax.np; ++p)
    while (T < kMaxT && T < ax.m / ax.radix(p)) T *= 2;
  while (T * kLines * kPer < ax.n) T *= 2;
  return T * kLines;
}
// f(shape) for the axis's shape
template <class F>
auto with_shape(const LineAxis &ax, F f) {
  switch (ax.np ? ax.m : 0) {
#define X(m_, t_, a_, b_, c_) case m_: return f(Fixed<m_, t_, a_, b_, c_>());
    QSS_FIXED_CHAINS(X)
#undef X
  }
  return line_big(ax) ? f(Loose<true>()) : f(Loose<false>());
}
inline size_t tables_lds(const LineAxis &ax) { return ax.np ? (size_t)ax.m * (ax.np - 1) * 16 : 0; }
inline size_t rows_lds(const LineAxis &ax, int lines) {
  return (size_t)line_pitch(ax) * 16 * 2 * lines + tables_lds(ax);
}

}  // namespace

hipError_t launch_line_cols(const ColArgs &a, hipStream_t s, hipEvent_t ev0, hipEvent_t ev1) {
  bool resid = false, push = false;
  for (int f = 0; f < a.nbatch; ++f) {
    resid = resid || a.resid[f] >= 0;
    push = push || a.push[f] >= 0 || !a.store[f];
  }
  const bool add = a.beta != 0.0;
  if (add && (resid || push)) return hipErrorInvalidValue;   // no caller has both
  const auto grid = [&](int L) { return (unsigned)((a.ny + L - 1) / L) * a.nbatch * a.nw; };
  if (!a.ax.np)
    return launch(add             ? k_line_cols_dense<3>
                  : resid && push ? k_line_cols_dense<4>
                  : resid         ? k_line_cols_dense<2>
                  : push          ? k_line_cols_dense<1>
                                  : k_line_cols_dense<0>,
                  grid(kDenseL), kDenseNT, (size_t)a.ax.n * kDenseL * 8, s, ev0, ev1,
                  a);
  auto fn = with_shape(a.ax, [&](auto shape) {
    using C = decltype(shape);
    return add             ? k_line_cols<3, C>
           : resid && push ? k_line_cols<4, C>
           : resid         ? k_line_cols<2, C>
           : push          ? k_line_cols<1, C>
                           : k_line_cols<0, C>;
  });
  return launch(fn, grid(kLines), line_threads(a.ax), (size_t)a.ax.m * 16 * 2 * kLines + tables_lds(a.ax),
                s, ev0, ev1, a);
}

hipError_t launch_line_rows(const RowArgs &a, hipStream_t s, hipEvent_t ev0, hipEvent_t ev1) {
  const long rows = (long)a.nz * a.nbatch * a.nw;
  if (!a.ax.np) return hipErrorInvalidValue;
  return launch(with_shape(a.ax, [&](auto shape) { return k_line_rows<decltype(shape)>; }),
                (unsigned)((rows + kLines - 1) / kLines), line_threads(a.ax),
                rows_lds(a.ax, kLines), s, ev0, ev1, a);
}

bool line_plane_ok(const LineAxis &y, const LineAxis &z) {
  const auto small = [](const LineAxis &ax) {
    return ax.np && with_shape(ax, [](auto shape) { return decltype(shape)::small; });
  };
  return small(y) && small(z);
}

hipError_t launch_line_plane(const SmallPlaneArgs &a, hipStream_t s, hipEvent_t ev0, hipEvent_t ev1) {
  if (!line_plane_ok(a.y, a.z)) return hipErrorInvalidValue;
  using Fn = void (*)(SmallPlaneArgs);
  const Fn fn = with_shape(a.y, [&](auto sy) -> Fn {
    return with_shape(a.z, [&](auto sz) -> Fn {
      using CY = decltype(sy);
      using CZ = decltype(sz);
      if constexpr (CY::small && CZ::small) return k_line_plane<CY, CZ>;
      else return nullptr;
    });
  });
  return launch(fn, (unsigned)(a.nbatch * a.nw), kSmallN * 8, 0, s, ev0, ev1, a);
}

hipError_t launch_line_modes(const ModeArgs &a, bool guess, hipStream_t s, hipEvent_t ev0,
                             hipEvent_t ev1) {
  const auto pick = [&](auto dense, auto shape) {
    constexpr bool D = decltype(dense)::value;
    using C = decltype(shape);
    return guess   ? k_line_modes<true, 6, D, C>
           : a.psi ? k_line_modes<false, 8, D, C>
                   : k_line_modes<false, 6, D, C>;
  };
  auto fn = with_shape(a.ax, [&](auto shape) { return pick(std::false_type(), shape); });
  return launch(a.ax.np ? fn : pick(std::true_type(), Loose<false>()),
                (unsigned)(a.nz * a.nw), a.ax.np ? line_threads(a.ax) : kDenseModesNT,
                rows_lds(a.ax, a.psi && !guess ? 8 : 6), s, ev0, ev1, a);
}
