// noalloc.hip — qss_transform2d_noalloc: the 2-D half-integer transform of
// qss_transform2d for callers that cannot allocate device memory (code under
// HIP graph capture, tight serving loops, harnesses that forbid hipMalloc).
//
// qss_transform2d runs on a context, whose creation allocates the transform
// tables and the intermediate plane of the two GEMM passes.  This entry point
// needs no context: tables and intermediate live in `scratch`, a fixed device
// array of this file (3 planes of kMaxN^2 doubles, 6 MiB per device, held until
// the process ends).  Each call rebuilds the tables in it (the same exact integer
// argument reduction as the context's host-built tables), runs the y pass into the
// intermediate and the z pass into the caller's output, all enqueued on the
// caller's stream: no allocation, no synchronisation.  Every call on a device
// shares that device's scratch, so calls that overlap on one device race; one
// stream serialises them.
//
// A side that has a chain of radices (even, no prime factor of the half above 13)
// goes through the line transforms (line.hip): a chain's tables are a few
// hundred entries where the dense ones are n^2 cosines, and the passes a fraction of
// the dense products' work; beside a side without one, from kLinePassMin on.  Dense
// against lines, us a call: 512 x 512 54.5 / 16.5, 312 x 200 38.5 / 15.7, 240 x 240 35.9 /
// 15.5, 100 x 100 22.4 / 14.3, 66 x 66 19.0 / 17.0, 12 x 10 14.3 / 12.3 (a context,
// whose tables stand ready, keeps dense products for loose chains
// below 192); what is left is three launches and two passes over the plane.
//
// The array's name is not a device address in host code: its per-device
// address comes from hipGetSymbolAddress, taken once per device with that
// device current, and only that address is handed to kernels.

#include <algorithm>
#include <exception>
#include <mutex>

#include "line_plan.h"
#include "qss_internal.h"

namespace {

constexpr int kMaxN = 512;
constexpr size_t kPlane = (size_t)kMaxN * kMaxN;
constexpr int kMaxDevices = 64;

// T_y (ny x ny), T_z (nz x nz), the y pass's result (nz x ny)
__device__ __align__(256) double scratch[3 * kPlane];

std::mutex g_mu;
double *g_scratch[kMaxDevices] = {};

// 2 cos / 2 sin (pi (2j+1)(2k+1) / (4n)), argument reduced exactly mod 2 pi
// through (2j+1)(2k+1) mod 8n (the host tables of a context, make_tables)
__global__ __launch_bounds__(256) void k_half_integer_table(double *T, int n, int kind) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= (long)n * n) return;
  const int j = (int)(i / n), k = (int)(i - (long)j * n);
  const long m = ((long)(2 * j + 1) * (2 * k + 1)) % (8L * n);
  const double a = M_PI * (double)m / (4.0 * n);
  T[i] = 2.0 * (kind == QSS_KIND_C ? cos(a) : sin(a));
}

// 2 cos, -2 sin and the like of whole multiples q of pi / 4n: the first quadrant's
// value (its half nearer to zero), turned by quadrants
__device__ inline void phase(int q, int n, double &c, double &s) {
  q %= 8 * n;
  const int quad = q / (2 * n), r = q - quad * 2 * n;
  const bool far = r > n;
  const double x = (double)(far ? 2 * n - r : r) / (4.0 * n);   // at most 1/4
  const double cx = cospi(x), sx = sinpi(x), c0 = far ? sx : cx, s0 = far ? cx : sx;
  c = quad == 0 ? c0 : quad == 1 ? -s0 : quad == 2 ? -c0 : s0;
  s = quad == 0 ? s0 : quad == 1 ? c0 : quad == 2 ? -s0 : -c0;
}

// the tables of both axes' chains (line_table in line_plan.h); blockIdx.y: axis
__global__ __launch_bounds__(256) void k_line_tables(LineAxis y, LineAxis z, double *ty,
                                                     double *tz) {
  const LineAxis ax = blockIdx.y ? z : y;
  double *const tw = blockIdx.y ? tz : ty;
  const int e = blockIdx.x * 256 + threadIdx.x, n = ax.n, m = ax.m;
  if (!ax.np || e >= (ax.np - 1) * m) return;
  const int p = 1 + e / m, i = e - (p - 1) * m;
  int ns = ax.radix(0);
  for (int q = 1; q < p; ++q) ns *= ax.radix(q);
  const int R = ax.radix(p), mr = m / R, b = i % mr, r = i / mr;
  int q = (b % ns) * r % (ns * R) * (8 * n / (ns * R));
  double scale = 1.0;
  if (p == 1) q += 4 * (i / ax.radix(0)) + 1;
  if (p == ax.np - 1) {
    q += 4 * b;
    scale = 2.0;
  }
  double c, s;
  phase(q, n, c, s);
  tw[2 * e] = scale * c;
  tw[2 * e + 1] = -scale * s;
}

// The chain of a length, searched for once per process (guarded by g_mu); np = 0
// where it has none.
struct Chain {
  bool known = false;
  LineAxis ax;
};
Chain g_chain[kMaxN + 1];
LineAxis chain_of(int n) {
  Chain &c = g_chain[n];
  if (!c.known) {
    LineAxis ax;
    try {
      if (line_chain(n, &ax)) c.ax = ax;
    } catch (const std::exception &) {   // no memory for the search: dense this time
      return LineAxis{};
    }
    c.known = true;
  }
  return c.ax;
}

int fail(const std::string &m, int code) {
  qss_set_error("qss_transform2d_noalloc: " + m);
  return code;
}

}  // namespace

extern "C" int qss_transform2d_noalloc(int ny, int nz, int kind_z, int kind_y,
                                       const double *in_dev, double *out_dev, double scale,
                                       void *stream) {
  if (ny < 2 || nz < 2 || ny > kMaxN || nz > kMaxN)
    return fail("ny, nz must be in [2, " + std::to_string(kMaxN) + "] (the scratch holds " +
                    std::to_string(kMaxN) + "^2 planes)",
                QSS_E_ARG);
  if ((kind_z != QSS_KIND_C && kind_z != QSS_KIND_S) ||
      (kind_y != QSS_KIND_C && kind_y != QSS_KIND_S))
    return fail("unknown transform kind", QSS_E_ARG);
  if (!in_dev || !out_dev || ((uintptr_t)in_dev & 15) || ((uintptr_t)out_dev & 15))
    return fail("planes must be non-null and 16-byte aligned", QSS_E_ARG);
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return fail(hipGetErrorString(e), QSS_E_HIP);
  if (dev < 0 || dev >= kMaxDevices) return fail("device index out of range", QSS_E_ARG);
  double *base = nullptr;
  LineAxis y, z;
  {
    std::lock_guard<std::mutex> lk(g_mu);
    y = chain_of(ny);
    z = chain_of(nz);
    if (!g_scratch[dev]) {   // first call on this device, the device current
      void *p = nullptr;
      e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
      if (e != hipSuccess) return fail(hipGetErrorString(e), QSS_E_HIP);
      g_scratch[dev] = static_cast<double *>(p);
    }
    base = g_scratch[dev];
  }
  double *Ty = base, *Tz = base + kPlane, *mid = base + 2 * kPlane;
  hipStream_t s = static_cast<hipStream_t>(stream);
  // a short y side with a factor of 11 or 13: its rows spill registers and take longer
  // than the dense pass (22 x 22 13.1 / 16.6 us, 52 x 52 17.2 / 17.9, 26 x 64 15.6 / 17.0;
  // 66 x 66 19.3 / 17.4)
  if (y.np && line_big(y) && ny < 56) y.np = 0;
  // one side without a chain: the other one's is worth it from kLinePassMin on
  // (121 x 256 30.3 / 18.9 us, 300 x 97 32.2 / 21.9, 200 x 35 23.3 / 20.4; 64 x 35 16.7
  // / 16.8, 26 x 35 16.5 / 19.8)
  if (!(y.np && z.np)) {
    if (ny < kLinePassMin) y.np = 0;
    if (nz < kLinePassMin) z.np = 0;
  }
  y.tw = Ty;
  z.tw = Tz;
  if (y.np || z.np) {
    const int most = std::max(y.np ? (y.np - 1) * y.m : 0, z.np ? (z.np - 1) * z.m : 0);
    hipLaunchKernelGGL(k_line_tables, dim3((unsigned)(most + 255) / 256, 2), dim3(256), 0, s, y, z,
                       Ty, Tz);
  }
  if (!y.np)
    hipLaunchKernelGGL(k_half_integer_table, dim3((unsigned)(((long)ny * ny + 255) / 256)),
                       dim3(256), 0, s, Ty, ny, kind_y);
  if (!z.np)
    hipLaunchKernelGGL(k_half_integer_table, dim3((unsigned)(((long)nz * nz + 255) / 256)),
                       dim3(256), 0, s, Tz, nz, kind_z);
  if ((e = hipGetLastError()) != hipSuccess) return fail(hipGetErrorString(e), QSS_E_HIP);
  if (y.np && z.np && line_plane_ok(y, z)) {
    SmallPlaneArgs a{};
    a.y = y; a.z = z;
    a.nbatch = a.nw = 1; a.alpha = scale;
    a.in[0] = in_dev; a.out[0] = out_dev;
    a.ky[0] = kind_y; a.kz[0] = kind_z;
    e = launch_line_plane(a, s);
    return e == hipSuccess ? QSS_OK : fail(hipGetErrorString(e), QSS_E_HIP);
  }
  // a dense pass: transform_batch's for one FP64 plane, default tile shape
  GemmArgs g{};
  g.nbatch = 1;
  g.nw = 1;
  g.b[0].resid = -1;
  g.b[0].push = -1;
  if (y.np) {
    RowArgs r{};
    r.ax = y;
    r.nz = nz; r.nbatch = r.nw = 1;
    r.in[0] = in_dev; r.out[0] = mid; r.ky[0] = kind_y;
    e = launch_line_rows(r, s);
  } else {
    g.M = nz; g.N = ny; g.K = ny;
    g.alpha = 1.0;
    g.b[0].A = in_dev;
    g.b[0].B = Ty;
    g.b[0].C = mid;
    e = launch_gemm(g, s, QSS_PREC_FP64, 0);
  }
  if (e != hipSuccess) return fail(hipGetErrorString(e), QSS_E_HIP);
  if (z.np) {
    ColArgs c{};
    c.ax = z;
    c.ny = ny; c.nbatch = c.nw = 1;
    c.in[0] = mid; c.out[0] = out_dev; c.kz[0] = kind_z;
    c.resid[0] = c.push[0] = -1;
    c.store[0] = 1;
    c.alpha = scale;
    e = launch_line_cols(c, s);
  } else {
    g.M = nz; g.N = ny; g.K = nz;
    g.alpha = scale;
    g.b[0].A = Tz;
    g.b[0].B = mid;
    g.b[0].C = out_dev;
    e = launch_gemm(g, s, QSS_PREC_FP64, 0);
  }
  return e == hipSuccess ? QSS_OK : fail(hipGetErrorString(e), QSS_E_HIP);
}
