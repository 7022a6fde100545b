// push_tile.hip — tiled predictor-corrector push with a deterministic
// LDS deposit (the default particle path).
//
// Particles are stored sorted by 16x16-cell tile (tile_start[] gives each
// tile's slot range).  One work-group owns one tile for a whole pass:
//   1. it stages the tile's (P+C)/2 field window (17x17 nodes) in LDS, so
//      the CIC/NGP gathers of MoveParticlesLayerSplit
//      (movepart_splitlayer.cpp:1101-1217, movepart_layer_CIC.cpp:166-203)
//      never leave the CU;
//   2. each thread pushes one particle per chunk of 256 (same arithmetic as
//      the reference, -ffp-contract=off);
//   3. every deposit event (one per sub-step, :1391-1466) enters the list of its
//      window cell; the lane that owns the cell orders the list by event index and
//      sums the events over the cell's four nodes in registers, and the four
//      corners go to the window's node sums in LDS in four turns
//      (DepositCurrentsInCellSplit :1547-1655 / MoveInCell
//      movepart_layer_CIC.cpp:449-496).  The float form has every node add the
//      events of its four cells' lists instead, and a round with a crowded cell
//      sorts the chunk's events by cell and index;
//   4. the 21x21 node window (tile + 2-cell halo + 1) goes to HBM and
//      k_combine adds the windows overlapping each node in a fixed order,
//      which is the periodic ghost fold of ExchangeCurrentsSplit (:1685-1711).
// With the reference's sub-cycle restart every sub-step lands within one
// cell of the start cell, so every event falls inside the window.
//
// Full step: the pushed particle is staged with its destination tile
// direction and its rank among the tile's particles going that way (slot
// order); tile_scan / k_permute rebuild the tile-sorted storage: each
// destination tile holds the groups from its 9 source directions in a fixed
// order, each group in source slot order.  The storage order, and so every
// summation order, is a pure function of the input.

#include <hip/hip_ext.h>

#include <type_traits>

#include "qss_internal.h"
#include "split_bf16.h"
#include "inv_gamma.h"
#include "tile_sort.h"

namespace {

constexpr int NT = 256;
constexpr int T = kTile;          // cells per tile edge
constexpr int H = 2;              // halo cells
constexpr int W = T + 2 * H + 1;  // window nodes per edge (21)
constexpr int NWIN = W * W;       // 441
constexpr int FW = T + 1;         // gathered field nodes per edge (17)
constexpr int NF = FW * FW;       // 289
constexpr int kMaxSub = 64;
constexpr int kInvalid = 0x7fffffff;

enum { ST_PARTICLE = 1, ST_OVERFLOW = 2, ST_SUBSTEPS = 4, ST_FAR = 8 };

struct TileArgs {
  const double *y, *z, *px, *py, *pz;
  const int32_t *cell;
  const int64_t *pid;
  const int32_t *tile_start;
  int ntj, ntk, ny, nz;
  const double *F;
  const float *Ff;        // fp32 push field (mixed modes)
  // products of uniform values, made on the host: there is no scalar FP64 unit, so
  // in the kernel each would sit in a vector register pair for its whole run
  double kick;            // charge over mass (-1) times half the slice step
  double mweight;         // -weight: the deposit factor of an electron
  double hxy, hxz;        // hx / hy, hx / hz
  double nyd, nzd;        // ny, nz
  double lo[2], hi[2];    // -2 ny, -2 nz; 3 ny, 3 nz: positions past these are errors
  double bext[3];         // uniform external B (movepart_splitlayer.cpp:1271-1273)
  int shape;
  double *win;            // per tile and part 4 components (rho last) of NWIN nodes
  // full step staging (indexed by the old slot)
  double *sy, *sz, *spx, *spy, *spz;
  int32_t *scell, *sdest;  // sdest = direction | rank << 4
  int32_t *tcount;         // 9 directions x nsplit x ntiles
  int32_t *counters;
  long npw;                // particle slots per wake (batched contexts)
  int nsplit;              // work-groups per tile (each takes every nsplit-th chunk)
  uint64_t ny_magic;       // ceil(2^44 / ny): cell / ny = (cell * ny_magic) >> 44
};

// cell -> (j, k) without a division: for 0 <= c < 2^28 and ny <= 2^14,
// c * ceil(2^44/ny) / 2^44 exceeds c/ny by less than 2^-16 < 1/ny, so the
// floor is exact
__device__ inline void cell_jk(int32_t c, int ny, uint64_t magic, int &j, int &k) {
  k = (int)(((uint64_t)(uint32_t)c * magic) >> 44);
  j = c - k * ny;
}

// the arguments of wake w of a batch: every per-wake array is stored
// wake-major with a fixed stride
__host__ __device__ inline TileArgs wake_view(const TileArgs &a0, int w) {
  TileArgs a = a0;
  const long pw = (long)w * a0.npw, nt = (long)a0.ntj * a0.ntk;
  const long plane = (long)a0.ny * a0.nz;
  a.y += pw; a.z += pw; a.px += pw; a.py += pw; a.pz += pw;
  a.cell += pw; a.pid += pw;
  a.tile_start += w * (nt + 1);
  if (a.F) a.F += w * kPushComp * plane;
  if (a.Ff) a.Ff += w * kPushComp * plane;
  a.win += w * nt * a0.nsplit * NWIN * 4;
  a.sy += pw; a.sz += pw; a.spx += pw; a.spy += pw; a.spz += pw;
  a.scell += pw; a.sdest += pw;
  a.tcount += w * nt * a0.nsplit * 9;
  return a;
}

using qss_tile::cell_order;
using qss_tile::kCell;
using qss_tile::sort256;
using qss_tile::thread_index;

template <typename T>
struct alignas(2 * sizeof(T)) pair_t {
  T x, y;
};
template <typename FT>
__device__ inline const FT *field_of(const TileArgs &a) {
  if constexpr (sizeof(FT) == 8) return a.F;
  else return a.Ff;
}

// ---- deposit of one round (at most one event per thread) ----------------------
// By cells: 256 particles of 4 per cell make lists of about 4, and each event is
// read once, where the sort of 256 keys (36 exchange stages, six of them through LDS
// with two barriers each) and the four reads of each event by its nodes took a third
// of a chunk's time.  Pushes of a 512^2 plane, 4 per cell: 44.5 us (full: 54.7) with
// the sort, 34.4 (42.7) by cells, all else as it is here.
// kCell: events of a cell that its owner lane sums directly: the bytes of one 8-byte
// list, and past 8 the longest list sets the pace of its wave.

template <int NQ>
__device__ inline void add_corners(double yp, double zp, const double *w, double (*s)[NQ]) {
  const double yc = 1. - yp, zc = 1. - zp;
  const double c[4] = {yc * zc, yp * zc, yc * zp, yp * zp};
#pragma unroll
  for (int k = 0; k < 4; ++k)
#pragma unroll
    for (int q = 0; q < NQ; ++q) s[k][q] = __builtin_fma(c[k], w[q], s[k][q]);
}

// A cell's corner sums onto the window's nodes, one corner after the other with a barrier
// between: in one corner's turn no two cells share a node.
template <int NQ>
__device__ inline void corner_turns(bool on, int cell, const double (*s)[NQ],
                                    double (*wacc)[NWIN], bool cic) {
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    if (k > 0 && !cic) break;
    if (on) {
      const int node = cell + (k & 1) + (k >> 1) * W;
#pragma unroll
      for (int q = 0; q < NQ; ++q) wacc[q][node] += s[k][q];
    }
    __syncthreads();
  }
}

// Sums of one cell's events over its four nodes, in the order of the events'
// indices: the order in which they reached the list does not matter.
template <int N, int NQ>
__device__ inline void cell_sums(uint2 bytes, int n, const double *ev_y, const double *ev_z,
                                 const double (*ev_w)[NT], bool cic, double (*s)[NQ]) {
  int e[N];
  cell_order<N>(bytes, n, e);
#pragma unroll
  for (int i = 0; i < N; ++i) {
    if (i >= n) break;
    const int ei = e[i];
    double w[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) w[q] = ev_w[q][ei];
    // NGP: all of it in corner 0
    const double yp = cic ? ev_y[ei] : 0., zp = cic ? ev_z[ei] : 0.;
    add_corners<NQ>(yp, zp, w, s);
  }
}

// A lane sums the events of the window cell it owns in this half (cells 0 .. NT - 1
// or the rest) over the four corners in registers, each event read once.  A chunk's
// events lie in few neighbouring rows, so with the cells in order some waves have all
// the work and the others none to issue (dealt to the waves in turn: 34.4 us a push at
// 512^2 against 32.0).
// Leaves the counts at zero.
template <int NQ>
__device__ inline void deposit_cells(int half, int *cnt, const uint2 *list, const double *ev_y,
                                     const double *ev_z, const double (*ev_w)[NT],
                                     double (*wacc)[NWIN], bool cic) {
  const int t = thread_index();
  const int cell = t + NT * half;
  double s[4][NQ];
  const int n = cell < NWIN ? cnt[cell] : 0;
#pragma unroll
  for (int k = 0; k < 4; ++k)
#pragma unroll
    for (int q = 0; q < NQ; ++q) s[k][q] = 0.0;
  if (n) {
    cnt[cell] = 0;
    const uint2 bytes = list[cell];
    if (n <= 4) cell_sums<4, NQ>(bytes, n, ev_y, ev_z, ev_w, cic, s);
    else cell_sums<8, NQ>(bytes, n, ev_y, ev_z, ev_w, cic, s);
  }
  corner_turns<NQ>(n > 0, cell, s, wacc, cic);
}

// The float form's round: the owner lanes put the lists in order, then every node
// adds the events of its four corner cells one after the other.  The sums are the
// sort's below, bit by bit (the same events in the same order): the fields of the
// split modes are rounded to float between the steps, and another order of these
// FP64 sums would flip some of those roundings.  512^2, 4 per cell: 39.9 us a push
// (full: 43.8), by the sort 41.1 (50.4).  Leaves the counts at zero.
template <int NQ>
__device__ inline void deposit_lists(int *cnt, uint2 *list, const double *ev_y, const double *ev_z,
                                     const double (*ev_w)[NT], double (*wacc)[NWIN], bool cic) {
  const int t = thread_index();
#pragma unroll 1
  for (int cell = t; cell < NWIN; cell += NT) {
    const int n = cnt[cell];
    if (n < 2) continue;
    int e[kCell];
    cell_order<kCell>(list[cell], n, e);
    uint2 b = {0, 0};
#pragma unroll
    for (int i = 0; i < kCell; ++i) (i < 4 ? b.x : b.y) |= (unsigned)(e[i] & 255) << 8 * (i % 4);
    list[cell] = b;
  }
  __syncthreads();
#pragma unroll 1
  for (int n = t; n < NWIN; n += NT) {
    double acc[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) acc[q] = wacc[q][n];
    const int nl_j = n % W, nl_k = n / W;
    int c[4];
    uint2 b[4];
#pragma unroll
    for (int cn = 0; cn < 4; ++cn) {
      const int cj = nl_j - (cn & 1), ck = nl_k - (cn >> 1);
      const bool in = cj >= 0 && ck >= 0 && (cic || cn == 0);
      c[cn] = in ? cnt[ck * W + cj] : 0;
      b[cn] = list[in ? ck * W + cj : 0];
    }
#pragma unroll
    for (int cn = 0; cn < 4; ++cn) {
      // four events at a time, their loads together
#pragma unroll 1
      for (int i = 0; i < c[cn]; i += 4) {
        const unsigned four = i ? b[cn].y : b[cn].x;
        double w[4][NQ], y[4], z[4];
#pragma unroll
        for (int h = 0; h < 4; ++h) {
          const int e = i + h < c[cn] ? four >> 8 * h & 255 : four & 255;
#pragma unroll
          for (int q = 0; q < NQ; ++q) w[h][q] = ev_w[q][e];
          y[h] = ev_y[e];
          z[h] = ev_z[e];
        }
#pragma unroll
        for (int h = 0; h < 4; ++h) {
          const double wy = (cn & 1) ? y[h] : 1. - y[h];
          const double wz = (cn >> 1) ? z[h] : 1. - z[h];
#pragma unroll
          for (int q = 0; q < NQ; ++q) {
            const double v = cic ? w[h][q] * wy * wz : w[h][q];
            acc[q] = i + h < c[cn] ? acc[q] + v : acc[q];
          }
        }
      }
    }
#pragma unroll
    for (int q = 0; q < NQ; ++q) wacc[q][n] = acc[q];
  }
  __syncthreads();
  for (int i = t; i < NWIN; i += NT) cnt[i] = 0;
  __syncthreads();
}

// A round with more than kCell events in some cell: the events sorted by cell and
// index.  BY_CELL (the double form): the owner lane sums its cell's run as
// deposit_cells does its list; else every node sums the runs of its four corner cells,
// event by event, in the order that deposit_lists keeps.  ev: y, z and the NQ weights by
// rows; the sorted events take the same memory in pairs, (y, z), (w0, w1), which are
// read at once.  halves: bit h set where half h of the cells has events.  *still is set
// where a cell is crowded: the next round is then sorted without trying the lists (a
// per cent of a push).  Both ways give a node the same sums, bit by bit.
// Bound by the chain of a lane's events (their reads' latency; with the chip full, the
// reads themselves), so the reads are paired, spread over the banks (run_slot) and two
// events in flight.  A layer's three pushes of 512^2, us: 9 per cell 387 with every chunk
// sorted, 395 with lists tried first and single reads, 333 like this; 16 811, 889, 605; 25
// 1318, 1430, 1040.  By nodes (float) 9 357, 362, 365; 16 772, 846, 708; 25 1239, 1369, 1298.
template <int NQ, bool BY_CELL>
__device__ inline void deposit_sorted(int cellw, int *keys, int *sorted, short *cstart,
                                      short *cend, double (*ev)[NT], double (*wacc)[NWIN],
                                      bool cic, int halves, int *still) {
  typedef double pair __attribute__((ext_vector_type(2)));
  const int t = thread_index();
  for (int i = t; i < NWIN; i += NT) { cstart[i] = 0; cend[i] = 0; }
  const int sk = sort256(cellw < 0 ? kInvalid : cellw << 8 | t, keys);
  sorted[t] = sk;
  // the event at sorted position t, moved there in place: gathered before the
  // barrier, stored after it, so the node sums below read events without the
  // sorted[] indirection
  double g[2 + NQ];
  if (sk != kInvalid) {
    const int e = sk & 255;
#pragma unroll
    for (int q = 0; q < 2 + NQ; ++q) g[q] = ev[q][e];
  }
  pair *const yz = reinterpret_cast<pair *>(ev[0]), *const w01 = reinterpret_cast<pair *>(ev[2]);
  __syncthreads();
  if (sk != kInvalid) {
    const int at = qss_tile::run_slot(t);
    yz[at] = pair{g[0], g[1]};
    w01[at] = pair{g[2], g[3]};
    if constexpr (NQ == 4) reinterpret_cast<pair *>(ev[4])[at] = pair{g[4], g[5]};
    else ev[4][at] = g[4];
    const int c = sk >> 8;
    const int prev = t > 0 ? sorted[t - 1] : kInvalid;
    const int next = t + 1 < NT ? sorted[t + 1] : kInvalid;
    if (t == 0 || (prev >> 8) != c) cstart[c] = (short)t;
    if (next == kInvalid || (next >> 8) != c) cend[c] = (short)(t + 1);
    if (t + kCell < NT && sorted[t + kCell] >> 8 == c) *still = 1;   // more than kCell of them
  }
  __syncthreads();
  const auto event = [&](int e, double &y, double &z, double *w) {
    const int at = qss_tile::run_slot(e);
    const pair p = yz[at], a = w01[at];
    y = p.x; z = p.y;
    w[0] = a.x; w[1] = a.y;
    if constexpr (NQ == 4) {
      const pair b = reinterpret_cast<const pair *>(ev[4])[at];
      w[2] = b.x; w[3] = b.y;
    } else {
      w[2] = ev[4][at];
    }
  };
  if constexpr (BY_CELL) {
#pragma unroll 1
    for (int half = 0; half < 2; ++half) {
      if (!(halves >> half & 1)) continue;
      const int cell = t + NT * half;
      const int e0 = cell < NWIN ? cstart[cell] : 0, e1 = cell < NWIN ? cend[cell] : 0;
      double s[4][NQ] = {};
#pragma unroll 2
      for (int e = e0; e < e1; ++e) {
        double y, z, w[4];
        event(e, y, z, w);
        add_corners<NQ>(cic ? y : 0., cic ? z : 0., w, s);   // NGP: all of it in corner 0
      }
      corner_turns<NQ>(e1 > e0, cell, s, wacc, cic);
    }
    return;
  }
  for (int n = t; n < NWIN; n += NT) {
    double acc[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) acc[q] = wacc[q][n];
    const int nl_j = n % W, nl_k = n / W;
    // corners: own cell (1-y)(1-z); left y(1-z); below (1-y)z; both yz
#pragma unroll
    for (int cn = 0; cn < 4; ++cn) {
      if (!cic && cn > 0) break;
      const int cj = nl_j - (cn & 1), ck = nl_k - (cn >> 1);
      if (cj < 0 || ck < 0) continue;
      const int cw = ck * W + cj;
      const int e1 = cend[cw];
#pragma unroll 2
      for (int e = cstart[cw]; e < e1; ++e) {
        double y, z, w[4];
        event(e, y, z, w);
        const double wy = (cn & 1) ? y : 1. - y;
        const double wz = (cn >> 1) ? z : 1. - z;
#pragma unroll
        for (int q = 0; q < NQ; ++q) acc[q] += cic ? w[q] * wy * wz : w[q];
      }
    }
#pragma unroll
    for (int q = 0; q < NQ; ++q) wacc[q][n] = acc[q];
  }
}

// R: arithmetic of the push (double: the reference's; float: mixed modes).
// FT: storage of the push field.  Positions and momenta are carried in
// double in both: the float form computes each slice's kick, rotation and
// displacement in float and adds them to the double state, and the deposit
// weights are summed in double.  With R = double every expression of the push
// evaluates exactly as the reference's (no contraction, same association).
//
// A tile's particles may be shared by nsplit work-groups (part p takes
// chunks p, p + nsplit, ...): each part writes its own window, direction
// counts and ranks, and the combine / reorder kernels visit the parts in
// order, so results are a pure function of the input and nsplit.
// A layer step's forms (no RHO) hold at most 128 VGPRs and 40 KB of LDS: four waves per
// SIMD, so all the tiles of a 512^2 grid (4 work-groups per CU) are resident at once;
// with the density 132 VGPRs (FULL: 144) and 46 KB, three.  The bound is
// instruction issue and latency, not memory: at 512^2 and 4 per cell 58 MB in and
// 15 MB out (full: 61 MB) in 31.8 us (full: 38.0), half of the wave cycles waiting at
// barriers and for LDS.  What spilled registers here cost most: with uniform FP64
// products made on the host, the sort's lane masks not kept over the loop and
// machine LICM off (it keeps FP64 literals in registers) no vector register spills and
// only the FULL forms keep scalar ones in vector lanes (30, float 12): 37 us on average
// of a step's three pushes at that point, against 42.6 with 104 scalar registers spilled.
// FULL: the pushed particles are staged for the reorder.
// RHO = false: the deposit sums Jx, Jy, Jz only and the windows' density
// component stays 0 (inside a layer step nothing reads the deposited density:
// the corrector takes rho from continuity in spectral space).
template <typename R, typename FT, bool RHO, bool FULL>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4)))
void k_push_tile(TileArgs a0) {
  const TileArgs a = wake_view(a0, blockIdx.y);   // wake of a batch
  const long pw = (long)blockIdx.y * a0.npw;
  // components in pairs and events component by component: neighbouring cells
  // and neighbouring events then lie side by side, one access of a wave free of
  // bank conflicts (a node's six or an event's four together cost 362 conflict
  // cycles per wave and chunk, a third of the LDS time)
  __shared__ pair_t<FT> Fw[3][NF];
  constexpr int NQ = RHO ? 4 : 3;
  __shared__ __attribute__((aligned(16))) double ev[2 + NQ][NT];   // y, z, weights
  double *const ev_y = ev[0], *const ev_z = ev[1];
  double(*const ev_w)[NT] = ev + 2;
  __shared__ double wacc[NQ][NWIN];   // the window's node sums
  // the round's events of each cell, or the sort's arrays in a crowded round
  __shared__ union {
    struct {
      int cnt[NWIN];
      uint2 list[NWIN];   // kCell event indices, a byte each
    } cell;
    struct {
      int keys[NT], sorted[NT];
      short cstart[NWIN], cend[NWIN];
    } sort;
  } sh;
  __shared__ int dir_total[9];
  __shared__ int wave_cnt[NT / 64][9];
  // what a round's events say to all: some cell is crowded, some particle has
  // another sub-step, events in the first and in the second half of the cells.
  // Two sets: one is cleared while the other is read.
  enum { FL_CROWDED, FL_MORE, FL_HALF0, FL_HALF1, FL_N };
  __shared__ int flag_sh[2][FL_N];

  const int t = threadIdx.x;
  const int tile = blockIdx.x / a.nsplit, part = blockIdx.x - tile * a.nsplit;
  const int tj = tile % a.ntj, tk = tile / a.ntj;
  const int j0 = tj * T, k0 = tk * T;
  const int ny = a.ny, nz = a.nz;
  const R kick = (R)a.kick, mweight = (R)a.mweight;
  const bool cic = a.shape == QSS_SHAPE_CIC;
  int status = 0;   // ST_* bits met by this thread, reported once at the end

  const int base = __builtin_amdgcn_readfirstlane(a.tile_start[tile]);
  const int np = __builtin_amdgcn_readfirstlane(a.tile_start[tile + 1]) - base;

  // 1. field window: nodes (j0..j0+T, k0..k0+T), periodic
  {
    // both nodes of a thread asked for before either is stored
    constexpr int PER = (NF + NT - 1) / NT;
    const long plane = (long)ny * nz;
    const FT *const F = field_of<FT>(a);
    FT v[PER][6];
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      const int i = t + NT * e < NF ? t + NT * e : NF - 1;
      const int lj = i % FW, lk = i / FW;
      const int gj = j0 + lj < ny ? j0 + lj : 0, gk = k0 + lk < nz ? k0 + lk : 0;   // at most one past
      const unsigned g = gj + ny * gk;
#pragma unroll
      for (int q = 0; q < 6; ++q) v[e][q] = (F + q * plane)[g];
    }
#pragma unroll
    for (int e = 0; e < PER; ++e)
      if (t + NT * e < NF)
#pragma unroll
        for (int q = 0; q < 3; ++q) Fw[q][t + NT * e] = {v[e][2 * q], v[e][2 * q + 1]};
  }
  if (t < 9) dir_total[t] = 0;
  if (t < 2 * FL_N) flag_sh[t / FL_N][t % FL_N] = 0;
  int par = 0;
  int sorting = 0;   // the round before was crowded
  for (int i = t; i < NWIN; i += NT) {
    sh.cell.cnt[i] = 0;
#pragma unroll
    for (int q = 0; q < NQ; ++q) wacc[q][i] = 0.0;
  }
  __syncthreads();

  for (int c0 = part * NT; c0 < np; c0 += a.nsplit * NT) {
    // the chunk's place in the wake's particle arrays, unmoved pointers: one for the
    // whole work-group, so that a lane's address is its index beside it (opaque: 13
    // pointers per lane carried from chunk to chunk would spill)
    const long g0 = pw + base + c0;
    const unsigned tl = thread_index();
    const bool active = c0 + t < np;
    int j = 0, k = 0;
    double yp = 0, zp = 0, px = 0, py = 0, pz = 0;
    R djx = 0, djy = 0, djz = 0, drho = 0, dy = 0, dz = 0, partdx = 0, step = 1;
    if (active) {
      cell_jk((a0.cell + g0)[tl], ny, a.ny_magic, j, k);
      yp = (a0.y + g0)[tl];
      zp = (a0.z + g0)[tl];
      if (!(yp >= 0 && yp <= 1 && zp >= 0 && zp <= 1)) status |= (ST_PARTICLE);
      px = (a0.px + g0)[tl]; py = (a0.py + g0)[tl]; pz = (a0.pz + g0)[tl];
      const R rpx = (R)px, rpy = (R)py, rpz = (R)pz;
      // one reciprocal per denominator, then products: the reference divides by
      // the same gamma and 1 - Vx many times over (movepart_splitlayer.cpp:
      // 1239-1330); results agree to an ulp per step
      const R igp = inv_gamma(rpx, rpy, rpz);
      R Vx = rpx * igp;
      const R Vxp = Vx, Vyp = rpy * igp, Vzp = rpz * igp;
      // gather from the staged window: local node (j - j0, k - k0)
      int lj = j - j0, lk = k - k0;
      if (lj < 0 || lj >= T || lk < 0 || lk >= T) {   // not in this tile: never expected
        status |= (ST_FAR);
        lj = min(max(lj, 0), T - 1);
        lk = min(max(lk, 0), T - 1);
      }
      R f[6];
      const int i00 = lj + FW * lk;
      if (!cic) {
#pragma unroll
        for (int q = 0; q < 3; ++q) {
          const pair_t<FT> v = Fw[q][i00];
          f[2 * q] = (R)v.x;
          f[2 * q + 1] = (R)v.y;
        }
      } else {
        const R ayc = R(1. - yp), ayp = R(yp), azc = R(1. - zp), azp = R(zp);
        const R acc = ayc * azc, apc = ayp * azc, acp = ayc * azp, app = ayp * azp;
#pragma unroll
        for (int q = 0; q < 3; ++q) {
          const pair_t<FT> f00 = Fw[q][i00], f10 = Fw[q][i00 + 1], f01 = Fw[q][i00 + FW],
                           f11 = Fw[q][i00 + FW + 1];
          f[2 * q] = acc * (R)f00.x + apc * (R)f10.x + acp * (R)f01.x + app * (R)f11.x;
          f[2 * q + 1] = acc * (R)f00.y + apc * (R)f10.y + acp * (R)f01.y + app * (R)f11.y;
        }
      }
      R ex = f[0], ey = f[1], ez = f[2], bx = f[3], by = f[4], bz = f[5];
      ex *= kick;
      ey *= kick;
      ez *= kick;
      // half kick, carried in the double state
      const R iu = R(1) / (R(1) - Vx);
      const R kx = ex * iu, ky = ey * iu, kz = ez * iu;
      px += (double)kx;
      py += (double)ky;
      pz += (double)kz;
      const R hpx = (R)px, hpy = (R)py, hpz = (R)pz;
      const R gamma_r = inv_gamma(hpx, hpy, hpz);
      bx += R(a.bext[0]);
      by += R(a.bext[1]);
      bz += R(a.bext[2]);
      const R beta = gamma_r * iu * kick;
      bx = bx * beta;
      by = by * beta;
      bz = bz * beta;
      const R co = R(2) / (R(1) + (bx * bx) + (by * by) + (bz * bz));
      R p3x = hpy * bz - hpz * by + hpx;
      R p3y = hpz * bx - hpx * bz + hpy;
      R p3z = hpx * by - hpy * bx + hpz;
      p3x *= co;
      p3y *= co;
      p3z *= co;
      const R px_new = p3y * bz - p3z * by;
      const R py_new = p3z * bx - p3x * bz;
      const R pz_new = p3x * by - p3y * bx;
      px += (double)(kx + px_new);
      py += (double)(ky + py_new);
      pz += (double)(kz + pz_new);
      const R npx = (R)px, npy = (R)py, npz = (R)pz;
      const R ig = inv_gamma(npx, npy, npz);
      const R Vxm = npx * ig, Vym = npy * ig, Vzm = npz * ig;
      Vx = R(0.5) * (Vxm + Vxp);
      const R Vy = R(0.5) * (Vym + Vyp), Vz = R(0.5) * (Vzm + Vzp);
      const R iv = R(1) / (R(1) - Vx);
      djx = mweight * Vxm * iv;
      djy = mweight * Vym * iv;
      djz = mweight * Vzm * iv;
      drho = mweight * iv;
      dy = Vy * R(a.hxy) * iv;
      dz = Vz * R(a.hxz) * iv;
      if (fabs(dy) > R(1) || fabs(dz) > R(1)) {
        if (fabs(dy) > fabs(dz)) step = partdx = fabs(dy);
        else step = partdx = fabs(dz);
      }
      if (partdx < R(1)) partdx = step = R(1);
      if (!(step < (R)(kMaxSub - 1))) {
        status |= (ST_SUBSTEPS);
        partdx = step = R(1);
        dy = R(0);
        dz = R(0);
      }
    }
    double ytmp = yp, ztmp = zp;
    int jj = j, kk = k;
    // sub-step rounds: round r deposits every particle's r-th sub-step
    for (;;) {
      const bool have = active && partdx > 0.;
      int cellw = -1;   // this round's window cell
      if (have) {
        R part_step;
        if (step == R(1)) { part_step = R(1); partdx = R(0); }   // partdx is 1: one step
        else if (partdx > R(1)) { partdx -= R(1); part_step = R(1) / step; }
        else { part_step = partdx / step; partdx = R(0); }
        // the reference restarts every sub-step from the start cell
        ytmp += (double)(dy * part_step) + j;
        ztmp += (double)(dz * part_step) + k;
        if (!(ytmp > a.lo[0] && ytmp < a.hi[0] && ztmp > a.lo[1] && ztmp < a.hi[1])) {
          status |= (ST_PARTICLE);
          ytmp = 0.0;
          ztmp = 0.0;
        }
        while (ytmp > a.nyd) ytmp -= a.nyd;
        while (ytmp < 0) ytmp += a.nyd;
        while (ztmp > a.nzd) ztmp -= a.nzd;
        while (ztmp < 0) ztmp += a.nzd;
        jj = (int)ytmp;
        kk = (int)ztmp;
        ytmp -= jj;
        ztmp -= kk;
        if (jj >= ny) jj -= ny;
        if (kk >= nz) kk -= nz;
        // window cell: any periodic image with both CIC nodes inside
        int dj = jj - j0, dk = kk - k0;
        if (dj + H < 0) dj += ny;
        else if (dj + H > W - 2) dj -= ny;
        if (dk + H < 0) dk += nz;
        else if (dk + H > W - 2) dk -= nz;
        const int lj = dj + H, lk = dk + H;
        if (lj >= 0 && lj <= W - 2 && lk >= 0 && lk <= W - 2) {
          cellw = lk * W + lj;
          ev_y[t] = ytmp;
          ev_z[t] = ztmp;
          ev_w[0][t] = (double)(djx * part_step);
          ev_w[1][t] = (double)(djy * part_step);
          ev_w[2][t] = (double)(djz * part_step);
          if constexpr (RHO) ev_w[3][t] = (double)(drho * part_step);
          if (!sorting) {
            const int r = atomicAdd(&sh.cell.cnt[cellw], 1);
            if (r < kCell) reinterpret_cast<uint8_t *>(&sh.cell.list[cellw])[r] = (uint8_t)t;
            else flag_sh[par][FL_CROWDED] = 1;
          }
          flag_sh[par][cellw < NT ? FL_HALF0 : FL_HALF1] = 1;
        } else {
          status |= (ST_FAR);
        }
      }
      if (active && partdx > 0.) flag_sh[par][FL_MORE] = 1;
      __syncthreads();
      const int *fl = flag_sh[par];
      const bool more = fl[FL_MORE], crowded = sorting || fl[FL_CROWDED];
      const bool half0 = fl[FL_HALF0], half1 = fl[FL_HALF1];
      par ^= 1;
      if (t < FL_N) flag_sh[par][t] = 0;   // last read a barrier ago
      if (crowded) {
        if (!sorting) __syncthreads();   // the lists give way to the sort
        deposit_sorted<NQ, sizeof(R) == 8>(cellw, sh.sort.keys, sh.sort.sorted, sh.sort.cstart,
                                           sh.sort.cend, ev, wacc, cic, half0 | half1 << 1,
                                           &flag_sh[par][FL_CROWDED]);
        __syncthreads();
        // crowded still: the next round is sorted without trying the lists
        sorting = __builtin_amdgcn_readfirstlane(flag_sh[par][FL_CROWDED]);
        if (!sorting) {
          for (int i = t; i < NWIN; i += NT) sh.cell.cnt[i] = 0;
          __syncthreads();
        }
      } else if constexpr (sizeof(R) == 4) {
        deposit_lists<NQ>(sh.cell.cnt, sh.cell.list, ev_y, ev_z, ev_w, wacc, cic);
      } else {
        // rolled: the code of a work-group's first pass comes from L2 line by line
#pragma unroll 1
        for (int half = half0 ? 0 : 1; half < (half1 ? 2 : 1); ++half)
          deposit_cells<NQ>(half, sh.cell.cnt, sh.cell.list, ev_y, ev_z, ev_w, wacc, cic);
        if (!half0 && !half1) __syncthreads();   // the flags are clear before the next round
      }
      if (!more) break;
    }
    if constexpr (FULL) {
      // destination tile direction (canonical for 1 or 2 tiles per axis)
      int dtj = 0, dtk = 0;
      if (active) {
        const int ntj_ = a.ntj, ntk_ = a.ntk;
        // |jj/T - tj| < ntj: one correction wraps it
        int d1 = jj / T - tj, d2 = kk / T - tk;
        d1 += d1 < 0 ? ntj_ : 0;
        d2 += d2 < 0 ? ntk_ : 0;
        dtj = d1 == 0 ? 0 : (d1 == ntj_ - 1 && ntj_ > 2 ? -1 : 1);
        dtk = d2 == 0 ? 0 : (d2 == ntk_ - 1 && ntk_ > 2 ? -1 : 1);
        if (d1 > 1 && d1 < ntj_ - 1) status |= (ST_FAR);
        if (d2 > 1 && d2 < ntk_ - 1) status |= (ST_FAR);
      }
      const int dir = (dtj + 1) + 3 * (dtk + 1);
      // rank among this tile's particles with the same direction, slot order: a turn
      // for each direction that the wave has (most particles stay in the tile)
      const unsigned ti = thread_index();
      const int lane = ti & 63, wv = ti >> 6;
      int myrank_w = 0;
      if (lane < 9) wave_cnt[wv][lane] = 0;
      unsigned long long left = __ballot(active);
      while (left) {
        const int d = __builtin_amdgcn_readlane(dir, __builtin_ctzll(left));
        const unsigned long long m = __ballot(active && dir == d);
        if (lane == 0) wave_cnt[wv][d] = __popcll(m);
        if (dir == d)
          myrank_w = __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32),
                                               __builtin_amdgcn_mbcnt_lo((unsigned)m, 0));
        left &= ~m;
      }
      __syncthreads();
      int off = dir_total[dir];
      for (int q = 0; q < wv; ++q) off += wave_cnt[q][dir];
      if (active) {
        (a0.sy + g0)[ti] = ytmp;
        (a0.sz + g0)[ti] = ztmp;
        (a0.spx + g0)[ti] = px;
        (a0.spy + g0)[ti] = py;
        (a0.spz + g0)[ti] = pz;
        (a0.scell + g0)[ti] = jj + ny * kk;
        (a0.sdest + g0)[ti] = dir | (part << 4) | ((off + myrank_w) << 8);
      }
      __syncthreads();
      if (t < 9) {
        int s = 0;
        for (int q = 0; q < NT / 64; ++q) s += wave_cnt[q][t];
        dir_total[t] += s;
      }
      __syncthreads();
    }
  }
  if (status) atomicOr(&a.counters[1], status);
  // 4. window to HBM
  double4 *wout = reinterpret_cast<double4 *>(a.win + (long)blockIdx.x * NWIN * 4);
  for (int i = t; i < NWIN; i += NT)
    wout[i] = make_double4(wacc[0][i], wacc[1][i], wacc[2][i], RHO ? wacc[NQ - 1][i] : 0.0);
  if (FULL && t < 9)
    a.tcount[(t * a.nsplit + part) * (a.ntj * a.ntk) + tile] = dir_total[t];
}

// New tile starts and group offsets: destination tile u receives the groups
// of source tiles u - dir(d) for d = 0..8 in that order, each as the groups
// of the source's parts 0..NS-1.  One work-group per wake takes one or two tiles a
// thread at a time (as many as the combine's registers allow), all loads together; counts and
// offsets are stored direction by direction, so that neighbouring lanes read
// neighbouring tiles.  It depends on the push only, as the combine does, and takes
// less time than a plane's combine at every size (per 1024 tiles 2.5 us against
// 5.6), so it is that launch's first work-group: by itself it was 3.6 us at 64^2,
// 9.5 at 256^2 (four parts) and 6.6 at 512^2.
template <int NS>
__device__ inline void tile_scan(const int32_t *tcount, int ntj, int ntk, int32_t *tile_start,
                                 int32_t *goff) {
  constexpr int B = NS == 1 ? 2 : 1, NG = 9 * NS, NW = NT / 64;
  __shared__ int wsum[B][NW];
  const int nt = ntj * ntk;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  int carry = 0;
  for (int b0 = 0; b0 < nt; b0 += NT * B) {
    int g[B][NG], tot[B], incl[B];
#pragma unroll
    for (int b = 0; b < B; ++b) {
      const int u = b0 + b * NT + (int)threadIdx.x;
      tot[b] = 0;
      const int uu = u < nt ? u : 0;
      const int uk = uu / ntj, uj = uu - uk * ntj;
#pragma unroll
      for (int d = 0; d < 9; ++d) {
        int sj = uj - (d % 3 - 1), sk = uk - (d / 3 - 1);
        sj = sj < 0 ? sj + ntj : (sj >= ntj ? sj - ntj : sj);
        sk = sk < 0 ? sk + ntk : (sk >= ntk ? sk - ntk : sk);
#pragma unroll
        for (int q = 0; q < NS; ++q) {
          const int v = tcount[(d * NS + q) * nt + sk * ntj + sj];
          g[b][d * NS + q] = u < nt ? v : 0;
        }
      }
    }
    // exclusive scan over the tiles: inclusive scans within each wave, then
    // the totals of the waves before this one (integer sums: exact)
#pragma unroll
    for (int b = 0; b < B; ++b) {
#pragma unroll
      for (int e = 0; e < NG; ++e) tot[b] += g[b][e];
      incl[b] = tot[b];
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int v = __shfl_up(incl[b], o, 64);
        if (lane >= o) incl[b] += v;
      }
      if (lane == 63) wsum[b][wv] = incl[b];
    }
    __syncthreads();
#pragma unroll
    for (int b = 0; b < B; ++b) {
      const int u = b0 + b * NT + (int)threadIdx.x;
      int before = 0, all = 0;
#pragma unroll
      for (int q = 0; q < NW; ++q) {
        const int v = wsum[b][q];
        before += q < wv ? v : 0;
        all += v;
      }
      int o = carry + before + incl[b] - tot[b];
      if (u < nt) {
        tile_start[u] = o;
#pragma unroll
        for (int e = 0; e < NG; ++e) {
          goff[e * nt + u] = o;
          o += g[b][e];
        }
      }
      carry += all;
    }
    __syncthreads();   // wsum is rewritten by the next tiles
  }
  if (threadIdx.x == 0) tile_start[nt] = carry;
}

// sum of the windows covering each node, fixed (dtk, dtj, part) order.  Per
// axis a node lies in its own tile's window (dt = 0) and in at most one
// neighbour's (dt = -1 within W - T - H nodes of the tile's low edge, +1 within
// H of its high edge; the two ranges are disjoint), so at most 4 x NS windows
// cover it: all their loads are issued before the first add.  An absent window
// reads the own tile's entry and adds +0.0 instead, which leaves the sum bitwise
// unchanged (the sum starts at +0.0, so it is never -0.0).
// xs0..xs2 (split-bf16 modes, one wake): Jx, Jy, Jz also written as the split
// operands of the forward transform that follows.
// grid: (node blocks of one plane, wakes); 32-bit node index (ny, nz <= 2^14); with
// tcount one more work-group, the first, does the full step's tile scan
static_assert(W - T - H <= T - H, "at most two tiles per axis cover a node");
// RHO = false: the density plane J3 is neither summed nor written
template <int NS, bool RHO>
__global__ __launch_bounds__(NT) void k_combine(const double *win, int ntj, int ntk, int ny,
                                                int nz, uint64_t ny_magic, double *J0,
                                                double *J1, double *J2, double *J3,
                                                uint16_t *xs0, uint16_t *xs1, uint16_t *xs2,
                                                int npc, const int32_t *tcount,
                                                int32_t *tile_start, int32_t *goff) {
  int block = blockIdx.x;
  if (tcount && block-- == 0) {
    const long nt = (long)ntj * ntk, w = blockIdx.y;
    tile_scan<NS>(tcount + w * nt * NS * 9, ntj, ntk, tile_start + w * (nt + 1),
                  goff + w * nt * NS * 9);
    return;
  }
  const int plane = ny * nz;
  const int n1 = block * NT + threadIdx.x;   // node of the wake's plane
  if (n1 >= plane) return;
  const double4 *w4 = reinterpret_cast<const double4 *>(win) +
                      (long)blockIdx.y * ntj * ntk * NS * NWIN;   // the wake's windows
  const long n = (long)blockIdx.y * plane + n1;                   // wake-major node index
  int nj, nk;
  cell_jk(n1, ny, ny_magic, nj, nk);
  const int tj = nj / T, tk = nk / T;
  const int rj = nj - tj * T, rk = nk - tk * T;   // position in the tile, [0, T)
  // covering tiles per axis, in increasing order: (d0, d0 + 1), the second
  // present when the node is near either edge
  const int dk0 = rk < W - T - H ? -1 : 0, dj0 = rj < W - T - H ? -1 : 0;
  const bool hk = rk < W - T - H || rk >= T - H, hj = rj < W - T - H || rj >= T - H;
  long idx[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a) {
    const int utk = tk + dk0 + a;                 // unwrapped tile row, in [-1, ntk]
    const int wtk = utk < 0 ? utk + ntk : (utk >= ntk ? utk - ntk : utk);
    const int lk = nk - (utk * T - H);
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const int utj = tj + dj0 + b;
      const int wtj = utj < 0 ? utj + ntj : (utj >= ntj ? utj - ntj : utj);
      const int lj = nj - (utj * T - H);
      idx[a][b] = (long)(wtk * ntj + wtj) * NS * NWIN + lk * W + lj;
    }
  }
  const bool ok[2][2] = {{true, hj}, {hk, hk && hj}};
  double4 v[2][2][NS];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int q = 0; q < NS; ++q)
        v[a][b][q] = w4[(ok[a][b] ? idx[a][b] : idx[0][0]) + (long)q * NWIN];
  double s[4] = {0, 0, 0, 0};
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int q = 0; q < NS; ++q) {
        const double4 u = ok[a][b] ? v[a][b][q] : make_double4(0.0, 0.0, 0.0, 0.0);
        s[0] += u.x; s[1] += u.y; s[2] += u.z;
        if (RHO) s[3] += u.w;
      }
  J0[n] = s[0]; J1[n] = s[1]; J2[n] = s[2];
  if (RHO) J3[n] = s[3];
  if (npc) {
    qss_split::store(xs0, plane, n, s[0], npc);
    qss_split::store(xs1, plane, n, s[1], npc);
    qss_split::store(xs2, plane, n, s[2], npc);
  }
}

__global__ __launch_bounds__(NT) void k_permute(TileArgs a0, const int32_t *goff, long np,
                                                int nw, double *y, double *z, double *px,
                                                double *py, double *pz, int32_t *cell,
                                                int64_t *pid) {
  const long sg = (long)blockIdx.x * NT + threadIdx.x;   // wake-major slot
  if (sg >= np * nw) return;
  const int w = (int)(sg / np);
  const long s = sg - (long)w * np;
  const TileArgs a = wake_view(a0, w);
  goff += (long)w * a.ntj * a.ntk * a.nsplit * 9;
  const long pw = (long)w * a0.npw;
  y += pw; z += pw; px += pw; py += pw; pz += pw; cell += pw; pid += pw;
  const int32_t c = a.scell[s];
  int cj, ck;
  cell_jk(c, a.ny, a.ny_magic, cj, ck);
  const int dst_tile = (ck / T) * a.ntj + cj / T;
  const int sd = a.sdest[s];   // direction | part << 4 | rank << 8
  const int group = (sd & 15) * a.nsplit + ((sd >> 4) & 15);
  const long o = goff[group * (a.ntj * a.ntk) + dst_tile] + (sd >> 8);
  y[o] = a.sy[s];
  z[o] = a.sz[s];
  px[o] = a.spx[s];
  py[o] = a.spy[s];
  pz[o] = a.spz[s];
  cell[o] = c;
  pid[o] = a.pid[s];   // ids are not staged: the old storage still holds them
}

// seeding in tile-major slot order: tile, local cell (j fastest), seed
__global__ void k_seed_tiled(double *y, double *z, double *px, double *py, double *pz,
                             int32_t *cell, int64_t *pid, long np, int nw, int ny, int ntj,
                             int ppc_y, int ppc_z, double jitter, uint64_t seed) {
  const long ng = (long)blockIdx.x * NT + threadIdx.x;   // wake-major slot
  if (ng >= np * nw) return;
  // every wake of a batch starts from the same plasma
  const long n = ng % np;
  y += ng - n; z += ng - n; px += ng - n; py += ng - n; pz += ng - n;
  cell += ng - n; pid += ng - n;
  const int ppc = ppc_y * ppc_z;
  const long per_tile = (long)T * T * ppc;
  const long tile = n / per_tile;
  const long r = n - tile * per_tile;
  const int lc = (int)(r / ppc), is = (int)(r - (long)lc * ppc);
  const int gj = (int)(tile % ntj) * T + lc % T;
  const int gk = (int)(tile / ntj) * T + lc / T;
  const long c = gj + (long)ny * gk;
  const long id = c * ppc + is;
  const int iy = is % ppc_y, iz = is / ppc_y;
  double yy = (iy + 1.0) / (ppc_y + 1.0);
  double zz = (iz + 1.0) / (ppc_z + 1.0);
  if (jitter != 0.0) {
    // the same counter-based draws as the cell-ordered seeding (by id)
    auto mix64 = [](uint64_t x) {
      x += 0x9E3779B97F4A7C15ull;
      x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
      x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
      return x ^ (x >> 31);
    };
    auto unif = [&](uint64_t a2, uint64_t b2) {
      const uint64_t h = mix64(seed ^ mix64(a2 ^ mix64(b2)));
      return (double)(h >> 11) * (1.0 / 9007199254740992.0) * 2.0 - 1.0;
    };
    yy += jitter * unif((uint64_t)id, 1);
    zz += jitter * unif((uint64_t)id, 2);
  }
  y[n] = yy;
  z[n] = zz;
  px[n] = 0.0;
  py[n] = 0.0;
  pz[n] = 0.0;
  cell[n] = (int32_t)c;
  pid[n] = id;
}

__global__ void k_uniform_tile_start(int32_t *ts, int nt, int nw, int per_tile) {
  const int i = blockIdx.x * NT + threadIdx.x;   // wake-major
  if (i < (nt + 1) * nw) ts[i] = (i % (nt + 1)) * per_tile;
}

inline dim3 grid1(long n) { return dim3((unsigned)((n + NT - 1) / NT)); }

TileArgs make_args(qss_ctx *c) {
  TileArgs a;
  const int b = c->cur;
  a.y = c->py_[b]; a.z = c->pz_[b]; a.px = c->ppx[b]; a.py = c->ppy[b]; a.pz = c->ppz[b];
  a.cell = c->pcell[b]; a.pid = c->pid[b];
  a.tile_start = c->tile_start[b];
  a.ntj = c->ntj; a.ntk = c->ntk; a.ny = c->ny; a.nz = c->nz;
  a.F = c->F;
  a.Ff = c->Ff;
  a.kick = -0.5 * c->hxs;
  a.mweight = -c->pweight;
  a.nyd = c->ny; a.nzd = c->nz;
  a.lo[0] = -2.0 * c->ny; a.lo[1] = -2.0 * c->nz;
  a.hi[0] = 3.0 * c->ny; a.hi[1] = 3.0 * c->nz;
  a.hxy = c->hxs / c->hy; a.hxz = c->hxs / c->hz;
  for (int q = 0; q < 3; ++q) a.bext[q] = c->p.b_ext[q];
  a.shape = c->p.shape;
  a.win = c->win;
  const long npall = c->np_cap * c->nw;
  a.sy = c->ev_y; a.sz = c->ev_z; a.spx = c->ev_p; a.spy = c->ev_p + npall;
  a.spz = c->ev_p + 2 * npall;
  a.scell = c->ev_cell; a.sdest = c->ev_rank;
  a.tcount = c->tcount;
  a.counters = c->d_counters;
  a.npw = c->np_cap;
  a.nsplit = c->nsplit;
  a.ny_magic = ((1ull << 44) + (uint64_t)c->ny - 1) / (uint64_t)c->ny;
  return a;
}

}  // namespace

hipError_t launch_push_tile(qss_ctx *c, int full, bool rho, hipEvent_t ev0, hipEvent_t ev1) {
  const dim3 grid(c->ntj * c->ntk * c->nsplit, c->nw), block(NT);
  const auto pick = [&](auto r, auto f) {
    using T = decltype(r);
    constexpr bool F = decltype(f)::value;
    return rho ? k_push_tile<T, T, true, F> : k_push_tile<T, T, false, F>;
  };
  const std::true_type yes;
  const std::false_type no;
  auto fn = c->mixed ? (full ? pick(0.0f, yes) : pick(0.0f, no))
                     : (full ? pick(0.0, yes) : pick(0.0, no));
  if (ev0 || ev1)
    hipExtLaunchKernelGGL(fn, grid, block, 0, c->stream, ev0, ev1, 0, make_args(c));
  else
    hipLaunchKernelGGL(fn, grid, block, 0, c->stream, make_args(c));
  return hipGetLastError();
}

hipError_t launch_combine(qss_ctx *c, bool rho, double *const *out, bool scan) {
  double *const J[4] = {c->C[QSS_JX], c->C[QSS_JY], c->C[QSS_JZ], c->C[QSS_RHO]};
  const bool split = c->npc && !out;   // sweep deposits only (not the tuning runs)
  if (!out) out = J;
  if (split)
    for (int b = 0; b < 3; ++b) c->xs_src[b] = J[b];
  const uint64_t ny_magic = ((1ull << 44) + (uint64_t)c->ny - 1) / (uint64_t)c->ny;
  auto fn = rho ? (c->nsplit == 1   ? k_combine<1, true>
                   : c->nsplit == 2 ? k_combine<2, true>
                                    : k_combine<4, true>)
                : (c->nsplit == 1   ? k_combine<1, false>
                   : c->nsplit == 2 ? k_combine<2, false>
                                    : k_combine<4, false>);
  if (c->nsplit != 1 && c->nsplit != 2 && c->nsplit != 4) return hipErrorInvalidValue;
  hipLaunchKernelGGL(fn, dim3(grid1(c->ncell).x + (scan ? 1 : 0), c->nw), dim3(NT), 0, c->stream,
                     c->win, c->ntj, c->ntk, c->ny, c->nz, ny_magic, out[0], out[1], out[2], out[3],
                     c->xs[0], c->xs[1], c->xs[2], split ? c->npc : 0,
                     scan ? c->tcount : nullptr, c->tile_start[c->cur ^ 1], c->goff);
  return hipGetLastError();
}

hipError_t launch_tile_reorder(qss_ctx *c) {
  const int nb = c->cur ^ 1;
  hipLaunchKernelGGL(k_permute, grid1(c->np * c->nw), dim3(NT), 0, c->stream, make_args(c),
                     c->goff, c->np, c->nw, c->py_[nb], c->pz_[nb], c->ppx[nb], c->ppy[nb],
                     c->ppz[nb], c->pcell[nb], c->pid[nb]);
  return hipGetLastError();
}

hipError_t launch_seed_tiled(qss_ctx *c) {
  const int b = c->cur;
  hipLaunchKernelGGL(k_seed_tiled, grid1(c->np * c->nw), dim3(NT), 0, c->stream, c->py_[b],
                     c->pz_[b], c->ppx[b], c->ppy[b], c->ppz[b], c->pcell[b], c->pid[b], c->np,
                     c->nw, c->ny, c->ntj, c->p.ppc_y, c->p.ppc_z, c->p.jitter,
                     (uint64_t)c->p.seed);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const int nt = c->ntj * c->ntk;
  hipLaunchKernelGGL(k_uniform_tile_start, grid1((long)(nt + 1) * c->nw), dim3(NT), 0,
                     c->stream, c->tile_start[b], nt, c->nw, T * T * c->p.ppc_y * c->p.ppc_z);
  return hipGetLastError();
}
