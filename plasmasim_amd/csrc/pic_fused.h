// Shared pieces of the step's fused field kernels (both forms).
//
// A step's field work is three launches instead of eleven: the first B half
// step with renew_grid and sr_b, the second with sr_b and sr_current2, the E
// step with sr_e.  On small grids every launch costs its latency (about 5 us
// on the stream, whatever it does), on large ones the guards and folds are
// strided passes of their own: at 64^3 FP32 the eleven took 140 us per step.
//  - Guards: sr_b / sr_e copy only interior columns into guard columns, so
//    the thread that owns an interior cell writes its images as well.  Of
//    columns, since m runs over the whole array: the z guards are copied as
//    they are.  nx, ny >= 4 keeps the source layers of both faces apart.
//  - Folds: the layers of sr_current2 form independent groups of two columns
//    (four in the corners); one thread takes a group at one m, in the
//    reference's order (x over all columns, then y).
#pragma once
#include <hip/hip_runtime.h>

#include "pic_internal.h"

namespace pic {

// The blocks of a step's field launch, of 256 threads, as a grid of rows: a
// launch may not have 2^32 threads along one dimension, which short columns
// reach first (nz = 8: at 6.7e7 columns, 64 threads each).  Blocks past the
// last one have no cell.
constexpr int64_t kGridRow = (int64_t)1 << 23;
__host__ inline dim3 block_grid(int64_t blocks) {
  const int64_t rows = div_up(blocks, kGridRow);
  return dim3((unsigned)(rows > 1 ? kGridRow : blocks), (unsigned)rows);
}
__device__ inline int block_index() { return (int)(blockIdx.y * gridDim.x + blockIdx.x); }

// cell of thread t of cell block b: 64 x 4 threads over (m, l), one k
struct CellBlocks {
  int gx, gy;  // blocks along m and l
  __host__ inline CellBlocks(const Geom &g)
      : gx((g.SZ + 63) / 64), gy((g.SY + 3) / 4) {}
  __host__ inline int64_t count(const Geom &g) const { return (int64_t)gx * gy * g.SX; }
  __host__ __device__ inline bool cell(const Geom &g, int b, int t, int &k, int &l,
                                       int &m) const {
    m = (b % gx) * 64 + (t & 63);
    l = (b / gx) % gy * 4 + (t >> 6);
    k = b / (gx * gy);
    return m < g.SZ && l < g.SY && k < g.SX;
  }
};

__device__ inline bool interior_column(const Geom &g, int k, int l) {
  return k >= 2 && k < g.NX + 2 && l >= 2 && l < g.NY + 2;
}

// The images of cell c of interior column (k, l): put(dst, src) in the
// reference's order, the corner from the x image.
template <typename Put>
__device__ inline void images(const Geom &g, int k, int l, int64_t c, Put put) {
  const int64_t dk = (int64_t)g.SY * g.SZ, dl = g.SZ;
  const int64_t x = k < 4 ? g.NX * dk : k >= g.NX ? -g.NX * dk : 0;
  const int64_t y = l < 4 ? g.NY * dl : l >= g.NY ? -g.NY * dl : 0;
  if (x) put(c + x, c);
  if (y) put(c + y, c);
  if (x && y) put(c + x + y, c + x);
}

// interior column e < fold_groups(g) that has images
__device__ inline void edge_column(const Geom &g, int e, int &k, int &l) {
  const auto edge = [](int p, int n) { return p < 2 ? 2 + p : n + p - 2; };
  if (e < 4 * g.NY) {
    k = edge(e & 3, g.NX);
    l = 2 + (e >> 2);
  } else {
    e -= 4 * g.NY;
    k = 4 + (e >> 2);
    l = edge(e & 3, g.NY);
  }
}

// columns that no fold reads or writes
__device__ inline bool unfolded_column(const Geom &g, int k, int l) {
  return k >= 4 && k < g.NX && l >= 4 && l < g.NY;
}

__host__ __device__ inline int fold_groups(const Geom &g) { return 4 * (g.NX + g.NY) - 16; }

// Fold group t of one plane at one m: load(i) reads the deposit, store(i, v)
// writes the plane (store(.., false): a value that the fold only reads).
template <typename Load, typename Store>
__device__ inline void fold_group(const Geom &g, int t, int m, Load load, Store store) {
  // pair p along an axis of n cells: layer d takes in guard layer s
  const auto dst = [](int p, int n) { return p < 2 ? 2 + p : n + p - 2; };
  const auto src = [](int p, int n) { return p < 2 ? n + 2 + p : p - 2; };
  const int ne = 4 * (g.NY - 4), nf = 4 * (g.NX - 4);
  if (t < ne + nf) {
    int64_t a, b;
    if (t < ne) {
      const int p = t & 3, l = 4 + (t >> 2);
      a = g.idx(dst(p, g.NX), l, m);
      b = g.idx(src(p, g.NX), l, m);
    } else {
      const int p = (t - ne) & 3, k = 4 + ((t - ne) >> 2);
      a = g.idx(k, dst(p, g.NY), m);
      b = g.idx(k, src(p, g.NY), m);
    }
    const auto vb = load(b);
    store(a, load(a) + vb, true);
    store(b, vb, false);
    return;
  }
  const int p = (t - ne - nf) & 3, q = (t - ne - nf) >> 2;
  const int kd = dst(p, g.NX), ks = src(p, g.NX), ld = dst(q, g.NY), ls = src(q, g.NY);
  const int64_t a = g.idx(kd, ld, m), x = g.idx(ks, ld, m), y = g.idx(kd, ls, m),
                xy = g.idx(ks, ls, m);
  const auto vx = load(x), vxy = load(xy);
  const auto vy = load(y) + vxy;
  store(a, (load(a) + vx) + vy, true);
  store(y, vy, true);
  store(x, vx + vxy, true);
  store(xy, vxy, false);
}

// thrust_fave: the running sums' share of both passes (6 partials per
// workgroup), one block per species and quantity, in a fixed order
struct ThrustFinish {
  const double *part[2];
  int nb[2];  // workgroups of the pass; 0: no pass ran
  double qn[2];
  double *acc;
};

__device__ inline void thrust_finish(const ThrustFinish &f, int b) {
  __shared__ double sh[256];
  const int sp = b / 6, q = b % 6;
  if (f.nb[sp] == 0) return;
  double v = 0.0;
  for (int i = threadIdx.x; i < f.nb[sp]; i += 256) v += f.part[sp][(int64_t)i * 6 + q];
  sh[threadIdx.x] = v;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) sh[threadIdx.x] += sh[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) f.acc[6 * sp + q] += f.qn[sp] * sh[0];
}

ThrustFinish thrust_finish_args(const pic_ctx *ctx);

}  // namespace pic
