// Plain FP64 form of the step on gfx950.
//
// Arithmetic mirrors ashida-lab/PLASMAsim PIC/3d_pic458_domain.c expression
// by expression; this translation unit is compiled with -ffp-contract=off so
// that no multiply-add is fused and every operation rounds as the
// reference's C does.  Layout: one plane per field component (m contiguous),
// particles in SoA per species; a dead particle carries z = NaN until the
// next compaction (inflow or sort).
#include <hip/hip_runtime.h>
#include <new>
#include <math.h>
#include <stdlib.h>
#include <string.h>

#include "philox.h"
#include "pic_fused.h"
#include "pic_internal.h"
#include "pic_tsort.h"
#include "pic_tiles.h"

namespace pic {
namespace f64 {

// ---------------------------------------------------------------------------
// field kernels

__global__ void k_zero(double *__restrict__ p, int64_t n) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (; i < n; i += stride) p[i] = 0.0;
}

__device__ inline double sigma_at(const SigmaProfile &s, int k2, int l2,
                                  int m2) {
  const double a4 = s.d4[0][k2] + s.d4[1][l2] + s.d4[2][m2];
  if (a4 == 0.0) return 0.0;  // outside every layer: all depths are zero
  const double a12 = s.d12[0][k2] + s.d12[1][l2] + s.d12[2][m2];
  return s.amp * (0.1 * sqrt(a4) + 0.01 * sqrt(a12));
}

struct FieldConst {
  double dt, dx, eps0, mu0, c;
};

// renew_b4_2 (:2580-2611) at interior cell c
__device__ inline void renew_b_cell(const Geom &g, const Fields<double> &F,
                                    const SigmaProfile &sg, const FieldConst &fc, int k,
                                    int l, int m, int64_t c, double out[3]) {
  const double temp = 1. / fc.eps0 * fc.dt * 0.5 * 0.5;
  const double dth = 0.5 * fc.dt;
  const double temp_24 = 1. / 24.;
  const double inv_dx = 1. / fc.dx;
  const int64_t dl = g.SZ, dk = (int64_t)g.SY * g.SZ;
  const double *ex = F.f[PIC_EX], *ey = F.f[PIC_EY], *ez = F.f[PIC_EZ];
  double f, h, s;

  s = sigma_at(sg, 2 * k + 1, 2 * l, 2 * m);
  f = s == 0.0 ? 1.0 : (1. - s * temp) / (1. + s * temp);
  h = s == 0.0 ? dth : dth / (1. + s * temp);
  {
    const double b0 = F.f[PIC_B0X][c];
    out[0] =
        b0 + f * (F.f[PIC_BX][c] - b0) -
        h * temp_24 *
            (27. * (ez[c] - ez[c - dl] - ey[c] + ey[c - 1]) -
             (ez[c + dl] - ez[c - 2 * dl] - ey[c + 1] + ey[c - 2])) *
            inv_dx;
  }
  s = sigma_at(sg, 2 * k, 2 * l + 1, 2 * m);
  f = s == 0.0 ? 1.0 : (1. - s * temp) / (1. + s * temp);
  h = s == 0.0 ? dth : dth / (1. + s * temp);
  {
    const double b0 = F.f[PIC_B0Y][c];
    out[1] =
        b0 + f * (F.f[PIC_BY][c] - b0) -
        h * temp_24 *
            (27. * (ex[c] - ex[c - 1] - ez[c] + ez[c - dk]) -
             (ex[c + 1] - ex[c - 2] - ez[c + dk] + ez[c - 2 * dk])) *
            inv_dx;
  }
  s = sigma_at(sg, 2 * k, 2 * l, 2 * m + 1);
  f = s == 0.0 ? 1.0 : (1. - s * temp) / (1. + s * temp);
  h = s == 0.0 ? dth : dth / (1. + s * temp);
  {
    const double b0 = F.f[PIC_B0Z][c];
    out[2] =
        b0 + f * (F.f[PIC_BZ][c] - b0) -
        h * temp_24 *
            (27. * (ey[c] - ey[c - dk] - ex[c] + ex[c - dl]) -
             (ey[c + dk] - ey[c - 2 * dk] - ex[c + dl] + ex[c - 2 * dl])) *
            inv_dx;
  }
}

__global__ __launch_bounds__(256) void k_renew_b(Geom g, Fields<double> F, SigmaProfile sg,
                                                 FieldConst fc) {
  const int m = 2 + blockIdx.x * blockDim.x + threadIdx.x;
  const int l = 2 + blockIdx.y * blockDim.y + threadIdx.y;
  const int k = 2 + blockIdx.z;
  if (m >= g.NZ + 2 || l >= g.NY + 2) return;
  const int64_t c = g.idx(k, l, m);
  double b[3];
  renew_b_cell(g, F, sg, fc, k, l, m, c, b);
#pragma unroll
  for (int q = 0; q < 3; ++q) F.f[PIC_BX + q][c] = b[q];
}

// renew_e4_2 (:2613-2652) at interior cell c; the curl acts on B - B0
// recomputed per term, as the reference writes it.
__device__ inline void renew_e_cell(const Geom &g, const Fields<double> &F,
                                    const SigmaProfile &sg, const FieldConst &fc, int k,
                                    int l, int m, int64_t c, double out[3]) {
  const double temp = fc.c * fc.c * fc.dt;
  const double temp_24 = 1. / 24.;
  const double inv_dx = 1. / fc.dx;
  const int64_t dl = g.SZ, dk = (int64_t)g.SY * g.SZ;
  const double *bx = F.f[PIC_BX], *by = F.f[PIC_BY], *bz = F.f[PIC_BZ];
  const double *b0x = F.f[PIC_B0X], *b0y = F.f[PIC_B0Y], *b0z = F.f[PIC_B0Z];
  double s, f, h;
#define D1(B, B0, a, b) (B[a] - B0[a] - B[b] + B0[b])

  s = sigma_at(sg, 2 * k, 2 * l + 1, 2 * m + 1);
  f = s == 0.0 ? 1.0 : (1. - 0.5 * fc.mu0 * s * temp) / (1. + 0.5 * fc.mu0 * s * temp);
  h = s == 0.0 ? temp : temp / (1. + 0.5 * fc.mu0 * s * temp);
  out[0] =
      f * F.f[PIC_EX][c] +
      h * (temp_24 *
               (27. * (D1(bz, b0z, c + dl, c) - D1(by, b0y, c + 1, c)) -
                (D1(bz, b0z, c + 2 * dl, c - dl) - D1(by, b0y, c + 2, c - 1))) *
               inv_dx -
           fc.mu0 * (F.f[PIC_JIX][c] - F.f[PIC_JEX][c]));

  s = sigma_at(sg, 2 * k + 1, 2 * l, 2 * m + 1);
  f = s == 0.0 ? 1.0 : (1. - 0.5 * fc.mu0 * s * temp) / (1. + 0.5 * fc.mu0 * s * temp);
  h = s == 0.0 ? temp : temp / (1. + 0.5 * fc.mu0 * s * temp);
  out[1] =
      f * F.f[PIC_EY][c] +
      h * (temp_24 *
               (27. * (D1(bx, b0x, c + 1, c) - D1(bz, b0z, c + dk, c)) -
                (D1(bx, b0x, c + 2, c - 1) - D1(bz, b0z, c + 2 * dk, c - dk))) *
               inv_dx -
           fc.mu0 * (F.f[PIC_JIY][c] - F.f[PIC_JEY][c]));

  s = sigma_at(sg, 2 * k + 1, 2 * l + 1, 2 * m);
  f = s == 0.0 ? 1.0 : (1. - 0.5 * fc.mu0 * s * temp) / (1. + 0.5 * fc.mu0 * s * temp);
  h = s == 0.0 ? temp : temp / (1. + 0.5 * fc.mu0 * s * temp);
  out[2] =
      f * F.f[PIC_EZ][c] +
      h * (temp_24 *
               (27. * (D1(by, b0y, c + dk, c) - D1(bx, b0x, c + dl, c)) -
                (D1(by, b0y, c + 2 * dk, c - dk) - D1(bx, b0x, c + 2 * dl, c - dl))) *
               inv_dx -
           fc.mu0 * (F.f[PIC_JIZ][c] - F.f[PIC_JEZ][c]));
#undef D1
}

__global__ __launch_bounds__(256) void k_renew_e(Geom g, Fields<double> F, SigmaProfile sg,
                                                 FieldConst fc) {
  const int m = 2 + blockIdx.x * blockDim.x + threadIdx.x;
  const int l = 2 + blockIdx.y * blockDim.y + threadIdx.y;
  const int k = 2 + blockIdx.z;
  if (m >= g.NZ + 2 || l >= g.NY + 2) return;
  const int64_t c = g.idx(k, l, m);
  double e[3];
  renew_e_cell(g, F, sg, fc, k, l, m, c, e);
#pragma unroll
  for (int q = 0; q < 3; ++q) F.f[PIC_EX + q][c] = e[q];
}

// sr_b / sr_e on one rank (:1001-1387): the guard columns of the three planes
// from `first`
__global__ void k_halo(Geom g, Fields<double> F, int first) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (int64_t)fold_groups(g) * g.SZ) return;
  int k, l;
  edge_column(g, (int)(i / g.SZ), k, l);
  const int64_t c = g.idx(k, l, (int)(i % g.SZ));
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    double *f = F.f[first + q];
    const double v = f[c];
    images(g, k, l, c, [&](int64_t d, int64_t) { f[d] = v; });
  }
}

// sr_current2 (:1805-2039) on one rank, 8 planes
__global__ void k_fold(Geom g, Fields<double> F) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (int64_t)fold_groups(g) * g.SZ) return;
#pragma unroll
  for (int q = PIC_JIX; q <= PIC_NE; ++q) {
    double *f = F.f[q];
    fold_group(
        g, (int)(i / g.SZ), (int)(i % g.SZ), [&](int64_t j) { return f[j]; },
        [&](int64_t j, double v, bool changed) {
          if (changed) f[j] = v;
        });
  }
}

// ---------------------------------------------------------------------------
// the step's field launches (pic_fused.h)

// B half step and sr_b of cell (k, l, m); kept (3 planes, or null): the
// end-of-step total B goes there first
__device__ inline void b_and_guards(const Geom &g, const Fields<double> &F, double *kept,
                                    const SigmaProfile &sg, const FieldConst &fc, int k, int l,
                                    int m) {
  const int64_t c = g.idx(k, l, m);
  const bool in = m >= 2 && m < g.NZ + 2;
  double b[3];
  if (in) renew_b_cell(g, F, sg, fc, k, l, m, c, b);
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    double *B = F.f[PIC_BX + q], *K = kept ? kept + q * g.plane : nullptr;
    const double old = B[c], v = in ? b[q] : old;
    if (K) K[c] = old;
    if (in) B[c] = v;
    images(g, k, l, c, [&](int64_t d, int64_t) {
      if (K) K[d] = B[d];
      B[d] = v;
    });
  }
}

// renew_grid, thrust_fave's copy of the total B, the first B half step, sr_b
__global__ __launch_bounds__(256) void k_step_b1(Geom g, CellBlocks cb, Fields<double> F,
                                                 double *kept, SigmaProfile sg,
                                                 FieldConst fc) {
  int k, l, m;
  if (!cb.cell(g, block_index(), threadIdx.x, k, l, m)) return;
  const int64_t c = g.idx(k, l, m);
#pragma unroll
  for (int q = 0; q < 8; ++q) F.f[PIC_JIX + q][c] = 0.0;
  if (interior_column(g, k, l)) b_and_guards(g, F, kept, sg, fc, k, l, m);
}

// The second B half step and sr_b, sr_current2, thrust_fave's sums: blocks
// below tb finish the thrust, then fb blocks fold, the rest are cells.
__global__ __launch_bounds__(256) void k_step_b2(Geom g, CellBlocks cb, Fields<double> F,
                                                 SigmaProfile sg, FieldConst fc, int tb,
                                                 ThrustFinish tf, int fb) {
  int b = block_index();
  if (b < tb) {
    thrust_finish(tf, b);
    return;
  }
  b -= tb;
  if (b < fb) {
    const int64_t t = (int64_t)b * 256 + threadIdx.x;
    if (t >= (int64_t)fold_groups(g) * g.SZ) return;
    const int m = (int)(t % g.SZ), grp = (int)(t / g.SZ);
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      double *f = F.f[PIC_JIX + q];
      fold_group(
          g, grp, m, [&](int64_t i) { return f[i]; },
          [&](int64_t i, double v, bool changed) {
            if (changed) f[i] = v;
          });
    }
    return;
  }
  b -= fb;
  int k, l, m;
  if (!cb.cell(g, b, threadIdx.x, k, l, m) || !interior_column(g, k, l)) return;
  b_and_guards(g, F, nullptr, sg, fc, k, l, m);
}

// the E step and sr_e
__global__ __launch_bounds__(256) void k_step_e(Geom g, CellBlocks cb, Fields<double> F,
                                                SigmaProfile sg, FieldConst fc) {
  int k, l, m;
  if (!cb.cell(g, block_index(), threadIdx.x, k, l, m) || !interior_column(g, k, l)) return;
  const int64_t c = g.idx(k, l, m);
  const bool in = m >= 2 && m < g.NZ + 2;
  double e[3];
  if (in) renew_e_cell(g, F, sg, fc, k, l, m, c, e);
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    double *E = F.f[PIC_EX + q];
    const double v = in ? e[q] : E[c];
    if (in) E[c] = v;
    images(g, k, l, c, [&](int64_t d, int64_t) { E[d] = v; });
  }
}

// ---------------------------------------------------------------------------
// particle kernels

// Gather of one staggered component (shape_func_v2 :3223-3273): the eight
// products are formed and summed in the reference's order.
__device__ inline double gather1(const double *__restrict__ F, const Geom &g,
                                 int a, int b, int c, double wa0, double wa1,
                                 double wb0, double wb1, double wc0,
                                 double wc1) {
  const int64_t i = g.idx(a, b, c);
  const int64_t dl = g.SZ, dk = (int64_t)g.SY * g.SZ;
  const double p1 = F[i] * (wa0 * wb0 * wc0) + F[i + 1] * (wa0 * wb0 * wc1);
  const double p2 =
      F[i + dl] * (wa0 * wb1 * wc0) + F[i + dl + 1] * (wa0 * wb1 * wc1);
  const double p3 =
      F[i + dk] * (wa1 * wb0 * wc0) + F[i + dk + 1] * (wa1 * wb0 * wc1);
  const double p4 = F[i + dk + dl] * (wa1 * wb1 * wc0) +
                    F[i + dk + dl + 1] * (wa1 * wb1 * wc1);
  return p1 + p2 + p3 + p4;
}

struct AxisW {
  int bi, bh;        // (int)(x/dx), (int)(x/dx - 0.5)
  double iu, il;     // integer-located weights: upper, lower
  double hu, hl;     // half-located weights
};

__device__ inline AxisW axis_weights(double x, double dx) {
  AxisW w;
  w.bi = (int)(x / dx);
  w.iu = ((w.bi + 1) * dx - x);
  w.il = (x - w.bi * dx);
  w.bh = (int)(x / dx - 0.5);
  w.hu = (((w.bh + 1) + 0.5) * dx - x);
  w.hl = (x - (w.bh + 0.5) * dx);
  return w;
}

// shape_func_v2 (:3017-3326): out = ex, ey, ez, bx, by, bz
__device__ inline void gather(const Fields<double> &F, const Geom &g, double x,
                              double y, double z, double dx, double out[6]) {
  const double inv_dx3 = 1. / (dx * dx * dx);
  const AxisW X = axis_weights(x, dx), Y = axis_weights(y, dx),
              Z = axis_weights(z, dx);
  out[0] = gather1(F.f[PIC_EX], g, X.bi, Y.bh, Z.bh, X.iu, X.il, Y.hu, Y.hl,
                   Z.hu, Z.hl) * inv_dx3;
  out[1] = gather1(F.f[PIC_EY], g, X.bh, Y.bi, Z.bh, X.hu, X.hl, Y.iu, Y.il,
                   Z.hu, Z.hl) * inv_dx3;
  out[2] = gather1(F.f[PIC_EZ], g, X.bh, Y.bh, Z.bi, X.hu, X.hl, Y.hu, Y.hl,
                   Z.iu, Z.il) * inv_dx3;
  out[3] = gather1(F.f[PIC_BX], g, X.bh, Y.bi, Z.bi, X.hu, X.hl, Y.iu, Y.il,
                   Z.iu, Z.il) * inv_dx3;
  out[4] = gather1(F.f[PIC_BY], g, X.bi, Y.bh, Z.bi, X.iu, X.il, Y.hu, Y.hl,
                   Z.iu, Z.il) * inv_dx3;
  out[5] = gather1(F.f[PIC_BZ], g, X.bi, Y.bi, Z.bh, X.iu, X.il, Y.iu, Y.il,
                   Z.hu, Z.hl) * inv_dx3;
}

// Constants of one species' pass, formed on the host by the reference's
// operations (a uniform FP64 product on the device would hold two vector
// registers through the whole loop).
struct PassConst {
  double dx, dt, dth, c;
  double cc;              // C^2
  double T, TT, T2;       // q dt / (2 m), its square, 2 T
  double eimf_x, eimf_y;  // V * IMF terms of E (:2817-2818)
  double qn, wn;          // q w / dx^3, w / dx^3
  double blo[3], bhi[3];  // ballistic zone
  double box_lo[3], box_hi[3];  // thrust_fave's box (open)
  int periodic[2];
};

// cal_track4 (:2804-2870), velocity
__device__ inline void boris(const PassConst &k, const double f[6], double &vx,
                             double &vy, double &vz) {
  const double C = k.c, T = k.T;
  double ex = f[0], ey = f[1], ez = f[2];
  const double bx = f[3], by = f[4], bz = f[5];
  ex += k.eimf_x;
  ey += k.eimf_y;
  double gamma1 = C / sqrt(k.cc - vx * vx - vy * vy - vz * vz);
  if (isnan(gamma1)) gamma1 = 0.;
  double ux = gamma1 * vx, uy = gamma1 * vy, uz = gamma1 * vz;
  double gamma2 = C / sqrt(k.cc + ux * ux + uy * uy + uz * uz);
  const double bux = gamma2 * (bx), buy = gamma2 * (by), buz = gamma2 * (bz);
  const double S = k.T2 / (1. + k.TT * (bux * bux + buy * buy + buz * buz));
  ux += (ex) * T;
  uy += (ey) * T;
  uz += (ez) * T;
  const double uox = ux + T * (uy * buz - uz * buy);
  const double uoy = uy + T * (uz * bux - ux * buz);
  const double uoz = uz + T * (ux * buy - uy * bux);
  double upx = ux + S * (uoy * buz - uoz * buy);
  double upy = uy + S * (uoz * bux - uox * buz);
  double upz = uz + S * (uox * buy - uoy * bux);
  upx += (ex) * T;
  upy += (ey) * T;
  upz += (ez) * T;
  gamma2 = C / sqrt(k.cc + upx * upx + upy * upy + upz * upz);
  vx = gamma2 * upx;
  vy = gamma2 * upy;
  vz = gamma2 * upz;
}

// Array-safety rule (the oracle states the same): nodes base..base+1 stay
// inside the array when -0.5 < x/dx < S-1 on every axis.
__device__ inline bool in_array(const Geom &g, double x, double y, double z,
                                double dx) {
  const double xd = x / dx, yd = y / dx, zd = z / dx;
  return xd > -0.5 && xd < g.SX - 1 && yd > -0.5 && yd < g.SY - 1 &&
         zd > -0.5 && zd < g.SZ - 1;
}

// ---------------------------------------------------------------------------
// particle pass: one workgroup per sort tile, J and n accumulated in an LDS
// window with FP64 atomics, then added to the planes (see pic_tiles.h)
//
// No unit is saturated (128^3 x 64 ppc with the force: VALU and LDS 47 % busy
// at three waves per SIMD), half of the waves' cycles are waits for memory; the
// pass is written for few instructions (867 per particle) with the reference's
// operations and rounding: one stencil per position shared by the gathers and the previous
// step's force; constants formed on the host; each lane's walk of the
// stencils set up once per workgroup, one swap of the weights per axis; and
// in normalised units (UNIT: dx = 1, where x / dx and w * dx are x and w
// exactly; planes and arrays below 4 GiB) no divisions by dx and 32-bit byte
// offsets from uniform bases.  165 VGPRs, from 239 at two waves per SIMD.
// 20 steps at 128^3 x 64 ppc 377 -> 345 ms, at 32^3 x 16 ppc 7.1 -> 5.8 ms; with
// the ordered gathers (gather6o) 295 ms.

constexpr int kWin64 = 1400;  // window capacity in nodes (4 x double each)

#define PIC_LDS __attribute__((address_space(3)))
#define PIC_GLB __attribute__((address_space(1)))

typedef unsigned long long u64;

__device__ __forceinline__ void lds_add64(char *acc, int byte, double v) {
  __hip_atomic_fetch_add((PIC_LDS double *)(acc + byte), v, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void glob_add64(double *p, double v) {
  __hip_atomic_fetch_add((PIC_GLB double *)p, v, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
}

template <bool UNIT>
struct Off {
  using T = int64_t;
};
template <>
struct Off<true> {
  using T = uint32_t;
};
template <typename T, typename O>
__device__ __forceinline__ T *at(T *base, O byte) {
  return (T *)((char *)base + byte);
}

// Gather of one staggered component around the byte offset i of its stencil
// base (shape_func_v2 :3223-3273): the products and sums of gather1.
template <typename O>
__device__ __forceinline__ double gather1o(const double *F, O i, O dl, O dk, double wa0,
                                           double wa1, double wb0, double wb1,
                                           double wc0, double wc1) {
  const double *f0 = at(F, i), *f1 = at(F, i + dl), *f2 = at(F, i + dk),
               *f3 = at(F, i + dk + dl);
  const double p1 = f0[0] * (wa0 * wb0 * wc0) + f0[1] * (wa0 * wb0 * wc1);
  const double p2 = f1[0] * (wa0 * wb1 * wc0) + f1[1] * (wa0 * wb1 * wc1);
  const double p3 = f2[0] * (wa1 * wb0 * wc0) + f2[1] * (wa1 * wb0 * wc1);
  const double p4 = f3[0] * (wa1 * wb1 * wc0) + f3[1] * (wa1 * wb1 * wc1);
  return p1 + p2 + p3 + p4;
}

// gather1o's loads and its products and sums, apart from each other
template <typename O>
__device__ __forceinline__ void load8o(const double *F, O i, O dl, O dk, double (&v)[8]) {
  const double *f0 = at(F, i), *f1 = at(F, i + dl), *f2 = at(F, i + dk),
               *f3 = at(F, i + dk + dl);
  v[0] = f0[0], v[1] = f0[1], v[2] = f1[0], v[3] = f1[1];
  v[4] = f2[0], v[5] = f2[1], v[6] = f3[0], v[7] = f3[1];
}
__device__ __forceinline__ double sum8o(const double (&v)[8], double wa0, double wa1,
                                        double wb0, double wb1, double wc0, double wc1) {
  const double p1 = v[0] * (wa0 * wb0 * wc0) + v[1] * (wa0 * wb0 * wc1);
  const double p2 = v[2] * (wa0 * wb1 * wc0) + v[3] * (wa0 * wb1 * wc1);
  const double p3 = v[4] * (wa1 * wb0 * wc0) + v[5] * (wa1 * wb0 * wc1);
  const double p4 = v[6] * (wa1 * wb1 * wc0) + v[7] * (wa1 * wb1 * wc1);
  return p1 + p2 + p3 + p4;
}

// The six components at a particle in a stated order: two components' loads
// are in flight ahead of the one summed.  Left alone, the compiler waits for
// each load before it issues the next in a kernel with the force; all six at
// once take 249 registers, which costs a wave per SIMD, two take 165.
template <typename O>
__device__ __forceinline__ void gather6o(const double *const (&E)[3],
                                         const double *const (&B)[3], O o, O hx, O hy, O hz,
                                         O dl, O dk, const AxisW &X, const AxisW &Y,
                                         const AxisW &Z, double inv_dx3, double (&f)[6]) {
  const O ox = o - hx, oy = o - hy, oz = o - hz;
  double u[8], v[8];
  load8o<O>(E[0], oy - hz, dl, dk, u);
  load8o<O>(E[1], ox - hz, dl, dk, v);
  __builtin_amdgcn_sched_barrier(0);
  f[0] = sum8o(u, X.iu, X.il, Y.hu, Y.hl, Z.hu, Z.hl) * inv_dx3;
  __builtin_amdgcn_sched_barrier(0);
  load8o<O>(E[2], ox - hy, dl, dk, u);
  __builtin_amdgcn_sched_barrier(0);
  f[1] = sum8o(v, X.hu, X.hl, Y.iu, Y.il, Z.hu, Z.hl) * inv_dx3;
  __builtin_amdgcn_sched_barrier(0);
  load8o<O>(B[0], ox, dl, dk, v);
  __builtin_amdgcn_sched_barrier(0);
  f[2] = sum8o(u, X.hu, X.hl, Y.hu, Y.hl, Z.iu, Z.il) * inv_dx3;
  __builtin_amdgcn_sched_barrier(0);
  load8o<O>(B[1], oy, dl, dk, u);
  __builtin_amdgcn_sched_barrier(0);
  f[3] = sum8o(v, X.hu, X.hl, Y.iu, Y.il, Z.iu, Z.il) * inv_dx3;
  __builtin_amdgcn_sched_barrier(0);
  load8o<O>(B[2], oz, dl, dk, v);
  __builtin_amdgcn_sched_barrier(0);
  f[4] = sum8o(u, X.iu, X.il, Y.hu, Y.hl, Z.iu, Z.il) * inv_dx3;
  f[5] = sum8o(v, X.iu, X.il, Y.iu, Y.il, Z.hu, Z.hl) * inv_dx3;
}

// The lane's walk over the 8 nodes of a stencil in the LDS window: lane j
// takes them mirrored along the axes set in j & 7, so that lanes holding
// particles of one cell add to different nodes.
struct Walk64 {
  int first;   // byte offset of the first visited node from the stencil base
  int off[8];  // byte offsets of the visits from the first node
  bool mx, my, mz;
};

__device__ inline Walk64 make_walk64(int WY, int WZ) {
  Walk64 k;
  const int sw = threadIdx.x & 7;
  k.mx = sw & 4;
  k.my = sw & 2;
  k.mz = sw & 1;
  const int sz = 8, sy = 8 * WZ, sx = 8 * WY * WZ;
  const int dx = k.mx ? -sx : sx, dy = k.my ? -sy : sy, dz = k.mz ? -sz : sz;
  k.first = (k.mx ? sx : 0) + (k.my ? sy : 0) + (k.mz ? sz : 0);
  k.off[0] = 0;
  k.off[1] = dz;
  k.off[2] = dy;
  k.off[3] = dy + dz;
  k.off[4] = dx;
  k.off[5] = dx + dz;
  k.off[6] = dx + dy;
  k.off[7] = dx + dy + dz;
  return k;
}

// The 8 contributions (temp*wa)*(wb*wc) of one component, as the reference
// forms them (:3412-3425), in the lane's walk order.
__device__ __forceinline__ void lds_dep8_64(char *acc, int base, const Walk64 &k,
                                            double temp, double wa0, double wa1,
                                            double wb0, double wb1, double wc0,
                                            double wc1) {
  const double A0 = k.mx ? wa1 : wa0, A1 = k.mx ? wa0 : wa1;
  const double B0 = k.my ? wb1 : wb0, B1 = k.my ? wb0 : wb1;
  const double C0 = k.mz ? wc1 : wc0, C1 = k.mz ? wc0 : wc1;
  const double ta0 = temp * A0, ta1 = temp * A1;
  const double bc00 = B0 * C0, bc01 = B0 * C1, bc10 = B1 * C0, bc11 = B1 * C1;
  const int p = base + k.first;
  lds_add64(acc, p + k.off[0], ta0 * bc00);
  lds_add64(acc, p + k.off[1], ta0 * bc01);
  lds_add64(acc, p + k.off[2], ta0 * bc10);
  lds_add64(acc, p + k.off[3], ta0 * bc11);
  lds_add64(acc, p + k.off[4], ta1 * bc00);
  lds_add64(acc, p + k.off[5], ta1 * bc01);
  lds_add64(acc, p + k.off[6], ta1 * bc10);
  lds_add64(acc, p + k.off[7], ta1 * bc11);
}

// the same stencil straight into a global plane
__device__ __noinline__ void glob_dep8_64(double *glob, int64_t i, int64_t dl, int64_t dk,
                                          double temp, double wa0, double wa1, double wb0,
                                          double wb1, double wc0, double wc1) {
  const double ta0 = temp * wa0, ta1 = temp * wa1;
  glob_add64(glob + i, (ta0) * (wb0 * wc0));
  glob_add64(glob + i + 1, (ta0) * (wb0 * wc1));
  glob_add64(glob + i + dl, (ta0) * (wb1 * wc0));
  glob_add64(glob + i + dl + 1, (ta0) * (wb1 * wc1));
  glob_add64(glob + i + dk, (ta1) * (wb0 * wc0));
  glob_add64(glob + i + dk + 1, (ta1) * (wb0 * wc1));
  glob_add64(glob + i + dk + dl, (ta1) * (wb1 * wc0));
  glob_add64(glob + i + dk + dl + 1, (ta1) * (wb1 * wc1));
}

// The particles outside the window (pend), straight into the global planes.
// A few, scattered over the waves: the wave takes them one at a time, each
// active lane adding one node of one component, instead of idling behind a
// lane's 8 or 24 atomics; more than kCoopMax in one wave go lane by lane (as
// in the FP32 pass).  Reached by every active lane of the wave.
constexpr int kCoopMax = 8;

__device__ __forceinline__ double lane_get(double v, int src) {
  const u64 b = (u64)__double_as_longlong(v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, src);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), src);
  return __longlong_as_double((long long)(((u64)hi << 32) | lo));
}

__device__ __forceinline__ void glob_coop64(const Geom &g, bool pend, bool current,
                                            double dx, double x, double y, double z,
                                            double q0, double q1, double q2, double *jx,
                                            double *jy, double *jz, double *nd) {
  u64 todo = __builtin_amdgcn_ballot_w64(pend);
  if (todo == 0) return;
  const int64_t dl = g.SZ, dk = (int64_t)g.SY * g.SZ;
  if (__builtin_popcountll(todo) > kCoopMax) {
    if (pend) {
      const AxisW X = axis_weights(x, dx), Y = axis_weights(y, dx), Z = axis_weights(z, dx);
      if (current) {
        glob_dep8_64(jx, g.idx(X.bi, Y.bh, Z.bh), dl, dk, q0, X.iu, X.il, Y.hu, Y.hl, Z.hu,
                     Z.hl);
        glob_dep8_64(jy, g.idx(X.bh, Y.bi, Z.bh), dl, dk, q1, X.hu, X.hl, Y.iu, Y.il, Z.hu,
                     Z.hl);
        glob_dep8_64(jz, g.idx(X.bh, Y.bh, Z.bi), dl, dk, q2, X.hu, X.hl, Y.hu, Y.hl, Z.iu,
                     Z.il);
      } else {
        glob_dep8_64(nd, g.idx(X.bh, Y.bh, Z.bh), dl, dk, q0, X.hu, X.hl, Y.hu, Y.hl, Z.hu,
                     Z.hl);
      }
    }
    return;
  }
  const u64 ex = __builtin_amdgcn_read_exec();
  const int rank = (int)__builtin_amdgcn_mbcnt_hi(
      (uint32_t)(ex >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)ex, 0u));
  const int nact = __builtin_popcountll(ex);
  const int nn = current ? 24 : 8;
  do {
    const int src = __builtin_ctzll(todo);
    todo &= todo - 1;
    const AxisW X = axis_weights(lane_get(x, src), dx), Y = axis_weights(lane_get(y, src), dx),
                Z = axis_weights(lane_get(z, src), dx);
    const double s0 = lane_get(q0, src);
    double s1 = 0.0, s2 = 0.0;
    if (current) {
      s1 = lane_get(q1, src);
      s2 = lane_get(q2, src);
    }
    for (int t = rank; t < nn; t += nact) {
      // node t: component t >> 3 (3: density), corner bits (x, y, z) of
      // t & 7; the component's own axis takes the integer-node weights
      const int c = current ? t >> 3 : 3;
      const bool ux = t & 4, uy = t & 2, uz = t & 1;
      const double wx = c == 0 ? (ux ? X.il : X.iu) : (ux ? X.hl : X.hu);
      const double wy = c == 1 ? (uy ? Y.il : Y.iu) : (uy ? Y.hl : Y.hu);
      const double wz = c == 2 ? (uz ? Z.il : Z.iu) : (uz ? Z.hl : Z.hu);
      const double q = c == 1 ? s1 : c == 2 ? s2 : s0;
      double *dst = c == 0 ? jx : c == 1 ? jy : c == 2 ? jz : nd;
      const int64_t i = g.idx(c == 0 ? X.bi : X.bh, c == 1 ? Y.bi : Y.bh, c == 2 ? Z.bi : Z.bh) +
                        (ux ? dk : 0) + (uy ? dl : 0) + (uz ? 1 : 0);
      glob_add64(dst + i, (q * wx) * (wy * wz));
    }
  } while (todo);
}

// A deposit's place: inside the array and the gate (:747-749), which reduce
// to 0 <= x and x/dx < S-1 per axis.
__device__ __forceinline__ bool dep_ok(const Geom &g, double x, double y, double z, int k,
                                       int l, int m) {
  return x >= 0. && k < g.SX - 1 && y >= 0. && l < g.SY - 1 && z >= 0. && m < g.SZ - 1;
}

// a deposit at cell c touches the nodes c - 1 to c + 1: cells within the
// anchor +- (kMargin - 1) keep them inside the window
__device__ __forceinline__ bool win_holds(const Win &w, int k, int l, int m) {
  return w.on && (unsigned)(k - w.vk0 + 1) <= (unsigned)(w.vk1 - w.vk0 + 2) &&
         (unsigned)(l - w.vl0 + 1) <= (unsigned)(w.vl1 - w.vl0 + 2) &&
         (unsigned)(m - w.vm0 + 1) <= (unsigned)(w.vm1 - w.vm0 + 2);
}

__device__ __forceinline__ int win_byte(const Win &w, int k, int l, int m) {
  return (((k - w.k0) * w.WY + (l - w.l0)) * w.WZ + (m - w.m0)) * 8;
}

// sr_particle (:2041-2531) of one particle: x and y shifted into the box;
// false when it drops out
template <bool UNIT>
__device__ __forceinline__ bool bounded(const Geom &g, double dx, const int (&periodic)[2],
                                        double &x, double &y, double z) {
  bool dead, xhi, xlo, yhi, ylo;
  if (UNIT) {  // the upper faces by the cells: the same comparisons
    dead = !(z >= 2.) || (int)z >= g.NZ + 2;
    xhi = (int)x >= g.NX + 2;
    xlo = x < 2.;
    yhi = (int)y >= g.NY + 2;
    ylo = y < 2.;
  } else {
    const double dx2 = 2. * dx;
    dead = !(z < (g.NZ + 2) * dx && z >= dx2);
    xhi = x >= (g.NX + 2) * dx;
    xlo = x < dx2;
    yhi = y >= (g.NY + 2) * dx;
    ylo = y < dx2;
  }
  dead = dead || ((xhi || xlo) && !periodic[0]) || ((yhi || ylo) && !periodic[1]);
  if (xhi) x = x - g.NX * dx;
  else if (xlo) x = x + g.NX * dx;
  if (yhi) y = y - g.NY * dx;
  else if (ylo) y = y + g.NY * dx;
  return !dead;
}

// sr_particle on its own, both species: reads the positions, writes what
// changes
struct Bound64 {
  Particles64 P[2];
  int64_t n[2];
  int nb0;  // workgroups of the ions
  int periodic[2];
};

__global__ void k_boundary(Geom g, Bound64 b, double dx) {
  const int sp = (int)blockIdx.x >= b.nb0 ? 1 : 0;
  const int64_t i = (int64_t)((int)blockIdx.x - (sp ? b.nb0 : 0)) * blockDim.x + threadIdx.x;
  if (i >= b.n[sp]) return;
  const Particles64 &P = b.P[sp];
  const double z = P.z[i];
  if (isnan(z)) return;
  const double x0 = P.x[i], y0 = P.y[i];
  double x = x0, y = y0;
  if (!bounded<false>(g, dx, b.periodic, x, y, z)) {
    P.z[i] = __longlong_as_double(0x7ff8000000000000LL);
    return;
  }
  if (x != x0) P.x[i] = x;
  if (y != y0) P.y[i] = y;
}

// thrust_fave partials of one workgroup (six per-thread sums added over the
// workgroup in a fixed order), stored at slot bid
__device__ inline void thrust_store64(const double (&th)[6], double *out, int bid) {
  __shared__ double sh[6][kBlock / 64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int q = 0; q < 6; ++q) {
    double a = th[q];
    for (int o = 32; o > 0; o >>= 1) a += __shfl_xor(a, o);
    if (lane == 0) sh[q][w] = a;
  }
  __syncthreads();
  if (threadIdx.x < 6) {
    double a = sh[threadIdx.x][0];
    for (int j = 1; j < kBlock / 64; ++j) a += sh[threadIdx.x][j];
    out[(int64_t)bid * 6 + threadIdx.x] = a;
  }
}

// the planes a pass reads and adds to: E, total B, the total B at the end of
// the previous step (THRUST)
struct PassFields {
  const double *e[3], *b[3], *bp[3];
  double *jx, *jy, *jz, *nd;
};

// One species' arguments of a pass; a launch takes one species or both.
struct SpeciesArgs64 {
  TileGeom tg;
  TileRun tr;
  PassFields F;
  Particles64 P;
  PassConst kc;
  double *thrust_part;
};
struct PassArgs64 {
  SpeciesArgs64 s[2];
};

// One particle pass.  PUSH_J: hot loop A (:731-812); DRIFT_N: hot loop B
// (:818-867); BOUNDARY: sr_particle (:2041-2531) on one rank.  The fused
// form (all three) is exact because none of the field updates between those
// loops in fdtd() reads or writes particle state.
// THRUST: also add thrust_fave (:5124-5285) of the previous step for the
// particles of the central box: their positions and velocities at the start
// of the pass are that step's end state, E is unchanged since, and bp holds
// the total B of its end.
// ROWS: as in the FP32 form, boxes of cell columns of a store sorted as one
// tile, the threads divided evenly over a box's columns.  32^3 x 16 ppc in
// chunks of 2048 slots, whose boxes fit no window, took 475 us per launch
// and in boxes 90 us; 8 x 8 x 16 x 4 ppc 70 us and 18 us.
// BOTH: the launch holds both species, the first nb0 workgroups the ions'.
template <bool PUSH_J, bool DRIFT_N, bool BOUNDARY, bool THRUST, bool ROWS, bool UNIT,
          bool BOTH>
__global__ __launch_bounds__(256) void k_particles_tiled(
    Geom g, PassArgs64 args, int nb0) {
  using O = typename Off<UNIT>::T;
  const int sp = BOTH && (int)blockIdx.x >= nb0 ? 1 : 0;
  const SpeciesArgs64 &sa = args.s[sp];
  const TileGeom &tg = sa.tg;
  const TileRun &tr = sa.tr;
  const PassFields &F = sa.F;
  const Particles64 &P = sa.P;
  const PassConst &kc = sa.kc;
  double *const thrust_part = sa.thrust_part;
  __shared__ double acc_mem[4 * kWin64];
  __shared__ Win sw;
  __shared__ int64_t s_range[2];
  const int tid = threadIdx.x;
  const int bid = sp == 0 ? xcd_remap(blockIdx.x, tr.parts(), BOTH ? nb0 : (int)gridDim.x)
                          : xcd_remap(blockIdx.x - nb0, tr.parts(), (int)gridDim.x - nb0);
  const double dx = UNIT ? 1.0 : kc.dx;
  if (tid == 0) {
    int64_t s, e;
    Win w;
    tile_setup<ROWS>(bid, tr, tg, kWin64,
               [&](int64_t i, int &k, int &l, int &m) {
                 const double x = P.x[i], y = P.y[i], z = P.z[i];
                 if (!in_array(g, x, y, z, dx)) return false;
                 k = (int)(x / dx);
                 l = (int)(y / dx);
                 m = (int)(z / dx);
                 return true;
               },
               s, e, w);
    sw = w;
    s_range[0] = s;
    s_range[1] = e;
  }
  __syncthreads();
  const int64_t s = s_range[0], e = s_range[1];
  double th[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  if (s >= e) {
    if (THRUST && tid < 6) thrust_part[(int64_t)bid * 6 + tid] = 0.0;
    return;
  }
  // the window into scalar registers
  Win w;
  w.on = __builtin_amdgcn_readfirstlane(sw.on ? 1 : 0) != 0;
  w.k0 = __builtin_amdgcn_readfirstlane(sw.k0);
  w.l0 = __builtin_amdgcn_readfirstlane(sw.l0);
  w.m0 = __builtin_amdgcn_readfirstlane(sw.m0);
  w.WX = __builtin_amdgcn_readfirstlane(sw.WX);
  w.WY = __builtin_amdgcn_readfirstlane(sw.WY);
  w.WZ = __builtin_amdgcn_readfirstlane(sw.WZ);
  w.vk0 = __builtin_amdgcn_readfirstlane(sw.vk0);
  w.vk1 = __builtin_amdgcn_readfirstlane(sw.vk1);
  w.vl0 = __builtin_amdgcn_readfirstlane(sw.vl0);
  w.vl1 = __builtin_amdgcn_readfirstlane(sw.vl1);
  w.vm0 = __builtin_amdgcn_readfirstlane(sw.vm0);
  w.vm1 = __builtin_amdgcn_readfirstlane(sw.vm1);
  const int WN = w.on ? w.WX * w.WY * w.WZ : 0;
  for (int i = tid; i < 4 * WN; i += blockDim.x) acc_mem[(i / WN) * kWin64 + i % WN] = 0.0;
  __syncthreads();
  char *acc = (char *)acc_mem;
  const Walk64 wk = make_walk64(w.WY, w.WZ);
  const int wsl = 8 * w.WZ, wsk = 8 * w.WY * w.WZ;  // window strides
  const O fl = (O)g.SZ * 8, fk = (O)g.SY * g.SZ * 8;  // plane strides
  const double dth = kc.dth;
  int64_t i0 = s + tid, i1 = e;
  int lanes = blockDim.x;
  if (ROWS && bid < tr.parts()) {
    lanes = kBlock / (tg.TX * tg.TY);
    int rs, re;
    row_range(tr, tg, g.NX, g.NY, g.NZ, bid, tid / lanes, rs, re);
    i0 = rs + tid % lanes;
    i1 = re;
  }
  for (int64_t i = i0; i < i1; i += lanes) {
    const O pb = (O)i * 8;
    double z = *at(P.z, pb);
    if (isnan(z)) continue;  // dead until the next compaction
    double x = *at(P.x, pb), y = *at(P.y, pb);
    double vx = *at(P.vx, pb), vy = *at(P.vy, pb), vz = *at(P.vz, pb);
    if (PUSH_J) {
      AxisW X = axis_weights(x, dx), Y = axis_weights(y, dx), Z = axis_weights(z, dx);
      // in_array by the cells: x/dx < S-1 for the cell below S-1
      const bool safe0 = x / dx > -0.5 && X.bi < g.SX - 1 && y / dx > -0.5 &&
                         Y.bi < g.SY - 1 && z / dx > -0.5 && Z.bi < g.SZ - 1;
      const bool push = safe0 && !(x < kc.blo[0] || x > kc.bhi[0] || y < kc.blo[1] ||
                                   y > kc.bhi[1] || z < kc.blo[2] || z > kc.bhi[2]);
      const bool box = THRUST && safe0 && x < kc.box_hi[0] && x > kc.box_lo[0] &&
                       y < kc.box_hi[1] && y > kc.box_lo[1] && z < kc.box_hi[2] &&
                       z > kc.box_lo[2];
      if (push || box) {
        const double inv_dx3 = 1. / (dx * dx * dx);
        // byte offset of the cell's node and of one node down per axis
        const O o = (((O)X.bi * g.SY + Y.bi) * g.SZ + Z.bi) * 8;
        const O hx = X.bh != X.bi ? fk : 0, hy = Y.bh != Y.bi ? fl : 0,
                hz = Z.bh != Z.bi ? 8 : 0;
        // (not with both species in one launch or dx != 1: the form below
        // keeps three waves there, this one takes 169 to 209 registers)
        if (THRUST && UNIT && !BOTH) {
          double f[6];
          // the force takes its own E: shared with the push, the E gather
          // comes before the force's branch and the push's B after it, and
          // every particle waits for memory twice (128^3 x 64 ppc, 20 steps:
          // 324 ms in the other branch's form, so 301 ms)
          if (box) {
            // the weights of x and the offset renamed, so that neither the
            // node weights nor the E loads are formed once for both
            AxisW XB = X;
            O ob = o;
            asm("" : "+v"(XB.iu), "+v"(XB.il), "+v"(XB.hu), "+v"(XB.hl), "+v"(ob));
            gather6o<O>(F.e, F.bp, ob, hx, hy, hz, fl, fk, XB, Y, Z, inv_dx3, f);
            th[0] += f[0];
            th[1] += f[1];
            th[2] += f[2];
            th[3] += vy * f[5] - vz * f[4];
            th[4] += vz * f[3] - vx * f[5];
            th[5] += vx * f[4] - vy * f[3];
          }
          if (push) {
            gather6o<O>(F.e, F.b, o, hx, hy, hz, fl, fk, X, Y, Z, inv_dx3, f);
            boris(kc, f, vx, vy, vz);
          }
        } else {
          const O ox = o - hx, oy = o - hy, oz = o - hz;
          double f[6];
          const auto take_e = [&]() {
            f[0] = gather1o<O>(F.e[0], oy - hz, fl, fk, X.iu, X.il, Y.hu, Y.hl, Z.hu, Z.hl) * inv_dx3;
            f[1] = gather1o<O>(F.e[1], ox - hz, fl, fk, X.hu, X.hl, Y.iu, Y.il, Z.hu, Z.hl) * inv_dx3;
            f[2] = gather1o<O>(F.e[2], ox - hy, fl, fk, X.hu, X.hl, Y.hu, Y.hl, Z.iu, Z.il) * inv_dx3;
          };
          const auto take_b = [&](const double *const (&B)[3], double (&o3)[3]) {
            o3[0] = gather1o<O>(B[0], ox, fl, fk, X.hu, X.hl, Y.iu, Y.il, Z.iu, Z.il) * inv_dx3;
            o3[1] = gather1o<O>(B[1], oy, fl, fk, X.iu, X.il, Y.hu, Y.hl, Z.iu, Z.il) * inv_dx3;
            o3[2] = gather1o<O>(B[2], oz, fl, fk, X.iu, X.il, Y.iu, Y.il, Z.hu, Z.hl) * inv_dx3;
          };
          double b3[3];
          // a wave without box particles does not enter the force's branch
          // (128^3 x 64 ppc, 20 steps with the force: 346 ms, so 324 ms)
          if (THRUST && __builtin_amdgcn_ballot_w64(box) != 0) {
            take_e();
            if (box) {
              double bp[3];
              take_b(F.bp, bp);
              th[0] += f[0];
              th[1] += f[1];
              th[2] += f[2];
              th[3] += vy * bp[2] - vz * bp[1];
              th[4] += vz * bp[0] - vx * bp[2];
              th[5] += vx * bp[1] - vy * bp[0];
            }
            // (kept apart from the push's: the compiler would otherwise form
            // the node weights once for both and hold them in 70 registers)
            asm("" : "+v"(X.iu), "+v"(X.il), "+v"(X.hu), "+v"(X.hl));
            if (push) take_b(F.b, b3);
          } else {
            take_e();
            take_b(F.b, b3);
          }
          if (push) {
            for (int q = 0; q < 3; ++q) f[3 + q] = b3[q];
            boris(kc, f, vx, vy, vz);
          }
        }
      }
      x += vx * kc.dt * 0.5;
      y += vy * kc.dt * 0.5;
      z += vz * kc.dt * 0.5;
    }
    if (PUSH_J) {
      // shape_func_*0_j_2 (:3397-3553) with the reference's weights
      const AxisW X = axis_weights(x, dx), Y = axis_weights(y, dx), Z = axis_weights(z, dx);
      const bool dep = dep_ok(g, x, y, z, X.bi, Y.bi, Z.bi);
      const bool in_lds = win_holds(w, X.bi, Y.bi, Z.bi);
      const double qn = kc.qn;
      if (dep && in_lds) {
        const int c = win_byte(w, X.bi, Y.bi, Z.bi);
        const int hx = X.bh != X.bi ? wsk : 0, hy = Y.bh != Y.bi ? wsl : 0,
                  hz = Z.bh != Z.bi ? 8 : 0;
        lds_dep8_64(acc + 0 * 8 * kWin64, c - hy - hz, wk, qn * vx, X.iu, X.il, Y.hu, Y.hl,
                    Z.hu, Z.hl);
        lds_dep8_64(acc + 1 * 8 * kWin64, c - hx - hz, wk, qn * vy, X.hu, X.hl, Y.iu, Y.il,
                    Z.hu, Z.hl);
        lds_dep8_64(acc + 2 * 8 * kWin64, c - hx - hy, wk, qn * vz, X.hu, X.hl, Y.hu, Y.hl,
                    Z.iu, Z.il);
      }
      glob_coop64(g, dep && !in_lds, true, dx, x, y, z, qn * vx, qn * vy, qn * vz, F.jx, F.jy,
                  F.jz, F.nd);
    }
    if (DRIFT_N) {
      x += vx * dth;
      y += vy * dth;
      z += vz * dth;
      // shape_func_*0_n_2 (:3333-3395)
      const AxisW X = axis_weights(x, dx), Y = axis_weights(y, dx), Z = axis_weights(z, dx);
      const bool dep = dep_ok(g, x, y, z, X.bi, Y.bi, Z.bi);
      const bool in_lds = win_holds(w, X.bi, Y.bi, Z.bi);
      const double wn = kc.wn;
      if (dep && in_lds) {
        const int c = win_byte(w, X.bi, Y.bi, Z.bi) - (X.bh != X.bi ? wsk : 0) -
                      (Y.bh != Y.bi ? wsl : 0) - (Z.bh != Z.bi ? 8 : 0);
        lds_dep8_64(acc + 3 * 8 * kWin64, c, wk, wn, X.hu, X.hl, Y.hu, Y.hl, Z.hu, Z.hl);
      }
      glob_coop64(g, dep && !in_lds, false, dx, x, y, z, wn, 0.0, 0.0, F.jx, F.jy, F.jz, F.nd);
    }
    if (BOUNDARY) {
      const bool dead = !bounded<UNIT>(g, dx, kc.periodic, x, y, z);
      if (dead) {
        *at(P.z, pb) = __longlong_as_double(0x7ff8000000000000LL);
        continue;
      }
    }
    *at(P.x, pb) = x;
    *at(P.y, pb) = y;
    *at(P.z, pb) = z;
    if (PUSH_J) {
      *at(P.vx, pb) = vx;
      *at(P.vy, pb) = vy;
      *at(P.vz, pb) = vz;
    }
  }
  if (THRUST) thrust_store64(th, thrust_part, bid);
  if (!w.on) return;
  __syncthreads();
  const int WYZ = w.WY * w.WZ;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    if (!PUSH_J && c < 3) continue;
    if (!DRIFT_N && c == 3) continue;
    double *dst = c == 0 ? F.jx : c == 1 ? F.jy : c == 2 ? F.jz : F.nd;
    for (int j = tid; j < WN; j += blockDim.x) {
      const double v = acc_mem[c * kWin64 + j];
      if (v == 0.0) continue;
      const int kk = w.k0 + j / WYZ, ll = w.l0 + (j / w.WZ) % w.WY,
                mm = w.m0 + j % w.WZ;
      if (kk < 0 || ll < 0 || mm < 0 || kk >= g.SX || ll >= g.SY || mm >= g.SZ)
        continue;
      glob_add64(dst + g.idx(kk, ll, mm), v);
    }
  }
}

// init_particle_flat (:412-625): particle p sits in interior cell p/ppc,
// cells in (k,l,m) order with m fastest; Philox event 0.
__global__ void k_load(Geom g, Particles64 P, int64_t n, int ppc, double dx,
                       double vth, double mu0, double mu1, double mu2,
                       uint64_t seed, int sp) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int64_t cell = i / ppc;
  const int m = (int)(cell % g.NZ);
  const int l = (int)((cell / g.NZ) % g.NY);
  const int k = (int)(cell / ((int64_t)g.NZ * g.NY));
  const ParticleDraw d = draw_particle(seed, sp, 0u, (uint64_t)i);
  P.x[i] = (k + 2) * dx + d.ux * dx;
  P.y[i] = (l + 2) * dx + d.uy * dx;
  P.z[i] = (m + 2) * dx + d.uz * dx;
  P.vx[i] = vth * d.n0 + mu0;
  P.vy[i] = vth * d.n1 + mu1;
  P.vz[i] = vth * d.n2 + mu2;
}

// add_*_flat refill (:6042-6104): batch index b = ((face*NX + k)*NY + l)*2*ppc
// + m*ppc + j, written after the survivors at offset base.
__global__ void k_refill(Geom g, Particles64 P, int64_t base, int64_t count,
                         int ppc, double dx, double vth, double mu0, double mu1,
                         double mu2, uint64_t seed, int sp, uint32_t event) {
  const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= count) return;
  const int64_t per_face = (int64_t)g.NX * g.NY * 2 * ppc;
  const int face = (int)(b / per_face);
  const int64_t r = b - face * per_face;
  const int m = (int)((r / ppc) % 2);
  const int l = (int)((r / (2 * ppc)) % g.NY);
  const int k = (int)(r / ((int64_t)2 * ppc * g.NY));
  const ParticleDraw d = draw_particle(seed, sp, event, (uint64_t)b);
  const double zlo = face == 0 ? (m + 2) * dx : (m + g.NZ) * dx;
  const int64_t o = base + b;
  P.x[o] = (k + 2) * dx + d.ux * dx;
  P.y[o] = (l + 2) * dx + d.uy * dx;
  P.z[o] = zlo + d.uz * dx;
  P.vx[o] = vth * d.n0 + mu0;
  P.vy[o] = vth * d.n1 + mu1;
  P.vz[o] = vth * d.n2 + mu2;
}

// inflow deletion flags (:6019-6021): keep live particles outside the slabs
__global__ void k_inflow_flags(const double *__restrict__ z, int64_t n,
                               double lo, double hi, uint8_t *flags) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double v = z[i];
  flags[i] = (!isnan(v) && !(v < lo || v > hi)) ? 1 : 0;
}

__global__ void k_live_flags(const double *__restrict__ z, int64_t n,
                             uint8_t *flags) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  flags[i] = isnan(z[i]) ? 0 : 1;
}

__global__ void k_gather_particles(Particles64 dst, Particles64 src,
                                   const uint32_t *__restrict__ idx,
                                   int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint32_t j = idx[i];
  dst.x[i] = src.x[j];
  dst.y[i] = src.y[j];
  dst.z[i] = src.z[j];
  dst.vx[i] = src.vx[j];
  dst.vy[i] = src.vy[j];
  dst.vz[i] = src.vz[j];
}

// sorting key (:7488-7497): ((int)(x/dx)-2, (int)(y/dx)-2, (int)(z/dx)-2),
// tile-major (the reference's lexicographic order with m fastest when one
// tile spans the interior); particles outside the interior (and dead ones)
// get the key ncell and are dropped after the sort.  zero (may be null): a
// word to clear for the kernels that follow.
__global__ __launch_bounds__(256) void k_sort_keys(Geom g, TileGeom tg,
                                                   Particles64 P, int64_t n,
                                                   double dx, uint32_t *keys,
                                                   uint32_t *zero) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  if (i == 0 && zero) *zero = 0;
  const uint32_t ncell = (uint32_t)g.NX * g.NY * g.NZ;
  uint32_t key = ncell;
  const double x = P.x[i], y = P.y[i], z = P.z[i];
  const double xd = x / dx, yd = y / dx, zd = z / dx;
  // range test before the conversions so that (int) never sees a value
  // outside int range or NaN
  if (xd > -1.0 && xd < g.NX + 3 && yd > -1.0 && yd < g.NY + 3 &&
      zd > -1.0 && zd < g.NZ + 3) {
    const int k = (int)(xd) - 2, l = (int)(yd) - 2, m = (int)(zd) - 2;
    if (k >= 0 && k < g.NX && l >= 0 && l < g.NY && m >= 0 && m < g.NZ)
      key = tg.key(k, l, m);
  }
  keys[i] = key;
}

__global__ __launch_bounds__(256) void k_count_live(
    const double *__restrict__ z, int64_t n, int64_t *count) {
  unsigned int t = 0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    t += !isnan(z[i]);
  for (int o = 32; o > 0; o >>= 1) t += __shfl_xor(t, o);
  __shared__ unsigned int part[kBlock / 64];
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = t;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long s = 0;
    for (int w = 0; w < kBlock / 64; ++w) s += part[w];
    if (s) atomicAdd((unsigned long long *)count, s);
  }
}

// ---------------------------------------------------------------------------
// diagnostics: per-block partial sums, summed on the host in block order

constexpr int kDiagField = 7;  // E2, B2, B1^2, charge, gauss^2, gauss max, -
constexpr int kDiagBox = 2;
constexpr int kDiagPart = 1 + 1 + 3 + 15 + 1;  // kin, kin_nr, mom, force, box

template <int NQ>
__device__ inline void block_reduce_store(double (&v)[NQ], double *out,
                                          const bool *is_max) {
  __shared__ double sh[NQ][kBlock / 64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    double a = v[q];
    for (int o = 32; o > 0; o >>= 1) {
      const double b = __shfl_xor(a, o);
      a = is_max[q] ? fmax(a, b) : a + b;
    }
    if (lane == 0) sh[q][w] = a;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      double a = sh[q][0];
      for (int j = 1; j < kBlock / 64; ++j)
        a = is_max[q] ? fmax(a, sh[q][j]) : a + sh[q][j];
      out[(int64_t)blockIdx.x * NQ + q] = a;
    }
  }
}

__global__ __launch_bounds__(256) void k_diag_fields(Geom g, Fields<double> F,
                                                     double dx, double eps0,
                                                     double mu0, double q,
                                                     double *out) {
  constexpr int NQ = kDiagField + kDiagBox;
  double v[NQ] = {0};
  const int64_t ncell = (int64_t)g.NX * g.NY * g.NZ;
  const double dx3 = dx * dx * dx;
  for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < ncell;
       t += (int64_t)gridDim.x * blockDim.x) {
    const int m = 2 + (int)(t % g.NZ);
    const int l = 2 + (int)((t / g.NZ) % g.NY);
    const int k = 2 + (int)(t / ((int64_t)g.NZ * g.NY));
    const int64_t c = g.idx(k, l, m);
    const int64_t dl = g.SZ, dk = (int64_t)g.SY * g.SZ;
    const double ex = F.f[PIC_EX][c], ey = F.f[PIC_EY][c], ez = F.f[PIC_EZ][c];
    const double bx = F.f[PIC_BX][c], by = F.f[PIC_BY][c], bz = F.f[PIC_BZ][c];
    const double b1x = bx - F.f[PIC_B0X][c], b1y = by - F.f[PIC_B0Y][c],
                 b1z = bz - F.f[PIC_B0Z][c];
    const double e2 = 0.5 * (ex * ex + ey * ey + ez * ez) * eps0;
    const double b2 = 0.5 * (bx * bx + by * by + bz * bz) / mu0;
    v[0] += e2 * dx3;
    v[1] += b2 * dx3;
    v[2] += 0.5 * (b1x * b1x + b1y * b1y + b1z * b1z) / mu0 * dx3;
    const double rho = F.f[PIC_NI][c] - F.f[PIC_NE][c];
    v[3] += q * rho * dx3;
    const double *Ex = F.f[PIC_EX], *Ey = F.f[PIC_EY], *Ez = F.f[PIC_EZ];
    const double r =
        -q * rho / eps0 +
        (-Ex[c + 2 * dk] + 27 * Ex[c + dk] - 27 * Ex[c] + Ex[c - dk] -
         Ey[c + 2 * dl] + 27 * Ey[c + dl] - 27 * Ey[c] + Ey[c - dl] -
         Ez[c + 2] + 27 * Ez[c + 1] - 27 * Ez[c] + Ez[c - 1]) /
            (24. * dx);
    v[4] += r * r;
    v[5] = fmax(v[5], fabs(r));
    if (k - 2 < g.NX * 0.8 && k - 2 > g.NX * 0.2 && l - 2 < g.NY * 0.8 &&
        l - 2 > g.NY * 0.2 && m - 2 < g.NZ * 0.8 && m - 2 > g.NZ * 0.2) {
      v[7] += e2;
      v[8] += b2;
    }
  }
  const bool is_max[NQ] = {false, false, false, false, false, true,
                           false, false, false};
  block_reduce_store<NQ>(v, out, is_max);
}

__global__ __launch_bounds__(256) void k_diag_particles(
    Geom g, Fields<double> F, Particles64 P, int64_t n, double dx, double c,
    double mass, double w, double qs, double *out) {
  constexpr int NQ = kDiagPart;
  double v[NQ] = {0};
  const double dx3 = dx * dx * dx;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const double z = P.z[i];
    if (isnan(z)) continue;
    const double x = P.x[i], y = P.y[i];
    const double vx = P.vx[i], vy = P.vy[i], vz = P.vz[i];
    const double v2 = vx * vx + vy * vy + vz * vz;
    const double gm = 1.0 / sqrt(1.0 - v2 / (c * c));
    v[0] += (gm - 1.0) * mass * c * c * w * dx3;
    v[1] += 0.5 * mass * w * dx3 * v2;
    v[2] += gm * mass * vx * w * dx3;
    v[3] += gm * mass * vy * w * dx3;
    v[4] += gm * mass * vz * w * dx3;
    if (x < g.NX * dx * 0.8 && x > g.NX * dx * 0.2 && y < g.NY * dx * 0.8 &&
        y > g.NY * dx * 0.2 && z < g.NZ * dx * 0.8 && z > g.NZ * dx * 0.2 &&
        in_array(g, x, y, z, dx)) {
      double f[6];
      gather(F, g, x, y, z, dx, f);
      const double qn = qs * w * dx3;
      v[5] += qn * (f[0] + vy * f[5] - vz * f[4]);
      v[6] += qn * (f[1] + vz * f[3] - vx * f[5]);
      v[7] += qn * (f[2] + vx * f[4] - vy * f[3]);
      v[8] += qn * f[0];
      v[9] += qn * f[1];
      v[10] += qn * f[2];
      v[11] += qn * (vy * f[5] - vz * f[4]);
      v[12] += qn * (vz * f[3] - vx * f[5]);
      v[13] += qn * (vx * f[4] - vy * f[3]);
      v[14 + 6] += 0.5 * mass * w * dx3 * v2;
    }
  }
  bool is_max[NQ];
  for (int q = 0; q < NQ; ++q) is_max[q] = false;
  block_reduce_store<NQ>(v, out, is_max);
}

// ---------------------------------------------------------------------------
// host side

static dim3 interior_grid(const Geom &g, dim3 &block) {
  block = dim3(64, 4, 1);
  return dim3((unsigned)div_up(g.NZ, 64), (unsigned)div_up(g.NY, 4),
              (unsigned)g.NX);
}

int renew_grid(pic_ctx *ctx) {
  Fields<double> F = fields<double>(ctx);
  // J (6 planes) and n (2 planes) are contiguous: PIC_JIX..PIC_NE
  const int64_t n = 8 * ctx->geom.plane;
  k_zero<<<2048, kBlock, 0, ctx->stream>>>(F.f[PIC_JIX], n);
  PIC_LAUNCH_CHECK(ctx);
  return 0;
}

static FieldConst field_const(const pic_ctx *ctx) {
  const pic_config &c = ctx->cfg;
  return FieldConst{c.dt, c.dx, c.eps0, c.mu0, c.c};
}

int renew_b_half(pic_ctx *ctx) {
  dim3 b, gr = interior_grid(ctx->geom, b);
  k_renew_b<<<gr, b, 0, ctx->stream>>>(ctx->geom, fields<double>(ctx),
                                       sigma(ctx), field_const(ctx));
  PIC_LAUNCH_CHECK(ctx);
  return 0;
}

int renew_e(pic_ctx *ctx) {
  dim3 b, gr = interior_grid(ctx->geom, b);
  k_renew_e<<<gr, b, 0, ctx->stream>>>(ctx->geom, fields<double>(ctx),
                                       sigma(ctx), field_const(ctx));
  PIC_LAUNCH_CHECK(ctx);
  return 0;
}

int halo(pic_ctx *ctx, int first) {
  const Geom &g = ctx->geom;
  k_halo<<<(unsigned)div_up((int64_t)fold_groups(g) * g.SZ, kBlock), kBlock, 0,
           ctx->stream>>>(g, fields<double>(ctx), first);
  PIC_LAUNCH_CHECK(ctx);
  return 0;
}

int fold_current(pic_ctx *ctx) {
  const Geom &g = ctx->geom;
  k_fold<<<(unsigned)div_up((int64_t)fold_groups(g) * g.SZ, kBlock), kBlock, 0,
           ctx->stream>>>(g, fields<double>(ctx));
  PIC_LAUNCH_CHECK(ctx);
  return 0;
}

int step_b1(pic_ctx *ctx, bool keep_b) {
  const Geom &g = ctx->geom;
  const CellBlocks cb(g);
  k_step_b1<<<block_grid(cb.count(g)), kBlock, 0, ctx->stream>>>(
      g, cb, fields<double>(ctx), keep_b ? (double *)ctx->thrust_bprev : nullptr, sigma(ctx),
      field_const(ctx));
  PIC_LAUNCH_CHECK(ctx);
  return 0;
}

int step_b2(pic_ctx *ctx) {
  const Geom &g = ctx->geom;
  const CellBlocks cb(g);
  const int tb = ctx->thrust_now ? 12 : 0;
  const int fb = (int)div_up((int64_t)fold_groups(g) * g.SZ, kBlock);
  k_step_b2<<<block_grid(tb + fb + cb.count(g)), kBlock, 0, ctx->stream>>>(
      g, cb, fields<double>(ctx), sigma(ctx), field_const(ctx), tb, thrust_finish_args(ctx), fb);
  PIC_LAUNCH_CHECK(ctx);
  return 0;
}

int step_e(pic_ctx *ctx) {
  const Geom &g = ctx->geom;
  const CellBlocks cb(g);
  k_step_e<<<block_grid(cb.count(g)), kBlock, 0, ctx->stream>>>(
      g, cb, fields<double>(ctx), sigma(ctx), field_const(ctx));
  PIC_LAUNCH_CHECK(ctx);
  return 0;
}

int load_particles(pic_ctx *ctx) {
  const pic_config &c = ctx->cfg;
  const int64_t n = (int64_t)c.nx * c.ny * c.nz * c.ppc;
  if (n > ctx->cap)
    return set_error(ctx, PIC_E_CAPACITY, "load: %lld particles > capacity %lld",
                     (long long)n, (long long)ctx->cap);
  for (int sp = 0; sp < 2; ++sp) {
    Particles64 P = p64(ctx, sp, ctx->cur[sp]);
    if (n > 0)
      k_load<<<(unsigned)div_up(n, kBlock), kBlock, 0, ctx->stream>>>(
          ctx->geom, P, n, c.ppc, c.dx, c.vth[sp], c.vdrift[0], c.vdrift[1],
          c.vdrift[2], c.seed, sp);
    ctx->n[sp] = n;
    ctx->sorted_end[sp] = 0;
  }
  PIC_LAUNCH_CHECK(ctx);
  // the loaded order is the reference's; bring it to tile order (the same
  // order when one tile spans the interior)
  for (int sp = 0; sp < 2; ++sp) {
    int rc = sort(ctx, sp);
    if (rc) return rc;
  }
  return 0;
}

// One species' arguments of a pass (push J / drift n / boundary); *nb is its
// number of workgroups, 0 when there is nothing to do.
static int prepare_pass(pic_ctx *ctx, int sp, int sel, SpeciesArgs64 &a, bool *rows,
                        unsigned *nb) {
  *nb = 0;
  const int64_t n = ctx->n[sp];
  if (n == 0) return 0;
  Fields<double> F = fields<double>(ctx);
  a.P = p64(ctx, sp, ctx->cur[sp]);
  const StepConst sc = step_const(ctx, sp);
  PassConst &kc = a.kc;
  {
    const double dx = sc.dx;
    kc.dx = dx;
    kc.dt = sc.dt;
    kc.dth = sc.dt * 0.5;
    kc.c = sc.c;
    kc.cc = sc.c * sc.c;
    kc.T = 0.5 * sc.q * sc.dt / sc.mass;
    kc.TT = kc.T * kc.T;
    kc.T2 = 2. * kc.T;
    kc.eimf_x = sc.vdrift_z * sc.imf_y;
    kc.eimf_y = -sc.vdrift_z * sc.imf_x;
    kc.qn = sc.q * sc.weight / (dx * dx * dx);
    kc.wn = sc.weight / (dx * dx * dx);
    const int N[3] = {ctx->geom.NX, ctx->geom.NY, ctx->geom.NZ};
    for (int x = 0; x < 3; ++x) {
      kc.blo[x] = sc.blo[x];
      kc.bhi[x] = sc.bhi[x];
      kc.box_lo[x] = N[x] * dx * 0.2;
      kc.box_hi[x] = N[x] * dx * 0.8;
    }
    kc.periodic[0] = sc.periodic[0];
    kc.periodic[1] = sc.periodic[1];
  }
  const double *kept = (const double *)ctx->thrust_bprev;
  for (int q = 0; q < 3; ++q) {
    a.F.e[q] = F.f[PIC_EX + q];
    a.F.b[q] = F.f[PIC_BX + q];
    a.F.bp[q] = kept + q * ctx->geom.plane;
  }
  a.F.jx = F.f[sp == PIC_ION ? PIC_JIX : PIC_JEX];
  a.F.jy = F.f[sp == PIC_ION ? PIC_JIY : PIC_JEY];
  a.F.jz = F.f[sp == PIC_ION ? PIC_JIZ : PIC_JEZ];
  a.F.nd = F.f[sp == PIC_ION ? PIC_NI : PIC_NE];
  TileGeom tg = tile_geom(ctx);
  add_drift_shift(tg, ctx->cfg, ctx->drift_halves[sp]);
  ctx->drift_halves[sp] += (sel & 4 ? 1 : 0) + (sel & 2 ? 1 : 0);
  TileRun tr;
  tr.tile_start = ctx->tile_start[sp];
  tr.sorted_end = ctx->sorted_end[sp];
  tr.ntiles = tr.sorted_end > 0 ? tg.ntiles() : 0;
  // a single tile (the reference's order): boxes of rows while the sort's
  // cell starts are current, otherwise chunks as an unsorted tail (slots of
  // the rows are 32-bit)
  *rows = tr.ntiles == 1 && ctx->row_start[sp] && ctx->row_end[sp] == tr.sorted_end &&
          n <= ((int64_t)1 << 30);
  if (*rows) {
    tg = row_geom(tg);
    tr.tile_start = ctx->row_start[sp];
    tr.ntiles = tg.ntiles();
  } else if (tr.ntiles == 1) {
    tr.ntiles = 0;
  }
  if (tr.ntiles == 0) tr.sorted_end = 0;
  tr.n = n;
  tr.chunk = tail_chunk(ctx->cfg.ppc, false, n - tr.sorted_end);
  tr.ntail = (int)div_up(n - tr.sorted_end, tr.chunk);
  tr.split = *rows || tr.ntiles == 0 ? 1 : pass_split(ctx);
  a.tg = tg;
  a.tr = tr;
  const unsigned blocks = (unsigned)(tr.parts() + tr.ntail);
  // the fused pass of pic_step adds the previous step's thrust_fave
  a.thrust_part = nullptr;
  if (ctx->thrust_now && sel == 7) {
    if ((int64_t)blocks > ctx->thrust_part_slots)
      return set_error(ctx, PIC_E_CAPACITY, "thrust: %u workgroups, %lld partial slots",
                       blocks, (long long)ctx->thrust_part_slots);
    a.thrust_part = ctx->thrust_part + (int64_t)sp * 6 * ctx->thrust_part_slots;
    ctx->thrust_nb[sp] = (int)blocks;  // finished by step_b2
  }
  *nb = blocks;
  return 0;
}

// the pass sel of one species (args.s[0], nb[1] = 0) or, fused, of both
static int launch_pass(pic_ctx *ctx, int sel, bool rows, const PassArgs64 &args,
                       const unsigned nb[2]) {
  const unsigned n = nb[0] + nb[1];
  if (n == 0) return 0;
  // normalised units with 32-bit byte offsets, or any dx with 64-bit ones
  const int64_t most = ctx->n[0] > ctx->n[1] ? ctx->n[0] : ctx->n[1];
  const bool unit = ctx->cfg.dx == 1.0 && most < ((int64_t)1 << 29) &&
                    ctx->geom.plane < ((int64_t)1 << 29);
#define F(ROWS, UNIT, BOTH)                                                           \
  (ctx->thrust_now ? k_particles_tiled<true, true, true, true, ROWS, UNIT, BOTH>      \
                   : k_particles_tiled<true, true, true, false, ROWS, UNIT, BOTH>)
#define L(ROWS, UNIT)                                                                 \
  (sel == 7 ? (nb[1] ? F(ROWS, UNIT, true) : F(ROWS, UNIT, false))                    \
   : sel == 4 ? k_particles_tiled<true, false, false, false, ROWS, UNIT, false>       \
              : k_particles_tiled<false, true, false, false, ROWS, UNIT, false>)
  const auto kern = unit ? (rows ? L(true, true) : L(false, true))
                         : (rows ? L(true, false) : L(false, false));
#undef L
#undef F
  kern<<<n, kBlock, 0, ctx->stream>>>(ctx->geom, args, (int)nb[0]);
  PIC_LAUNCH_CHECK(ctx);
  return 0;
}

// one routine's pass: push and J, or drift and n
int push(pic_ctx *ctx, int sp, bool drift) {
  const int sel = drift ? 2 : 4;
  PassArgs64 args;
  memset(&args, 0, sizeof args);
  bool rows = false;
  unsigned nb[2] = {0, 0};
  int rc = prepare_pass(ctx, sp, sel, args.s[0], &rows, &nb[0]);
  return rc ? rc : launch_pass(ctx, sel, rows, args, nb);
}

// The fused passes of both species, in one launch where both are in the same
// state (tiles, boxes or chunks) and leave places empty (kBothBlocks).
int push_both(pic_ctx *ctx) {
  PassArgs64 args;
  memset(&args, 0, sizeof args);
  bool rows[2] = {false, false};
  unsigned nb[2] = {0, 0};
  for (int sp = 0; sp < 2; ++sp) {
    int rc = prepare_pass(ctx, sp, 7, args.s[sp], &rows[sp], &nb[sp]);
    if (rc) return rc;
  }
  if (nb[0] && nb[1] && rows[0] == rows[1] && nb[0] + nb[1] < kBothBlocks) {
    timing_begin(ctx, PIC_T_PUSH);
    int rc = launch_pass(ctx, 7, rows[0], args, nb);
    timing_end(ctx, PIC_T_PUSH, 2);
    return rc;
  }
  for (int sp = 0; sp < 2; ++sp) {
    PassArgs64 one = args;
    one.s[0] = args.s[sp];
    const unsigned n[2] = {nb[sp], 0};
    timing_begin(ctx, PIC_T_PUSH);
    int rc = launch_pass(ctx, 7, rows[sp], one, n);
    timing_end(ctx, PIC_T_PUSH);
    if (rc) return rc;
  }
  return 0;
}

int particle_boundary(pic_ctx *ctx) {
  Bound64 b;
  int64_t nb[2];
  for (int sp = 0; sp < 2; ++sp) {
    b.P[sp] = p64(ctx, sp, ctx->cur[sp]);
    b.n[sp] = ctx->n[sp];
    b.periodic[sp] = ctx->cfg.periodic[sp];
    nb[sp] = div_up(ctx->n[sp], kBlock);
  }
  b.nb0 = (int)nb[0];
  if (nb[0] + nb[1] == 0) return 0;
  k_boundary<<<(unsigned)(nb[0] + nb[1]), kBlock, 0, ctx->stream>>>(ctx->geom, b, ctx->cfg.dx);
  PIC_LAUNCH_CHECK(ctx);
  return 0;
}

// Stable compaction of the current buffer into the other one through the
// flags already written to ctx->flags; returns the survivor count.
static int compact(pic_ctx *ctx, int sp, int64_t *kept) {
  const int64_t n = ctx->n[sp];
  int rc = select_flagged(ctx, ctx->flags, ctx->idx, n, kept);
  if (rc) return rc;
  Particles64 src = p64(ctx, sp, ctx->cur[sp]);
  Particles64 dst = p64(ctx, sp, 1 - ctx->cur[sp]);
  if (*kept > 0)
    k_gather_particles<<<(unsigned)div_up(*kept, kBlock), kBlock, 0,
                         ctx->stream>>>(dst, src, ctx->idx, *kept);
  PIC_LAUNCH_CHECK(ctx);
  ctx->cur[sp] = 1 - ctx->cur[sp];
  ctx->n[sp] = *kept;
  return 0;
}

// add_*_flat: slab particles become dead slots (z = NaN) in place and the
// refill is appended, so tile ranges stay valid until the next sort; the
// store is compacted first only when the refill would not fit
__global__ void k_inflow_kill(double *z, int64_t n, double lo, double hi) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double v = z[i];
  if (!isnan(v) && (v < lo || v > hi)) z[i] = __longlong_as_double(0x7ff8000000000000LL);
}

int inflow(pic_ctx *ctx, int sp, uint32_t event) {
  const pic_config &c = ctx->cfg;
  const Geom &g = ctx->geom;
  if (ctx->n[sp] > 0) {
    Particles64 P = p64(ctx, sp, ctx->cur[sp]);
    k_inflow_kill<<<(unsigned)div_up(ctx->n[sp], kBlock), kBlock, 0,
                    ctx->stream>>>(P.z, ctx->n[sp], 4 * c.dx, g.NZ * c.dx);
    PIC_LAUNCH_CHECK(ctx);
  }
  const int nface = c.refill_far ? 2 : 1;
  const int64_t add = (int64_t)g.NX * g.NY * 2 * c.ppc * nface;
  if (ctx->n[sp] + add > ctx->cap) {
    Particles64 P = p64(ctx, sp, ctx->cur[sp]);
    k_live_flags<<<(unsigned)div_up(ctx->n[sp], kBlock), kBlock, 0,
                   ctx->stream>>>(P.z, ctx->n[sp], ctx->flags);
    PIC_LAUNCH_CHECK(ctx);
    int64_t kept = 0;
    int rc = compact(ctx, sp, &kept);
    if (rc) return rc;
    ctx->sorted_end[sp] = 0;
  }
  if (ctx->n[sp] + add > ctx->cap)
    return set_error(ctx, PIC_E_CAPACITY,
                     "inflow: %lld + %lld particles exceed capacity %lld",
                     (long long)ctx->n[sp], (long long)add, (long long)ctx->cap);
  if (add > 0) {
    Particles64 P = p64(ctx, sp, ctx->cur[sp]);
    k_refill<<<(unsigned)div_up(add, kBlock), kBlock, 0, ctx->stream>>>(
        g, P, ctx->n[sp], add, c.ppc, c.dx, c.vth[sp], c.vdrift[0],
        c.vdrift[1], c.vdrift[2], c.seed, sp, event);
    PIC_LAUNCH_CHECK(ctx);
  }
  ctx->n[sp] += add;
  return 0;
}

// The tile sort's destination map of the FP64 form (pic_tsort.h): the
// particles carry no cell index, so the sort runs on the key array of
// k_sort_keys (tile * cells per tile + cell in the tile, or the drop key);
// the home slot is the tile coordinates modulo 4, as in the FP32 form.
struct KeyMapKey {
  TileGeom tg;
  uint32_t drop;  // tiles x cells per tile
  __host__ __device__ uint32_t cells() const { return (uint32_t)(tg.TX * tg.TY * tg.TZ); }
  __device__ bool dest(int32_t c, uint32_t &t, uint32_t &cin, int &h) const {
    const uint32_t key = (uint32_t)c;
    if (key >= drop) return false;
    t = tg.tile_of(key);
    cin = tg.cell_of(key);
    const uint32_t tz = t % (uint32_t)tg.NTZ, r = t / (uint32_t)tg.NTZ;
    const uint32_t ty = r % (uint32_t)tg.NTY, tx = r / (uint32_t)tg.NTY;
    h = (int)(((tx & 3u) << 4) | ((ty & 3u) << 2) | (tz & 3u));
    return true;
  }
};

int tsort_setup(pic_ctx *ctx) {
  const TileGeom tg = tile_geom(ctx);
  // (slots are 32-bit in the tile sort: larger stores take the radix sort)
  if (tg.ntiles() <= 1 || tg.TX * tg.TY * tg.TZ > tsort::kTileCells ||
      ctx->cap > ((int64_t)1 << 30))
    return 0;
  ctx->ts64 = new (std::nothrow) tsort::Bufs();
  if (!ctx->ts64) return set_error(ctx, PIC_E_NOMEM, "tile sort lists");
  return tsort::reserve(ctx, *ctx->ts64, tg.ntiles(), ctx->cap);
}

void tsort_free(pic_ctx *ctx) {
  if (!ctx->ts64) return;
  tsort::release(*ctx->ts64);
  delete ctx->ts64;
  ctx->ts64 = nullptr;
}

int sort(pic_ctx *ctx, int sp) {
  const Geom &g = ctx->geom;
  const int64_t n = ctx->n[sp];
  ctx->drift_halves[sp] = 0;
  if (n == 0) return 0;
  Particles64 src = p64(ctx, sp, ctx->cur[sp]);
  const TileGeom tg = tile_geom(ctx);
  const int nt = tg.ntiles();
  const TileGeom bg = row_geom(tg);
  const bool boxes = ctx->row_start[sp] && boxes_filled(n, bg.ntiles());
  k_sort_keys<<<(unsigned)div_up(n, kBlock), kBlock, 0, ctx->stream>>>(
      g, tg, src, n, ctx->cfg.dx, ctx->keys, boxes ? ctx->tile_start[sp] + nt + 1 : nullptr);
  PIC_LAUNCH_CHECK(ctx);
  const uint32_t ncell = (uint32_t)g.NX * g.NY * g.NZ;
  if (ctx->ts64 && ctx->sorted_end[sp] > 0 && ctx->sorted_end[sp] <= n) {
    // the tiles of the last sort are current: the tile sort of the keys
    const KeyMapKey km{tg, (uint32_t)nt * (uint32_t)(tg.TX * tg.TY * tg.TZ)};
    bool done = false;
    int64_t valid = 0;
    int rc = tsort::run(ctx, km, nt, ctx->tile_start[sp], ctx->sorted_end[sp], n,
                        (const int32_t *)ctx->keys, *ctx->ts64, ctx->idx, &done, &valid);
    if (rc) return rc;
    if (done) {
      Particles64 dst = p64(ctx, sp, 1 - ctx->cur[sp]);
      if (valid > 0)
        k_gather_particles<<<(unsigned)div_up(valid, kBlock), kBlock, 0, ctx->stream>>>(
            dst, src, ctx->idx, valid);
      PIC_LAUNCH_CHECK(ctx);
      ctx->cur[sp] = 1 - ctx->cur[sp];
      ctx->n[sp] = valid;
      ctx->sorted_end[sp] = valid;
      ctx->sort_tile_count++;
      return 0;
    }
  }
  ctx->sort_radix_count++;
  int bits = 1;
  while (bits < 32 && ((uint64_t)1 << bits) <= ncell) ++bits;
  int rc = sort_keys(ctx, ctx->keys, ctx->keys_alt, ctx->idx, n, bits);
  if (rc) return rc;
  rc = boxes ? cell_starts(ctx, ctx->keys_alt, n, bg, ctx->row_start[sp], ctx->tile_start[sp])
             : tile_bounds(ctx, ctx->keys_alt, n, (uint32_t)(tg.TX * tg.TY * tg.TZ), nt,
                           ctx->tile_start[sp]);
  if (rc) return rc;
  // the kept count is the start of the drop tile
  PIC_HIP(ctx, hipMemcpyAsync(ctx->host_counter, ctx->tile_start[sp] + nt,
                              2 * sizeof(uint32_t), hipMemcpyDeviceToHost,
                              ctx->stream));
  PIC_HIP(ctx, hipStreamSynchronize(ctx->stream));
  const int64_t valid = (int64_t)((uint32_t *)ctx->host_counter)[0];
  const int64_t most = (int64_t)((uint32_t *)ctx->host_counter)[1];
  Particles64 dst = p64(ctx, sp, 1 - ctx->cur[sp]);
  if (valid > 0)
    k_gather_particles<<<(unsigned)div_up(valid, kBlock), kBlock, 0,
                         ctx->stream>>>(dst, src, ctx->idx, valid);
  PIC_LAUNCH_CHECK(ctx);
  ctx->cur[sp] = 1 - ctx->cur[sp];
  ctx->n[sp] = valid;
  ctx->sorted_end[sp] = valid;
  ctx->row_end[sp] = boxes && boxes_even(valid, bg.ntiles(), most) ? valid : 0;
  return 0;
}

int count_live(pic_ctx *ctx, int sp, int64_t *out) {
  const int64_t n = ctx->n[sp];
  *out = 0;
  if (n == 0) return 0;
  Particles64 P = p64(ctx, sp, ctx->cur[sp]);
  PIC_HIP(ctx, hipMemsetAsync(ctx->dev_counter, 0, sizeof(int64_t), ctx->stream));
  k_count_live<<<(unsigned)(div_up(n, kBlock) < 2048 ? div_up(n, kBlock) : 2048),
                 kBlock, 0, ctx->stream>>>(P.z, n, ctx->dev_counter);
  PIC_LAUNCH_CHECK(ctx);
  PIC_HIP(ctx, hipMemcpyAsync(ctx->host_counter, ctx->dev_counter,
                              sizeof(int64_t), hipMemcpyDeviceToHost,
                              ctx->stream));
  PIC_HIP(ctx, hipStreamSynchronize(ctx->stream));
  *out = ctx->host_counter[0];
  return 0;
}

static_assert(kDiagField + kDiagBox == kDiagNQF && kDiagPart == kDiagNQP,
              "diagnostics layout");

int diagnose_partials(pic_ctx *ctx, double *pf, unsigned long long *counts) {
  const pic_config &c = ctx->cfg;
  const Geom &g = ctx->geom;
  Fields<double> F = fields<double>(ctx);
  double *pp[2] = {pf + (int64_t)kDiagNBF * kDiagNQF,
                   pf + (int64_t)kDiagNBF * kDiagNQF + (int64_t)kDiagNBP * kDiagNQP};
  k_diag_fields<<<kDiagNBF, kBlock, 0, ctx->stream>>>(g, F, c.dx, c.eps0, c.mu0,
                                                      c.q, pf);
  PIC_LAUNCH_CHECK(ctx);
  for (int sp = 0; sp < 2; ++sp) {
    Particles64 P = p64(ctx, sp, ctx->cur[sp]);
    k_diag_particles<<<kDiagNBP, kBlock, 0, ctx->stream>>>(
        g, F, P, ctx->n[sp], c.dx, c.c, c.mass[sp], c.weight[sp],
        sp == PIC_ION ? c.q : -c.q, pp[sp]);
    PIC_LAUNCH_CHECK(ctx);
    if (counts && ctx->n[sp] > 0) {
      k_count_live<<<(unsigned)(div_up(ctx->n[sp], kBlock) < 2048
                                    ? div_up(ctx->n[sp], kBlock) : 2048),
                     kBlock, 0, ctx->stream>>>(P.z, ctx->n[sp],
                                               (int64_t *)(counts + sp));
      PIC_LAUNCH_CHECK(ctx);
    }
  }
  return 0;
}

int diagnose(pic_ctx *ctx, pic_diag *out) {
  const int nbf = kDiagNBF, nbp = kDiagNBP;
  constexpr int NQF = kDiagNQF, NQP = kDiagNQP;
  const int64_t need = kDiagPartials;
  if (ctx->diag_partial_cap < need) {
    if (ctx->diag_partial) (void)hipFree(ctx->diag_partial);
    ctx->diag_partial = nullptr;
    PIC_HIP(ctx, device_malloc(ctx, &ctx->diag_partial, need * sizeof(double)));
    ctx->diag_partial_cap = need;
  }
  double *pf = ctx->diag_partial;
  double *pp[2] = {pf + (int64_t)nbf * NQF, pf + (int64_t)nbf * NQF + (int64_t)nbp * NQP};
  int rc0 = diagnose_partials(ctx, pf, nullptr);
  if (rc0) return rc0;
  double *h = (double *)malloc(need * sizeof(double));
  if (!h) return set_error(ctx, PIC_E_NOMEM, "diagnose: host buffer");
  hipError_t e = hipMemcpyAsync(h, pf, need * sizeof(double),
                                hipMemcpyDeviceToHost, ctx->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
  if (e != hipSuccess) {
    free(h);
    return set_error(ctx, PIC_E_HIP, "diagnose: %s", hipGetErrorString(e));
  }
  memset(out, 0, sizeof(*out));
  double s[NQF] = {0};
  for (int b = 0; b < nbf; ++b)
    for (int q = 0; q < NQF; ++q) {
      const double v = h[(int64_t)b * NQF + q];
      s[q] = q == 5 ? fmax(s[q], v) : s[q] + v;
    }
  out->field_energy_e = s[0];
  out->field_energy_b = s[1];
  out->field_energy_b1 = s[2];
  out->charge = s[3];
  out->gauss_l2 = sqrt(s[4]);
  out->gauss_max = s[5];
  out->energy_box[0] = s[7];
  out->energy_box[1] = s[8];
  for (int sp = 0; sp < 2; ++sp) {
    double t[NQP] = {0};
    const double *hp = h + (pp[sp] - pf);
    for (int b = 0; b < nbp; ++b)
      for (int q = 0; q < NQP; ++q) t[q] += hp[(int64_t)b * NQP + q];
    out->kinetic[sp] = t[0];
    out->kinetic_nr[sp] = t[1];
    out->momentum[sp][0] = t[2];
    out->momentum[sp][1] = t[3];
    out->momentum[sp][2] = t[4];
    for (int j = 0; j < 3; ++j) out->force[j] += t[5 + j];
    const int b0 = sp == PIC_ION ? 3 : 9;
    for (int j = 0; j < 6; ++j) out->force[b0 + j] = t[8 + j];
    out->energy_box[2 + sp] = t[20];
  }
  free(h);
  for (int sp = 0; sp < 2; ++sp) {
    int rc = count_live(ctx, sp, &out->count[sp]);
    if (rc) return rc;
  }
  return 0;
}

}  // namespace f64
}  // namespace pic
