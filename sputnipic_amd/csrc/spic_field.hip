// spic_field.hip -- the field-solve side that consumes the deposit, on the
// device and in FP64 (the field solve stays in the reference's FP64):
//   ghost updates of scalar arrays   applyBCscalarDensN / FieldNzero / DensC /
//                                    FieldC (src/BC.cpp:11-123, 242-352,
//                                    623-735, 737-850)
//   net rhoc from the net rhon       src/sputniPIC_CPU.cpp:276-277
//                                    (applyBCscalarDensN + interpN2Cinterp,
//                                    src/Grid.cpp:164-185)
//   hat densities                    calculateHatDensities
//                                    (src/MaxwellSolver.cpp:465-604)
//   implicit field operator          MaxwellImage (src/MaxwellSolver.cpp:95-257)
// This file is compiled without FMA contraction and keeps the reference's
// operation order in every expression, so results are bit-identical to the
// reference's FP64 build.  Volume work is one thread per interior node or
// cell; where the reference makes a temporary array and then transforms it
// (scale, interpolate, add, negate, scale, sum), the transform is applied
// in the kernel that produces the value, in the same order.
#include <hip/hip_runtime.h>

#include "spic.h"
#include "spic_binned.hpp"
#include "spic_internal.hpp"

namespace spic {
namespace {

// Ghost updates, the reference's sequence (periodic faces x, y, z; edges
// along x, y, z; corners; non-periodic faces x, y, z, copied from the
// adjacent plane or zeroed) in two launches with the same result:
//  * k_bc_periodic: the periodic faces, edges and corners.  A node array
//    takes its ghosts from planes n-3 and 2, a cell array from n-2 and 1.
//    Every element these steps read is interior and no two steps write the
//    same element, so they run together.  The reference runs the y-edge
//    loop to the node count (j < nyn - 1), which for a cell array also
//    writes the four corners at j = nyc - 1; the corner step, which runs
//    whenever the y-edge step does, overwrites those, so they are skipped.
//  * k_bc_faces: the non-periodic faces.  Applied in x, y, z order, the
//    plane copies leave at every element with a ghost index on a
//    non-periodic axis the value of the element with those indices moved
//    one plane inward (clamped), read after the periodic steps; zeroed
//    faces leave zero there.
__global__ void k_bc_periodic(double *arr, int n0, int n1, int n2, int nyn, int nodes,
                              int px, int py, int pz) {
  SPIC_GLOBAL double *a = gmem(arr);
  const int lo = nodes ? 3 : 2, hi = nodes ? 2 : 1;
#define A(i, j, k) a[((int64_t)(i) * n1 + (j)) * n2 + (k)]
  const int64_t fx = px ? (int64_t)(n1 - 2) * (n2 - 2) : 0;
  const int64_t fy = py ? (int64_t)(n0 - 2) * (n2 - 2) : 0;
  const int64_t fz = pz ? (int64_t)(n0 - 2) * (n1 - 2) : 0;
  const int64_t ex = (py || pz) ? n0 - 2 : 0;
  // y-edge rows j = 1 .. nyn - 2, without the cell corner row j = n1 - 1
  const int yend = nyn - 1 < n1 - 1 ? nyn - 1 : n1 - 1;
  const int64_t ey = (px || pz) ? yend - 1 : 0;
  const int64_t ez = (px || py) ? n2 - 2 : 0;
  const int64_t co = (px || py || pz) ? 1 : 0;
  const int64_t total = fx + fy + fz + ex + ey + ez + co;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total;
       e += (int64_t)gridDim.x * blockDim.x) {
    int64_t r = e;
    if (r < fx) {
      const int j = 1 + (int)(r / (n2 - 2)), k = 1 + (int)(r % (n2 - 2));
      A(0, j, k) = A(n0 - lo, j, k);
      A(n0 - 1, j, k) = A(hi, j, k);
      continue;
    }
    r -= fx;
    if (r < fy) {
      const int i = 1 + (int)(r / (n2 - 2)), k = 1 + (int)(r % (n2 - 2));
      A(i, 0, k) = A(i, n1 - lo, k);
      A(i, n1 - 1, k) = A(i, hi, k);
      continue;
    }
    r -= fy;
    if (r < fz) {
      const int i = 1 + (int)(r / (n1 - 2)), j = 1 + (int)(r % (n1 - 2));
      A(i, j, 0) = A(i, j, n2 - lo);
      A(i, j, n2 - 1) = A(i, j, hi);
      continue;
    }
    r -= fz;
    if (r < ex) {
      const int i = 1 + (int)r;
      A(i, n1 - 1, n2 - 1) = A(i, hi, hi);
      A(i, 0, 0) = A(i, n1 - lo, n2 - lo);
      A(i, 0, n2 - 1) = A(i, n1 - lo, hi);
      A(i, n1 - 1, 0) = A(i, hi, n2 - lo);
      continue;
    }
    r -= ex;
    if (r < ey) {
      const int j = 1 + (int)r;
      A(n0 - 1, j, n2 - 1) = A(hi, j, hi);
      A(0, j, 0) = A(n0 - lo, j, n2 - lo);
      A(0, j, n2 - 1) = A(n0 - lo, j, hi);
      A(n0 - 1, j, 0) = A(hi, j, n2 - lo);
      continue;
    }
    r -= ey;
    if (r < ez) {
      const int k = 1 + (int)r;
      A(n0 - 1, n1 - 1, k) = A(hi, hi, k);
      A(0, 0, k) = A(n0 - lo, n1 - lo, k);
      A(n0 - 1, 0, k) = A(hi, n1 - lo, k);
      A(0, n1 - 1, k) = A(n0 - lo, hi, k);
      continue;
    }
    A(n0 - 1, n1 - 1, n2 - 1) = A(hi, hi, hi);
    A(0, n1 - 1, n2 - 1) = A(n0 - lo, hi, hi);
    A(n0 - 1, 0, n2 - 1) = A(hi, n1 - lo, hi);
    A(0, 0, n2 - 1) = A(n0 - lo, n1 - lo, hi);
    A(n0 - 1, n1 - 1, 0) = A(hi, hi, n2 - lo);
    A(0, n1 - 1, 0) = A(n0 - lo, hi, n2 - lo);
    A(n0 - 1, 0, 0) = A(hi, n1 - lo, n2 - lo);
    A(0, 0, 0) = A(n0 - lo, n1 - lo, n2 - lo);
  }
}

// Index moved one plane inward if it is a ghost of a non-periodic axis.
__device__ __forceinline__ int clamp_ghost(int v, int n, int periodic) {
  if (periodic) return v;
  return v == 0 ? 1 : (v == n - 1 ? n - 2 : v);
}

// Every element on the ghost planes of the non-periodic axes (an element
// on two such planes is visited twice and written the same value twice).
__global__ void k_bc_faces(double *arr, int n0, int n1, int n2, int zero_faces, int px,
                           int py, int pz) {
  SPIC_GLOBAL double *a = gmem(arr);
  const int64_t sx = px ? 0 : 2 * (int64_t)n1 * n2;
  const int64_t sy = py ? 0 : 2 * (int64_t)n0 * n2;
  const int64_t sz = pz ? 0 : 2 * (int64_t)n0 * n1;
  const int64_t total = sx + sy + sz;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total;
       e += (int64_t)gridDim.x * blockDim.x) {
    int i, j, k;
    int64_t r = e;
    if (r < sx) {
      const int64_t plane = (int64_t)n1 * n2;
      i = r < plane ? 0 : n0 - 1;
      r %= plane;
      j = (int)(r / n2);
      k = (int)(r % n2);
    } else if ((r -= sx) < sy) {
      const int64_t plane = (int64_t)n0 * n2;
      j = r < plane ? 0 : n1 - 1;
      r %= plane;
      i = (int)(r / n2);
      k = (int)(r % n2);
    } else {
      r -= sy;
      const int64_t plane = (int64_t)n0 * n1;
      k = r < plane ? 0 : n2 - 1;
      r %= plane;
      i = (int)(r / n1);
      j = (int)(r % n1);
    }
    A(i, j, k) = zero_faces ? 0.0
                            : A(clamp_ghost(i, n0, px), clamp_ghost(j, n1, py),
                                clamp_ghost(k, n2, pz));
  }
#undef A
}

// Interior point (i, j, k) of an n0 x n1 x n2 array for thread index t
// (t < (n0 - 2)(n1 - 2)(n2 - 2)).
__device__ __forceinline__ void interior(int64_t t, int n1, int n2, int &i, int &j, int &k) {
  const int m1 = n1 - 2, m2 = n2 - 2;
  k = 1 + (int)(t % m2);
  j = 1 + (int)((t / m2) % m1);
  i = 1 + (int)(t / ((int64_t)m2 * m1));
}

// Stencil kernels work on runs of neighbouring blocks per die: consecutive
// workgroups go to the eight dies in turn, each with an L2 of its own, so
// workgroup b of 8 r takes block (b % 8) r + b / 8.  On 128x64x64 cells one
// application of the Maxwell operator takes 32 us instead of 36.
constexpr unsigned kXcds = 8;

inline unsigned xcd_grid(int64_t blocks) {
  return (unsigned)((blocks + kXcds - 1) / kXcds * kXcds);
}
__device__ __forceinline__ unsigned xcd_block() {
  return (blockIdx.x % kXcds) * (gridDim.x / kXcds) + blockIdx.x / kXcds;
}

// The interior index whose value a ghost index takes, per axis (the ghost
// updates above as a map): periodic axes wrap, the others take the plane
// inside.  A ghost on several axes takes the element with every one mapped.
struct GhostMap {
  int lo[3], hi[3];  // source of index 0 and of index n - 1
};

inline GhostMap ghost_map(int n0, int n1, int n2, bool nodes, const spic_solve_params *p) {
  const int n[3] = {n0, n1, n2};
  const bool per[3] = {p->PERIODICX != 0, p->PERIODICY != 0, p->PERIODICZ != 0};
  GhostMap g;
  for (int a = 0; a < 3; ++a) {
    g.lo[a] = per[a] ? n[a] - (nodes ? 3 : 2) : 1;
    g.hi[a] = per[a] ? (nodes ? 2 : 1) : n[a] - 2;
  }
  return g;
}

__device__ __forceinline__ int ghost_src(int v, int n, int lo, int hi) {
  return v == 0 ? lo : (v == n - 1 ? hi : v);
}

// Stores v, the value of interior element (i, j, k), to the ghosts that take
// it, and with SELF to the element itself.  Every ghost has one source, so
// one pass over the interior writes a whole array.
template <bool SELF>
__device__ __forceinline__ void put_ghosts(SPIC_GLOBAL double *a, int n0, int n1, int n2,
                                           const GhostMap &g, int i, int j, int k, double v) {
  if (SELF) a[((int64_t)i * n1 + j) * n2 + k] = v;
  const bool any = i == g.lo[0] || i == g.hi[0] || j == g.lo[1] || j == g.hi[1] ||
                   k == g.lo[2] || k == g.hi[2];
  if (!any) return;
  for (int ti = 0; ti < 3; ++ti) {
    if ((ti == 1 && i != g.lo[0]) || (ti == 2 && i != g.hi[0])) continue;
    const int gi = ti == 0 ? i : (ti == 1 ? 0 : n0 - 1);
    for (int tj = 0; tj < 3; ++tj) {
      if ((tj == 1 && j != g.lo[1]) || (tj == 2 && j != g.hi[1])) continue;
      const int gj = tj == 0 ? j : (tj == 1 ? 0 : n1 - 1);
      for (int tk = 0; tk < 3; ++tk) {
        if ((tk == 1 && k != g.lo[2]) || (tk == 2 && k != g.hi[2])) continue;
        if (ti == 0 && tj == 0 && tk == 0) continue;
        const int gk = tk == 0 ? k : (tk == 1 ? 0 : n2 - 1);
        a[((int64_t)gi * n1 + gj) * n2 + gk] = v;
      }
    }
  }
}

struct Dims {
  int nxn, nyn, nzn, nxc, nyc, nzc;
  int64_t nn, nc;
  int64_t in_nodes, in_cells;  // interior counts
};

inline Dims dims_of(const spic_grid *g) {
  Dims d;
  d.nxn = g->nxn; d.nyn = g->nyn; d.nzn = g->nzn;
  d.nxc = g->nxc; d.nyc = g->nyc; d.nzc = g->nzc;
  d.nn = (int64_t)d.nxn * d.nyn * d.nzn;
  d.nc = (int64_t)d.nxc * d.nyc * d.nzc;
  d.in_nodes = (int64_t)(d.nxn - 2) * (d.nyn - 2) * (d.nzn - 2);
  d.in_cells = (int64_t)(d.nxc - 2) * (d.nyc - 2) * (d.nzc - 2);
  return d;
}

#define NIDX(i, j, k) (((int64_t)(i) * d.nyn + (j)) * d.nzn + (k))
#define CIDX(i, j, k) (((int64_t)(i) * d.nyc + (j)) * d.nzc + (k))

// applyBCscalarDensN of rhon (its ghosts, from its interior) and
// interpN2Cinterp (src/Grid.cpp:164-185) on the interior cells, which read
// interior nodes only: one thread per interior node, one launch where the
// ghost updates took two before it.
__global__ void k_rhoc(Dims d, GhostMap g, double *rhon, double *__restrict__ rhoc) {
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (t >= d.in_nodes) return;
  int i, j, k;
  interior(t, d.nyn, d.nzn, i, j, k);
  SPIC_GLOBAL double *n = gmem(rhon);
  put_ghosts<false>(n, d.nxn, d.nyn, d.nzn, g, i, j, k, n[NIDX(i, j, k)]);
  if (i > d.nxc - 2 || j > d.nyc - 2 || k > d.nzc - 2) return;
  gmem(rhoc)[CIDX(i, j, k)] =
      .125 * (n[NIDX(i, j, k)] + n[NIDX(i + 1, j, k)] + n[NIDX(i, j + 1, k)] +
              n[NIDX(i, j, k + 1)] + n[NIDX(i + 1, j + 1, k)] + n[NIDX(i + 1, j, k + 1)] +
              n[NIDX(i, j + 1, k + 1)] + n[NIDX(i + 1, j + 1, k + 1)]);
}

// .25 * (a - b) * inv, one term of the reference's divergence stencils, with
// inv4 = .25 * inv: a factor of a power of two commutes with the rounding, so
// the value is the same as long as nothing underflows.  Multiplying by .25
// here becomes a v_ldexp_f64 per term (36 per cell and species in k_divsymm).
__device__ __forceinline__ double q4(double a, double b, double inv4) {
  return (a - b) * inv4;
}

// Difference quotients of an array at the cell whose lower node is element o
// (strides si, sj, 1): along x the nodes (i+1, ., .) against (i, ., .) over
// the corners (j,k), (j,k+1), (j+1,k), (j+1,k+1); y and z alike, in the
// reference's order (src/Grid.cpp:267-398).
template <typename A>
__device__ __forceinline__ double diff_x(const A &a, int64_t o, int64_t si, int64_t sj, double inv4) {
  return q4(a[o + si], a[o], inv4) + q4(a[o + si + 1], a[o + 1], inv4) +
         q4(a[o + si + sj], a[o + sj], inv4) + q4(a[o + si + sj + 1], a[o + sj + 1], inv4);
}
template <typename A>
__device__ __forceinline__ double diff_y(const A &a, int64_t o, int64_t si, int64_t sj, double inv4) {
  return q4(a[o + sj], a[o], inv4) + q4(a[o + sj + 1], a[o + 1], inv4) +
         q4(a[o + si + sj], a[o + si], inv4) + q4(a[o + si + sj + 1], a[o + si + 1], inv4);
}
template <typename A>
__device__ __forceinline__ double diff_z(const A &a, int64_t o, int64_t si, int64_t sj, double inv4) {
  return q4(a[o + 1], a[o], inv4) + q4(a[o + si + 1], a[o + si], inv4) +
         q4(a[o + sj + 1], a[o + sj], inv4) + q4(a[o + si + sj + 1], a[o + si + sj], inv4);
}

// divSymmTensorN2C (src/Grid.cpp:322-398) at one cell, then scaled by
// alfa = -dt/2 (src/MaxwellSolver.cpp:518-520); P: pxx pxy pxz pyy pyz pzz.
template <typename A>
__device__ __forceinline__ void div_symm(const A (&P)[6], int64_t o, int64_t si, int64_t sj,
                                         double invdx, double invdy, double invdz, double alfa,
                                         double out[3]) {
  const double c1X = diff_x(P[0], o, si, sj, invdx), c2X = diff_x(P[1], o, si, sj, invdx),
               c3X = diff_x(P[2], o, si, sj, invdx);
  const double c1Y = diff_y(P[1], o, si, sj, invdy), c2Y = diff_y(P[3], o, si, sj, invdy),
               c3Y = diff_y(P[4], o, si, sj, invdy);
  const double c1Z = diff_z(P[2], o, si, sj, invdz), c2Z = diff_z(P[4], o, si, sj, invdz),
               c3Z = diff_z(P[5], o, si, sj, invdz);
  out[0] = (c1X + c1Y + c1Z) * alfa;
  out[1] = (c2X + c2Y + c2Z) * alfa;
  out[2] = (c3X + c3Y + c3Z) * alfa;
}

// Workgroup tiles of the image's first kernel: FX x 4 x 16 cells.
constexpr int kFY = 4, kFZ = 16;
// One thread per node of the tile, in whole waves.
template <int FX>
constexpr int kFieldThreads = ((FX + 1) * (kFY + 1) * (kFZ + 1) + 63) / 64 * 64;

struct Tiles {
  int ny, nz;  // tiles per axis
  unsigned total;
  unsigned first = 0, end = 0;  // of one launch
};
// Tiles per launch: a thin grid has tiles that are mostly empty, and a launch fewer
// than 2^32 threads.
constexpr unsigned kMaxTiles = 1u << 16;

inline Tiles tiles_of(int fx, int n0, int n1, int n2) {
  Tiles t;
  t.ny = (n1 + kFY - 1) / kFY;
  t.nz = (n2 + kFZ - 1) / kFZ;
  t.total = (unsigned)((n0 + fx - 1) / fx * t.ny * t.nz);
  return t;
}

struct HatArgs {
  const double *P[6 * kMaxSpecies];  // pxx pxy pxz pyy pyz pzz, nodes
  const double *J[3 * kMaxSpecies];  // species currents Jx Jy Jz, nodes
  double *tc[3 * kMaxSpecies];       // scaled tensor divergence, interior cells
  double beta[kMaxSpecies];          // .5 * qom * dt / c
  const double *Bx, *By, *Bz;
  double *Jh[3];
  int ns;
};

// The scaled tensor divergence on the interior cells; blockIdx.y is the
// species, blockIdx.z a run of `planes` cell planes.  A thread walks along x
// and keeps the upper plane's four nodes of the six components for the next
// cell: 24 loads per cell instead of 48 (49 us against 60 on 128x64x64 cells
// and four species).
__global__ __launch_bounds__(256) void k_divsymm(Dims d, HatArgs a, int planes, double invdx,
                                                 double invdy, double invdz, double alfa) {
  const int ny = d.nyc - 2, nz = d.nzc - 2;
  const int t = blockIdx.x * 256 + threadIdx.x;
  if (t >= ny * nz) return;
  const int j = 1 + t / nz, k = 1 + t % nz;
  const int i0 = 1 + blockIdx.z * planes, i1 = min(i0 + planes, d.nxc - 1);
  const int s = blockIdx.y;
  // element (di, dj, dk) of a cell's eight nodes at 4 di + 2 dj + dk
  double P[6][8];
  const int64_t plane = (int64_t)d.nyn * d.nzn;
  int64_t n = NIDX(i0, j, k), c = CIDX(i0, j, k);
#pragma unroll
  for (int q = 0; q < 6; ++q) {
    const SPIC_GLOBAL double *p = gmem(a.P[6 * s + q]) + n;
    P[q][4] = p[0]; P[q][5] = p[1]; P[q][6] = p[d.nzn]; P[q][7] = p[d.nzn + 1];
  }
  for (int i = i0; i < i1; ++i) {
    n += plane;
#pragma unroll
    for (int q = 0; q < 6; ++q) {
      const SPIC_GLOBAL double *p = gmem(a.P[6 * s + q]) + n;
#pragma unroll
      for (int e = 0; e < 4; ++e) P[q][e] = P[q][4 + e];
      P[q][4] = p[0]; P[q][5] = p[1]; P[q][6] = p[d.nzn]; P[q][7] = p[d.nzn + 1];
    }
    double out[3];
    div_symm(P, 0, 4, 2, invdx, invdy, invdz, alfa, out);
#pragma unroll
    for (int m = 0; m < 3; ++m) gmem(a.tc[3 * s + m])[c] = out[m];
    c += (int64_t)d.nyc * d.nzc;
  }
}

// The hat current with its ghosts: per interior node, species in order,
// interpC2Ninterp of the three divergences (src/Grid.cpp:122-141), their ghost
// cells read at their sources (applyBCscalarDensC), plus the species current,
// then the PIdot update (src/MaxwellSolver.cpp:531-566); the hat current starts
// at zero, as the reference zeroes it.  One kernel for both steps, the tensors
// staged in LDS per 4x4x16 tile, was slower (135-146 us against 98 for the two
// on 128x64x64 cells and four species): 1.7 cells formed per node and three
// workgroups per CU.
__global__ __launch_bounds__(256) void k_pidot(Dims d, HatArgs a, GhostMap gc, GhostMap gn) {
  const int64_t t = xcd_block() * (int64_t)blockDim.x + threadIdx.x;
  if (t >= d.in_nodes) return;
  int i, j, k;
  interior(t, d.nyn, d.nzn, i, j, k);
  const int64_t n = NIDX(i, j, k);
  const int ci[2] = {ghost_src(i - 1, d.nxc, gc.lo[0], gc.hi[0]),
                     ghost_src(i, d.nxc, gc.lo[0], gc.hi[0])};
  const int cj[2] = {ghost_src(j - 1, d.nyc, gc.lo[1], gc.hi[1]),
                     ghost_src(j, d.nyc, gc.lo[1], gc.hi[1])};
  const int ck[2] = {ghost_src(k - 1, d.nzc, gc.lo[2], gc.hi[2]),
                     ghost_src(k, d.nzc, gc.lo[2], gc.hi[2])};
  const double bx = gmem(a.Bx)[n], by = gmem(a.By)[n], bz = gmem(a.Bz)[n];
  double hx = 0.0, hy = 0.0, hz = 0.0;
  for (int s = 0; s < a.ns; ++s) {
    double tn[3];
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      const SPIC_GLOBAL double *c = gmem(a.tc[3 * s + m]);
#define TC(x, y, z) c[CIDX(ci[1 - x], cj[1 - y], ck[1 - z])]
      tn[m] = .125 * (TC(0, 0, 0) + TC(1, 0, 0) + TC(0, 1, 0) + TC(0, 0, 1) + TC(1, 1, 0) +
                      TC(1, 0, 1) + TC(0, 1, 1) + TC(1, 1, 1));
#undef TC
      tn[m] += gmem(a.J[3 * s + m])[n];
    }
    const double beta = a.beta[s];
    const double omcx = beta * bx, omcy = beta * by, omcz = beta * bz;
    const double edotb = tn[0] * omcx + tn[1] * omcy + tn[2] * omcz;
    const double denom = 1 / (1.0 + omcx * omcx + omcy * omcy + omcz * omcz);
    hx += (tn[0] + (tn[1] * omcz - tn[2] * omcy + edotb * omcx)) * denom;
    hy += (tn[1] + (tn[2] * omcx - tn[0] * omcz + edotb * omcy)) * denom;
    hz += (tn[2] + (tn[0] * omcy - tn[1] * omcx + edotb * omcz)) * denom;
  }
  put_ghosts<true>(gmem(a.Jh[0]), d.nxn, d.nyn, d.nzn, gn, i, j, k, hx);
  put_ghosts<true>(gmem(a.Jh[1]), d.nxn, d.nyn, d.nzn, gn, i, j, k, hy);
  put_ghosts<true>(gmem(a.Jh[2]), d.nxn, d.nyn, d.nzn, gn, i, j, k, hz);
}

// rhoh = rhoc - dt * th * divN2C(Jh) (src/MaxwellSolver.cpp:586-596, divN2C:
// src/Grid.cpp:267-319) on the interior cells, which read interior nodes
// only, and its ghosts.
__global__ void k_rhoh(Dims d, GhostMap g, const double *Jx, const double *Jy, const double *Jz,
                       const double *rhoc, double *rhoh, double invdx, double invdy,
                       double invdz, double dt, double th) {
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (t >= d.in_cells) return;
  int i, j, k;
  interior(t, d.nyc, d.nzc, i, j, k);
  const int64_t o = NIDX(i, j, k), si = (int64_t)d.nyn * d.nzn, sj = d.nzn;
  const double div = diff_x(gmem(Jx), o, si, sj, invdx) + diff_y(gmem(Jy), o, si, sj, invdy) +
                     diff_z(gmem(Jz), o, si, sj, invdz);
  put_ghosts<true>(gmem(rhoh), d.nxc, d.nyc, d.nzc, g, i, j, k,
                   gmem(rhoc)[CIDX(i, j, k)] - dt * th * div);
}

struct ImageArgs {
  const double *vec;                  // E(n + theta): the Krylov vector
  const double *Bx, *By, *Bz;
  const double *rhon[kMaxSpecies];
  double beta[kMaxSpecies];           // .5 * qom * dt / c
  double coef[kMaxSpecies];           // fourpi / 2 * delt * dt / c * qom
  double *D[3];
  int ns;
  int per[3];
};

// Element of the Krylov vector's node (i, j, k): its interior nodes,
// components interleaved (solver2phys, src/Basic.cpp:365-375).
__device__ __forceinline__ int64_t vec_at(const Dims &d, int i, int j, int k) {
  return 3 * (((int64_t)(i - 1) * (d.nyn - 2) + (j - 1)) * (d.nzn - 2) + (k - 1));
}

// D = sum over species of mu . E (src/MaxwellSolver.cpp:169-198) at the
// interior nodes, species in order from zero, and divN2C of D on the interior
// cells (its stencil reads interior nodes only, so D's ghost update, which
// the reference applies first, does not change it).  One workgroup per tile
// of cells; D of the tile's nodes passes through LDS, so the nodes of the upper
// faces are computed twice (1.66 nodes per cell with FX 4, 1.49 with 8) and a
// launch and a read of D are saved.  Latency bounds it: one node per thread
// instead of two in turn (17.4 against 24 us on 128x64x64 cells, FX 4).
template <int FX>
__global__ __launch_bounds__(kFieldThreads<FX>) void k_image_d(Dims d, ImageArgs a, Tiles tiles,
                                                           double *divc, double invdx,
                                                           double invdy, double invdz) {
  constexpr int NX = FX + 1, NY = kFY + 1, NZ = kFZ + 1;
  __shared__ double s_d[3][NX * NY * NZ];
  const int tid = threadIdx.x;
  const unsigned tile = tiles.first + xcd_block();
  if (tile >= tiles.end) return;
  const int bz = tile % tiles.nz, by = (tile / tiles.nz) % tiles.ny,
            bx = tile / (tiles.nz * tiles.ny);
  const int i0 = 1 + bx * FX, j0 = 1 + by * kFY, k0 = 1 + bz * kFZ;
  for (int e = tid; e < NX * NY * NZ; e += kFieldThreads<FX>) {
    const int ex = e / (NY * NZ), ey = (e / NZ) % NY, ez = e % NZ;
    const int i = i0 + ex, j = j0 + ey, k = k0 + ez;
    if (i > d.nxn - 2 || j > d.nyn - 2 || k > d.nzn - 2) continue;
    const int64_t n = NIDX(i, j, k), t = vec_at(d, i, j, k);
    const double vx = gmem(a.vec)[t], vy = gmem(a.vec)[t + 1], vz = gmem(a.vec)[t + 2];
    const double bX = gmem(a.Bx)[n], bY = gmem(a.By)[n], bZ = gmem(a.Bz)[n];
    // every species' density before the first is used: one wait, not ns
    double rho[kMaxSpecies];
#pragma unroll
    for (int s = 0; s < kMaxSpecies; ++s)
      if (s < a.ns) rho[s] = gmem(a.rhon[s])[n];
    double dx = 0.0, dy = 0.0, dz = 0.0;
#pragma unroll
    for (int s = 0; s < kMaxSpecies; ++s) {
      if (s >= a.ns) break;
      const double beta = a.beta[s];
      const double omcx = beta * bX, omcy = beta * bY, omcz = beta * bZ;
      const double edotb = vx * omcx + vy * omcy + vz * omcz;
      const double denom =
          a.coef[s] * rho[s] / (1.0 + omcx * omcx + omcy * omcy + omcz * omcz);
      dx += (vx + (vy * omcz - vz * omcy + edotb * omcx)) * denom;
      dy += (vy + (vz * omcx - vx * omcz + edotb * omcy)) * denom;
      dz += (vz + (vx * omcy - vy * omcx + edotb * omcz)) * denom;
    }
    s_d[0][e] = dx;
    s_d[1][e] = dy;
    s_d[2][e] = dz;
    // a node belongs to the tile of the cell it starts; the last plane's
    // nodes start no interior cell and belong to the last tile
    if ((ex < FX || i == d.nxn - 2) && (ey < kFY || j == d.nyn - 2) &&
        (ez < kFZ || k == d.nzn - 2)) {
      gmem(a.D[0])[n] = dx;
      gmem(a.D[1])[n] = dy;
      gmem(a.D[2])[n] = dz;
    }
  }
  __syncthreads();
  if (tid >= FX * kFY * kFZ) return;
  const int lx = tid / (kFY * kFZ), ly = (tid / kFZ) % kFY, lz = tid % kFZ;
  const int i = i0 + lx, j = j0 + ly, k = k0 + lz;
  if (i > d.nxc - 2 || j > d.nyc - 2 || k > d.nzc - 2) return;
  const double *X = s_d[0], *Y = s_d[1], *Z = s_d[2];
  const int64_t o = (lx * NY + ly) * NZ + lz;
  gmem(divc)[CIDX(i, j, k)] = diff_x(X, o, NY * NZ, NZ, invdx) +
                              diff_y(Y, o, NY * NZ, NZ, invdy) +
                              diff_z(Z, o, NY * NZ, NZ, invdz);
}

// Three consecutive doubles in two loads (an address that is 8-byte aligned
// serves a 16-byte load).
__device__ __forceinline__ void load3(const SPIC_GLOBAL double *p, double v[3]) {
  typedef double d2 __attribute__((ext_vector_type(2), aligned(8)));
  const d2 a = *(const SPIC_GLOBAL d2 *)p;
  v[0] = a.x;
  v[1] = a.y;
  v[2] = p[2];
}

// The image at an interior node, packed as phys2solver does
// (src/Basic.cpp:385-392): ((-lapN2N_V(v) - gradC2N(divC)) * delt^2 + D) + v
// (src/MaxwellSolver.cpp:168-231, src/Grid.cpp:187-225 and 668-717).  The
// ghosts of v (applyBCscalarFieldNzero) and of divC (applyBCscalarFieldC)
// are read at their sources: no unpacked copy of v and no ghost update runs.
// The operator takes two launches instead of eight: 28 us per application on
// 128x64x64 cells against 53.
__global__ void k_image(Dims d, ImageArgs a, GhostMap gn, GhostMap gc, const double *divc,
                        double *im, double invdx, double invdy, double invdz, double dd) {
  const int64_t t = xcd_block() * (int64_t)blockDim.x + threadIdx.x;
  if (t >= d.in_nodes) return;
  int i, j, k;
  interior(t, d.nyn, d.nzn, i, j, k);
  const int64_t n = NIDX(i, j, k);
  const SPIC_GLOBAL double *S = gmem(divc);
  // cells i - 1 and i of node i, at their sources
  const int ci[2] = {ghost_src(i - 1, d.nxc, gc.lo[0], gc.hi[0]),
                     ghost_src(i, d.nxc, gc.lo[0], gc.hi[0])};
  const int cj[2] = {ghost_src(j - 1, d.nyc, gc.lo[1], gc.hi[1]),
                     ghost_src(j, d.nyc, gc.lo[1], gc.hi[1])};
  const int ck[2] = {ghost_src(k - 1, d.nzc, gc.lo[2], gc.hi[2]),
                     ghost_src(k, d.nzc, gc.lo[2], gc.hi[2])};
  double c[2][2][2];
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
      for (int z = 0; z < 2; ++z) c[x][y][z] = S[CIDX(ci[x], cj[y], ck[z])];
  const double qx = .25 * invdx, qy = .25 * invdy, qz = .25 * invdz;
  double grad[3];
  grad[0] = q4(c[1][1][1], c[0][1][1], qx) + q4(c[1][1][0], c[0][1][0], qx) +
            q4(c[1][0][1], c[0][0][1], qx) + q4(c[1][0][0], c[0][0][0], qx);
  grad[1] = q4(c[1][1][1], c[1][0][1], qy) + q4(c[1][1][0], c[1][0][0], qy) +
            q4(c[0][1][1], c[0][0][1], qy) + q4(c[0][1][0], c[0][0][0], qy);
  grad[2] = q4(c[1][1][1], c[1][1][0], qz) + q4(c[0][1][1], c[0][1][0], qz) +
            q4(c[1][0][1], c[1][0][0], qz) + q4(c[0][0][1], c[0][0][0], qz);
  const SPIC_GLOBAL double *v = gmem(a.vec);
  // the six neighbours' elements of v; a ghost of a non-periodic axis is zero
  const int64_t at[6] = {
      vec_at(d, ghost_src(i - 1, d.nxn, gn.lo[0], gn.hi[0]), j, k),
      vec_at(d, ghost_src(i + 1, d.nxn, gn.lo[0], gn.hi[0]), j, k),
      vec_at(d, i, ghost_src(j - 1, d.nyn, gn.lo[1], gn.hi[1]), k),
      vec_at(d, i, ghost_src(j + 1, d.nyn, gn.lo[1], gn.hi[1]), k),
      vec_at(d, i, j, ghost_src(k - 1, d.nzn, gn.lo[2], gn.hi[2])),
      vec_at(d, i, j, ghost_src(k + 1, d.nzn, gn.lo[2], gn.hi[2]))};
  const bool zero[6] = {!a.per[0] && i == 1,         !a.per[0] && i == d.nxn - 2,
                        !a.per[1] && j == 1,         !a.per[1] && j == d.nyn - 2,
                        !a.per[2] && k == 1,         !a.per[2] && k == d.nzn - 2};
  double nb[6][3], own[3];
  load3(v + 3 * t, own);
#pragma unroll
  for (int q = 0; q < 6; ++q) load3(v + at[q], nb[q]);
#pragma unroll
  for (int m = 0; m < 3; ++m) {
    const double c0 = own[m];
    double e[6];
#pragma unroll
    for (int q = 0; q < 6; ++q) e[q] = zero[q] ? 0.0 : nb[q][m];
    const double lap = (e[0] - 2 * c0 + e[1]) * invdx * invdx +
                       (e[2] - 2 * c0 + e[3]) * invdy * invdy +
                       (e[4] - 2 * c0 + e[5]) * invdz * invdz;
    double img = -lap;
    img -= grad[m];
    img *= dd;
    img += gmem(a.D[m])[n];
    img += c0;
    gmem(im)[3 * t + m] = img;
  }
}

#undef NIDX
#undef CIDX

inline unsigned grid1(int64_t n) { return (unsigned)((n + 255) / 256); }

// Whether two arrays of na and nb doubles share memory.
inline bool overlap(const double *a, int64_t na, const double *b, int64_t nb) {
  const uintptr_t x = (uintptr_t)a, y = (uintptr_t)b;
  return x < y + (uintptr_t)nb * sizeof(double) && y < x + (uintptr_t)na * sizeof(double);
}

hipError_t launch_bc(double *a, const Dims &d, bool nodes, bool zero_faces,
                     const spic_solve_params *p, hipStream_t s) {
  const int n0 = nodes ? d.nxn : d.nxc, n1 = nodes ? d.nyn : d.nyc,
            n2 = nodes ? d.nzn : d.nzc;
  const int px = p->PERIODICX ? 1 : 0, py = p->PERIODICY ? 1 : 0, pz = p->PERIODICZ ? 1 : 0;
  // enough threads for the largest face pair; grid-stride loops do the rest
  const int64_t faces = 2 * ((int64_t)n0 * n1 + (int64_t)n0 * n2 + (int64_t)n1 * n2);
  unsigned blocks = (unsigned)((faces + 255) / 256);
  if (blocks > 1024) blocks = 1024;
  if (px || py || pz)
    hipLaunchKernelGGL(k_bc_periodic, dim3(blocks), dim3(256), 0, s, a, n0, n1, n2,
                       d.nyn, nodes ? 1 : 0, px, py, pz);
  if (!px || !py || !pz)
    hipLaunchKernelGGL(k_bc_faces, dim3(blocks), dim3(256), 0, s, a, n0, n1, n2,
                       zero_faces ? 1 : 0, px, py, pz);
  return hipGetLastError();
}

int check_solve(const spic_grid *grd, const spic_solve_params *p, int ns) {
  int rc = check_grid(grd);
  if (rc) return rc;
  if (grd->prec != SPIC_F64)
    return fail(SPIC_EINVAL, "the field-solve operators run in FP64 (grid prec must be F64)");
  if (!p) return fail(SPIC_EINVAL, "solve parameters are NULL");
  if (ns < 0 || ns > kMaxSpecies)
    return fail(SPIC_EINVAL, "species count must be 0..%d", kMaxSpecies);
  if (grd->nxc < 3 || grd->nyc < 3 || grd->nzc < 3)
    return fail(SPIC_EINVAL, "grid needs at least one physical cell per axis");
  return SPIC_OK;
}

int finish(hipStream_t s, hipError_t e, const char *what) {
  if (e == hipSuccess) e = hipGetLastError();
  if (e == hipSuccess && !async_mode()) e = hipStreamSynchronize(s);
  return e == hipSuccess ? SPIC_OK : hip_fail(e, what);
}

}  // namespace
}  // namespace spic

using spic::Dims;

extern "C" {

size_t spic_field_workspace_bytes(const spic_grid *grd, int ns) {
  if (!grd || ns < 0) return 0;
  const Dims d = spic::dims_of(grd);
  const int64_t hat = 3 * (int64_t)ns * d.nc;
  const int64_t image = 6 * d.nn + d.nc;
  return sizeof(double) * (size_t)(hat > image ? hat : image);
}

int spic_bc_scalar(const spic_grid *grd, double *a, int kind, const spic_solve_params *p,
                   void *stream) {
  int rc = spic::check_solve(grd, p, 0);
  if (rc) return rc;
  if (!a) return spic::fail(SPIC_EINVAL, "array is NULL");
  if (kind < 0 || kind > 3) return spic::fail(SPIC_EINVAL, "BC kind must be 0..3");
  hipStream_t s = (hipStream_t)stream;
  const Dims d = spic::dims_of(grd);
  return spic::finish(s, spic::launch_bc(a, d, kind <= 1, kind == 1, p, s), "BC");
}

int spic_rhoc_from_rhon(const spic_grid *grd, double *rhon, double *rhoc,
                        const spic_solve_params *p, void *stream) {
  int rc = spic::check_solve(grd, p, 0);
  if (rc) return rc;
  if (!rhon || !rhoc) return spic::fail(SPIC_EINVAL, "rhon or rhoc is NULL");
  hipStream_t s = (hipStream_t)stream;
  const Dims d = spic::dims_of(grd);
  const spic::GhostMap g = spic::ghost_map(d.nxn, d.nyn, d.nzn, true, p);
  hipLaunchKernelGGL(spic::k_rhoc, dim3(spic::grid1(d.in_nodes)), dim3(256), 0, s, d, g, rhon,
                     rhoc);
  const hipError_t e = hipGetLastError();
  return spic::finish(s, e, "rhoc from rhon");
}

int spic_hat_densities(const spic_grid *grd, const spic_field *field,
                       const spic_moments *ids, int ns, const double *rhoc,
                       const spic_solve_params *p, const spic_hat *out, void *work,
                       size_t work_bytes, void *stream) {
  int rc = spic::check_solve(grd, p, ns);
  if (rc) return rc;
  if ((rc = spic::check_field(field))) return rc;
  if (!ids || !rhoc || !out || !out->rhoh || !out->Jxh || !out->Jyh || !out->Jzh)
    return spic::fail(SPIC_EINVAL, "moments, rhoc or hat arrays are NULL");
  if (ns < 1) return spic::fail(SPIC_EINVAL, "species count must be 1..%d", spic::kMaxSpecies);
  for (int is = 0; is < ns; ++is)
    if ((rc = spic::check_moments(&ids[is]))) return rc;
  if (!work || work_bytes < spic_field_workspace_bytes(grd, ns))
    return spic::fail(SPIC_EINVAL, "workspace of %zu bytes needed",
                      spic_field_workspace_bytes(grd, ns));
  hipStream_t s = (hipStream_t)stream;
  const Dims d = spic::dims_of(grd);
  spic::HatArgs a;
  for (int is = 0; is < ns; ++is) {
    const spic_moments &m = ids[is];
    const double *P[6] = {m.pxx, m.pxy, m.pxz, m.pyy, m.pyz, m.pzz};
    for (int c = 0; c < 6; ++c) a.P[6 * is + c] = P[c];
    for (int c = 0; c < 3; ++c) a.tc[3 * is + c] = (double *)work + (3 * is + c) * d.nc;
    a.J[3 * is] = m.Jx;
    a.J[3 * is + 1] = m.Jy;
    a.J[3 * is + 2] = m.Jz;
    a.beta[is] = .5 * p->qom[is] * p->dt / p->c;
  }
  a.Bx = (const double *)field->Bxn;
  a.By = (const double *)field->Byn;
  a.Bz = (const double *)field->Bzn;
  a.Jh[0] = out->Jxh;
  a.Jh[1] = out->Jyh;
  a.Jh[2] = out->Jzh;
  a.ns = ns;
  const double alfa = -p->dt / 2.0;
  const spic::GhostMap gc = spic::ghost_map(d.nxc, d.nyc, d.nzc, false, p),
                       gn = spic::ghost_map(d.nxn, d.nyn, d.nzn, true, p);
  // planes per thread: as many as leave a thousand workgroups
  const unsigned sheet = spic::grid1((int64_t)(d.nyc - 2) * (d.nzc - 2));
  int planes = (int)((int64_t)sheet * ns * (d.nxc - 2) / 1024);
  planes = planes < 1 ? 1 : planes > 16 ? 16 : planes;
  hipLaunchKernelGGL(spic::k_divsymm, dim3(sheet, ns, (d.nxc - 2 + planes - 1) / planes),
                     dim3(256), 0, s, d, a, planes, .25 * grd->invdx, .25 * grd->invdy,
                     .25 * grd->invdz, alfa);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) {
    hipLaunchKernelGGL(spic::k_pidot, dim3(spic::xcd_grid(spic::grid1(d.in_nodes))), dim3(256), 0, s, d, a, gc,
                       gn);
    e = hipGetLastError();
  }
  if (e == hipSuccess) {
    hipLaunchKernelGGL(spic::k_rhoh, dim3(spic::grid1(d.in_cells)), dim3(256), 0, s, d, gc,
                       out->Jxh, out->Jyh, out->Jzh, rhoc, out->rhoh, .25 * grd->invdx,
                       .25 * grd->invdy, .25 * grd->invdz, p->dt, p->th);
    e = hipGetLastError();
  }
  return spic::finish(s, e, "hat densities");
}

int spic_maxwell_image(const spic_grid *grd, const spic_field *field,
                       const spic_moments *ids, int ns, const spic_solve_params *p,
                       const double *vec, double *im, void *work, size_t work_bytes,
                       void *stream) {
  int rc = spic::check_solve(grd, p, ns);
  if (rc) return rc;
  if ((rc = spic::check_field(field))) return rc;
  if (!vec || !im || (ns > 0 && !ids))
    return spic::fail(SPIC_EINVAL, "vector, image or moments are NULL");
  for (int is = 0; is < ns; ++is)
    if (!ids[is].rhon) return spic::fail(SPIC_EINVAL, "species %d rhon is NULL", is);
  if (!work || work_bytes < spic_field_workspace_bytes(grd, ns))
    return spic::fail(SPIC_EINVAL, "workspace of %zu bytes needed",
                      spic_field_workspace_bytes(grd, ns));
  hipStream_t s = (hipStream_t)stream;
  const Dims d = spic::dims_of(grd);
  double *w = (double *)work;
  double *D[3] = {w, w + d.nn, w + 2 * d.nn};
  double *divc = w + 3 * d.nn;
  const double delt = p->c * p->th * p->dt;
  spic::ImageArgs a;
  a.vec = vec;
  for (int m = 0; m < 3; ++m) a.D[m] = D[m];
  a.per[0] = p->PERIODICX != 0;
  a.per[1] = p->PERIODICY != 0;
  a.per[2] = p->PERIODICZ != 0;
  a.Bx = (const double *)field->Bxn;
  a.By = (const double *)field->Byn;
  a.Bz = (const double *)field->Bzn;
  for (int is = 0; is < ns; ++is) {
    a.rhon[is] = ids[is].rhon;
    a.beta[is] = .5 * p->qom[is] * p->dt / p->c;
    a.coef[is] = p->fourpi / 2 * delt * p->dt / p->c * p->qom[is];
  }
  a.ns = ns;
  const spic::GhostMap gn = spic::ghost_map(d.nxn, d.nyn, d.nzn, true, p),
                       gc = spic::ghost_map(d.nxc, d.nyc, d.nzc, false, p);
  // Larger tiles compute fewer nodes twice but leave a small grid with fewer
  // workgroups: the operator takes 28.3 us with FX 8 on 128x64x64 cells (1024
  // workgroups of it) and 29.6 with FX 4, but a cycle with eight of them on
  // 33x17x19 cells (32) 300 and 293; on 64x32x32 (128) they do not differ.
  spic::Tiles tiles = spic::tiles_of(8, d.nxc - 2, d.nyc - 2, d.nzc - 2);
  const bool wide = tiles.total >= 256;
  if (!wide) tiles = spic::tiles_of(4, d.nxc - 2, d.nyc - 2, d.nzc - 2);
  // the image's nodes read their neighbours' unknowns: an image in the
  // vector's own memory is formed from a copy
  hipError_t e = hipSuccess;
  if (spic::overlap(vec, 3 * d.in_nodes, im, 3 * d.in_nodes)) {
    a.vec = divc + d.nc;
    e = hipMemcpyAsync(divc + d.nc, vec, sizeof(double) * 3 * d.in_nodes,
                       hipMemcpyDeviceToDevice, s);
    if (e != hipSuccess) return spic::hip_fail(e, "MaxwellImage");
  }
  for (tiles.first = 0; tiles.first < tiles.total; tiles.first = tiles.end) {
    tiles.end = tiles.total - tiles.first > spic::kMaxTiles ? tiles.first + spic::kMaxTiles
                                                            : tiles.total;
    const dim3 grid(spic::xcd_grid(tiles.end - tiles.first));
    if (wide)
      hipLaunchKernelGGL(spic::k_image_d<8>, grid, dim3(spic::kFieldThreads<8>), 0, s, d, a, tiles,
                         divc, .25 * grd->invdx, .25 * grd->invdy, .25 * grd->invdz);
    else
      hipLaunchKernelGGL(spic::k_image_d<4>, grid, dim3(spic::kFieldThreads<4>), 0, s, d, a, tiles,
                         divc, .25 * grd->invdx, .25 * grd->invdy, .25 * grd->invdz);
  }
  e = hipGetLastError();
  if (e == hipSuccess) {
    hipLaunchKernelGGL(spic::k_image, dim3(spic::xcd_grid(spic::grid1(d.in_nodes))), dim3(256), 0, s, d, a, gn,
                       gc, divc, im, grd->invdx, grd->invdy, grd->invdz, delt * delt);
    e = hipGetLastError();
  }
  return spic::finish(s, e, "MaxwellImage");
}

}  // extern "C"
