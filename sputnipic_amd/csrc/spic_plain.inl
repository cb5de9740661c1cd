// spic_plain.inl -- caller-order ("plain") gfx950 kernels for mover_PC,
// interpP2G and the fused mover_interp.  The push takes one lane per particle;
// SoA loads and stores are coalesced; field and node-coordinate gathers go
// through L2.  The deposit sums per cell in registers, by tile or by wave, and
// adds its sums in FP64 with hardware global atomics.
//
// Included by two translation units: spic_plain_fast.hip (SPIC_STRICT 0,
// FMA contraction allowed) and spic_plain_strict.hip (SPIC_STRICT 1, built
// with -ffp-contract=off).  In strict mode every operation keeps the
// reference's operand types and order (src/Mover.cpp:4-162, 385-572), so an
// FP64 or FP32 particle state matches the CPU reference bit for bit.
#include "spic_internal.hpp"
#include "spic_wave.hpp"

#ifndef SPIC_NS
#error "define SPIC_NS and SPIC_STRICT before including spic_plain.inl"
#endif

namespace spic {
namespace SPIC_NS {

constexpr bool kStrict = (SPIC_STRICT != 0);

// Mover cell index: 2 + int((x - xStart) * invdx), truncating toward zero
// (src/Mover.cpp:39-41).  The reference evaluates the product in double
// (xStart is double).  The argument is clamped first so that the int
// conversion is defined for any input; any index outside [1, n-1] is
// flagged by the caller.
template <typename T>
__device__ __forceinline__ int cell_trunc(T p, double start, T inv, int n) {
  if (kStrict || sizeof(T) == 8) {
    double c = ((double)p - start) * (double)inv;
    c = fmin(fmax(c, -8.0), (double)n + 8.0);
    return 2 + (int)c;
  } else {
    float c = ((float)p - (float)start) * (float)inv;
    c = fminf(fmaxf(c, -8.0f), (float)n + 8.0f);
    return 2 + (int)c;
  }
}

// Deposit cell index: 2 + int(floor((x - xStart) * invdx))
// (src/Mover.cpp:399-401).
template <typename T>
__device__ __forceinline__ int cell_floor(T p, double start, T inv, int n) {
  if (kStrict || sizeof(T) == 8) {
    double c = ((double)p - start) * (double)inv;
    c = fmin(fmax(c, -8.0), (double)n + 8.0);
    return 2 + (int)floor(c);
  } else {
    float c = ((float)p - (float)start) * (float)inv;
    c = fminf(fmaxf(c, -8.0f), (float)n + 8.0f);
    return 2 + (int)floorf(c);
  }
}

// Both nodes ix-1 and ix must exist: 1 <= ix <= n-1.  Out-of-range indices
// are clamped (so no access leaves the arrays) and reported.
__device__ __forceinline__ bool clamp_index(int &ix, int n) {
  bool bad = (ix < 1) | (ix > n - 1);
  ix = min(max(ix, 1), n - 1);
  return bad;
}

// The six field components of every node together (kRec values each, FP32
// padded to 16-byte alignment), as the mover's gather reads them: a node is
// one line instead of six, and the two nodes of a z pair mostly share it.
template <typename T>
struct PackedField {
  static constexpr int kRec = sizeof(T) == 8 ? 6 : 8;
  const T *rec;
};

template <typename T>
__global__ __launch_bounds__(256) void k_pack_fields(KField<T> f, T *__restrict__ rec, int nn) {
  constexpr int kRec = PackedField<T>::kRec;
  const int n = blockIdx.x * 256 + threadIdx.x;
  if (n >= nn) return;
  T *r = rec + (size_t)n * kRec;
  r[0] = f.Ex[n]; r[1] = f.Ey[n]; r[2] = f.Ez[n];
  r[3] = f.Bx[n]; r[4] = f.By[n]; r[5] = f.Bz[n];
}

// The stencil of the cell whose upper node is `base`: F[a][b][c] holds node
// base - a * sx - b * sy - c.
template <typename T>
__device__ __forceinline__ void load_stencil(const KField<T> &f, int base, int sx, int sy,
                                             T (&F)[2][2][2][6]) {
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const int n = base - a * sx - b * sy - c;
        F[a][b][c][0] = f.Ex[n]; F[a][b][c][1] = f.Ey[n]; F[a][b][c][2] = f.Ez[n];
        F[a][b][c][3] = f.Bx[n]; F[a][b][c][4] = f.By[n]; F[a][b][c][5] = f.Bz[n];
      }
}

template <typename T>
__device__ __forceinline__ void load_stencil(const PackedField<T> &f, int base, int sx, int sy,
                                             T (&F)[2][2][2][6]) {
  constexpr int kVec = 16 / sizeof(T);  // 16-byte loads
  typedef T Vec __attribute__((ext_vector_type(kVec)));
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const T *r = f.rec + (size_t)(base - a * sx - b * sy - c) * PackedField<T>::kRec;
#pragma unroll
        for (int i = 0; i < 6; i += kVec) {
          const Vec v = *reinterpret_cast<const Vec *>(r + i);
#pragma unroll
          for (int j = 0; j < kVec; ++j)
            if (i + j < 6) F[a][b][c][i + j] = v[j];
        }
      }
}

// One particle's predictor-corrector push and particle BC
// (src/Mover.cpp:33-157).  Returns true if an iterate left the grid by
// more than one cell.
// The gathers bound it: 48 field values per particle from L2, a cache line
// per lane and load once the particles have mixed.  They stay in registers
// while the iterate stays in its cell (nine in ten do), so most particles
// gather once instead of once per iteration: 5.97M FP64 particles of a mixed
// order in 1.70 ms against 3.62, three waves per SIMD in FP64 (168 VGPRs,
// the limit; unlimited it takes 176 and two).  From packed fields 24 loads of
// 16 bytes on a sixth of the lines: a million in random order on 257499 nodes
// 110 us against 419, in cell order 54 against 65.
template <typename T, typename FV>
__device__ __forceinline__ bool push_particle_once(const KGrid<T> &g,
                                              const FV &f,
                                              const KPush<T> &k, T &x, T &y,
                                              T &z, T &u, T &v, T &w) {
  const int nyn = g.nyn, nzn = g.nzn;
  const int sx = nyn * nzn, sy = nzn;
  const T xt = x, yt = y, zt = z;
  T upt = T(0), vpt = T(0), wpt = T(0);
  T xc = x, yc = y, zc = z;
  bool bad = false;
  // the stencil of the last cell: nodes ix - a, iy - b, iz - c
  int cix = -1, ciy = -1, ciz = -1;
  T F[2][2][2][6];
  T X0 = T(0), X1 = T(0), Y0 = T(0), Y1 = T(0), Z0 = T(0), Z1 = T(0);
  for (int it = 0; it < k.niter; ++it) {
    int ix = cell_trunc<T>(xc, g.xStart, g.invdx, g.nxn);
    int iy = cell_trunc<T>(yc, g.yStart, g.invdy, g.nyn);
    int iz = cell_trunc<T>(zc, g.zStart, g.invdz, g.nzn);
    bad |= clamp_index(ix, g.nxn);
    bad |= clamp_index(iy, g.nyn);
    bad |= clamp_index(iz, g.nzn);
    if (ix != cix || iy != ciy || iz != ciz) {
      cix = ix; ciy = iy; ciz = iz;
      X0 = g.xn[ix - 1]; X1 = g.xn[ix];
      Y0 = g.yn[iy - 1]; Y1 = g.yn[iy];
      Z0 = g.zn[iz - 1]; Z1 = g.zn[iz];
      load_stencil(f, (ix * nyn + iy) * nzn + iz, sx, sy, F);
    }
    const T xi[2] = {xc - X0, X1 - xc};
    const T eta[2] = {yc - Y0, Y1 - yc};
    const T zeta[2] = {zc - Z0, Z1 - zc};
    T Exl = T(0), Eyl = T(0), Ezl = T(0), Bxl = T(0), Byl = T(0), Bzl = T(0);
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          const T wgt = xi[a] * eta[b] * zeta[c] * g.invVOL;
          Exl += wgt * F[a][b][c][0];
          Eyl += wgt * F[a][b][c][1];
          Ezl += wgt * F[a][b][c][2];
          Bxl += wgt * F[a][b][c][3];
          Byl += wgt * F[a][b][c][4];
          Bzl += wgt * F[a][b][c][5];
        }
    const T q2 = k.qomdt2;
    const T omdtsq = q2 * q2 * (Bxl * Bxl + Byl * Byl + Bzl * Bzl);
    T denom;
    if (kStrict || sizeof(T) == 8)
      denom = (T)(1.0 / (1.0 + (double)omdtsq));  // double, as Mover.cpp:71
    else
      denom = T(1) / (T(1) + omdtsq);
    const T ut = u + q2 * Exl;
    const T vt = v + q2 * Eyl;
    const T wt = w + q2 * Ezl;
    const T udotb = ut * Bxl + vt * Byl + wt * Bzl;
    upt = (ut + q2 * (vt * Bzl - wt * Byl + q2 * udotb * Bxl)) * denom;
    vpt = (vt + q2 * (wt * Bxl - ut * Bzl + q2 * udotb * Byl)) * denom;
    wpt = (wt + q2 * (ut * Byl - vt * Bxl + q2 * udotb * Bzl)) * denom;
    xc = xt + upt * k.dto2;
    yc = yt + vpt * k.dto2;
    zc = zt + wpt * k.dto2;
  }
  if (kStrict || sizeof(T) == 8) {
    // 2.0 * uptilde - u in double, then narrowed (Mover.cpp:91-93)
    u = (T)(2.0 * (double)upt - (double)u);
    v = (T)(2.0 * (double)vpt - (double)v);
    w = (T)(2.0 * (double)wpt - (double)w);
  } else {
    u = T(2) * upt - u;
    v = T(2) * vpt - v;
    w = T(2) * wpt - w;
  }
  x = xt + upt * k.dt_sub;
  y = yt + vpt * k.dt_sub;
  z = zt + wpt * k.dt_sub;
  // Particle BC: two independent tests per axis, compared and updated in
  // double as the reference does (Lx is double; Mover.cpp:103-157).
  if ((double)x > g.Lx) {
    if (k.perx) x = (T)((double)x - g.Lx);
    else { u = -u; x = (T)(2 * g.Lx - (double)x); }
  }
  if (x < T(0)) {
    if (k.perx) x = (T)((double)x + g.Lx);
    else { u = -u; x = -x; }
  }
  if ((double)y > g.Ly) {
    if (k.pery) y = (T)((double)y - g.Ly);
    else { v = -v; y = (T)(2 * g.Ly - (double)y); }
  }
  if (y < T(0)) {
    if (k.pery) y = (T)((double)y + g.Ly);
    else { v = -v; y = -y; }
  }
  if ((double)z > g.Lz) {
    if (k.perz) z = (T)((double)z - g.Lz);
    else { w = -w; z = (T)(2 * g.Lz - (double)z); }
  }
  if (z < T(0)) {
    if (k.perz) z = (T)((double)z + g.Lz);
    else { w = -w; z = -z; }
  }
  return bad;
}

// The push of one particle: once, or k.nloop times with the particle BC
// after each (the reference GPU mover's sub-cycle loop,
// src/gpu/Particles_gpu.cu:336-437).
template <typename T, typename FV>
__device__ __forceinline__ bool push_particle(const KGrid<T> &g, const FV &f,
                                              const KPush<T> &k, T &x, T &y, T &z, T &u,
                                              T &v, T &w) {
  bool bad = false;
#pragma unroll 1
  for (int isub = 0; isub < k.nloop; ++isub)
    bad |= push_particle_once<T, FV>(g, f, k, x, y, z, u, v, w);
  return bad;
}

constexpr int kBlock = 256;

template <typename T, typename FV>
__global__ __launch_bounds__(kBlock)
__attribute__((amdgpu_waves_per_eu(sizeof(T) == 8 ? 3 : 4)))
void k_mover(KGrid<T> g, FV f, KPart<T> p, KPush<T> k, unsigned int *status) {
  bool bad = false;
  // unsigned: the last index plus the grid does not fit an int near 2^31
  for (unsigned int i = blockIdx.x * kBlock + threadIdx.x; i < (unsigned)p.n;
       i += gridDim.x * kBlock) {
    T x = p.x[i], y = p.y[i], z = p.z[i], u = p.u[i], v = p.v[i], w = p.w[i];
    bad |= push_particle(g, f, k, x, y, z, u, v, w);
    p.x[i] = x; p.y[i] = y; p.z[i] = z;
    p.u[i] = u; p.v[i] = v; p.w[i] = w;
  }
  if (bad) atomicAdd(status, 1u);
}

// The ten-moment CIC deposit (src/Mover.cpp:399-570) of small species and of
// captured calls: per node weight q*xi*eta*zeta*invVOL, every moment term times
// invVOL again, added in FP64.  A wave takes kRun particles one after another:
// lane l sums moment l % 8 of node l / 8 (and moments 8 and 9 in the lanes of
// moments 0 and 1) in registers while the cell stays the same, then adds its
// sums to the arrays, so that particles in cell order cost 80 atomics per cell
// they meet, each to an address of its own.  Bound by the atomics (20 to 33 G/s).
// 8192 particles on 2299 nodes, FP64, against one particle per lane: 8.0 us in
// cell order instead of 88 (lanes of one cell then met at one address), 28
// instead of 44 in random order; 500 particles 10 instead of 15 to 27.
constexpr int kRun = 32;

template <typename T>
__global__ __launch_bounds__(64) void k_deposit(KGrid<T> g, KPart<T> p, KMom m,
                                                unsigned int *status) {
  // x y z u v w q 1, then the node coordinates X0 X1 Y0 Y1 Z0 Z1 of the cell
  __shared__ T s_p[14][kRun];
  __shared__ double *s_mom[10];
  const int lane = threadIdx.x;
  if (lane == 0) {
#pragma unroll
    for (int k = 0; k < 10; ++k) s_mom[k] = m.m[k];
  }
  const int first = blockIdx.x * kRun;
  const int n = min(kRun, p.n - first);
  int base = 0;
  bool bad = false;
  if (lane < n) {
    const int i = first + lane;
    const T x = p.x[i], y = p.y[i], z = p.z[i];
    int ix = cell_floor<T>(x, g.xStart, g.invdx, g.nxn);
    int iy = cell_floor<T>(y, g.yStart, g.invdy, g.nyn);
    int iz = cell_floor<T>(z, g.zStart, g.invdz, g.nzn);
    bad = clamp_index(ix, g.nxn);
    bad |= clamp_index(iy, g.nyn);
    bad |= clamp_index(iz, g.nzn);
    base = (ix * g.nyn + iy) * g.nzn + iz;
    s_p[0][lane] = x; s_p[1][lane] = y; s_p[2][lane] = z;
    s_p[3][lane] = p.u[i]; s_p[4][lane] = p.v[i]; s_p[5][lane] = p.w[i];
    s_p[6][lane] = p.q[i]; s_p[7][lane] = T(1);
    s_p[8][lane] = g.xn[ix - 1]; s_p[9][lane] = g.xn[ix];
    s_p[10][lane] = g.yn[iy - 1]; s_p[11][lane] = g.yn[iy];
    s_p[12][lane] = g.zn[iz - 1]; s_p[13][lane] = g.zn[iz];
  }
  if (bad) atomicAdd(status + 1, 1u);
  __syncthreads();
  // this lane's node (ix - a, iy - b, iz - c): weight x - X0 (a = 0) or
  // X1 - x, which is the exact negative of x - X1
  const int a = lane >> 5, b = (lane >> 4) & 1, c = (lane >> 3) & 1, mm = lane & 7;
  const T sign = ((a + b + c) & 1) ? -g.invVOL : g.invVOL;
  const int off = -(a * g.nyn + b) * g.nzn - c;
  // its moments as products of two of 1 u v w (rows 7 3 4 5)
  const int row1 = mm == 0 ? 7 : mm < 4 ? mm + 2 : mm < 7 ? 3 : 4;
  const int row2 = mm < 4 ? 7 : mm < 7 ? mm - 1 : 4;
  const int row3 = mm == 0 ? 4 : 5;  // second moment: v w or w w
  double sum = 0.0, sum2 = 0.0;
  int cur = __builtin_amdgcn_readlane(base, 0);
  auto flush = [&]() {
    if (sum != 0.0) unsafeAtomicAdd(s_mom[mm] + cur + off, sum);
    if (mm < 2 && sum2 != 0.0) unsafeAtomicAdd(s_mom[8 + mm] + cur + off, sum2);
    sum = sum2 = 0.0;
  };
  for (int j = 0; j < n; ++j) {
    const int cell = __builtin_amdgcn_readlane(base, j);
    if (cell != cur) {
      flush();
      cur = cell;
    }
    const T wgt = s_p[6][j] * (s_p[0][j] - s_p[8 + a][j]) * (s_p[1][j] - s_p[10 + b][j]) *
                  (s_p[2][j] - s_p[12 + c][j]) * sign;
    sum += (double)((s_p[row1][j] * s_p[row2][j]) * wgt * g.invVOL);
    sum2 += (double)((s_p[row3][j] * s_p[5][j]) * wgt * g.invVOL);
  }
  flush();
}

// Calls f(first, count) for n items in runs of at most `slice`, until it returns
// false.  In 64 bits: the run after the last one of a species of 2^31 - 1
// particles starts beyond an int.
template <typename F>
constexpr void for_slices(int64_t n, int64_t slice, F f) {
  for (int64_t first = 0; first < n; first += slice)
    if (!f(first, n - first < slice ? n - first : slice)) return;
}
constexpr int64_t slices_sum(int64_t n, int64_t slice) {
  int64_t sum = 0;
  for_slices(n, slice, [&sum, slice](int64_t first, int64_t count) {
    const bool next = first == sum && count > 0 && count <= slice;
    sum += count;
    return next;
  });
  return sum;
}

template <typename T>
KPart<T> part_slice(const KPart<T> &p, int64_t first, int64_t count) {
  KPart<T> q = p;
  q.x += first; q.y += first; q.z += first;
  q.u += first; q.v += first; q.w += first;
  q.q += first;
  q.n = (int)count;
  return q;
}

static inline unsigned grid_for(int n) {
  long blocks = ((long)n + kBlock - 1) / kBlock;
  if (blocks < 1) blocks = 1;
  if (blocks > (1L << 20)) blocks = 1L << 20;
  return (unsigned)blocks;
}

// ---- deposit through tiles -------------------------------------------------
//
// 80 global FP64 atomics per particle bound the direct deposit: 0.4 G
// particles/s, 14.4 ms for 5.97M FP64 particles in bin order.  Here the
// particles of a species are first counted into tiles of 4x4x4 cells (each
// gets its rank in its tile), their indices are placed tile by tile, and one
// workgroup per run of a tile's particles gathers them, sums their moments
// per cell in registers and adds 5x5x5 nodes to the arrays: about 1250 atomics
// per run instead of 80 per particle.  The particles themselves do not move.
// Tiles cover the deposit cells ix - 1 = 0 .. nxn - 2, guard cells included.
// Five launches and the scratch take 39 us whatever the size; k_deposit takes
// 36 for 12288 particles in random order, 57 for 20000, and with few particles
// per tile stays ahead longer (20000 on 4225 tiles: 42 / 53 us; 65536: 130 / 80).
constexpr int kDepMinParticles = 16384, kDepMinPerTile = 8;
constexpr int kDepTile = 4;
constexpr int kDepCells = kDepTile * kDepTile * kDepTile;
constexpr int kDepBatch = 512;         // particles staged in LDS at a time
constexpr int kDepMaxRun = 4096;       // particles per workgroup at most
constexpr int kDepSlice = 1 << 24;     // particles binned at a time (24-bit indices)
// Tiles at most: each may be a work item of its own, of 4 * kDepCells threads, and a
// launch has fewer than 2^32.
constexpr long kDepMaxTiles = 1 << 23;
static_assert((kDepMaxTiles + kDepSlice / kDepBatch) * 4 * kDepCells < (1ll << 32), "one launch");
constexpr uint32_t kDepIndexMask = (1u << 24) - 1u;
static_assert(slices_sum(2147483647, kDepSlice) == 2147483647 &&
                  slices_sum(kDepSlice, kDepSlice) == kDepSlice &&
                  slices_sum(kDepSlice + 1, kDepSlice) == kDepSlice + 1 &&
                  slices_sum(127 * (int64_t)kDepSlice + 1, kDepSlice) ==
                      127 * (int64_t)kDepSlice + 1,
              "every particle in one slice");

struct DepBins {
  int nty, ntz, ntiles;
  int run;                // particles per work item
  int per;                // particles per thread of the count
  int in_lds;             // the tiles' counters fit in LDS (kLdsTiles)
  unsigned int *cnt;      // [ntiles + 2]: particles per tile, total, items
  unsigned int *next;     // [ntiles]: next free place of each tile
  uint4 *items;           // tile, first place, particles
  unsigned int *where;    // [n]: cell in the tile | tile << 6
  unsigned int *perm;     // [n] by place: index | cell in the tile << 24
};

// Tile and cell within the tile of a (clamped) deposit cell.
__device__ __forceinline__ void dep_tile(const DepBins &b, int ix, int iy, int iz,
                                         unsigned int &tile, unsigned int &cell) {
  const int cx = ix - 1, cy = iy - 1, cz = iz - 1;
  tile = ((cx / kDepTile) * b.nty + cy / kDepTile) * b.ntz + cz / kDepTile;
  cell = ((cx % kDepTile) * kDepTile + cy % kDepTile) * kDepTile + cz % kDepTile;
}

template <typename T>
__device__ __forceinline__ bool dep_cell(const KGrid<T> &g, T x, T y, T z, int &ix, int &iy,
                                         int &iz) {
  ix = cell_floor<T>(x, g.xStart, g.invdx, g.nxn);
  iy = cell_floor<T>(y, g.yStart, g.invdy, g.nyn);
  iz = cell_floor<T>(z, g.zStart, g.invdz, g.nzn);
  bool bad = clamp_index(ix, g.nxn);
  bad |= clamp_index(iy, g.nyn);
  bad |= clamp_index(iz, g.nzn);
  return bad;
}

// Counts the particles into tiles; with PUSH, pushes them first.  Up to
// kLdsTiles tiles a workgroup counts its particles in LDS and adds each
// tile it met once: with counters in global memory alone, a million
// particles in random order on 45 tiles took 1.3 ms in contended atomics.
template <typename T, bool PUSH, typename FV>
__global__ __launch_bounds__(kBlock)
__attribute__((amdgpu_waves_per_eu(sizeof(T) == 8 && PUSH ? 3 : 4)))
void k_dep_count(KGrid<T> g, FV f, KPart<T> p, KPush<T> k, DepBins b,
                 unsigned int *status) {
  __shared__ unsigned int s_cnt[kLdsTiles];
  const int tid = threadIdx.x;
  if (b.in_lds) {
    for (int t = tid; t < b.ntiles; t += kBlock) s_cnt[t] = 0u;
    __syncthreads();
  }
  const int first = blockIdx.x * kBlock * b.per;
  bool bad = false, bad_dep = false;
  for (int e = 0; e < b.per; ++e) {
    const int i = first + e * kBlock + tid;
    const bool active = i < p.n;
    unsigned int tile = 0, cell = 0;
    if (active) {
      T x = p.x[i], y = p.y[i], z = p.z[i];
      if constexpr (PUSH) {
        T u = p.u[i], v = p.v[i], w = p.w[i];
        bad |= push_particle(g, f, k, x, y, z, u, v, w);
        p.x[i] = x; p.y[i] = y; p.z[i] = z;
        p.u[i] = u; p.v[i] = v; p.w[i] = w;
      }
      int ix, iy, iz;
      bad_dep |= dep_cell<T>(g, x, y, z, ix, iy, iz);
      dep_tile(b, ix, iy, iz, tile, cell);
      b.where[i] = cell | (tile << 6);
    }
    if (b.in_lds) key_rank(s_cnt, tile, active);
    else key_rank(b.cnt, tile, active);
  }
  if (bad) atomicAdd(status, 1u);
  if (bad_dep) atomicAdd(status + 1, 1u);
  if (b.in_lds) {
    __syncthreads();
    for (int t = tid; t < b.ntiles; t += kBlock)
      if (s_cnt[t]) atomicAdd(b.cnt + t, s_cnt[t]);
  }
}

// Places of the tiles (in no particular order) and their work items.
static __global__ __launch_bounds__(kBlock) void k_dep_bounds(DepBins b) {
  const int t = blockIdx.x * kBlock + threadIdx.x, lane = threadIdx.x & 63;
  const unsigned int c = t < b.ntiles ? b.cnt[t] : 0u;
  const unsigned int ni = (c + b.run - 1) / b.run;
  unsigned int sc = c, si = ni;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const unsigned int vc = __shfl_up(sc, d), vi = __shfl_up(si, d);
    if (lane >= d) { sc += vc; si += vi; }
  }
  unsigned int bc = 0, bi = 0;
  if (lane == 63 && sc) {
    bc = atomicAdd(b.cnt + b.ntiles, sc);
    bi = atomicAdd(b.cnt + b.ntiles + 1, si);
  }
  const unsigned int first = __shfl(bc, 63) + sc - c, item = __shfl(bi, 63) + si - ni;
  if (c) b.next[t] = first;
  for (unsigned int j = 0; j < ni; ++j)
    b.items[item + j] = make_uint4((unsigned int)t, first + j * b.run,
                                   min((unsigned int)b.run, c - j * b.run), 0u);
}

// Places each particle's index in its tile, the places taken as the count
// took its counters: each tile's places at once per workgroup (IN_LDS), PER
// particles per thread, or per wave.
template <int PER, bool IN_LDS>
static __global__ __launch_bounds__(kBlock) void k_dep_place(DepBins b, int n) {
  __shared__ unsigned int s_cnt[IN_LDS ? kLdsTiles : 1];
  const int tid = threadIdx.x;
  const int first = blockIdx.x * kBlock * PER;
  unsigned int w[PER], r[PER];
#pragma unroll
  for (int e = 0; e < PER; ++e) {
    const int i = first + e * kBlock + tid;
    w[e] = i < n ? b.where[i] : 0u;
  }
  if constexpr (IN_LDS) {
    for (int t = tid; t < b.ntiles; t += kBlock) s_cnt[t] = 0u;
    __syncthreads();
  }
#pragma unroll
  for (int e = 0; e < PER; ++e)
    r[e] = key_rank(IN_LDS ? s_cnt : b.next, w[e] >> 6, first + e * kBlock + tid < n);
  if constexpr (IN_LDS) {
    __syncthreads();
    for (int t = tid; t < b.ntiles; t += kBlock)
      if (s_cnt[t]) s_cnt[t] = atomicAdd(b.next + t, s_cnt[t]);
    __syncthreads();
  }
#pragma unroll
  for (int e = 0; e < PER; ++e) {
    const int i = first + e * kBlock + tid;
    if (i < n)
      b.perm[(IN_LDS ? s_cnt[w[e] >> 6] : 0u) + r[e]] = (unsigned int)i | ((w[e] & 63u) << 24);
  }
}

// One work item per workgroup: batches of kDepBatch particles are gathered
// into LDS sorted by cell (a count, a wave scan and a placement; every
// batch's particles fit, unlike fixed buckets), then the four threads of a
// cell, two of its eight nodes each, sum them in FP64 registers that live
// until the item's end.  39 KB of LDS and 126 VGPRs in FP64: four workgroups
// per CU cover each other's gathers.  5.97M FP64 particles in bin order: 231 us
// (64 B each, 1.65 TB/s); loading the next batch ahead needs 140 VGPRs, three
// workgroups, and takes 250 us.
template <typename T>
__global__ __launch_bounds__(4 * kDepCells)
__attribute__((amdgpu_waves_per_eu(4)))
void k_tile_deposit(KGrid<T> g, KPart<T> p, KMom m,
                                                                 DepBins b) {
  constexpr int NT = 4 * kDepCells, PER = kDepBatch / NT, NB = kDepTile + 1;
  // strict arithmetic, and FP32 particles as the direct kernel adds them:
  // every term rounded in T before it is added in FP64
  constexpr bool kTerms = kStrict || sizeof(T) == 4;
  __shared__ T s_p[7][kDepBatch];
  __shared__ double s_mom[10][NB * NB * NB];
  __shared__ unsigned int s_cnt[kDepCells], s_off[kDepCells + 1];
  if (blockIdx.x >= b.cnt[b.ntiles + 1]) return;
  const uint4 item = b.items[blockIdx.x];
  const int tid = threadIdx.x;
  const int c0z = (int)(item.x % b.ntz) * kDepTile;
  const int c0y = (int)((item.x / b.ntz) % b.nty) * kDepTile;
  const int c0x = (int)(item.x / (b.ntz * b.nty)) * kDepTile;
  for (int i = tid; i < 10 * NB * NB * NB; i += NT) (&s_mom[0][0])[i] = 0.0;
  if (tid < kDepCells) s_cnt[tid] = 0u;
  // this thread's cell and its node pair, corners (a, b, 0) and (a, b, 1)
  const int my = tid >> 2, ma = (tid >> 1) & 1, mb = tid & 1;
  const int lx = my / (kDepTile * kDepTile), ly = (my / kDepTile) % kDepTile,
            lz = my % kDepTile;
  // nodes of cells beyond the grid are never used; their index is bounded
  const int nx1 = min(c0x + lx + 1, g.nxn - 1), ny1 = min(c0y + ly + 1, g.nyn - 1),
            nz1 = min(c0z + lz + 1, g.nzn - 1);
  const T X0 = g.xn[nx1 - 1], X1 = g.xn[nx1];
  const T Y0 = g.yn[ny1 - 1], Y1 = g.yn[ny1];
  const T Z0 = g.zn[nz1 - 1], Z1 = g.zn[nz1];
  const T iv = g.invVOL;
  double acc[20];
#pragma unroll
  for (int j = 0; j < 20; ++j) acc[j] = 0.0;
  __syncthreads();
  for (unsigned int o = 0; o < item.z; o += kDepBatch) {
    T val[PER][7];
    unsigned int cell[PER], rank[PER];
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      const unsigned int j = o + e * NT + tid;
      cell[e] = kDepCells;
      if (j < item.z) {
        const unsigned int w = b.perm[item.y + j];
        const unsigned int i = w & kDepIndexMask;
        cell[e] = w >> 24;
        val[e][0] = p.x[i]; val[e][1] = p.y[i]; val[e][2] = p.z[i];
        val[e][3] = p.q[i];
        val[e][4] = p.u[i]; val[e][5] = p.v[i]; val[e][6] = p.w[i];
        rank[e] = atomicAdd(&s_cnt[cell[e]], 1u);
      }
    }
    __syncthreads();
    if (tid < 64) {
      const unsigned int c = s_cnt[tid];
      unsigned int sum = c;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const unsigned int v = __shfl_up(sum, d);
        if (tid >= d) sum += v;
      }
      s_off[tid] = sum - c;
      if (tid == 63) s_off[64] = sum;
      s_cnt[tid] = 0u;
    }
    __syncthreads();
#pragma unroll
    for (int e = 0; e < PER; ++e)
      if (cell[e] < (unsigned int)kDepCells) {
        const unsigned int at = s_off[cell[e]] + rank[e];
#pragma unroll
        for (int c = 0; c < 7; ++c) s_p[c][at] = val[e][c];
      }
    __syncthreads();
    const unsigned int end = s_off[my + 1];
    for (unsigned int j = s_off[my]; j < end; ++j) {
      const T x = s_p[0][j], y = s_p[1][j], z = s_p[2][j], q = s_p[3][j];
      const T u = s_p[4][j], v = s_p[5][j], w = s_p[6][j];
      const T xi = ma ? X1 - x : x - X0, eta = mb ? Y1 - y : y - Y0;
      if constexpr (kTerms) {
        // the reference's terms, each rounded in T (src/Mover.cpp:430-568)
        const T wg[2] = {q * xi * eta * (z - Z0) * iv, q * xi * eta * (Z1 - z) * iv};
        const T uu = u * u, uv = u * v, uw = u * w, vv = v * v, vw = v * w, ww = w * w;
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          double *a = acc + 10 * c;
          const T wgt = wg[c];
          a[0] += (double)(wgt * iv);
          a[1] += (double)((u * wgt) * iv);
          a[2] += (double)((v * wgt) * iv);
          a[3] += (double)((w * wgt) * iv);
          a[4] += (double)((uu * wgt) * iv);
          a[5] += (double)((uv * wgt) * iv);
          a[6] += (double)((uw * wgt) * iv);
          a[7] += (double)((vv * wgt) * iv);
          a[8] += (double)((vw * wgt) * iv);
          a[9] += (double)((ww * wgt) * iv);
        }
      } else {
        // sums of p_m (q xi eta zeta); invVOL^2 enters once at the end
        const double qxy = q * xi * eta;
        const double w0 = qxy * (z - Z0), w1 = qxy * (Z1 - z);
        const double pm[10] = {1.0, u, v, w, u * u, u * v, u * w, v * v, v * w, w * w};
#pragma unroll
        for (int j2 = 0; j2 < 10; ++j2) {
          acc[j2] += pm[j2] * w0;
          acc[10 + j2] += pm[j2] * w1;
        }
      }
    }
  }
  // corner (a, b, c) of cell (lx, ly, lz) is block node (lx + 1 - a, ...)
  const double scale = kTerms ? 1.0 : (double)iv * (double)iv;
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const int nb = ((lx + 1 - ma) * NB + (ly + 1 - mb)) * NB + (lz + 1 - c);
#pragma unroll
    for (int j = 0; j < 10; ++j)
      if (acc[10 * c + j] != 0.0) atomicAdd(&s_mom[j][nb], acc[10 * c + j] * scale);
  }
  __syncthreads();
  for (int i = tid; i < 10 * NB * NB * NB; i += NT) {
    const int j = i / (NB * NB * NB), nb = i % (NB * NB * NB);
    const double v = s_mom[j][nb];
    const int nx = c0x + nb / (NB * NB), ny = c0y + (nb / NB) % NB, nz = c0z + nb % NB;
    if (v != 0.0 && nx < g.nxn && ny < g.nyn && nz < g.nzn)
      unsafeAtomicAdd(m.m[j] + (size_t)((nx * g.nyn + ny) * g.nzn + nz), v);
  }
}

// Whether a species' deposit goes through tiles: enough particles to fill the
// workgroups' batches, and a stream that may allocate (a capture keeps the
// direct kernels).
inline bool dep_through_tiles(long ntiles, int n, hipStream_t s) {
  return n >= kDepMinParticles && (long)n >= ntiles * kDepMinPerTile &&
         ntiles <= kDepMaxTiles && stream_may_alloc(s);
}

// Whether the push packs the fields first.  Packing costs a launch and the
// scratch's allocation, 14 us per call, and 96 bytes per node: from 262144
// particles (131072 in cell order on 2197 nodes: 11.4 us as they are, 21.2
// packed; a million 59.7 / 48.9) and up to a node for two particles.
constexpr int kPackMin = 1 << 18;
inline bool pack_pays(int n, int nn) { return n >= kPackMin && nn <= n / 2; }

template <typename T>
void pack_fields(const KField<T> &f, const PackedField<T> &to, int nn, hipStream_t s) {
  hipLaunchKernelGGL(k_pack_fields<T>, dim3((nn + 255) / 256), dim3(256), 0, s, f,
                     const_cast<T *>(to.rec), nn);
}

// Deposit through tiles, with the push before it when `f` is given.  `taken`
// stays false when nothing has run: the caller then has the direct kernels.
template <typename T>
hipError_t tile_deposit(const KGrid<T> &g, const KField<T> *f, const KPart<T> &p,
                        const KPush<T> *k, const KMom &m, unsigned int *status,
                        hipStream_t s, bool &taken) {
  taken = false;
  DepBins b;
  const long ntx = (g.nxn - 2) / kDepTile + 1;
  b.nty = (g.nyn - 2) / kDepTile + 1;
  b.ntz = (g.nzn - 2) / kDepTile + 1;
  const long ntiles = ntx * b.nty * b.ntz;
  if (!dep_through_tiles(ntiles, p.n, s)) return hipSuccess;
  b.ntiles = (int)ntiles;
  const int slice = p.n < kDepSlice ? p.n : kDepSlice;
  // about a thousand items at least, so that small species fill the device
  int run = (slice / 1024 + kDepBatch - 1) / kDepBatch * kDepBatch;
  b.run = run < kDepBatch ? kDepBatch : run > kDepMaxRun ? kDepMaxRun : run;
  const size_t max_items = (size_t)slice / b.run + (size_t)(ntiles < slice ? ntiles : slice);
  auto up = [](size_t v) { return (v + 255) & ~size_t(255); };
  // the count's particles per thread: enough workgroups first, then few
  // enough that reading out their counters stays cheap
  b.per = slice / (kBlock * 2048);
  b.per = b.per < 1 ? 1 : b.per > 16 ? 16 : b.per;
  b.in_lds = ntiles <= kLdsTiles && ntiles <= 8 * kBlock * b.per ? 1 : 0;
  const int nn = g.nxn * g.nyn * g.nzn;
  const bool pack = f && pack_pays(p.n, nn);
  const size_t a_fld = pack ? up(sizeof(T) * PackedField<T>::kRec * (size_t)nn) : 0;
  const size_t a_cnt = up(4 * (size_t)(ntiles + 2)), a_next = up(4 * (size_t)ntiles),
               a_items = up(sizeof(uint4) * max_items), a_n = up(4 * (size_t)slice);
  char *w = nullptr;
  hipError_t e = stream_alloc((void **)&w, a_cnt + a_next + a_items + 2 * a_n + a_fld, s);
  if (e != hipSuccess) {
    (void)hipGetLastError();  // the direct kernels need no scratch
    return hipSuccess;
  }
  taken = true;
  b.cnt = (unsigned int *)w;
  b.next = (unsigned int *)(w + a_cnt);
  b.items = (uint4 *)(w + a_cnt + a_next);
  b.where = (unsigned int *)(w + a_cnt + a_next + a_items);
  b.perm = (unsigned int *)(w + a_cnt + a_next + a_items + a_n);
  const PackedField<T> packed{(const T *)(w + a_cnt + a_next + a_items + 2 * a_n)};
  if (pack) pack_fields(*f, packed, nn, s);
  for_slices(p.n, slice, [&](int64_t first, int64_t count) {
    const KPart<T> q = part_slice(p, first, count);
    if ((e = zero_u32(b.cnt, (size_t)ntiles + 2, s)) != hipSuccess) return false;
    const unsigned counts = (unsigned)((q.n + kBlock * b.per - 1) / (kBlock * b.per));
    if (pack)
      hipLaunchKernelGGL((k_dep_count<T, true, PackedField<T>>), dim3(counts), dim3(kBlock), 0,
                         s, g, packed, q, *k, b, status);
    else if (f)
      hipLaunchKernelGGL((k_dep_count<T, true, KField<T>>), dim3(counts), dim3(kBlock), 0, s, g,
                         *f, q, *k, b, status);
    else
      hipLaunchKernelGGL((k_dep_count<T, false, KField<T>>), dim3(counts), dim3(kBlock), 0, s,
                         g, KField<T>{}, q, KPush<T>{}, b, status);
    hipLaunchKernelGGL(k_dep_bounds, dim3(grid_for(b.ntiles)), dim3(kBlock), 0, s, b);
    // Places by workgroup: 4096 particles each where that leaves 128 of them,
    // 1024 where few tiles make one atomic per wave contend (131072 particles
    // on 45 tiles: 73 us per call against 291), else by wave (a million on 1377
    // tiles that a short workgroup would read out: 239 us against 511).
    if (ntiles <= kLdsTiles && q.n >= 128 * kBlock * 16)
      hipLaunchKernelGGL((k_dep_place<16, true>), dim3(grid_for((q.n + 15) / 16)), dim3(kBlock),
                         0, s, b, q.n);
    else if (ntiles <= 4 * kBlock)
      hipLaunchKernelGGL((k_dep_place<4, true>), dim3(grid_for((q.n + 3) / 4)), dim3(kBlock), 0,
                         s, b, q.n);
    else
      hipLaunchKernelGGL((k_dep_place<1, false>), dim3(grid_for(q.n)), dim3(kBlock), 0, s, b,
                         q.n);
    const size_t items = (size_t)q.n / b.run + (size_t)(ntiles < q.n ? ntiles : q.n);
    hipLaunchKernelGGL(k_tile_deposit<T>, dim3((unsigned)items), dim3(4 * kDepCells), 0, s, g,
                       q, m, b);
    e = hipGetLastError();
    return e == hipSuccess;
  });
  const hipError_t ef = stream_free(w, s);
  return e != hipSuccess ? e : ef;
}

template <typename T>
hipError_t launch_mover(const KGrid<T> &g, const KField<T> &f,
                        const KPart<T> &p, const KPush<T> &k,
                        unsigned int *status, hipStream_t s) {
  if (p.n <= 0) return hipSuccess;
  const int nn = g.nxn * g.nyn * g.nzn;
  T *rec = nullptr;
  if (pack_pays(p.n, nn) && stream_may_alloc(s) &&
      stream_alloc((void **)&rec, sizeof(T) * PackedField<T>::kRec * (size_t)nn, s) !=
          hipSuccess) {
    (void)hipGetLastError();  // the fields as they are need no scratch
    rec = nullptr;
  }
  if (!rec) {
    hipLaunchKernelGGL((k_mover<T, KField<T>>), dim3(grid_for(p.n)), dim3(kBlock), 0, s, g, f,
                       p, k, status);
    return hipGetLastError();
  }
  const PackedField<T> packed{rec};
  pack_fields(f, packed, nn, s);
  hipLaunchKernelGGL((k_mover<T, PackedField<T>>), dim3(grid_for(p.n)), dim3(kBlock), 0, s, g,
                     packed, p, k, status);
  const hipError_t e = hipGetLastError(), ef = stream_free(rec, s);
  return e != hipSuccess ? e : ef;
}

// k_deposit in launches of fewer than 2^32 threads.
template <typename T>
hipError_t direct_deposit(const KGrid<T> &g, const KPart<T> &p, const KMom &m,
                          unsigned int *status, hipStream_t s) {
  hipError_t e = hipSuccess;
  for_slices(p.n, 1 << 30, [&](int64_t first, int64_t count) {
    const KPart<T> q = part_slice(p, first, count);
    hipLaunchKernelGGL(k_deposit<T>, dim3((q.n - 1) / kRun + 1), dim3(64), 0, s, g, q, m, status);
    e = hipGetLastError();
    return e == hipSuccess;
  });
  return e;
}

template <typename T>
hipError_t launch_deposit(const KGrid<T> &g, const KPart<T> &p, const KMom &m,
                          unsigned int *status, hipStream_t s) {
  if (p.n <= 0) return hipSuccess;
  bool taken;
  const hipError_t e = tile_deposit<T>(g, nullptr, p, nullptr, m, status, s, taken);
  if (taken) return e;
  return direct_deposit<T>(g, p, m, status, s);
}

template <typename T>
hipError_t launch_mover_deposit(const KGrid<T> &g, const KField<T> &f,
                                const KPart<T> &p, const KPush<T> &k,
                                const KMom &m, unsigned int *status,
                                hipStream_t s) {
  if (p.n <= 0) return hipSuccess;
  bool taken;
  const hipError_t e = tile_deposit<T>(g, &f, p, &k, m, status, s, taken);
  if (taken) return e;
  const hipError_t em = launch_mover<T>(g, f, p, k, status, s);
  if (em != hipSuccess) return em;
  return direct_deposit<T>(g, p, m, status, s);
}

#define SPIC_INSTANTIATE(T)                                                   \
  template hipError_t launch_mover<T>(const KGrid<T> &, const KField<T> &,    \
                                      const KPart<T> &, const KPush<T> &,     \
                                      unsigned int *, hipStream_t);           \
  template hipError_t launch_deposit<T>(const KGrid<T> &, const KPart<T> &,   \
                                        const KMom &, unsigned int *,         \
                                        hipStream_t);                         \
  template hipError_t launch_mover_deposit<T>(                                \
      const KGrid<T> &, const KField<T> &, const KPart<T> &,                  \
      const KPush<T> &, const KMom &, unsigned int *, hipStream_t);
SPIC_INSTANTIATE(double)
SPIC_INSTANTIATE(float)
#undef SPIC_INSTANTIATE

}  // namespace SPIC_NS
}  // namespace spic
