// spic_binsort.hip -- binned particle storage: the sort that (re)builds it,
// the store back to the caller's order, the per-node reduction of the
// phase kernel's tile partials, and the count reset before each phase.
//
// Sort.  A particle's cell is its deposit cell 2 + floor((p - start) * inv)
// minus the two guard offsets, clamped to the physical cells; its rank is
// a per-cell counter taken with an atomic.  The key
//   tile | rank within the cell | cell within the tile
// orders each tile's particles round-robin over its cells (every cell's
// first particle, then every cell's second, ...), so that any run of
// 4 * cells-per-tile consecutive particles holds about four per cell: the
// phase kernel sums one such run per batch cell by cell, and
// particles that stay in their tile keep this order from phase to phase.
// Most loads get there by tiles (counts, places and one workgroup per tile;
// load_through_tiles); the others, and a binned source, by a stable LSD radix sort
// (rocPRIM) of (key, source slot) pairs, whose result is the
// permutation; the seven arrays and the particle id are gathered to sorted
// position i + tile * slack, so that every segment gets `slack` free slots
// after its particles.  A binned source is enumerated densely through an
// exclusive scan of its counts.
#include <cstring>

#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>

#include "spic_binned.hpp"
#include "spic_wave.hpp"

namespace spic {
namespace {

inline unsigned nblocks(long n, int tpb = 256) {
  long b = (n + tpb - 1) / tpb;
  if (b < 1) b = 1;
  if (b > (1L << 20)) b = 1L << 20;
  return (unsigned)b;
}

inline size_t align_up(size_t v) { return (v + 255) & ~size_t(255); }

template <typename TS, typename T>
__device__ __forceinline__ int phys_cell(TS p, double start, T inv, int nc) {
  double c = floor(((double)p - start) * (double)inv);
  c = fmin(fmax(c, 0.0), (double)(nc - 1));
  return (int)c;
}

// Fixed-point positions (FixedParams): a length from the caller's arrays
// to the int32 coordinate along axis a, rounded to nearest and bounded to
// the box plus 32 cells either side (a position farther out is reported
// by the phase as out of the grid); and back.
__device__ __forceinline__ int to_fixed_pos(double p, const FixedParams &f, int a) {
  const double ext = (double)(32 << f.k[a]);
  double X = rint((p - f.start[a]) * f.to_fixed[a]);
  X = fmin(fmax(X, -ext), (double)f.lim[a] + ext);
  return (int)X;
}

__device__ __forceinline__ double from_fixed_pos(int X, const FixedParams &f, int a) {
  return f.start[a] + (double)X * f.from_fixed[a];
}

// Particles per range of a binned source (tiles, then the overflow region).
__global__ void k_range_counts(const int64_t *__restrict__ seg,
                               const unsigned int *__restrict__ cnt,
                               unsigned int ovf_cap, int ntiles,
                               unsigned int *__restrict__ out) {
  for (int t = blockIdx.x * blockDim.x + threadIdx.x; t <= ntiles;
       t += gridDim.x * blockDim.x)
    out[t] = (unsigned int)range_view(seg, cnt, ntiles, ovf_cap, t).count;
}


// Rank of this lane's particle among the active lanes of its wave that
// share `key`, plus the count already in counter[key]: one atomic per
// distinct key in the wave (few when the input is in cell order).
__device__ __forceinline__ uint32_t wave_rank(unsigned int *counter, uint32_t key,
                                              bool active) {
  const int lane = __lane_id();
  const unsigned long long below = (1ull << lane) - 1ull;
  unsigned long long todo = __ballot(active);
  uint32_t rank = 0;
  while (todo) {
    const int leader = __ffsll((long long)todo) - 1;
    const uint32_t lkey = __shfl(key, leader);
    const unsigned long long same = __ballot(active && key == lkey);
    unsigned int base = 0;
    if (lane == leader) base = atomicAdd(&counter[lkey], (unsigned int)__popcll(same));
    base = __shfl(base, leader);
    if (active && key == lkey) rank = base + (uint32_t)__popcll(same & below);
    todo &= ~same;
  }
  return rank;
}

// Key of one particle: tile | rank of the particle within its cell | cell
// within the tile.  `binned`: the position comes from engine storage, in
// fixed point when the layout says so (else from the caller's arrays).
template <typename TS, typename T>
__device__ __forceinline__ void cell_of(const KGrid<T> &g, const BinLayout &L, TS x, TS y,
                                        TS z, int &cx, int &cy, int &cz, uint32_t &tile,
                                        uint32_t &cit, bool binned = true) {
  if constexpr (sizeof(TS) == 4) {
    if (binned && L.fixed) {
      cx = min(max(__float_as_int((float)x) >> L.fx.k[0], 0), L.ncx - 1);
      cy = min(max(__float_as_int((float)y) >> L.fx.k[1], 0), L.ncy - 1);
      cz = min(max(__float_as_int((float)z) >> L.fx.k[2], 0), L.ncz - 1);
    } else {
      cx = phys_cell(x, g.xStart, g.invdx, L.ncx);
      cy = phys_cell(y, g.yStart, g.invdy, L.ncy);
      cz = phys_cell(z, g.zStart, g.invdz, L.ncz);
    }
  } else {
    cx = phys_cell(x, g.xStart, g.invdx, L.ncx);
    cy = phys_cell(y, g.yStart, g.invdy, L.ncy);
    cz = phys_cell(z, g.zStart, g.invdz, L.ncz);
  }
  const int tx = cx / L.tx, ty = cy / L.ty, tz = cz / L.tz;
  tile = (uint32_t)((tx * L.nty + ty) * L.ntz + tz);
  cit = (uint32_t)(((cx - tx * L.tx) * L.ty + (cy - ty * L.ty)) * L.tz + (cz - tz * L.tz));
}

// Keys of a dense source (particles 0..n-1 in the caller's order, element
// type TS), ranks from per-cell counters with wave-aggregated atomics.
template <typename TS, typename T>
__global__ void k_bin_keys(KGrid<T> g, BinLayout L, int64_t n,
                           const TS *__restrict__ x, const TS *__restrict__ y,
                           const TS *__restrict__ z, unsigned int *__restrict__ cell_count,
                           uint32_t *__restrict__ key, uint32_t *__restrict__ idx) {
  const uint32_t rank_max = (1u << L.rank_bits) - 1u;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  const int64_t n_up = (n + 63) / 64 * 64;  // whole waves stay in the loop
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n_up; i += stride) {
    const bool active = i < n;
    int cx = 0, cy = 0, cz = 0;
    uint32_t tile = 0, cit = 0;
    if (active) cell_of(g, L, x[i], y[i], z[i], cx, cy, cz, tile, cit, false);
    const uint32_t cell = (uint32_t)(((int64_t)cx * L.ncy + cy) * L.ncz + cz);
    uint32_t r = wave_rank(cell_count, cell, active);
    if (!active) continue;
    r = r < rank_max ? r : rank_max;
    key[i] = (tile << (L.rank_bits + L.cell_bits)) | (r << L.cell_bits) | cit;
    idx[i] = (uint32_t)i;
  }
}

// Keys of a binned source: block t takes range t (a tile's segment, or
// t == ntiles: the overflow region), whose particles land at dense
// positions P[t] + r.  A tile's own particles take their rank from LDS
// counters of its cells; others (overflow region) from the global ones.
// Equal ranks of one cell from the two sources only make equal keys.
template <typename T>
__global__ __launch_bounds__(256) void k_bin_keys_binned(
    KGrid<T> g, BinLayout L, const T *__restrict__ x, const T *__restrict__ y,
    const T *__restrict__ z, const unsigned int *__restrict__ P,
    const int64_t *__restrict__ seg, const unsigned int *__restrict__ cnt,
    unsigned int ovf_cap, unsigned int *__restrict__ cell_count, uint32_t *__restrict__ key,
    uint32_t *__restrict__ idx) {
  __shared__ unsigned int s_cnt[kMaxTileCells];
  const uint32_t rank_max = (1u << L.rank_bits) - 1u;
  const int t = blockIdx.x;
  const int ncells = L.tx * L.ty * L.tz;
  for (int c = threadIdx.x; c < ncells; c += blockDim.x) s_cnt[c] = 0u;
  __syncthreads();
  const RangeView v = range_view(seg, cnt, L.ntiles, ovf_cap, t);
  const int64_t base = P[t];
  for (int64_t r = threadIdx.x; r < v.count; r += blockDim.x) {
    const int64_t j = v.slot(r);
    int cx, cy, cz;
    uint32_t tile, cit;
    cell_of(g, L, x[j], y[j], z[j], cx, cy, cz, tile, cit);
    uint32_t rk;
    if ((int)tile == t) rk = atomicAdd(&s_cnt[cit], 1u);
    else rk = atomicAdd(&cell_count[((size_t)cx * L.ncy + cy) * L.ncz + cz], 1u);
    rk = rk < rank_max ? rk : rank_max;
    key[base + r] = (tile << (L.rank_bits + L.cell_bits)) | (rk << L.cell_bits) | cit;
    idx[base + r] = (uint32_t)j;
  }
}

__global__ void k_zero_u32(unsigned int *p, int64_t n) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    p[i] = 0u;
}

template <typename T>
struct Arrays7 {
  T *p[7];
};

// The sorted gather into binned storage.  A dense source (src_id null)
// holds the caller's values in TS: with fixed-point storage (to_fixed) its
// positions are converted, the rest rounded to T; a binned source is the
// engine's own storage, copied word for word.
template <typename TS, typename T>
__global__ void k_bin_gather(Arrays7<TS> src, const uint32_t *__restrict__ src_id,
                             const uint32_t *__restrict__ perm,
                             const uint32_t *__restrict__ keys, int shift, int64_t n,
                             int64_t slack, Arrays7<T> dst, uint32_t *__restrict__ dst_id,
                             int to_fixed, FixedParams fx) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const uint32_t j = perm[i];
    const int64_t o = i + (int64_t)(keys[i] >> shift) * slack;
#pragma unroll
    for (int a = 0; a < 7; ++a) {
      if constexpr (sizeof(T) == 4) {
        if (a < 3 && to_fixed) {
          dst.p[a][o] = __int_as_float(to_fixed_pos((double)src.p[a][j], fx, a));
          continue;
        }
      }
      dst.p[a][o] = (T)src.p[a][j];
    }
    if (dst_id) dst_id[o] = src_id ? src_id[j] : j;
  }
}

// ---- load through tiles ----------------------------------------------------
//
// A dense source is counted into tiles, its indices are placed tile by tile,
// and one workgroup per tile ranks its particles per cell and gathers them in
// round-robin order.  4.0M FP64 particles that have drifted two cells from
// their cell order: 262 us (gather 193, the rest counts and places) against
// 735 us for keys, radix sort and gather.  Most of a line's particles then lie
// in different tiles: 490 MB are fetched for 232 MB of particles, 3.7 TB/s in
// all.  Gathering component by component over all tiles instead fetches 797 MB
// (281 us).  Which loads go this way: load_through_tiles.
constexpr int kLoadThreads = 1024;
constexpr int kLoadManyTiles = 16384;
constexpr int kLoadPer = 8;      // particles per thread that a tile's workgroup holds
constexpr int kLoadHeld = kLoadThreads * kLoadPer;
constexpr int kLoadRanks = 128;   // ranks in the slot tables
constexpr int kLoadSorted = 512;  // particles of a cell that are put in caller order
constexpr int kStoreThreads = 512;
constexpr int kStorePer = 8;
constexpr int kStoreHeld = kStoreThreads * kStorePer;
constexpr int kStoreLines = 512;  // line counters of a store
// Particles per tile from which a store groups them by line: with 128 a
// workgroup is mostly idle (230k FP64 particles: 25 us grouped, 19 direct), 512
// take 13.0 against 14.6, 1728 237 against 534 (3.1M).
constexpr int kStoreMinTile = 512;

struct LoadBins {
  int64_t n;
  int per;                 // particles per thread of the count
  unsigned int *count;     // [ntiles] particles per tile
  unsigned int *next;      // [ntiles] places taken in each tile
  const int64_t *seg;      // the segments: tile t's places begin at seg[t] - t * slack
  uint32_t *where;         // [n] tile | cell in the tile (cell_bits)
  uint32_t *perm;          // [n] by place: index of the particle
  // tiles of more than kLoadHeld particles, in pieces of that many
  unsigned int *big;       // [0] pieces, [1] such tiles
  uint4 *pieces;           // tile, number among those tiles, first place, 0
  unsigned int *cells;     // [2 NC] of each such tile: particles per cell, ranks taken
  int tile_blocks;         // workgroups of whole tiles, before those of pieces
};

// Counts the particles into tiles, NT threads per workgroup, which counts up to
// LT tiles in LDS and adds each tile it met once; LT = 0: one atomic per wave and
// tile in global memory.
template <typename TS, typename T, int NT, int LT>
__global__ __launch_bounds__(NT) void k_load_count(KGrid<T> g, BinLayout L, LoadBins b,
                                                   const TS *__restrict__ x,
                                                   const TS *__restrict__ y,
                                                   const TS *__restrict__ z) {
  __shared__ unsigned int s_cnt[LT > 0 ? LT : 1];
  const int tid = threadIdx.x;
  if constexpr (LT > 0) {
    for (int t = tid; t < L.ntiles; t += NT) s_cnt[t] = 0u;
    __syncthreads();
  }
  const int64_t first = blockIdx.x * (int64_t)(NT * b.per);
  for (int e = 0; e < b.per; ++e) {
    const int64_t i = first + e * NT + tid;
    const bool active = i < b.n;
    uint32_t tile = 0, cit = 0;
    if (active) {
      int cx, cy, cz;
      cell_of(g, L, x[i], y[i], z[i], cx, cy, cz, tile, cit, false);
      b.where[i] = (tile << L.cell_bits) | cit;
    }
    key_rank(LT > 0 ? s_cnt : b.count, tile, active);
  }
  if constexpr (LT > 0) {
    __syncthreads();
    for (int t = tid; t < L.ntiles; t += NT)
      if (s_cnt[t]) atomicAdd(b.count + t, s_cnt[t]);
  }
}

// Places each particle's index in its tile: each tile's places at once per
// workgroup (LT > 0), PER particles per thread, or per wave.
template <int PER, int NT, int LT>
__global__ __launch_bounds__(NT) void k_load_place(BinLayout L, LoadBins b) {
  __shared__ unsigned int s_cnt[LT > 0 ? LT : 1];
  const int tid = threadIdx.x;
  const int64_t first = blockIdx.x * (int64_t)(NT * PER);
  unsigned int t[PER], r[PER];
#pragma unroll
  for (int e = 0; e < PER; ++e) {
    const int64_t i = first + e * NT + tid;
    t[e] = i < b.n ? b.where[i] >> L.cell_bits : 0u;
  }
  if constexpr (LT > 0) {
    for (int k = tid; k < L.ntiles; k += NT) s_cnt[k] = 0u;
    __syncthreads();
  }
#pragma unroll
  for (int e = 0; e < PER; ++e)
    r[e] = key_rank(LT > 0 ? s_cnt : b.next, t[e], first + e * NT + tid < b.n);
  if constexpr (LT > 0) {
    __syncthreads();
    for (int k = tid; k < L.ntiles; k += NT)
      if (s_cnt[k]) s_cnt[k] = atomicAdd(b.next + k, s_cnt[k]);
    __syncthreads();
  }
#pragma unroll
  for (int e = 0; e < PER; ++e) {
    const int64_t i = first + e * NT + tid;
    if (i < b.n)
      b.perm[b.seg[t[e]] - (int64_t)t[e] * L.slack + (LT > 0 ? s_cnt[t[e]] : 0u) + r[e]] =
          (uint32_t)i;
  }
}

// A caller's value into binned storage: with fixed-point storage positions
// are converted, everything else is rounded to T.
template <typename TS, typename T>
__device__ __forceinline__ T load_value(TS v, int a, int fixed, const FixedParams &fx) {
  if constexpr (sizeof(T) == 4) {
    if (a < 3 && fixed) return __int_as_float(to_fixed_pos((double)v, fx, a));
  }
  return (T)v;
}

// One workgroup per tile, tiles in runs per XCD: counts its cells, ranks each
// particle within its cell, turns the rank into its slot in round-robin order
// (slot of the k-th particle of cell c: particles of rank < k over all cells,
// plus the cells before c that hold more than k; tables up to kLoadRanks ranks,
// a loop over the cells beyond), then takes the components one after another:
// read in the order of the places, where neighbours of the caller's arrays are
// mostly neighbours, put at their slots in LDS and written in order.
//
// The places come in no particular order (atomics, workgroup by workgroup), the
// ranks do: a cell's particles keep the caller's order, so that a load of the
// same arrays always gives the same storage.  The indices are put in LDS cell by cell and each counts the smaller ones
// of its cell, whole waves over one run of indices (the LDS reads are broadcast):
// 4.0M FP64 particles on 1024 tiles 1 to 3% more for the load.
// Cells of more than kLoadSorted particles keep the order of their places: the
// count grows with the square.
// A tile of more than kLoadHeld particles is taken in pieces, a workgroup each:
// the cells are counted over all of them first (k_load_pieces), a piece takes its
// ranks of each cell at once, in the order of the places, and writes every
// particle at its slot.  3.6M of 4.0M FP64 particles in one of 512 tiles:
// 0.94 ms (one workgroup for the tile 50, the radix sort 2.4), in one cell of it
// 0.32 (25, 1.08).  Where no tile is that full the two additions cost 3 us.
template <int NC>
__global__ __launch_bounds__(kLoadThreads) void k_load_pieces(BinLayout L, LoadBins b) {
  __shared__ unsigned int s_count[NC];
  if (blockIdx.x >= b.big[0]) return;
  const int tid = threadIdx.x;
  const uint4 piece = b.pieces[blockIdx.x];
  const int t = (int)piece.x;
  const int n = min(b.count[t] - piece.z, (unsigned)kLoadHeld);
  const uint32_t *perm = b.perm + (b.seg[t] - (int64_t)t * L.slack) + piece.z;
  const uint32_t mask = (1u << L.cell_bits) - 1u;
  if (tid < NC) s_count[tid] = 0u;
  __syncthreads();
  for (int r = tid; r < (n + 63) / 64 * 64; r += kLoadThreads)
    key_rank(s_count, r < n ? b.where[perm[r]] & mask : 0u, r < n);
  __syncthreads();
  if (tid < NC && s_count[tid]) atomicAdd(b.cells + (size_t)piece.y * 2 * NC + tid, s_count[tid]);
}

template <typename TS, typename T, int NC>
__global__ __launch_bounds__(kLoadThreads) __attribute__((amdgpu_waves_per_eu(8)))
void k_load_tile(BinLayout L, LoadBins b, Arrays7<TS> src, Arrays7<T> dst, uint32_t *dst_id) {
  // particles per cell; a whole tile's first place of each cell's indices, or
  // the first rank of a piece's in each cell
  __shared__ unsigned int s_count[NC], s_first[NC], s_A[kLoadRanks];
  __shared__ unsigned char s_T[NC][kLoadRanks];
  // the indices and their cells, cell by cell; then values by slot
  __shared__ unsigned char s_cell[kLoadHeld];
  constexpr int kStage = kLoadHeld * 4 / (int)sizeof(T);  // values: 32 KB
  __shared__ T s_stage[kStage];
  uint32_t *const s_key = reinterpret_cast<uint32_t *>(s_stage);
  const int tid = threadIdx.x;
  const bool whole = (int)blockIdx.x < b.tile_blocks;
  int t;
  uint4 piece = make_uint4(0u, 0u, 0u, 0u);
  if (whole) {
    t = (int)((blockIdx.x % 8) * (b.tile_blocks / 8) + blockIdx.x / 8);
    if (t >= L.ntiles || b.count[t] == 0u || b.count[t] > (unsigned)kLoadHeld) return;
  } else {
    if (blockIdx.x - b.tile_blocks >= b.big[0]) return;
    piece = b.pieces[blockIdx.x - b.tile_blocks];
    t = (int)piece.x;
  }
  const int64_t out0 = b.seg[t];
  const int n = min(b.count[t] - piece.z, (unsigned)kLoadHeld);
  const uint32_t *perm = b.perm + (out0 - (int64_t)t * L.slack) + piece.z;
  const uint32_t mask = (1u << L.cell_bits) - 1u;
  if (tid < NC) s_count[tid] = 0u;
  __syncthreads();
  uint32_t j[kLoadPer], pos[kLoadPer];  // index; rank and cell, then slot
#pragma unroll
  for (int e = 0; e < kLoadPer; ++e) {
    const int r = e * kLoadThreads + tid;
    if (r < n) j[e] = perm[r];
  }
#pragma unroll
  for (int e = 0; e < kLoadPer; ++e)
    if (e * kLoadThreads + tid < n) pos[e] = b.where[j[e]] & mask;
#pragma unroll
  for (int e = 0; e < kLoadPer; ++e)
    if (e * kLoadThreads + tid < n) pos[e] |= atomicAdd(&s_count[pos[e]], 1u) << 8;
  __syncthreads();
  if (!whole) {
    if (tid < NC) {
      unsigned int *cells = b.cells + (size_t)piece.y * 2 * NC;
      s_first[tid] = s_count[tid] ? atomicAdd(cells + NC + tid, s_count[tid]) : 0u;
      s_count[tid] = cells[tid];
    }
    __syncthreads();
  }
  if (tid < kLoadRanks) {
    unsigned int a = 0, before = 0;
#pragma unroll 8
    for (int c = 0; c < NC; ++c) {
      const unsigned int m = s_count[c];
      a += m < (unsigned)tid ? m : (unsigned)tid;
      s_T[c][tid] = (unsigned char)before;
      before += m > (unsigned)tid ? 1u : 0u;
    }
    s_A[tid] = a;
  } else if (whole && tid < kLoadRanks + NC) {
    unsigned int before = 0;
#pragma unroll 8
    for (int c = 0; c < NC; ++c) before += c < tid - kLoadRanks ? s_count[c] : 0u;
    s_first[tid - kLoadRanks] = before;
  }
  __syncthreads();
  auto slot = [&](unsigned int c, unsigned int k) -> unsigned int {
    if (k < (unsigned)kLoadRanks) return s_A[k] + s_T[c][k];
    unsigned int p = 0;
#pragma unroll 4
    for (int cc = 0; cc < NC; ++cc) {
      const unsigned int m = s_count[cc];
      p += m < k ? m : k;
      if (cc < (int)c && m > k) ++p;
    }
    return p;
  };
  if (!whole) {
#pragma unroll
    for (int e = 0; e < kLoadPer; ++e)
      if (e * kLoadThreads + tid < n) {
        const unsigned int c = pos[e] & 0xffu;
        const int64_t o = out0 + slot(c, s_first[c] + (pos[e] >> 8));
#pragma unroll
        for (int a = 0; a < 7; ++a) dst.p[a][o] = load_value<TS, T>(src.p[a][j[e]], a, L.fixed, L.fx);
        if (dst_id) dst_id[o] = j[e];
      }
    return;
  }
#pragma unroll
  for (int e = 0; e < kLoadPer; ++e)
    if (e * kLoadThreads + tid < n) {
      const unsigned int c = pos[e] & 0xffu, at = s_first[c] + (pos[e] >> 8);
      s_key[at] = j[e];
      s_cell[at] = (unsigned char)c;
      pos[e] = at;
    }
  __syncthreads();
  uint32_t rank[kLoadPer];  // of the index at place e * kLoadThreads + tid
#pragma unroll
  for (int e = 0; e < kLoadPer; ++e) {
    const int at = e * kLoadThreads + tid;
    if (at >= n) break;
    const unsigned int c = s_cell[at], first = s_first[c], m = s_count[c];
    rank[e] = (unsigned)at - first;
    if (m <= (unsigned)kLoadSorted) {
      const uint32_t key = s_key[at];
      rank[e] = 0u;
#pragma unroll 4
      for (unsigned int i = 0; i < m; ++i) rank[e] += s_key[first + i] < key ? 1u : 0u;
    }
  }
  __syncthreads();
#pragma unroll
  for (int e = 0; e < kLoadPer; ++e)
    if (e * kLoadThreads + tid < n) s_key[e * kLoadThreads + tid] = rank[e];
  __syncthreads();
#pragma unroll
  for (int e = 0; e < kLoadPer; ++e)
    if (e * kLoadThreads + tid < n) pos[e] = slot(s_cell[pos[e]], s_key[pos[e]]);
  __syncthreads();
#pragma unroll
  for (int a = 0; a < 7; ++a) {
    T val[kLoadPer];
#pragma unroll
    for (int e = 0; e < kLoadPer; ++e)
      if (e * kLoadThreads + tid < n)
        val[e] = load_value<TS, T>(src.p[a][j[e]], a, L.fixed, L.fx);
    T *__restrict__ to = dst.p[a] + out0;
    for (int c0 = 0; c0 < n; c0 += kStage) {
#pragma unroll
      for (int e = 0; e < kLoadPer; ++e)
        if (e * kLoadThreads + tid < n && pos[e] - c0 < (unsigned)kStage)
          s_stage[pos[e] - c0] = val[e];
      __syncthreads();
      const int m = min(n - c0, kStage);
      for (int p = tid; p < m; p += kLoadThreads) to[c0 + p] = s_stage[p];
      __syncthreads();
    }
  }
  if (!dst_id) return;
  uint32_t *s_id = reinterpret_cast<uint32_t *>(s_stage);
  for (int c0 = 0; c0 < n; c0 += kStage) {
#pragma unroll
    for (int e = 0; e < kLoadPer; ++e)
      if (e * kLoadThreads + tid < n && pos[e] - c0 < (unsigned)kStage)
        s_id[pos[e] - c0] = j[e];
    __syncthreads();
    const int m = min(n - c0, kStage);
    for (int p = tid; p < m; p += kLoadThreads) dst_id[out0 + c0 + p] = s_id[p];
    __syncthreads();
  }
}

// seg[t] = (first sorted position of tile >= t) + t * slack; cnt from the
// differences, no unused runs; the overflow region starts empty.
__global__ void k_bin_bounds(const uint32_t *__restrict__ keys, int shift, int64_t n,
                             int ntiles, int64_t slack, int64_t *__restrict__ seg,
                             unsigned int *__restrict__ cnt) {
  for (int t = blockIdx.x * blockDim.x + threadIdx.x; t <= ntiles;
       t += gridDim.x * blockDim.x) {
    int64_t b[2];
    for (int k = 0; k < 2; ++k) {
      const int64_t tt = t + k;
      int64_t lo = 0, hi = n;
      while (lo < hi) {
        const int64_t mid = lo + ((hi - lo) >> 1);
        if ((int64_t)(keys[mid] >> shift) < tt) lo = mid + 1;
        else hi = mid;
      }
      b[k] = lo;
    }
    seg[t] = b[0] + (int64_t)t * slack;
    cnt[t] = t < ntiles ? (unsigned int)(b[1] - b[0]) : 0u;
    cnt[(ntiles + 1) + t] = 0u;
    cnt[2 * (ntiles + 1) + t] = 0u;
    cnt[3 * (ntiles + 1) + t] = 0u;
  }
}

// Big-endian IEEE float32 bits of v rounded to float (H5T_IEEE_F32BE).
template <typename T>
__device__ __forceinline__ uint32_t be32(T v) {
  return __builtin_bswap32(__float_as_uint((float)v));
}

// A stored value out of binned storage in the caller's element type TD:
// fixed-point positions converted back; with NA = 6 (a snapshot) as big-endian
// float32 words.
template <typename T, typename TD, int NA>
__device__ __forceinline__ TD store_value(T v, int a, int fixed, const FixedParams &fx) {
  if constexpr (sizeof(T) == 4) {
    if (a < 3 && fixed) {
      const double p = from_fixed_pos(__float_as_int((float)v), fx, a);
      if constexpr (NA == 6) return be32(p);
      else return (TD)p;
    }
  }
  if constexpr (NA == 6) return be32(v);
  else return (TD)v;
}

// Each particle of a segment (one workgroup each, then the overflow region)
// straight to its place: dst[id] = src, or, in an engine without ids, densely
// in storage order.
template <typename T, typename TD, int NA>
__global__ __launch_bounds__(256) void k_bin_store(
    Arrays7<T> src, const uint32_t *__restrict__ id, const uint32_t *__restrict__ base,
    const int64_t *__restrict__ seg, const unsigned int *__restrict__ cnt,
    unsigned int ovf_cap, int ntiles, Arrays7<TD> dst, int fixed, FixedParams fx) {
  const RangeView v = range_view(seg, cnt, ntiles, ovf_cap, (int)blockIdx.x);
  for (int64_t r = threadIdx.x; r < v.count; r += 256) {
    const int64_t i = v.slot(r);
    const uint32_t k = id ? id[i] : base[blockIdx.x] + (uint32_t)r;
#pragma unroll
    for (int a = 0; a < NA; ++a)
      dst.p[a][k] = store_value<T, TD, NA>(src.p[a][i], a, fixed, fx);
  }
}

// One workgroup per segment (then the overflow region), in runs per XCD:
// dst[id] = src.  Particles of one line of the caller's arrays lie all over
// the segment (round-robin over the cells); written in storage order, a line
// goes out in parts, one per particle.  Here up to kStoreHeld particles are
// grouped by that line first (counts by line modulo kStoreLines, a scan, a
// placement), then the components follow one another: read in storage order,
// put at their places in LDS, written line by line.  4.0M FP64 particles, two
// cells from their cell order: 300 us against 601 straight to their places
// (particles of a line that lie in other tiles still make partial writes: 706
// MB go out for 224 MB).  Not faster: slots inverted first and the particles
// read at them in load order, 378 us; component by component over all tiles,
// 469; 1024 threads for up to 8192 particles, 294 to 312 with spills.
template <typename T, typename TD, int NA>
__global__ __launch_bounds__(kStoreThreads) __attribute__((amdgpu_waves_per_eu(6)))
void k_store_tile(Arrays7<T> src, const uint32_t *__restrict__ id,
                  const int64_t *__restrict__ seg, const unsigned int *__restrict__ cnt,
                  unsigned int ovf_cap, int ntiles, Arrays7<TD> dst, int fixed,
                  FixedParams fx) {
  constexpr unsigned int kLine = 128 / sizeof(TD);
  __shared__ unsigned int s_line[kStoreLines];
  __shared__ unsigned int s_wave[kStoreLines / 64];
  __shared__ uint32_t s_id[kStoreHeld];
  __shared__ T s_stage[kStoreHeld];
  __shared__ const T *s_from[NA];
  __shared__ TD *s_to[NA];
  static_assert(kStoreLines == kStoreThreads, "a thread per counter");
  const int t = (int)((blockIdx.x % 8) * (gridDim.x / 8) + blockIdx.x / 8);
  if (t > ntiles) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const RangeView v = range_view(seg, cnt, ntiles, ovf_cap, t);
  if (tid < NA) {
#pragma unroll
    for (int a = 0; a < NA; ++a)
      if (tid == a) {
        s_from[a] = src.p[a] + v.first;
        s_to[a] = dst.p[a];
      }
  }
  // a slot's offset within the range fits 32 bits
  auto at = [&v](uint32_t r) { return r < v.gap_lo ? r : r + v.gap_len; };
  const uint32_t count = (uint32_t)v.count;
  for (uint32_t first = 0; first < count; first += kStoreHeld) {
    const int n = (int)min(count - first, (uint32_t)kStoreHeld);
    s_line[tid] = 0u;
    __syncthreads();
    uint32_t k[kStorePer], pos[kStorePer];
#pragma unroll
    for (int e = 0; e < kStorePer; ++e) {
      const int r = e * kStoreThreads + tid;
      if (r < n) k[e] = (id + v.first)[at(first + r)];
    }
#pragma unroll
    for (int e = 0; e < kStorePer; ++e)
      if (e * kStoreThreads + tid < n)
        pos[e] = atomicAdd(&s_line[k[e] / kLine % kStoreLines], 1u);
    __syncthreads();
    const unsigned int c = s_line[tid];
    unsigned int sum = c;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const unsigned int u = __shfl_up(sum, d);
      if (lane >= d) sum += u;
    }
    if (lane == 63) s_wave[tid >> 6] = sum;
    __syncthreads();
    sum -= c;
    for (int w = 0; w < (tid >> 6); ++w) sum += s_wave[w];
    s_line[tid] = sum;
    __syncthreads();
#pragma unroll
    for (int e = 0; e < kStorePer; ++e)
      if (e * kStoreThreads + tid < n) {
        pos[e] += s_line[k[e] / kLine % kStoreLines];
        s_id[pos[e]] = k[e];
      }
    // a loop of its own per component: unrolled, the loads of the next ones
    // are moved ahead and spill
#pragma unroll 1
    for (int a = 0; a < NA; ++a) {
      const SPIC_GLOBAL T *from = gmem(s_from[a]);
      SPIC_GLOBAL TD *to = gmem(s_to[a]);
      T val[kStorePer];
#pragma unroll
      for (int e = 0; e < kStorePer; ++e) {
        const int r = e * kStoreThreads + tid;
        if (r < n) val[e] = from[at(first + r)];
      }
#pragma unroll
      for (int e = 0; e < kStorePer; ++e)
        if (e * kStoreThreads + tid < n) s_stage[pos[e]] = val[e];
      __syncthreads();
      for (int p = tid; p < n; p += kStoreThreads)
        to[s_id[p]] = store_value<T, TD, NA>(s_stage[p], a, fixed, fx);
      __syncthreads();
    }
  }
}

// Workgroup b of nb (layout_blocks), 256 threads each, writes its part of the
// output buffer's segments of a species: the input buffer's, or, when its
// overflow region holds more than kRelayoutOverflow particles, segments of each
// tile's particles plus its share of the slack, half of it even and half in
// proportion to the particles (arrivals grow with them).  Both halves are rounded
// down, so the segments take at most n + ntiles * slack slots and the overflow
// region after them stays inside the buffer.  A workgroup adds up the tiles before
// its own by itself: half a million tiles by one workgroup took 1.7 of 25.7 ms of a
// phase of 33.5M particles.
__device__ __forceinline__ void phase_layout(const LayoutArgs &l, int ntiles, int b, int nb) {
  __shared__ unsigned long long s_sum[4];
  const SPIC_GLOBAL int64_t *in = gmem(l.seg_in);
  SPIC_GLOBAL int64_t *out = gmem(l.seg_out);
  const SPIC_GLOBAL unsigned int *cnt = gmem(l.cnt_in);
  const int tid = threadIdx.x, lane = tid & 63;
  const int chunk = (ntiles + nb - 1) / nb;
  const int t0 = min(b * chunk, ntiles), t1 = min(t0 + chunk, ntiles);
  if (cnt[ntiles] <= kRelayoutOverflow) {
    for (int t = t0 + tid; t < t1; t += 256) out[t] = in[t];
    if (b == nb - 1 && tid == 0) out[ntiles] = in[ntiles];
    return;
  }
  const int64_t even = l.slack / 2;
  const double share = l.n > 0 ? 0.5 * (double)l.slack * (double)ntiles / (double)l.n : 0.0;
  auto slots = [&](int t) -> unsigned long long {
    const unsigned int held = cnt[t] - cnt[3 * (ntiles + 1) + t];
    return (unsigned long long)held + (unsigned long long)even +
           (unsigned long long)((double)held * share);
  };
  // inclusive sum over the workgroup's threads; total: of all of them
  auto scan = [&](unsigned long long v, unsigned long long &total) -> unsigned long long {
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const unsigned long long u = __shfl_up(v, d);
      if (lane >= d) v += u;
    }
    __syncthreads();  // the last scan's sums have been read
    if (lane == 63) s_sum[tid >> 6] = v;
    __syncthreads();
    total = 0;
    for (int w = 0; w < 4; ++w) {
      if (w == (tid >> 6)) v += total;
      total += s_sum[w];
    }
    return v;
  };
  unsigned long long before = 0, first, total;
#pragma unroll 4
  for (int t = tid; t < t0; t += 256) before += slots(t);
  (void)scan(before, first);
  for (int base = t0; base < t1; base += 256) {
    const int t = base + tid;
    const unsigned long long v = t < t1 ? slots(t) : 0;
    const unsigned long long at = first + scan(v, total) - v;
    if (t < t1) out[t] = (int64_t)at;
    first += total;
  }
  if (b == nb - 1 && tid == 0) out[ntiles] = (int64_t)first;
}

// Per species (blockIdx.y): the first layout_blocks workgroups write the output
// segments; thread i of the others zeroes counter i (i < n) and, with c.nn > 0,
// node i of the ten moment arrays (i < nn).
__global__ __launch_bounds__(256) void k_phase_start(CountArrays c) {
  const int s = blockIdx.y, nb = layout_blocks(c.ntiles);
  if (s >= c.ns) return;
  if ((int)blockIdx.x < nb) {
    if (c.lay[s].seg_out) phase_layout(c.lay[s], c.ntiles, blockIdx.x, nb);
    return;
  }
  const int64_t total = c.n > c.nn ? c.n : c.nn;
  for (int64_t i = (blockIdx.x - nb) * (int64_t)blockDim.x + threadIdx.x; i < total;
       i += (int64_t)(gridDim.x - nb) * blockDim.x) {
    if (i < c.n) gmem(c.p[s])[i] = 0u;
    if (i < c.nn) {
#pragma unroll
      for (int m = 0; m < 10; ++m) gmem(c.mom[s].m[m])[i] = 0.0;
    }
  }
}

// Per node and species: the sum of the partials of every tile whose staged
// block holds the node (at most two tiles per axis), in tile order, with
// Neumaier's compensated summation, added to the FP64 moment arrays.
// Tiles whose input segment held no particle of the species wrote no
// partials (their flag is 0) and are skipped.
template <typename P, int TX, int TY, int TZ>
__device__ __forceinline__ void reduce_node(int n, int s, int nyn, int nzn, int ntx, int nty,
                                            int ntz, int ntiles, int ns,
                                            const P *__restrict__ partials,
                                            const unsigned char *__restrict__ pflag,
                                            double *const *mom) {
  constexpr int BX = TX + 3, BY = TY + 3, BZ = TZ + 3, NB = BX * BY * BZ;
  const int gz = n % nzn, gy = (n / nzn) % nyn, gx = n / (nzn * nyn);
  const int xl = gx >= BX - 1 ? (gx - (BX - 1) + TX - 1) / TX : 0;
  const int xh = min(gx / TX, ntx - 1);
  const int yl = gy >= BY - 1 ? (gy - (BY - 1) + TY - 1) / TY : 0;
  const int yh = min(gy / TY, nty - 1);
  const int zl = gz >= BZ - 1 ? (gz - (BZ - 1) + TZ - 1) / TZ : 0;
  const int zh = min(gz / TZ, ntz - 1);
  double sum[10], cmp[10];
#pragma unroll
  for (int m = 0; m < 10; ++m) { sum[m] = 0.0; cmp[m] = 0.0; }
  bool any = false;
  for (int tx = xl; tx <= xh; ++tx)
    for (int ty = yl; ty <= yh; ++ty)
      for (int tz = zl; tz <= zh; ++tz) {
        const int tile = (tx * nty + ty) * ntz + tz;
        if (!gmem(pflag)[(size_t)tile * ns + s]) continue;
        any = true;
        const int b = ((gx - tx * TX) * BY + (gy - ty * TY)) * BZ + (gz - tz * TZ);
        const SPIC_GLOBAL P *src =
            gmem(partials) + ((size_t)tile * ns + s) * (10 * NB) + (size_t)b * 10;
#pragma unroll
        for (int m = 0; m < 10; ++m) {
          const double v = (double)src[m];
          const double t = sum[m] + v;
          cmp[m] += fabs(sum[m]) >= fabs(v) ? (sum[m] - t) + v : (v - t) + sum[m];
          sum[m] = t;
        }
      }
  if (!any) return;
#pragma unroll
  for (int m = 0; m < 10; ++m) gmem(mom[m])[n] += sum[m] + cmp[m];
}

template <typename P, int TX, int TY, int TZ>
__global__ __launch_bounds__(256) void k_binned_reduce(BinnedReduceArgs a, int nn) {
  const int s = blockIdx.y;
  const int n = blockIdx.x * 256 + threadIdx.x;
  if (n >= nn) return;
  reduce_node<P, TX, TY, TZ>(n, s, a.nyn, a.nzn, a.ntx, a.nty, a.ntz, a.ntiles, a.ns,
                             (const P *)a.partials, a.pflag, a.mom[s].m);
}

// The reduce of a batch: blockIdx.y is the species.
template <typename T, int TX, int TY, int TZ>
__global__ __launch_bounds__(256) void k_binned_reduce_batch(
    const BinnedArgs<T> *__restrict__ tab, BatchMap map) {
  int i = 0;
  for (int k = 1; k < map.n; ++k) i += (int)blockIdx.x >= map.start[k] ? 1 : 0;
  const BinnedArgs<T> &a = tab[i];
  const int s = blockIdx.y;
  const int n = (blockIdx.x - map.start[i]) * 256 + threadIdx.x;
  if (s >= a.ns || n >= a.g.nxn * a.g.nyn * a.g.nzn) return;
  reduce_node<PartialT<T>, TX, TY, TZ>(n, s, a.g.nyn, a.g.nzn, a.ntx, a.nty, a.ntz, a.ntiles,
                                       a.ns, (const PartialT<T> *)a.partials, a.pflag,
                                       a.sp[s].m.m);
}

// The same for a batch: the blocks of instance i are map.start[i] and up.
template <typename T>
__global__ __launch_bounds__(256) void k_phase_start_batch(
    const BinnedArgs<T> *__restrict__ tab, BatchMap map, int moments) {
  int i = 0;
  for (int k = 1; k < map.n; ++k) i += (int)blockIdx.x >= map.start[k] ? 1 : 0;
  const BinnedArgs<T> &a = tab[i];
  const int s = blockIdx.y;
  if (s >= a.ns) return;
  const int block = blockIdx.x - map.start[i];
  const int nb = layout_blocks(a.ntiles);
  if (block < nb) {
    const BinnedSpecies<T> &sp = a.sp[s];
    phase_layout(LayoutArgs{sp.seg_in, sp.seg_out, sp.cnt_in, sp.slack, sp.n}, a.ntiles, block,
                 nb);
    return;
  }
  const int64_t j = (int64_t)(block - nb) * 256 + threadIdx.x;
  if (j < kCntArrays * (int64_t)(a.ntiles + 1)) gmem(a.sp[s].cnt_out)[j] = 0u;
  if (moments && j < (int64_t)a.g.nxn * a.g.nyn * a.g.nzn) {
#pragma unroll
    for (int m = 0; m < 10; ++m) gmem(a.sp[s].m.m[m])[j] = 0.0;
  }
}

}  // namespace

hipError_t launch_binned_reduce(const BinnedReduceArgs &a, int tx, int ty, int tz,
                                int nn, hipStream_t s) {
  if (nn <= 0 || a.ns <= 0) return hipSuccess;
  dim3 grid((nn + 255) / 256, a.ns);
  const bool f = a.partials_fp32 != 0;
  if (tx == 4 && ty == 4 && tz == 4) {
    if (f) hipLaunchKernelGGL((k_binned_reduce<float, 4, 4, 4>), grid, dim3(256), 0, s, a, nn);
    else hipLaunchKernelGGL((k_binned_reduce<double, 4, 4, 4>), grid, dim3(256), 0, s, a, nn);
  } else if (tx == 8 && ty == 4 && tz == 4) {
    if (f) hipLaunchKernelGGL((k_binned_reduce<float, 8, 4, 4>), grid, dim3(256), 0, s, a, nn);
    else hipLaunchKernelGGL((k_binned_reduce<double, 8, 4, 4>), grid, dim3(256), 0, s, a, nn);
  } else {
    return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

template <typename T>
hipError_t launch_batch_reduce(const BinnedArgs<T> *tab, const BatchMap &nodes,
                               int max_ns, int tx, int ty, int tz, hipStream_t s) {
  if (nodes.n <= 0 || nodes.start[nodes.n] <= 0 || max_ns <= 0) return hipSuccess;
  dim3 grid(nodes.start[nodes.n], max_ns);
  if (tx == 4 && ty == 4 && tz == 4)
    hipLaunchKernelGGL((k_binned_reduce_batch<T, 4, 4, 4>), grid, dim3(256), 0, s, tab,
                       nodes);
  else if (tx == 8 && ty == 4 && tz == 4)
    hipLaunchKernelGGL((k_binned_reduce_batch<T, 8, 4, 4>), grid, dim3(256), 0, s, tab,
                       nodes);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

template <typename T>
hipError_t launch_batch_start(const BinnedArgs<T> *tab, const BatchMap &counts,
                                    int max_ns, int moments, hipStream_t s) {
  if (counts.n <= 0 || counts.start[counts.n] <= 0 || max_ns <= 0) return hipSuccess;
  hipLaunchKernelGGL((k_phase_start_batch<T>), dim3(counts.start[counts.n], max_ns),
                     dim3(256), 0, s, tab, counts, moments);
  return hipGetLastError();
}

template hipError_t launch_batch_reduce<double>(const BinnedArgs<double> *,
                                                const BatchMap &, int, int, int, int,
                                                hipStream_t);
template hipError_t launch_batch_reduce<float>(const BinnedArgs<float> *, const BatchMap &,
                                               int, int, int, int, hipStream_t);
template hipError_t launch_batch_start<double>(const BinnedArgs<double> *,
                                                     const BatchMap &, int, int,
                                                     hipStream_t);
template hipError_t launch_batch_start<float>(const BinnedArgs<float> *,
                                                    const BatchMap &, int, int, hipStream_t);

// Copy particle j of the source to slot o of the destination.
template <typename PS, typename PSI, typename PD, typename PDI>
__device__ __forceinline__ void copy_particle(PS src, PSI src_id, int64_t stride, int64_t j,
                                              PD dst, PDI dst_id, int64_t o) {
#pragma unroll
  for (int a = 0; a < 7; ++a) dst[a * stride + o] = src[a * stride + j];
  if (dst_id) dst_id[o] = src_id[j];  // engines that keep no ids have neither
}

constexpr int kTileThreads = 512;
constexpr unsigned int kTileStaged = 12288;  // particles a tile block stages in LDS
// Values of one component that a tile block stages at a time.  In FP32 its 16 KB
// (and slot tables of 256 ranks in them) leave room for a third workgroup per
// CU: 6.3M particles on 3072 tiles in 145 us against 187 with 8192 (a fourth, at
// 6144 staged slots, changes nothing).
constexpr int kTileChunk = 4096;
constexpr int kTileU = 4;                    // particles a thread loads at once
constexpr int kScanThreads = 1024;

// wave_rank on a global counter array (global atomics, not flat ones).
__device__ __forceinline__ uint32_t wave_rank_g(SPIC_GLOBAL unsigned int *counter,
                                                uint32_t key, bool active) {
  const int lane = __lane_id();
  const unsigned long long below = (1ull << lane) - 1ull;
  unsigned long long todo = __ballot(active);
  uint32_t rank = 0;
  while (todo) {
    const int leader = __ffsll((long long)todo) - 1;
    const uint32_t lkey = __shfl(key, leader);
    const unsigned long long same = __ballot(active && key == lkey);
    unsigned int base = 0;
    if (lane == leader)
      base = __hip_atomic_fetch_add(counter + lkey, (unsigned int)__popcll(same),
                                    __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    base = __shfl(base, leader);
    if (active && key == lkey) rank = base + (uint32_t)__popcll(same & below);
    todo &= ~same;
  }
  return rank;
}

// Job of block b in a tile-sort map (uniform across the workgroup).
__device__ __forceinline__ int sort_job(const TileSortMap &map, int b) {
  int j = 0;
  for (int k = 1; k < map.n; ++k) j += b >= map.start[k] ? 1 : 0;
  return j;
}

// Tile sort, step 1 (block b of nb of the job).  Block t < ntiles reads
// segment t: its particles that lie in tile t are tile t's own (own[t],
// added to count[t]); every other particle adds one to its tile's count.
// Blocks ntiles and up split the overflow region, whose particles all add
// one to their tile's count.
// BATCH: the launch covers every job of a map; the block's job, taken from
// the table, replaces the pointer and layout arguments.
template <typename T, bool BATCH>
__global__ __launch_bounds__(kTileThreads) void k_tile_count(
    KGrid<T> g, BinLayout L, const T *src_a, int64_t stride, const int64_t *seg_a,
    const unsigned int *cnt_a, unsigned int ovf_cap, unsigned int *count_a,
    unsigned int *own_a, const TileSortJob<T> *__restrict__ jobs, TileSortMap map) {
  __shared__ unsigned int s_own;
  int b = blockIdx.x;
  int nb = gridDim.x;
  if constexpr (BATCH) {
    const int j = sort_job(map, blockIdx.x);
    const TileSortJob<T> &J = jobs[j];
    g = J.g; L = J.L; src_a = J.src; stride = J.stride; seg_a = J.src_seg;
    cnt_a = J.src_cnt; ovf_cap = J.ovf_cap; count_a = J.count; own_a = J.own;
    b -= map.start[j];
    nb = map.start[j + 1] - map.start[j];
  }
  const SPIC_GLOBAL T *__restrict__ src = gmem(src_a);
  SPIC_GLOBAL unsigned int *__restrict__ count = gmem(count_a);
  const int tid = threadIdx.x;
  const bool ovf = b >= L.ntiles;
  const RangeView v = range_view(gmem(seg_a), gmem(cnt_a), L.ntiles, ovf_cap,
                                 ovf ? L.ntiles : b);
  const int64_t first = ovf ? (int64_t)(b - L.ntiles) * kTileThreads : 0;
  const int64_t step = ovf ? (int64_t)(nb - L.ntiles) * kTileThreads : (int64_t)kTileThreads;
  if (tid == 0) s_own = 0u;
  __syncthreads();
  unsigned int mine = 0;
  for (int64_t base = first; base < v.count; base += kTileU * step) {
    T px[kTileU], py[kTileU], pz[kTileU];
#pragma unroll
    for (int u = 0; u < kTileU; ++u) {
      const int64_t r = base + u * step + tid;
      if (r < v.count) {
        const int64_t j = v.slot(r);
        px[u] = src[j];
        py[u] = src[stride + j];
        pz[u] = src[2 * stride + j];
      }
    }
#pragma unroll
    for (int u = 0; u < kTileU; ++u) {
      const bool in = base + u * step + tid < v.count;
      uint32_t tile = 0;
      if (in) {
        int cx, cy, cz;
        uint32_t cit;
        cell_of(g, L, px[u], py[u], pz[u], cx, cy, cz, tile, cit);
      }
      const bool home = in && !ovf && (int)tile == b;
      mine += home ? 1u : 0u;
      (void)wave_rank_g(count, tile, in && !home);
    }
  }
  if (ovf) return;
  if (mine) atomicAdd(&s_own, mine);
  __syncthreads();
  if (tid == 0) {
    gmem(own_a)[b] = s_own;
    if (s_own)
      __hip_atomic_fetch_add(count + b, s_own, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// Tile sort, step 2 (one workgroup of kScanThreads): the exclusive scan P
// of the counts (P[ntiles] = n) and the destination layout,
// seg[t] = P[t] + t * slack, cnt[t] = count[t], no unused runs, an empty
// overflow region.
template <typename T>
__device__ __forceinline__ void tile_bounds_body(const TileSortJob<T> &J) {
  constexpr int NW = kScanThreads / 64;
  __shared__ unsigned int s_wsum[NW];
  __shared__ unsigned int s_carry;
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int nt = J.L.ntiles;
  if (tid == 0) s_carry = 0u;
  __syncthreads();
  for (int base = 0; base <= nt; base += kScanThreads) {
    const int t = base + tid;
    const unsigned int c = t < nt ? gmem(J.count)[t] : 0u;
    unsigned int v = c;  // inclusive scan within the wave
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const unsigned int u = __shfl_up(v, d);
      if (lane >= d) v += u;
    }
    if (lane == 63) s_wsum[wid] = v;
    __syncthreads();
    if (wid == 0) {
      unsigned int w = lane < NW ? s_wsum[lane] : 0u;
#pragma unroll
      for (int d = 1; d < NW; d <<= 1) {
        const unsigned int u = __shfl_up(w, d);
        if (lane >= d) w += u;
      }
      if (lane < NW) s_wsum[lane] = w;  // inclusive over the waves
    }
    __syncthreads();
    const unsigned int carry = s_carry;
    const unsigned int excl = carry + (wid ? s_wsum[wid - 1] : 0u) + v - c;
    if (t <= nt) {
      gmem(J.dst_seg)[t] = (int64_t)excl + (int64_t)t * J.L.slack;
      gmem(J.dst_cnt)[t] = c;
      gmem(J.dst_cnt)[(nt + 1) + t] = 0u;
      gmem(J.dst_cnt)[2 * (nt + 1) + t] = 0u;
      gmem(J.dst_cnt)[3 * (nt + 1) + t] = 0u;
    }
    if (J.big && c > (unsigned)kLoadHeld) {
      const unsigned int pieces = (c + kLoadHeld - 1) / kLoadHeld;
      const unsigned int number = atomicAdd(J.big + 1, 1u), at = atomicAdd(J.big, pieces);
      for (unsigned int k = 0; k < pieces; ++k)
        J.pieces[at + k] = make_uint4((unsigned)t, number, k * kLoadHeld, 0u);
    }
    __syncthreads();
    if (tid == 0) s_carry = carry + s_wsum[NW - 1];
    __syncthreads();
  }
}

// Tile sort, step 3 (block b of nb of the job).  Block t < ntiles writes
// tile t's own particles to the start of its destination segment in
// round-robin cell order -- rank 0 of every cell in cell order, then rank
// 1, and so on: bin_sort's order -- and every other particle of its source
// segment after the own particles of that particle's tile (slot
// dst_seg[tile] + own[tile] + k, k from the fill counters).  Blocks ntiles
// and up do the latter for the overflow region.  For the own particles:
//  1. each particle's cell within the tile (or "foreign") goes to LDS, and
//     LDS counters count each cell;
//  2. tables give the slot of the k-th particle of cell c as A[k] + T[c][k]
//     (A[k]: particles of rank < k over all cells; T[c][k]: cells before c
//     holding more than k particles); ranks beyond the tables' KT columns
//     take the slot by a loop over the cells; each particle's slot goes to
//     LDS;
//  3. per component and output chunk of the LDS stage, the chunk's
//     particles are read in source order (coalesced) into the stage at their
//     slots, and the stage is written out in slot order (coalesced).
// A segment of more than kTileStaged particles skips the stage and writes
// each particle at its slot directly.
// BATCH: the launch covers every job of a map; the block's job, taken from
// the table, replaces the pointer and layout arguments.
template <typename T, int NC, int KT, bool BATCH>
__global__ __launch_bounds__(kTileThreads) void k_tile_sort(
    KGrid<T> g, BinLayout L, const T *src_a, int64_t stride, const uint32_t *src_id_a,
    const int64_t *src_seg_a, const unsigned int *src_cnt_a, unsigned int ovf_cap, T *dst_a,
    uint32_t *dst_id_a, const int64_t *dst_seg_a, const unsigned int *own_a,
    unsigned int *fill_a, const TileSortJob<T> *__restrict__ jobs, TileSortMap map) {
  constexpr int kTileStageBytes = kTileChunk * (int)sizeof(T);
  static_assert(KT * NC <= kTileStageBytes, "slot table exceeds the stage");
  static_assert(NC <= 256, "counts of the cells before a cell must fit a byte");
  constexpr uint16_t kForeign = 0xFFFF;  // also "no slot": foreign particles take none
  constexpr uint16_t kNoSlot = 0xFFFF;
  constexpr int kChunk = kTileChunk;
  __shared__ unsigned int s_count[NC], s_rank[NC], s_kmax, s_own;
  __shared__ unsigned int s_A[KT];
  // each staged particle's cell (step 1), then its slot (step 2)
  __shared__ uint16_t s_slot[kTileStaged];
  __shared__ __align__(16) unsigned char s_raw[kTileStageBytes];
  unsigned char(*s_T)[KT] = reinterpret_cast<unsigned char(*)[KT]>(s_raw);
  int t = blockIdx.x;
  int nb = gridDim.x;
  if constexpr (BATCH) {
    const int j = sort_job(map, blockIdx.x);
    const TileSortJob<T> &J = jobs[j];
    g = J.g; L = J.L; src_a = J.src; stride = J.stride; src_id_a = J.src_id;
    src_seg_a = J.src_seg; src_cnt_a = J.src_cnt; ovf_cap = J.ovf_cap; dst_a = J.dst;
    dst_id_a = J.dst_id; dst_seg_a = J.dst_seg; own_a = J.own; fill_a = J.fill;
    t -= map.start[j];
    nb = map.start[j + 1] - map.start[j];
  }
  const SPIC_GLOBAL T *__restrict__ src = gmem(src_a);
  const SPIC_GLOBAL uint32_t *__restrict__ src_id = gmem(src_id_a);
  const SPIC_GLOBAL int64_t *__restrict__ src_seg = gmem(src_seg_a);
  const SPIC_GLOBAL unsigned int *__restrict__ src_cnt = gmem(src_cnt_a);
  SPIC_GLOBAL T *__restrict__ dst = gmem(dst_a);
  SPIC_GLOBAL uint32_t *__restrict__ dst_id = gmem(dst_id_a);
  const SPIC_GLOBAL int64_t *__restrict__ dst_seg = gmem(dst_seg_a);
  const SPIC_GLOBAL unsigned int *__restrict__ own = gmem(own_a);
  SPIC_GLOBAL unsigned int *__restrict__ fill = gmem(fill_a);
  const int tid = threadIdx.x;

  if (t >= L.ntiles) {
    const RangeView v = range_view(src_seg, src_cnt, L.ntiles, ovf_cap, L.ntiles);
    const int64_t step = (int64_t)(nb - L.ntiles) * kTileThreads;
    for (int64_t base = (int64_t)(t - L.ntiles) * kTileThreads; base < v.count;
         base += step) {
      const int64_t r = base + tid;
      const bool in = r < v.count;
      int64_t j = 0;
      uint32_t tile = 0;
      if (in) {
        j = v.slot(r);
        int cx, cy, cz;
        uint32_t cit;
        cell_of(g, L, src[j], src[stride + j], src[2 * stride + j], cx, cy, cz, tile,
                   cit);
      }
      const uint32_t k = wave_rank_g(fill, tile, in);
      if (in) copy_particle(src, src_id, stride, j, dst, dst_id, dst_seg[tile] + own[tile] + k);
    }
    return;
  }

  const RangeView v = range_view(src_seg, src_cnt, L.ntiles, ovf_cap, t);
  if (v.count == 0) return;
  const bool staged = v.count <= (int64_t)kTileStaged;
  for (int c = tid; c < NC; c += kTileThreads) {
    s_count[c] = 0u;
    s_rank[c] = 0u;
  }
  if (tid == 0) s_kmax = 0u;
  __syncthreads();

  // 1. cells and counts
  for (int64_t r0 = tid; r0 < v.count; r0 += kTileU * kTileThreads) {
    T px[kTileU], py[kTileU], pz[kTileU];
#pragma unroll
    for (int u = 0; u < kTileU; ++u) {
      const int64_t r = r0 + (int64_t)u * kTileThreads;
      if (r < v.count) {
        const int64_t j = v.slot(r);
        px[u] = src[j];
        py[u] = src[stride + j];
        pz[u] = src[2 * stride + j];
      }
    }
#pragma unroll
    for (int u = 0; u < kTileU; ++u) {
      const int64_t r = r0 + (int64_t)u * kTileThreads;
      if (r < v.count) {
        int cx, cy, cz;
        uint32_t tile, cit;
        cell_of(g, L, px[u], py[u], pz[u], cx, cy, cz, tile, cit);
        const bool home = (int)tile == t;
        if (home) atomicAdd(&s_count[cit], 1u);
        if (staged) s_slot[r] = home ? (uint16_t)cit : kForeign;
      }
    }
  }
  __syncthreads();
  for (int c = tid; c < NC; c += kTileThreads) atomicMax(&s_kmax, s_count[c]);
  __syncthreads();

  // 2. slot tables, then each particle's slot
  const int kmax = (int)(s_kmax < (unsigned)KT ? s_kmax : (unsigned)KT);
  for (int k = tid; k < kmax; k += kTileThreads) {
    unsigned int a = 0, before = 0;
#pragma unroll 8
    for (int c = 0; c < NC; ++c) {
      const unsigned int n = s_count[c];
      a += n < (unsigned)k ? n : (unsigned)k;
      s_T[c][k] = (unsigned char)before;
      before += n > (unsigned)k ? 1u : 0u;
    }
    s_A[k] = a;
  }
  if (tid == 0) {
    unsigned int n_own = 0;
    for (int c = 0; c < NC; ++c) n_own += s_count[c];
    s_own = n_own;
  }
  __syncthreads();
  const int64_t out0 = dst_seg[t];
  for (int64_t base = 0; base < v.count; base += kTileThreads) {
    const int64_t r = base + tid;
    const bool in = r < v.count;
    unsigned int c = kForeign;
    uint32_t tile = 0;
    if (in) {
      if (staged) c = s_slot[r];
      if (!staged || c == kForeign) {
        const int64_t j = v.slot(r);
        int cx, cy, cz;
        uint32_t cit;
        cell_of(g, L, src[j], src[stride + j], src[2 * stride + j], cx, cy, cz, tile,
                   cit);
        c = (int)tile == t ? cit : kForeign;
      }
    }
    const bool foreign = in && c == kForeign;
    const uint32_t kf = wave_rank_g(fill, tile, foreign);
    if (!in) continue;
    if (foreign) {
      copy_particle(src, src_id, stride, v.slot(r), dst, dst_id,
                    dst_seg[tile] + own[tile] + kf);
      if (staged) s_slot[r] = kNoSlot;
      continue;
    }
    const unsigned int k = atomicAdd(&s_rank[c], 1u);
    unsigned int pos;
    if (k < (unsigned)KT) {
      pos = s_A[k] + s_T[c][k];
    } else {
      pos = 0;
#pragma unroll 4
      for (int cc = 0; cc < NC; ++cc) {
        const unsigned int n = s_count[cc];
        pos += n < k ? n : k;
        if (cc < (int)c && n > k) ++pos;
      }
    }
    if (staged) s_slot[r] = (uint16_t)pos;
    else copy_particle(src, src_id, stride, v.slot(r), dst, dst_id, out0 + pos);
  }
  if (!staged) return;
  __syncthreads();  // slots complete; the tables' LDS becomes the stage

  // 3. per component and output chunk: gather into the stage, write out
  const unsigned int n_own = s_own;
  T *stage = reinterpret_cast<T *>(s_raw);
  uint32_t *stage_id = reinterpret_cast<uint32_t *>(s_raw);
  const int ncomp = dst_id ? 8 : 7;  // the ids are the eighth, when kept
  for (int a = 0; a < ncomp; ++a) {
    for (unsigned int c0 = 0; c0 < n_own; c0 += (unsigned)kChunk) {
      for (int64_t r0 = tid; r0 < v.count; r0 += kTileU * kTileThreads) {
        unsigned int p[kTileU];
        T val[kTileU];
        uint32_t idv[kTileU];
#pragma unroll
        for (int u = 0; u < kTileU; ++u) {
          const int64_t r = r0 + (int64_t)u * kTileThreads;
          p[u] = kChunk;
          if (r < v.count && s_slot[r] != kNoSlot) {
            p[u] = (unsigned int)s_slot[r] - c0;  // wraps above kChunk below c0
            if (p[u] < (unsigned)kChunk) {
              const int64_t j = v.slot(r);
              if (a < 7) val[u] = src[a * stride + j];
              else idv[u] = src_id[j];
            }
          }
        }
#pragma unroll
        for (int u = 0; u < kTileU; ++u) {
          if (p[u] < (unsigned)kChunk) {
            if (a < 7) stage[p[u]] = val[u];
            else stage_id[p[u]] = idv[u];
          }
        }
      }
      __syncthreads();
      const unsigned int m = n_own - c0 < (unsigned)kChunk ? n_own - c0 : (unsigned)kChunk;
      for (unsigned int p = tid; p < m; p += kTileThreads) {
        if (a < 7) dst[a * stride + out0 + c0 + p] = stage[p];
        else dst_id[out0 + c0 + p] = stage_id[p];
      }
      __syncthreads();
    }
  }
}

template <typename T>
__global__ __launch_bounds__(kScanThreads) void k_tile_bounds(TileSortJob<T> J) {
  tile_bounds_body<T>(J);
}

template <typename T>
__global__ __launch_bounds__(kScanThreads) void k_tile_bounds_batch(
    const TileSortJob<T> *__restrict__ jobs) {
  const TileSortJob<T> &J = jobs[blockIdx.x];
  tile_bounds_body<T>(J);
}

template <typename T>
hipError_t tile_sort(const TileSortJob<T> &J, hipStream_t s) {
  const int nc = J.L.tx * J.L.ty * J.L.tz;
  if (nc != 64 && nc != 128) return hipErrorInvalidValue;
  const int64_t nzero = 3 * ((int64_t)J.L.ntiles + 1);
  hipLaunchKernelGGL(k_zero_u32, dim3(nblocks(nzero)), dim3(256), 0, s, J.count, nzero);
  hipError_t e;
  if ((e = hipGetLastError()) != hipSuccess) return e;
  const dim3 grid(J.L.ntiles + kTileOvfBlocks);
  hipLaunchKernelGGL((k_tile_count<T, false>), grid, dim3(kTileThreads), 0, s, J.g, J.L, J.src,
                     J.stride, J.src_seg, J.src_cnt, J.ovf_cap, J.count, J.own,
                     (const TileSortJob<T> *)nullptr, TileSortMap{});
  if ((e = hipGetLastError()) != hipSuccess) return e;
  hipLaunchKernelGGL(k_tile_bounds<T>, dim3(1), dim3(kScanThreads), 0, s, J);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  if (nc == 64)
    hipLaunchKernelGGL((k_tile_sort<T, 64, 64 * sizeof(T), false>), grid, dim3(kTileThreads), 0, s, J.g, J.L,
                       J.src, J.stride, J.src_id, J.src_seg, J.src_cnt, J.ovf_cap, J.dst,
                       J.dst_id, (const int64_t *)J.dst_seg, (const unsigned int *)J.own,
                       J.fill, (const TileSortJob<T> *)nullptr, TileSortMap{});
  else
    hipLaunchKernelGGL((k_tile_sort<T, 128, 32 * sizeof(T), false>), grid, dim3(kTileThreads), 0, s, J.g, J.L,
                       J.src, J.stride, J.src_id, J.src_seg, J.src_cnt, J.ovf_cap, J.dst,
                       J.dst_id, (const int64_t *)J.dst_seg, (const unsigned int *)J.own,
                       J.fill, (const TileSortJob<T> *)nullptr, TileSortMap{});
  return hipGetLastError();
}

template <typename T>
hipError_t tile_sort_batch(const TileSortJob<T> *jobs, const TileSortMap &map, int tx,
                           int ty, int tz, unsigned int *ws, size_t ws_words,
                           hipStream_t s) {
  const int nc = tx * ty * tz;
  if (nc != 64 && nc != 128) return hipErrorInvalidValue;
  if (map.n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_zero_u32, dim3(nblocks((long)ws_words)), dim3(256), 0, s, ws,
                     (int64_t)ws_words);
  hipError_t e;
  if ((e = hipGetLastError()) != hipSuccess) return e;
  const dim3 grid(map.start[map.n]);
  const KGrid<T> g0{};
  const BinLayout L0{};
  hipLaunchKernelGGL((k_tile_count<T, true>), grid, dim3(kTileThreads), 0, s, g0, L0,
                     (const T *)nullptr, (int64_t)0, (const int64_t *)nullptr,
                     (const unsigned int *)nullptr, 0u, (unsigned int *)nullptr,
                     (unsigned int *)nullptr, jobs, map);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  hipLaunchKernelGGL(k_tile_bounds_batch<T>, dim3(map.n), dim3(kScanThreads), 0, s, jobs);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  // the batch instances take their arguments from the job table
  if (nc == 64)
    hipLaunchKernelGGL((k_tile_sort<T, 64, 64 * sizeof(T), true>), grid, dim3(kTileThreads), 0, s, g0, L0,
                       (const T *)nullptr, (int64_t)0, (const uint32_t *)nullptr,
                       (const int64_t *)nullptr, (const unsigned int *)nullptr, 0u,
                       (T *)nullptr, (uint32_t *)nullptr, (const int64_t *)nullptr,
                       (const unsigned int *)nullptr, (unsigned int *)nullptr, jobs, map);
  else
    hipLaunchKernelGGL((k_tile_sort<T, 128, 32 * sizeof(T), true>), grid, dim3(kTileThreads), 0, s, g0,
                       L0, (const T *)nullptr, (int64_t)0, (const uint32_t *)nullptr,
                       (const int64_t *)nullptr, (const unsigned int *)nullptr, 0u,
                       (T *)nullptr, (uint32_t *)nullptr, (const int64_t *)nullptr,
                       (const unsigned int *)nullptr, (unsigned int *)nullptr, jobs, map);
  return hipGetLastError();
}

template hipError_t tile_sort<double>(const TileSortJob<double> &, hipStream_t);
template hipError_t tile_sort<float>(const TileSortJob<float> &, hipStream_t);
template hipError_t tile_sort_batch<double>(const TileSortJob<double> *, const TileSortMap &,
                                            int, int, int, unsigned int *, size_t,
                                            hipStream_t);
template hipError_t tile_sort_batch<float>(const TileSortJob<float> *, const TileSortMap &,
                                           int, int, int, unsigned int *, size_t,
                                           hipStream_t);

hipError_t phase_start(const CountArrays &c, hipStream_t s) {
  if (c.ns <= 0 || c.n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_phase_start, dim3(layout_blocks(c.ntiles) + nblocks(c.n > c.nn ? c.n : c.nn), c.ns), dim3(256),
                     0, s, c);
  return hipGetLastError();
}

// Whether a load goes through tiles: they hold at most kLoadHeld particles on
// average, and workgroups can count them in LDS (beyond kLdsTiles those of 1024
// threads, for enough particles).  28.8M FP32 particles on 16640 tiles, counted
// with global atomics: 5.75 ms, 5.0 by the radix sort; 2.1M 505 / 390 us.
// Many tiles of a few particles each, whose workgroups are mostly tables, keep
// the radix sort too (FP64, tiles / radix, us): 2048 tiles of 1 / 8 / 32
// particles 61 / 71, 69 / 83, 73 / 99; 3072 75 / 70, 89 / 92, 98 / 113; 4096
// 89 / 71, 109 / 95, 121 / 120; 5120 105 / 83, 129 / 101, 145 / 128.  From 64 on
// tiles win (4096: 144 / 167, 5120: 171 / 192).
// FP32 engines take tiles from four particles per cell on (4.0M particles on 512
// tiles 519 / 969 us).  With fewer, a tile's deposit is one batch of a few
// waves, whose sums follow the load's order and repeat to the last bit; the radix
// sort's order there gives the roundings it always gave.
inline bool load_through_tiles(const BinLayout &L, int64_t n, bool fp32) {
  const int64_t nt = L.ntiles;
  if (fp32 && n < 4 * nt * (L.tx * L.ty * L.tz)) return false;
  if (nt > 2048 && n < 64 * nt) return false;
  return n <= kLoadHeld * nt &&
         (nt <= kLdsTiles || (nt <= kLoadManyTiles && n >= 256 * 1024 * 16));
}

// The workspace of such a load: two words per tile, the counters of the tiles
// taken in pieces (all of these zeroed first), the pieces, two words per particle.
struct LoadSpace {
  int64_t zeroed;       // words
  unsigned int pieces;  // at most
  size_t a_zeroed, a_pieces, a_n, total;
};

inline LoadSpace load_space(const BinLayout &L, int64_t n) {
  const int64_t big = n / kLoadHeld < L.ntiles ? n / kLoadHeld : L.ntiles;
  LoadSpace sp;
  sp.zeroed = 2 * ((int64_t)L.ntiles + 1) + 2 + big * 2 * (L.tx * L.ty * L.tz);
  sp.pieces = (unsigned)(n > kLoadHeld ? n / kLoadHeld + big : 0);
  sp.a_zeroed = align_up(sizeof(unsigned int) * (size_t)sp.zeroed);
  sp.a_pieces = align_up(sizeof(uint4) * (size_t)sp.pieces);
  sp.a_n = align_up(sizeof(uint32_t) * (size_t)(n > 0 ? n : 1));
  sp.total = sp.a_zeroed + sp.a_pieces + 2 * sp.a_n;
  return sp;
}

// The load of a dense source through tiles.
template <typename TS, typename T>
hipError_t load_tiles(const KGrid<T> &g, const BinLayout &L, int64_t n, const void *const src[7],
                      T *const dst[7], uint32_t *dst_id, int64_t *dst_seg,
                      unsigned int *dst_cnt, char *w, const LoadSpace &sp, hipStream_t s) {
  const int nc = L.tx * L.ty * L.tz;
  if (nc != 64 && nc != 128) return hipErrorInvalidValue;
  TileSortJob<T> J;
  std::memset(&J, 0, sizeof(J));
  J.L = L;
  J.dst_seg = dst_seg;
  J.dst_cnt = dst_cnt;
  J.count = (unsigned int *)w;
  LoadBins b;
  b.n = n;
  b.count = J.count;
  b.next = J.count + L.ntiles + 1;
  b.seg = dst_seg;
  b.big = b.next + L.ntiles + 1;
  b.cells = b.big + 2;
  b.pieces = (uint4 *)(w + sp.a_zeroed);
  b.where = (uint32_t *)(w + sp.a_zeroed + sp.a_pieces);
  b.perm = (uint32_t *)(w + sp.a_zeroed + sp.a_pieces + sp.a_n);
  b.tile_blocks = (L.ntiles + 7) / 8 * 8;
  J.big = sp.pieces ? b.big : nullptr;
  J.pieces = b.pieces;
  // many tiles: workgroups of 1024 threads and 64 KB of counters, 16384
  // particles each, where that leaves one per CU
  const bool many = L.ntiles > kLdsTiles;
  const int64_t per = n / (256 * 2048);
  b.per = many || per > 16 ? 16 : per < 1 ? 1 : (int)per;
  Arrays7<TS> as;
  Arrays7<T> ad;
  for (int a = 0; a < 7; ++a) {
    as.p[a] = (TS *)src[a];
    ad.p[a] = dst[a];
  }
  hipLaunchKernelGGL(k_zero_u32, dim3(nblocks((long)sp.zeroed)), dim3(256), 0, s, J.count,
                     sp.zeroed);
  hipError_t e;
  if ((e = hipGetLastError()) != hipSuccess) return e;
  if (n > 0) {
    const int nt = many ? 1024 : 256;
    const dim3 grid((unsigned)((n + nt * b.per - 1) / (nt * b.per)));
    if (many)
      hipLaunchKernelGGL((k_load_count<TS, T, 1024, kLoadManyTiles>), grid, dim3(1024), 0, s, g,
                         L, b, as.p[0], as.p[1], as.p[2]);
    else if (L.ntiles <= kLdsTiles && L.ntiles <= 8 * 256 * b.per)
      hipLaunchKernelGGL((k_load_count<TS, T, 256, kLdsTiles>), grid, dim3(256), 0, s, g, L, b,
                         as.p[0], as.p[1], as.p[2]);
    else
      hipLaunchKernelGGL((k_load_count<TS, T, 256, 0>), grid, dim3(256), 0, s, g, L, b, as.p[0],
                         as.p[1], as.p[2]);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  hipLaunchKernelGGL(k_tile_bounds<T>, dim3(1), dim3(kScanThreads), 0, s, J);
  if ((e = hipGetLastError()) != hipSuccess || n == 0) return e;
  // places by workgroup or by wave, as the deposit through tiles takes them
  auto blocks = [n](int per) { return dim3((unsigned)((n + 256 * per - 1) / (256 * per))); };
  if (many)
    hipLaunchKernelGGL((k_load_place<16, 1024, kLoadManyTiles>), blocks(64), dim3(1024), 0, s, L,
                       b);
  else if (L.ntiles <= kLdsTiles && n >= 128 * 256 * 16)
    hipLaunchKernelGGL((k_load_place<16, 256, kLdsTiles>), blocks(16), dim3(256), 0, s, L, b);
  else if (L.ntiles <= 4 * 256)
    hipLaunchKernelGGL((k_load_place<4, 256, kLdsTiles>), blocks(4), dim3(256), 0, s, L, b);
  else
    hipLaunchKernelGGL((k_load_place<1, 256, 0>), blocks(1), dim3(256), 0, s, L, b);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  const dim3 threads(kLoadThreads), grid(b.tile_blocks + sp.pieces);
  if (nc == 64) {
    if (sp.pieces) hipLaunchKernelGGL((k_load_pieces<64>), dim3(sp.pieces), threads, 0, s, L, b);
    hipLaunchKernelGGL((k_load_tile<TS, T, 64>), grid, threads, 0, s, L, b, as, ad, dst_id);
  } else {
    if (sp.pieces) hipLaunchKernelGGL((k_load_pieces<128>), dim3(sp.pieces), threads, 0, s, L, b);
    hipLaunchKernelGGL((k_load_tile<TS, T, 128>), grid, threads, 0, s, L, b, as, ad, dst_id);
  }
  return hipGetLastError();
}

template <typename T>
hipError_t bin_sort(const KGrid<T> &g, const BinLayout &L, int64_t n,
                    const void *const src[7], int src_f64, const uint32_t *src_id,
                    const int64_t *src_seg, const unsigned int *src_cnt,
                    unsigned int src_ovf_cap, T *const dst[7], uint32_t *dst_id,
                    int64_t *dst_seg, unsigned int *dst_cnt, void *workspace,
                    size_t workspace_bytes, size_t *needed, hipStream_t s) {
  if (n < 0 || n > 0xFFFFFFFFll) return hipErrorInvalidValue;
  const bool binned = src_seg != nullptr;
  // the caller's FP64 arrays into an FP32 engine (a binned source is always
  // the engine's own precision)
  const bool widened = !binned && src_f64 && sizeof(T) == 4;
  if (binned && src_f64 != (sizeof(T) == 8 ? 1 : 0)) return hipErrorInvalidValue;
  const size_t nt1 = (size_t)L.ntiles + 1;
  const size_t a_n = align_up(sizeof(uint32_t) * (size_t)(n > 0 ? n : 1));
  const size_t a_t = align_up(sizeof(uint32_t) * nt1);
  const int64_t ncell = (int64_t)L.ncx * L.ncy * L.ncz;
  const size_t a_c = align_up(sizeof(uint32_t) * (size_t)ncell);
  const int shift = L.rank_bits + L.cell_bits;
  const int key_bits = L.tile_bits + shift;
  if (!binned && load_through_tiles(L, n, sizeof(T) == 4)) {
    const LoadSpace sp = load_space(L, n);
    if (needed) *needed = sp.total;
    if (!workspace) return hipSuccess;
    if (workspace_bytes < sp.total) return hipErrorInvalidValue;
    return widened ? load_tiles<double, T>(g, L, n, src, dst, dst_id, dst_seg, dst_cnt,
                                           (char *)workspace, sp, s)
                   : load_tiles<T, T>(g, L, n, src, dst, dst_id, dst_seg, dst_cnt,
                                      (char *)workspace, sp, s);
  }
  size_t sort_bytes = 0, scan_bytes = 0;
  hipError_t e = rocprim::radix_sort_pairs(
      nullptr, sort_bytes, (uint32_t *)nullptr, (uint32_t *)nullptr,
      (uint32_t *)nullptr, (uint32_t *)nullptr, (size_t)n, 0, key_bits, s);
  if (e != hipSuccess) return e;
  e = rocprim::exclusive_scan(nullptr, scan_bytes, (const unsigned int *)nullptr,
                              (unsigned int *)nullptr, 0u, nt1,
                              rocprim::plus<unsigned int>(), s);
  if (e != hipSuccess) return e;
  const size_t total =
      4 * a_n + 2 * a_t + a_c + align_up(sort_bytes) + align_up(scan_bytes);
  if (needed) *needed = total;
  if (!workspace) return hipSuccess;
  if (workspace_bytes < total) return hipErrorInvalidValue;
  char *w = (char *)workspace;
  uint32_t *keys_in = (uint32_t *)w;
  uint32_t *keys_out = (uint32_t *)(w + a_n);
  uint32_t *idx_in = (uint32_t *)(w + 2 * a_n);
  uint32_t *perm = (uint32_t *)(w + 3 * a_n);
  unsigned int *clamped = (unsigned int *)(w + 4 * a_n);
  unsigned int *P = (unsigned int *)(w + 4 * a_n + a_t);
  unsigned int *cell_count = (unsigned int *)(w + 4 * a_n + 2 * a_t);
  void *sort_tmp = (void *)(w + 4 * a_n + 2 * a_t + a_c);
  void *scan_tmp = (void *)(w + 4 * a_n + 2 * a_t + a_c + align_up(sort_bytes));

  if (binned && n > 0) {
    hipLaunchKernelGGL(k_range_counts, dim3(nblocks((long)nt1)), dim3(256), 0, s,
                       src_seg, src_cnt, src_ovf_cap, L.ntiles, clamped);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    e = rocprim::exclusive_scan(scan_tmp, scan_bytes, (const unsigned int *)clamped,
                                P, 0u, nt1, rocprim::plus<unsigned int>(), s);
    if (e != hipSuccess) return e;
  }
  if (n > 0) {
    hipLaunchKernelGGL(k_zero_u32, dim3(nblocks(ncell)), dim3(256), 0, s, cell_count,
                       ncell);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if (binned)
      hipLaunchKernelGGL(k_bin_keys_binned<T>, dim3((unsigned)nt1), dim3(256), 0, s, g, L,
                         (const T *)src[0], (const T *)src[1], (const T *)src[2],
                         (const unsigned int *)P, src_seg, src_cnt, src_ovf_cap, cell_count,
                         keys_in, idx_in);
    else if (widened)
      hipLaunchKernelGGL((k_bin_keys<double, T>), dim3(nblocks(n)), dim3(256), 0, s, g, L, n,
                         (const double *)src[0], (const double *)src[1],
                         (const double *)src[2], cell_count, keys_in, idx_in);
    else
      hipLaunchKernelGGL((k_bin_keys<T, T>), dim3(nblocks(n)), dim3(256), 0, s, g, L, n,
                         (const T *)src[0], (const T *)src[1], (const T *)src[2],
                         cell_count, keys_in, idx_in);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    e = rocprim::radix_sort_pairs(sort_tmp, sort_bytes, keys_in, keys_out, idx_in,
                                  perm, (size_t)n, 0, key_bits, s);
    if (e != hipSuccess) return e;
    Arrays7<T> ad;
    for (int a = 0; a < 7; ++a) ad.p[a] = dst[a];
    const int conv = (!binned && L.fixed) ? 1 : 0;
    const uint32_t *sid = binned ? src_id : (const uint32_t *)nullptr;
    if (widened) {
      Arrays7<double> as;
      for (int a = 0; a < 7; ++a) as.p[a] = (double *)src[a];
      hipLaunchKernelGGL((k_bin_gather<double, T>), dim3(nblocks(n)), dim3(256), 0, s, as,
                         sid, (const uint32_t *)perm, (const uint32_t *)keys_out, shift, n,
                         L.slack, ad, dst_id, conv, L.fx);
    } else {
      Arrays7<T> as;
      for (int a = 0; a < 7; ++a) as.p[a] = (T *)src[a];
      hipLaunchKernelGGL((k_bin_gather<T, T>), dim3(nblocks(n)), dim3(256), 0, s, as, sid,
                         (const uint32_t *)perm, (const uint32_t *)keys_out, shift, n,
                         L.slack, ad, dst_id, conv, L.fx);
    }
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  hipLaunchKernelGGL(k_bin_bounds, dim3(nblocks((long)nt1)), dim3(256), 0, s,
                     (const uint32_t *)keys_out, shift, n, L.ntiles, L.slack, dst_seg,
                     dst_cnt);
  return hipGetLastError();
}

template hipError_t bin_sort<double>(const KGrid<double> &, const BinLayout &, int64_t,
                                     const void *const[7], int, const uint32_t *,
                                     const int64_t *, const unsigned int *,
                                     unsigned int, double *const[7], uint32_t *,
                                     int64_t *, unsigned int *, void *, size_t,
                                     size_t *, hipStream_t);
template hipError_t bin_sort<float>(const KGrid<float> &, const BinLayout &, int64_t,
                                    const void *const[7], int, const uint32_t *,
                                    const int64_t *, const unsigned int *,
                                    unsigned int, float *const[7], uint32_t *,
                                    int64_t *, unsigned int *, void *, size_t,
                                    size_t *, hipStream_t);

namespace {

template <typename T, typename TD, int NA>
hipError_t store_any(const BinLayout &L, int64_t n, T *const src[7], const uint32_t *id,
                     const uint32_t *base, const int64_t *seg, const unsigned int *cnt,
                     unsigned int ovf_cap, void *const *dst, hipStream_t s) {
  Arrays7<T> as;
  Arrays7<TD> ad;
  for (int a = 0; a < 7; ++a) as.p[a] = src[a];
  for (int a = 0; a < 7; ++a) ad.p[a] = a < NA ? (TD *)dst[a] : nullptr;
  if (id && n >= kStoreMinTile * (int64_t)L.ntiles)
    hipLaunchKernelGGL((k_store_tile<T, TD, NA>), dim3((unsigned)(L.ntiles / 8 + 1) * 8),
                       dim3(kStoreThreads), 0, s, as, id, seg, cnt, ovf_cap, L.ntiles, ad,
                       L.fixed, L.fx);
  else
    hipLaunchKernelGGL((k_bin_store<T, TD, NA>), dim3(L.ntiles + 1), dim3(256), 0, s, as, id, base,
                       seg, cnt, ovf_cap, L.ntiles, ad, L.fixed, L.fx);
  return hipGetLastError();
}

}  // namespace

template <typename T>
hipError_t bin_store(const BinLayout &L, int64_t n, T *const src[7], const uint32_t *id,
                     const uint32_t *base, const int64_t *seg, const unsigned int *cnt,
                     unsigned int ovf_cap, void *const dst[7], int dst_f64, hipStream_t s) {
  if (dst_f64) return store_any<T, double, 7>(L, n, src, id, base, seg, cnt, ovf_cap, dst, s);
  if constexpr (sizeof(T) == 8) return hipErrorInvalidValue;  // no narrowing store
  else return store_any<T, float, 7>(L, n, src, id, base, seg, cnt, ovf_cap, dst, s);
}

template <typename T>
hipError_t bin_store_be32(const BinLayout &L, int64_t n, T *const src[7], const uint32_t *id,
                          const uint32_t *base, const int64_t *seg, const unsigned int *cnt,
                          unsigned int ovf_cap, uint32_t *const dst[6], hipStream_t s) {
  return store_any<T, uint32_t, 6>(L, n, src, id, base, seg, cnt, ovf_cap, (void *const *)dst,
                                   s);
}

template hipError_t bin_store_be32<double>(const BinLayout &, int64_t, double *const[7],
                                           const uint32_t *, const uint32_t *, const int64_t *,
                                           const unsigned int *, unsigned int,
                                           uint32_t *const[6], hipStream_t);
template hipError_t bin_store_be32<float>(const BinLayout &, int64_t, float *const[7],
                                          const uint32_t *, const uint32_t *, const int64_t *,
                                          const unsigned int *, unsigned int,
                                          uint32_t *const[6], hipStream_t);

template hipError_t bin_store<double>(const BinLayout &, int64_t, double *const[7],
                                      const uint32_t *, const uint32_t *, const int64_t *,
                                      const unsigned int *, unsigned int,
                                      void *const[7], int, hipStream_t);
template hipError_t bin_store<float>(const BinLayout &, int64_t, float *const[7],
                                     const uint32_t *, const uint32_t *, const int64_t *,
                                     const unsigned int *, unsigned int,
                                     void *const[7], int, hipStream_t);

// Dense position of each range's first particle (tiles in order, then the
// overflow region), for stores of an engine that keeps no ids: range counts
// then an exclusive scan.  Workspace: counts | bases | rocPRIM storage; with
// workspace == nullptr only *needed is set.  *bases points into the
// workspace.
hipError_t range_bases(const int64_t *seg, const unsigned int *cnt, unsigned int ovf_cap,
                       int ntiles, void *workspace, size_t workspace_bytes, size_t *needed,
                       const uint32_t **bases, hipStream_t s) {
  const size_t n = (size_t)ntiles + 1;
  const size_t a = align_up(n * sizeof(unsigned int));
  size_t tmp = 0;
  hipError_t e = rocprim::exclusive_scan(nullptr, tmp, (const unsigned int *)nullptr,
                                         (unsigned int *)nullptr, 0u, n,
                                         rocprim::plus<unsigned int>(), s);
  if (e != hipSuccess) return e;
  if (needed) *needed = 2 * a + align_up(tmp);
  if (!workspace) return hipSuccess;
  if (workspace_bytes < 2 * a + align_up(tmp)) return hipErrorInvalidValue;
  unsigned int *counts = (unsigned int *)workspace;
  unsigned int *out = (unsigned int *)((char *)workspace + a);
  hipLaunchKernelGGL(k_range_counts, dim3(nblocks((long)n)), dim3(256), 0, s, seg,
                     cnt, ovf_cap, ntiles, counts);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  e = rocprim::exclusive_scan((char *)workspace + 2 * a, tmp, counts, out, 0u, n,
                              rocprim::plus<unsigned int>(), s);
  if (e != hipSuccess) return e;
  *bases = out;
  return hipSuccess;
}

}  // namespace spic
