// nebo_particles.hip -- particle <-> cell interpolation and point fields.
//
// CellToParticle is a gather: one thread per particle takes the cells its cube
// overlaps (k, then j, then i, as ParticleOperators.h:339-388 does) and sums
// src(i,j,k) * fraction into a register.  ParticleToCell is a scatter whose
// per-cell sums must come out in particle order to match the reference's serial
// loop bit for bit (ParticleOperators.h:184-270), so atomics on the cells are out.
// The scatter by bricks (below, "ParticleToCell by bricks") gathers the particles of
// one brick of cells in LDS and puts each cell's contributions in particle order
// there.  Particle sets it does not suit (dense in the window, or crowded into a few
// bricks of it) are sorted in device memory:
//   1. count the cells each particle overlaps, exclusive scan -> entry offsets;
//   2. each particle writes its entries in its own loop order: value
//      src[p] * fraction and key cell at entry e, so entries stand in the serial
//      loop's order;
//   3. stable radix sort of (cell, value) pairs on the cell's bits alone:
//      entries of one cell become contiguous and keep their serial order;
//   4. the first entry of each cell sums the cell's run onto the cell's value,
//      reading the sorted values in sequence.
//
// Point fields (pointfield/PointOperators.h:40-160) are an index gather and an
// index scatter; repeated scatter indices keep the last point, resolved on the
// host when the index list is uploaded.

#include "nebo_internal.h"
#include "nebo_device.h"

#include <hip/hip_runtime.h>
#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <unordered_map>
#include <vector>

namespace nebo {
namespace {

constexpr int kBlock = 256;

// One cell field as the particle loops see it: cell (i,j,k) of the window
// (0-based, ghosts included) lives at flat index (i+o0) + X*((j+o1) + Y*(k+o2)),
// an axis of glob extent 1 always at 0 (MemoryWindow::flat_index,
// MemoryWindow.h:121-131).
struct CellGrid {
  int nmax[3];       // window extent
  int off[3];        // window offset
  int glob[3];       // glob extents
  double h[3];       // spacing
  double loface[3];  // coordinate of the (-) face of window cell 0
  double rh[3];      // 1 / h, correctly rounded
  int stride[3];     // of the block; 0 along an axis of glob extent 1
  int origin;        // flat index of window cell 0 (stride 0 axes at 0)
};

CellGrid make_grid(const nebo_field_t* f, const nebo_particle_geom_t& g)
{
  CellGrid c;
  const double d[3] = {g.dx, g.dy, g.dz}, lo[3] = {g.xlo, g.ylo, g.zlo};
  for (int a = 0; a < 3; ++a) {
    c.nmax[a] = f->extent[a];
    c.off[a] = f->offset[a];
    // the constructor's defaults: spacing 1 and origin 0 where the spacing is <= 0
    c.h[a] = d[a] <= 0 ? 1.0 : d[a];
    const double o = d[a] <= 0 ? 0.0 : lo[a];
    // xlo - dx*ngm - dx/2, evaluated left to right
    c.loface[a] = o - c.h[a] * f->ghost_minus[a] - c.h[a] / 2;
  }
  int at = 1;
  c.origin = 0;
  for (int a = 0; a < 3; ++a) {
    c.glob[a] = f->glob[a];
    c.rh[a] = 1.0 / c.h[a];
    c.stride[a] = f->glob[a] > 1 ? at : 0;
    c.origin += c.stride[a] * c.off[a];
    at *= f->glob[a];
  }
  return c;
}

// The box of cells a particle overlaps and what the fractions need.
struct PBox {
  long lo[3], hi[3];
  double plo[3], phi[3];
  double pvol;
  bool has[3];
  bool skip;
};

__device__ __forceinline__ double dmin(double a, double b) { return (b < a) ? b : a; }   // std::min
__device__ __forceinline__ double dmax(double a, double b) { return (a < b) ? b : a; }   // std::max

__device__ __forceinline__ PBox particle_box(const CellGrid& g, const double* const coord[3],
                                             const double* psize, long p)
{
  PBox b;
  const double size = psize[p];
  const double rp = size * 0.5;
  b.skip = false;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    b.has[a] = coord[a] != nullptr;
    b.plo[a] = b.has[a] ? coord[a][p] - rp : 0;
    b.phi[a] = b.has[a] ? b.plo[a] + size : 0;
    // size_t conversion of the low index: exact for t > -1 (truncation); at
    // t <= -1 (or NaN) the reference's conversion wraps and its loop is empty
    const double t = (b.plo[a] - g.loface[a]) / g.h[a];
    if (!(t > -1.0)) b.skip = true;
    const double tc = t > 4.0e18 ? 4.0e18 : (t > 0.0 ? t : 0.0);
    b.lo[a] = (long)tc;
    if (b.has[a]) {
      // std::min(nmax, int(u) + 1), with u clamped where int(u) would overflow
      double u = (b.phi[a] - g.loface[a]) / g.h[a];
      u = u > 2.0e9 ? 2.0e9 : (u < -2.0e9 ? -2.0e9 : u);
      b.hi[a] = (long)u + 1;
    } else {
      b.hi[a] = b.lo[a] + 1;
    }
    // the reference bounds only a resolved axis by the window; bounding every
    // axis keeps each access inside the window (the same cells where the
    // reference's are in bounds)
    if (b.hi[a] > g.nmax[a]) b.hi[a] = g.nmax[a];
  }
  b.pvol = (b.has[0] ? 2 * rp : 1) * (b.has[1] ? 2 * rp : 1) * (b.has[2] ? 2 * rp : 1);
  return b;
}

__device__ __forceinline__ long box_cells(const PBox& b)
{
  if (b.skip) return 0;
  long n = 1;
#pragma unroll
  for (int a = 0; a < 3; ++a) n *= b.hi[a] > b.lo[a] ? b.hi[a] - b.lo[a] : 0;
  return n;
}

// Visit the cells of the box in the reference's order with (flat index, fraction).
template <typename F>
__device__ __forceinline__ void for_cells(const CellGrid& g, const PBox& b, F&& f)
{
  for (long k = b.lo[2]; k < b.hi[2]; ++k) {
    const double zcm = g.loface[2] + (double)k * g.h[2];
    const double zcp = zcm + g.h[2];
    const double zcont = b.has[2] ? dmin(zcp, b.phi[2]) - dmax(zcm, b.plo[2]) : 1;
    for (long j = b.lo[1]; j < b.hi[1]; ++j) {
      const double ycm = g.loface[1] + (double)j * g.h[1];
      const double ycp = ycm + g.h[1];
      const double ycont = b.has[1] ? dmin(ycp, b.phi[1]) - dmax(ycm, b.plo[1]) : 1;
      for (long i = b.lo[0]; i < b.hi[0]; ++i) {
        const double xcm = g.loface[0] + (double)i * g.h[0];
        const double xcp = xcm + g.h[0];
        const double xcont = b.has[0] ? dmin(xcp, b.phi[0]) - dmax(xcm, b.plo[0]) : 1;
        const double contribution = xcont * ycont * zcont / b.pvol;
        const long gi = g.glob[0] > 1 ? i + g.off[0] : 0;
        const long gj = g.glob[1] > 1 ? j + g.off[1] : 0;
        const long gk = g.glob[2] > 1 ? k + g.off[2] : 0;
        f(gi + (long)g.glob[0] * (gj + (long)g.glob[1] * gk), contribution);
      }
    }
  }
}

struct Coords {
  const double* c[3];
};

// a / b, correctly rounded, given r = 1 / b correctly rounded and the sizes of a and b
// such that no step can overflow or lose bits (P. Markstein, "Computation of elementary
// functions on the IBM RISC System/6000 processor", 1990: a quotient within one unit in
// the last place, corrected by its exact remainder, is the rounded quotient; the first
// correction brings it within one).  5 operations; a division takes 11, one of them at
// a quarter of the rate.
__device__ __forceinline__ double quotient(double a, double b, double r)
{
  double q = a * r;
  q = __builtin_fma(__builtin_fma(-b, q, a), r, q);
  return __builtin_fma(__builtin_fma(-b, q, a), r, q);
}
__device__ __forceinline__ bool quotient_safe(double a) { return fabs(a) > 1e-150 && fabs(a) < 1e150; }
__device__ __forceinline__ bool divisor_safe(double b) { return fabs(b) > 1e-100 && fabs(b) < 1e100; }

__device__ __forceinline__ double divide(double a, double b, double r, bool b_safe)
{
  return b_safe && quotient_safe(a) ? quotient(a, b, r) : a / b;
}

// A particle's cube and the cells [lo, hi) it overlaps, by particle_box's rules in
// 32-bit arithmetic (a value beyond 2^31 lies past any window either way).
struct PRange {
  int lo[3], hi[3];
  double plo[3];
  double size;
};

struct PIn {
  double c[3], size;
};

__device__ __forceinline__ PIn load_particle(const Coords& pc, const double* psize, long p)
{
  PIn v;
  v.size = psize[p];
#pragma unroll
  for (int a = 0; a < 3; ++a) v.c[a] = pc.c[a] ? pc.c[a][p] : 0;
  return v;
}

// False when the particle is skipped; the range may be empty.
__device__ __forceinline__ bool particle_range(const CellGrid& g, const bool (&has)[3], const PIn& v, PRange* r)
{
  r->size = v.size;
  const double rp = v.size * 0.5;
  bool ok = true;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const bool safe = divisor_safe(g.h[a]);
    r->plo[a] = has[a] ? v.c[a] - rp : 0;
    const double t = divide(r->plo[a] - g.loface[a], g.h[a], g.rh[a], safe);
    if (!(t > -1.0)) ok = false;
    r->lo[a] = (int)(t > 2147483646.0 ? 2147483646.0 : (t > 0.0 ? t : 0.0));
    if (has[a]) {
      double u = divide(r->plo[a] + v.size - g.loface[a], g.h[a], g.rh[a], safe);
      // an end below the window (a cube of negative size, or NaN) is 0: lo >= 0, so the
      // range is empty, and hi - lo cannot pass the range of an int
      u = u > 2147483646.0 ? 2147483646.0 : (u > -1.0 ? u : -1.0);
      r->hi[a] = (int)u + 1;
    } else {
      r->hi[a] = r->lo[a] + 1;
    }
    if (r->hi[a] > g.nmax[a]) r->hi[a] = g.nmax[a];
  }
  return ok;
}

__device__ __forceinline__ double cube_volume(const bool (&has)[3], double size)
{
  const double rp = size * 0.5;
  return (has[0] ? 2 * rp : 1) * (has[1] ? 2 * rp : 1) * (has[2] ? 2 * rp : 1);
}

// The gather: a thread per particle.  A particle of at most kSpan cells per axis forms
// its overlaps with them axis by axis once and then runs through the kSpan^3
// combinations in the reference's order (k, j, i), those no lane of the wave has being
// skipped; larger ones loop over their cells.  (Three nested loops ran for a wave's
// largest extent on each axis and formed all three overlaps in each round: about 25
// rounds of 55 vector instructions where a particle of 0.2-1.5 cells overlaps 6.3
// cells.)  4M particles on 64^3 cells, whose field fits the L2s: 100 us
// against 175; on 128^3 in random order, where 13M lines miss them (7.5 TB/s from the
// memory-side cache), 222 against 247, and 87 against 183 where the particles are in
// cell order.  AXES are the axes the particles resolve, bit a for axis a, and known to
// the compiler, since a particle reaches one cell along the others: 1M particles on 64
// cells of one axis 10.0 us, on 64 x 64 14.8 (15.1 and 19.9 where every axis takes kSpan
// cells; 12.9 and 23.6 by three nested loops).
constexpr int kSpan = 3;

template <int AXES>
__global__ __launch_bounds__(kBlock) void cell_to_particle_kernel(double* __restrict__ dest,
                                                                  const double* __restrict__ src, CellGrid g,
                                                                  Coords pc, const double* __restrict__ psize, long np,
                                                                  int* __restrict__ skipped)
{
  const long p = (long)blockIdx.x * kBlock + threadIdx.x;
  if (p >= np) return;
  constexpr bool has[3] = {(AXES & 1) != 0, (AXES & 2) != 0, (AXES & 4) != 0};
  constexpr int span[3] = {has[0] ? kSpan : 1, has[1] ? kSpan : 1, has[2] ? kSpan : 1};
  PRange r;
  if (!particle_range(g, has, load_particle(pc, psize, p), &r)) {
    if (skipped) atomicAdd(skipped, 1);
    dest[p] = 0.0;
    return;
  }
  const int nx = r.hi[0] - r.lo[0], ny = r.hi[1] - r.lo[1], nz = r.hi[2] - r.lo[2];
  double acc = 0.0;
  if (nx > 0 && ny > 0 && nz > 0) {
    const double vol = cube_volume(has, r.size), rvol = 1.0 / vol;
    double phi[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) phi[a] = has[a] ? r.plo[a] + r.size : 0;
    auto part = [&](int a, int i) {
      const double lo = g.loface[a] + (double)i * g.h[a], hi = lo + g.h[a];
      return has[a] ? __builtin_fmin(hi, phi[a]) - __builtin_fmax(lo, r.plo[a]) : 1.0;
    };
    const double* cell0 = src + (g.origin + r.lo[0] * g.stride[0] + r.lo[1] * g.stride[1] + r.lo[2] * g.stride[2]);
    double w[3][kSpan];
    bool fast = nx <= span[0] && ny <= span[1] && nz <= span[2] && divisor_safe(vol);
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int i = 0; i < span[a]; ++i) {
        w[a][i] = part(a, r.lo[a] + i);
        // an overlap of zero gives a quotient of zero (of either sign: the sum starts at
        // +0, so it never shows); three others multiply to a safe dividend
        fast = fast && (w[a][i] == 0.0 || (fabs(w[a][i]) > 1e-50 && fabs(w[a][i]) < 1e50));
      }
    if (fast) {
      double xy[kSpan][kSpan];
#pragma unroll
      for (int j = 0; j < span[1]; ++j)
#pragma unroll
        for (int i = 0; i < span[0]; ++i) xy[j][i] = w[0][i] * w[1][j];
#pragma unroll
      for (int k = 0; k < span[2]; ++k) {
        if (k < nz) {
          double v[kSpan][kSpan];
#pragma unroll
          for (int j = 0; j < span[1]; ++j)
#pragma unroll
            for (int i = 0; i < span[0]; ++i) {
              v[j][i] = 0.0;
              if (j < ny && i < nx) v[j][i] = cell0[i * g.stride[0] + j * g.stride[1] + k * g.stride[2]];
            }
#pragma unroll
          for (int j = 0; j < span[1]; ++j)
#pragma unroll
            for (int i = 0; i < span[0]; ++i)
              if (j < ny && i < nx) acc += v[j][i] * quotient(xy[j][i] * w[2][k], vol, rvol);
        }
      }
    } else {
      for (int k = 0; k < nz; ++k)
        for (int j = 0; j < ny; ++j)
          for (int i = 0; i < nx; ++i)
            acc += cell0[i * g.stride[0] + j * g.stride[1] + k * g.stride[2]] *
                   (part(0, r.lo[0] + i) * part(1, r.lo[1] + j) * part(2, r.lo[2] + k) / vol);
    }
  }
  dest[p] = acc;
}

__global__ void count_kernel(long* __restrict__ counts, CellGrid g, Coords pc, const double* __restrict__ psize,
                             long np, int* __restrict__ skipped)
{
  const long p = (long)blockIdx.x * kBlock + threadIdx.x;
  if (p >= np) return;
  const PBox b = particle_box(g, pc.c, psize, p);
  if (b.skip && skipped) atomicAdd(skipped, 1);
  counts[p] = box_cells(b);
}

// Entry e (the serial loop's e-th contribution: particles in order, each one's
// cells in k, j, i order) holds its cell and its value.
__global__ void fill_kernel(uint32_t* __restrict__ keys, double* __restrict__ vals,
                            const long* __restrict__ offsets, const double* __restrict__ src, CellGrid g,
                            Coords pc, const double* __restrict__ psize, long np)
{
  const long p = (long)blockIdx.x * kBlock + threadIdx.x;
  if (p >= np) return;
  const PBox b = particle_box(g, pc.c, psize, p);
  if (b.skip) return;
  long e = offsets[p];
  const double s = src[p];
  for_cells(g, b, [&](long cell, double c) {
    vals[e] = s * c;
    keys[e] = (uint32_t)cell;
    ++e;
  });
}

// After a stable sort by cell, each cell's entries are contiguous and in serial
// order; the first entry of each run adds the run, in order, onto the cell.
__global__ void run_sum_kernel(double* __restrict__ dest, const uint32_t* __restrict__ keys,
                               const double* __restrict__ vals, long total)
{
  const long s = (long)blockIdx.x * kBlock + threadIdx.x;
  if (s >= total) return;
  const uint32_t cell = keys[s];
  if (s > 0 && keys[s - 1] == cell) return;
  double acc = dest[cell];
  // The run is read U entries at a time, all loads issued before the adds, which
  // still go one by one in entry order up to the first entry of another cell
  // (cells are below 2^31, so the padding key 0xffffffff ends a run).
  constexpr int U = 8;
  for (long t = s;; t += U) {
    uint32_t k[U];
    double v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      k[u] = t + u < total ? keys[t + u] : 0xffffffffu;
      v[u] = t + u < total ? vals[t + u] : 0.0;
    }
    bool end = false;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      end = end || k[u] != cell;
      if (!end) acc += v[u];
    }
    if (end) break;
  }
  dest[cell] = acc;
}

// ---- ParticleToCell by bricks ------------------------------------------------------
// The window is cut into bricks of 64 to 1024 cells.
//   1. count_bricks: each block of a fixed share of the particles counts, in LDS, how
//      many of them reach into each brick (one row of counts per block);
//   2. scan_rows, scan_bricks: places of every block's records of every brick, by
//      prefix sums over the rows of a brick and over the bricks;
//   3. fill_bricks: the same blocks write a 48-byte record per particle and brick, or
//      one wave for each block, where a block has many in one brick (particles in an
//      order of space);
//   4. sum_bricks: one workgroup per brick, a thread per cell: the records set their
//      bits in the masks of the cells they reach, and each cell adds its contributions
//      in the order of the bits (the serial loop's order).
// Bound by the records' scattered writes (about 1.5 of them per particle of up to 1.5
// cells) and by the arithmetic per contribution (75 % of sum_bricks' time issues
// vector instructions), where a sort of the contributions moves 12 bytes of each (6.3
// per particle) through memory 7 times.  2M particles of 0.2-1.5 cells on 112x96x104
// cells: 336 us per call (sum_bricks 131, fill_bricks 128, count_bricks 25, the scans
// 30) against 870 us sorted; 4M on 128^3: 564 against 1622; 1M on 40^3: 302 against
// 713.  In cell order 395 against 870 (sum_bricks 188: successive records wait for the
// same threads; fill_bricks, one wave per block, 132), 4M on 128^3 702 and 1617.

struct Bricks {
  int sh[3];     // log2 of a brick's cells per axis (at most 5)
  int nb[3];     // bricks per axis
  int total;     // bricks
  bool has[3];   // axes the particles resolve
};

struct alignas(16) BrickRec {
  double plo[3];
  double size, src;
  uint32_t idx;     // the particle
  uint32_t range;   // first and last cell within the brick, 5 bits each, per axis
};
static_assert(sizeof(BrickRec) == 48, "record size");

struct BrickStats {
  uint64_t records;   // of all bricks
  uint32_t most;      // of the fullest brick
  uint32_t group;     // that one block writes into one brick, at most
};
static_assert(sizeof(BrickStats) <= kHostSlotBytes, "statistics are written to a slot");

constexpr int kBinThreads = 512;
constexpr int kBinBatch = 4;          // particles a thread loads at a time
constexpr int kBinRows = 512;          // blocks that bin the particles, at most
constexpr int kRowCols = 16;           // bricks per block of scan_rows
constexpr int kRowSegments = 64;
constexpr int kMaxBricks = 16384;      // 64 KB of LDS counters
constexpr int kBrickTarget = 512;      // particles per brick of up to 256 cells, at most
constexpr int kThinTarget = 128;       // of a larger one
constexpr int kMostGroup = 32;         // records of one block in one brick, in any order
constexpr int kGranule = 64;           // particles whose records one wave writes at a time
// Particles per cell of the window: denser sets are sorted, since a cell's thread walks
// its contributions alone (1M particles on 24^3 cells, 72 per cell: 1250 us by bricks,
// 700 sorted; on 40^3, 16 per cell: 340 and 711).
constexpr double kMostPerCell = 32;

// f(brick, bx, by, bz) for every brick the range reaches into.
template <typename F>
__device__ __forceinline__ void for_bricks(const Bricks& b, const PRange& r, F&& f)
{
  if (r.hi[0] <= r.lo[0] || r.hi[1] <= r.lo[1] || r.hi[2] <= r.lo[2]) return;
  for (int z = r.lo[2] >> b.sh[2]; z <= (r.hi[2] - 1) >> b.sh[2]; ++z)
    for (int y = r.lo[1] >> b.sh[1]; y <= (r.hi[1] - 1) >> b.sh[1]; ++y)
      for (int x = r.lo[0] >> b.sh[0]; x <= (r.hi[0] - 1) >> b.sh[0]; ++x)
        f(x + b.nb[0] * (y + b.nb[1] * z), x, y, z);
}

__global__ __launch_bounds__(kBinThreads) void count_bricks(uint32_t* __restrict__ rows, CellGrid g, Bricks b,
                                                            Coords pc, const double* __restrict__ psize, long np,
                                                            int share, int* __restrict__ skipped)
{
  extern __shared__ uint32_t bins[];
  for (int i = threadIdx.x; i < b.total; i += kBinThreads) bins[i] = 0;
  __syncthreads();
  const long first = (long)blockIdx.x * share, last = min(first + share, np);
  for (long p0 = first + threadIdx.x; p0 < last; p0 += kBinBatch * kBinThreads) {
    PIn in[kBinBatch];
#pragma unroll
    for (int u = 0; u < kBinBatch; ++u) in[u] = load_particle(pc, psize, min(p0 + u * kBinThreads, last - 1));
#pragma unroll
    for (int u = 0; u < kBinBatch; ++u) {
      if (p0 + u * kBinThreads >= last) continue;
      PRange r;
      if (!particle_range(g, b.has, in[u], &r)) {
        if (skipped) atomicAdd(skipped, 1);
        continue;
      }
      for_bricks(b, r, [&](int brick, int, int, int) { atomicAdd(&bins[brick], 1u); });
    }
  }
  __syncthreads();
  uint32_t* row = rows + (size_t)blockIdx.x * b.total;
  for (int i = threadIdx.x; i < b.total; i += kBinThreads) row[i] = bins[i];
}

// Each brick's counts become their exclusive prefix over the rows; totals[brick]
// their sum, group[block] the largest count.  kRowCols bricks per block, the rows in
// kRowSegments parts.
__global__ __launch_bounds__(kRowCols * kRowSegments) void scan_rows(uint32_t* __restrict__ rows,
                                                               uint32_t* __restrict__ totals,
                                                               uint32_t* __restrict__ group, int n_rows,
                                                               int n_bricks)
{
  constexpr int U = 8;   // loads in flight per thread
  __shared__ uint32_t part[kRowSegments][kRowCols], bigs[kRowCols * kRowSegments / 64];
  const int col = threadIdx.x % kRowCols, seg = threadIdx.x / kRowCols;
  const int brick = blockIdx.x * kRowCols + col;
  const int per = (n_rows + kRowSegments - 1) / kRowSegments;
  const int r0 = min(seg * per, n_rows), r1 = min(r0 + per, n_rows);
  uint32_t* mine = rows + min(brick, n_bricks - 1);
  uint32_t sum = 0, big = 0, v[U] = {};
  for (int r = r0; r < r1; r += U) {
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = mine[(size_t)min(r + u, r1 - 1) * n_bricks];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (r + u < r1) sum += v[u];
      big = max(big, v[u]);
    }
  }
  part[seg][col] = sum;
  big = brick < n_bricks ? big : 0;
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) big = max(big, (uint32_t)__shfl_xor((int)big, off, 64));
  if ((threadIdx.x & 63) == 0) bigs[threadIdx.x >> 6] = big;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kRowCols * kRowSegments / 64; ++w) big = max(big, bigs[w]);
    group[blockIdx.x] = big;
  }
  uint32_t at = 0;
#pragma unroll
  for (int q = 0; q < kRowSegments; ++q) at += q < seg ? part[q][col] : 0;
  if (brick >= n_bricks) return;
  for (int r = r0; r < r1; r += U) {
    if (per > U) {   // else v holds the whole part
#pragma unroll
      for (int u = 0; u < U; ++u) v[u] = mine[(size_t)min(r + u, r1 - 1) * n_bricks];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (r + u >= r1) continue;   // past the part v repeats its last row
      mine[(size_t)(r + u) * n_bricks] = at;
      at += v[u];
    }
  }
  if (seg == kRowSegments - 1) totals[brick] = at;
}

// base[brick]: records before the brick's first (base[n_bricks]: all of them), and
// the statistics the host chooses the next launch by.  One block, 1024 bricks at a
// time.  (Where the records pass 2^32, base is not used.)
__global__ __launch_bounds__(1024) void scan_bricks(uint32_t* __restrict__ base, const uint32_t* __restrict__ totals,
                                                    int n_bricks, const uint32_t* __restrict__ group, int n_group,
                                                    BrickStats* __restrict__ stats)
{
  __shared__ unsigned long long part[16];
  __shared__ uint32_t bigs[16], groups[16];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  unsigned long long before = 0;
  uint32_t big = 0;
  for (int i0 = 0; i0 < n_bricks; i0 += 1024) {
    const int i = i0 + t;
    const uint32_t own = i < n_bricks ? totals[i] : 0;
    big = max(big, own);
    unsigned long long sum = own;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const unsigned long long v = __shfl_up(sum, off, 64);
      if (lane >= off) sum += v;
    }
    if (lane == 63) part[wave] = sum;
    __syncthreads();
    unsigned long long all = 0;
#pragma unroll
    for (int w = 0; w < 16; ++w) {
      const unsigned long long v = part[w];
      if (w < wave) sum += v;
      all += v;
    }
    if (i < n_bricks) base[i] = (uint32_t)(before + sum - own);
    before += all;
    __syncthreads();
  }
  uint32_t grp = 0;
  for (int i = t; i < n_group; i += 1024) grp = max(grp, group[i]);
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    big = max(big, (uint32_t)__shfl_xor((int)big, off, 64));
    grp = max(grp, (uint32_t)__shfl_xor((int)grp, off, 64));
  }
  if (lane == 0) {
    bigs[wave] = big;
    groups[wave] = grp;
  }
  __syncthreads();
  if (t == 0) {
    for (int w = 1; w < 16; ++w) {
      big = max(big, bigs[w]);
      grp = max(grp, groups[w]);
    }
    base[n_bricks] = (uint32_t)before;
    stats->records = before;
    stats->most = big;
    stats->group = grp;
  }
}

// NT threads per block.  With kBinThreads a block's records of one brick come out in any
// order, which sum_bricks puts right where they are few.  With one wave (NT 64) they
// come out in order up to those of kGranule consecutive particles: a wave's LDS
// operations are executed one after the other.
template <int NT>
__global__ __launch_bounds__(NT) void fill_bricks(BrickRec* __restrict__ recs, const uint32_t* __restrict__ rows,
                                                  const uint32_t* __restrict__ base, CellGrid g, Bricks b, Coords pc,
                                                  const double* __restrict__ psize, const double* __restrict__ src,
                                                  long np, int share)
{
  extern __shared__ uint32_t bins[];
  const uint32_t* row = rows + (size_t)blockIdx.x * b.total;
  for (int i = threadIdx.x; i < b.total; i += NT) bins[i] = base[i] + row[i];
  __syncthreads();
  const long first = (long)blockIdx.x * share, last = min(first + share, np);
  for (long p0 = first + threadIdx.x; p0 - threadIdx.x < last; p0 += kBinBatch * NT) {
    PIn in[kBinBatch];
    double val[kBinBatch];
#pragma unroll
    for (int u = 0; u < kBinBatch; ++u) {
      const long p = min(p0 + u * NT, last - 1);
      in[u] = load_particle(pc, psize, p);
      val[u] = src[p];
    }
#pragma unroll
    for (int u = 0; u < kBinBatch; ++u) {
      const long p = p0 + u * NT;
      PRange r;
      if (p < last && particle_range(g, b.has, in[u], &r)) {
        BrickRec rec;
#pragma unroll
        for (int a = 0; a < 3; ++a) rec.plo[a] = r.plo[a];
        rec.size = r.size;
        rec.src = val[u];
        rec.idx = (uint32_t)p;
        for_bricks(b, r, [&](int brick, int x, int y, int z) {
          const int at[3] = {x, y, z};
          rec.range = 0;
#pragma unroll
          for (int a = 0; a < 3; ++a) {
            const int o = at[a] << b.sh[a], m = (1 << b.sh[a]) - 1;
            const int lo = max(r.lo[a] - o, 0), hi = min(r.hi[a] - 1 - o, m);
            rec.range |= (uint32_t)(lo | hi << 5) << (10 * a);
          }
          recs[atomicAdd(&bins[brick], 1u)] = rec;
        });
      }
      if constexpr (NT == kGranule) {   // one granule's places before the next one's
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
      }
    }
  }
}

// f(cell) for the cells of a record's range, x fastest.
template <typename F>
__device__ __forceinline__ void for_range(const Bricks& b, uint32_t range, F&& f)
{
  const int x0 = range & 31, x1 = (range >> 5) & 31, y0 = (range >> 10) & 31, y1 = (range >> 15) & 31;
  const int z0 = (range >> 20) & 31, z1 = (range >> 25) & 31;
  for (int z = z0; z <= z1; ++z)
    for (int y = y0; y <= y1; ++y)
      for (int x = x0; x <= x1; ++x) f(x | (y | z << b.sh[1]) << b.sh[0]);
}

// One workgroup per brick, NT threads with Q cells each.  The brick's records are
// taken R at a time in the order of their particles.  A record goes to LDS, where it
// also sets its bit in the mask of every cell it reaches; each cell's thread then
// walks its mask's bits upwards, which is particle order, and adds the contributions
// it forms from the records.
//
// A brick's list is in order up to the records of one granule, which are at most `group`:
// a record's place follows from its neighbours.  A granule is what one block of
// fill_bricks wrote (`share` consecutive particles, 1.4 records on average in the case
// above), or, where that is much, a part of 2^part of them.
template <int NT, int Q, int R>
__global__ __launch_bounds__(NT) void sum_bricks(double* __restrict__ dest, CellGrid g, Bricks b,
                                                 const uint32_t* __restrict__ base,
                                                 const BrickRec* __restrict__ recs, uint32_t share, int part,
                                                 int group)
{
  constexpr int C = NT * Q;      // cells, at most
  constexpr int W = R / 64;      // mask words per cell
  __shared__ double plo[3][R], size[R], val[R];
  __shared__ unsigned long long mask[W][C];
  __shared__ uint32_t idx[R + 4 * (kGranule - 1)];

  const int brick = xcd_tile(blockIdx.x, gridDim.x);
  const uint32_t first = base[brick];
  const int n = (int)(base[brick + 1] - first);
  if (n == 0) return;
  const BrickRec* mine = recs + first;
  const int t = threadIdx.x;
  const int cells = 1 << (b.sh[0] + b.sh[1] + b.sh[2]);
  const int ox = (brick % b.nb[0]) << b.sh[0];
  const int oy = (brick / b.nb[0] % b.nb[1]) << b.sh[1];
  const int oz = (brick / b.nb[0] / b.nb[1]) << b.sh[2];
  const int M = group - 1;       // a record is at most M places from its own

  double acc[Q], lo[Q][3], hi[Q][3];
  long at[Q];   // flat index of the cell, -1 outside the window
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    const int c = t + q * NT;
    const int x = ox + (c & ((1 << b.sh[0]) - 1)), y = oy + ((c >> b.sh[0]) & ((1 << b.sh[1]) - 1));
    const int z = oz + (c >> (b.sh[0] + b.sh[1]));
    const int xyz[3] = {x, y, z};
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      lo[q][a] = g.loface[a] + (double)xyz[a] * g.h[a];
      hi[q][a] = lo[q][a] + g.h[a];
    }
    at[q] = -1;
    acc[q] = 0.0;
    if (c < cells && x < g.nmax[0] && y < g.nmax[1] && z < g.nmax[2]) {
      const long gx = g.glob[0] > 1 ? x + g.off[0] : 0, gy = g.glob[1] > 1 ? y + g.off[1] : 0;
      const long gz = g.glob[2] > 1 ? z + g.off[2] : 0;
      at[q] = gx + (long)g.glob[0] * (gy + (long)g.glob[1] * gz);
      acc[q] = dest[at[q]];
    }
  }

  for (int r0 = 0; r0 < n; r0 += R) {
    // the particles of places r0 - 2M .. r0 + R + 2M, and empty masks
    for (int i = t; i < R + 4 * M; i += NT) {
      const int j = r0 - 2 * M + i;
      idx[i] = j >= 0 && j < n ? mine[j].idx : 0xffffffffu;   // no particle's block
    }
    for (int i = t; i < W * C; i += NT) mask[i / C][i % C] = 0;
    __syncthreads();
    for (int i = M + t; i < R + 3 * M; i += NT) {
      const int j = r0 - 2 * M + i;
      if (j < 0 || j >= n) continue;
      // the particles [g0, g0 + gn) are p's granule; "no particle" is in none (p < 2^31)
      const uint32_t p = idx[i], in = p % share, g0 = p - (in & ((1u << part) - 1));
      const uint32_t gn = min(1u << part, p - in + share - g0);
      int place = j - r0;
      for (int k = i - 1; k >= i - M && idx[k] - g0 < gn; --k) place -= idx[k] > p;
      for (int k = i + 1; k <= i + M && idx[k] - g0 < gn; ++k) place += idx[k] < p;
      if (place < 0 || place >= R) continue;
      const BrickRec r = mine[j];
#pragma unroll
      for (int a = 0; a < 3; ++a) plo[a][place] = r.plo[a];
      size[place] = r.size;
      val[place] = r.src;
      unsigned long long* word = mask[place >> 6];
      for_range(b, r.range, [&](int c) { atomicOr(&word[c], 1ull << (place & 63)); });
    }
    __syncthreads();
    const int words = min(W, (n - r0 + 63) / 64);
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int c = t + q * NT;
      int w = 0;
      unsigned long long m = mask[0][c];
      for (;;) {
        while (m == 0 && ++w < words) m = mask[w][c];
        if (w >= words) break;
        const int i = w * 64 + __builtin_ctzll(m);
        m &= m - 1;
        const double s = size[i];
        double part[3];
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          const double pl = plo[a][i], ph = pl + s;
          part[a] = b.has[a] ? __builtin_fmin(hi[q][a], ph) - __builtin_fmax(lo[q][a], pl) : 1;
        }
        acc[q] += val[i] * (part[0] * part[1] * part[2] / cube_volume(b.has, s));
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (int q = 0; q < Q; ++q)
    if (at[q] >= 0) dest[at[q]] = acc[q];
}

using SumBricksFn = void (*)(double*, CellGrid, Bricks, const uint32_t*, const BrickRec*, uint32_t, int, int);
SumBricksFn sum_bricks_fn(int cells, int* threads)
{
  *threads = cells <= 64 ? 64 : cells <= 128 ? 128 : 256;
  return cells <= 64    ? sum_bricks<64, 1, 128>
         : cells <= 128 ? sum_bricks<128, 1, 128>
         : cells <= 256 ? sum_bricks<256, 1, 256>
         : cells <= 512 ? sum_bricks<256, 2, 256>
                        : sum_bricks<256, 4, 128>;
}

// Brick shape for np particles on the window, within 64 to 1024 cells (fewer on windows
// of fewer resolved axes) and kMaxBricks bricks: up to 256 cells for at most kBrickTarget
// particles per brick, more for at most kThinTarget.  A cell thread of a larger brick
// holds 2 or 4 cells whose masks it walks one after the other, which pays only where
// there is little in them (per call, 256, 512 and 1024 cells: 1M particles on 128^3 212,
// 217 and 257 us, 100k on 64^3 69, 81 and 108; 500k on 160x160x80 155, 142 and 160, 200k on
// 128^3 124, 110 and 104).  False where kMaxBricks bricks do not cover the window.
bool choose_bricks(const CellGrid& g, const Coords& pc, int64_t np, Bricks* b)
{
  const double window = (double)g.nmax[0] * g.nmax[1] * g.nmax[2];
  // A brick's time goes with the particles per cell, the sort's with the particles: small
  // dense sets are sorted (per call, bricks and sort: 200k particles on 24^3 366 and 244 us,
  // 20k on 16^3 203 and 155, 8k on 12^3 175 and 132; 400k on 30^3 317 and 340, 200k 188 and
  // 226, 500k on 40^3 198 and 413), less soon where an axis has one cell or is not resolved
  // and a particle reaches fewer cells (60k on 100x60 140 and 190, 150k 278 and 261).
  double per_cell = np / window;
  for (int a = 0; a < 3; ++a)
    if (!pc.c[a] || g.nmax[a] == 1) per_cell *= 0.4;
  if (np > kMostPerCell * window || per_cell > 2.6 + np / 35000.0) return false;
  int bits = 6;
  while (bits < 10 && np / window * (double)(2 << bits) <= (bits < 8 ? kBrickTarget : kThinTarget)) ++bits;
  for (;; ++bits) {
    int used = 0;
    for (int a = 0; a < 3; ++a) b->sh[a] = 0;
    for (; used < bits; ++used) {
      int pick = -1;
      for (int a = 0; a < 3; ++a)
        if (b->sh[a] < 5 && (1 << b->sh[a]) < g.nmax[a] && (pick < 0 || b->sh[a] < b->sh[pick])) pick = a;
      if (pick < 0) break;
      ++b->sh[pick];
    }
    double total = 1;
    for (int a = 0; a < 3; ++a) {
      b->nb[a] = (g.nmax[a] + (1 << b->sh[a]) - 1) >> b->sh[a];
      b->has[a] = pc.c[a] != nullptr;
      total *= b->nb[a];
    }
    if (total <= kMaxBricks) {
      b->total = (int)total;
      return true;
    }
    if (bits >= 10 || used < bits) return false;
  }
}

// Whether a counted set goes on by bricks, from times in us on MI355X.  The fullest brick's
// workgroup walks its records alone, the longer for each the fewer waves share them,
// and much longer where the list is in an order of space, whose successive records belong
// to the same few cells: per record 0.06 us in bricks of 256 cells in random order, 0.18
// in cell order, 0.11 and 0.48 in bricks of 64.  A set in random order that is sorted
// all the same has a clear gain by it (1.25), one in order no loss.  Sets of 5k to 4M
// particles, some of them crowded into a part of the window, estimated, measured and
// sorted after the count: 2M in cell order 438, 396 and 917 us, with a fifth of them in
// 30^3 cells 1440, 1405 and 980; the same at random 714, 698 and 980; 1M on 64^3 in cell
// order 379, 324 and 605; 1M on 40^3 841, 904 and 737; 30% of 1M random in 20^3 cells 977,
// 979 and 635.
bool bricks_pay(const Bricks& b, const BrickStats& st, int64_t np)
{
  constexpr double any[] = {0.11, 0.09, 0.06, 0.08, 0.10}, ordered[] = {0.48, 0.28, 0.18, 0.30, 0.30};
  const int bits = std::max(b.sh[0] + b.sh[1] + b.sh[2], 6) - 6;
  const bool few = st.group <= kMostGroup;
  const double rest = st.most - 0.5 * (double)st.records / b.total;
  const double bricks = 50 + 1e-4 * (double)st.records + (few ? any : ordered)[bits] * rest;
  return bricks <= (few ? 1.25 : 1.0) * (150 + 4.2e-4 * (double)np);
}

// The scatter by bricks.  *counted: the particles were counted (and the skipped ones
// reported); *done: dest holds the sums.  Left to the sort when *done stays false:
// windows of too many bricks, dense sets, and, after the count (17 us for 5k particles, 40
// for 2M, 75 for 4M), sets crowded into few bricks.
int scatter_by_bricks(double* dest, const double* src, const CellGrid& g, const Coords& pc, const double* psize,
                      int64_t np, int32_t* skipped, hipStream_t s, const char* ctx, bool* counted, bool* done)
{
  *counted = *done = false;
  Bricks b;
  if (np >= (int64_t(1) << 31) || !choose_bricks(g, pc, np, &b)) return NEBO_OK;
  // a row per 1024 particles, and per 4 particles per brick, so that one block's records
  // of one brick stay few (5000 particles on 24^3 cells, 54 bricks: rows of 1000 left the
  // set to the sort, 150 us); at most kBinRows, more where the bricks are few (dense sets)
  const int64_t most_rows = std::max<int64_t>(kBinRows, (int64_t)kBinRows * 4096 / b.total);
  const int64_t rows_wanted = std::max((np + 1023) / 1024, np / (4 * (int64_t)b.total));
  const int n_rows = (int)std::min<int64_t>(most_rows, rows_wanted);
  const int share = (int)((np + n_rows - 1) / n_rows);
  const size_t row_bytes = sizeof(uint32_t) * (size_t)b.total;
  char* work = nullptr;
  BrickStats* stats = nullptr;
  int rc = host_slot_take((void**)&stats, ctx);
  if (rc) return rc;
  // rows, totals, base (+1), group (one per block of scan_rows)
  const int n_group = (b.total + kRowCols - 1) / kRowCols;
  if ((rc = scratch_alloc((void**)&work, row_bytes * (n_rows + 2) + sizeof(uint32_t) * (1 + n_group), s, ctx))) {
    host_slot_give(stats);
    return rc;
  }
  uint32_t* rows = reinterpret_cast<uint32_t*>(work);
  uint32_t* totals = rows + (size_t)n_rows * b.total;
  uint32_t* base = totals + b.total;
  uint32_t* group = base + b.total + 1;
  hipLaunchKernelGGL(count_bricks, dim3(n_rows), dim3(kBinThreads), row_bytes, s, rows, g, b, pc, psize, (long)np,
                     share, skipped);
  hipLaunchKernelGGL(scan_rows, dim3(n_group), dim3(kRowCols * kRowSegments), 0, s,
                     rows, totals, group, n_rows,
                     b.total);
  hipLaunchKernelGGL(scan_bricks, dim3(1), dim3(1024), 0, s, base, totals, b.total, group, n_group,
                     stats);
  rc = check_hip(hipGetLastError(), ctx);
  if (!rc) rc = check_hip(hipStreamSynchronize(s), ctx);
  const BrickStats st = *stats;
  host_slot_give(stats);
  if (rc) {
    scratch_free(work, s);
    return rc;
  }
  *counted = true;
  if (st.records > 0 && st.records < (uint64_t(1) << 31) && bricks_pay(b, st, np)) {
    BrickRec* recs = nullptr;
    if (!(rc = scratch_alloc((void**)&recs, sizeof(BrickRec) * st.records, s, ctx))) {
      const bool few = st.group <= kMostGroup;
      const auto fill = few ? fill_bricks<kBinThreads> : fill_bricks<kGranule>;
      hipLaunchKernelGGL(fill, dim3(n_rows), dim3(few ? kBinThreads : kGranule), row_bytes, s, recs, rows, base, g, b,
                         pc, psize, src, (long)np, share);
      int threads = 0;
      const SumBricksFn fn = sum_bricks_fn(1 << (b.sh[0] + b.sh[1] + b.sh[2]), &threads);
      hipLaunchKernelGGL(fn, dim3(b.total), dim3(threads), 0, s, dest, g, b, base, recs, (uint32_t)share,
                         few ? 31 : 6, few ? (int)st.group : std::min<int>(st.group, kGranule));
      rc = check_hip(hipGetLastError(), ctx);
      scratch_free(recs, s);
    }
    *done = rc == NEBO_OK;
  } else if (st.records == 0) {
    *done = true;
  }
  scratch_free(work, s);
  return rc;
}

int bits_for(uint64_t n)   // bits to hold 0..n-1
{
  int b = 0;
  while (b < 64 && (1ull << b) < n) ++b;
  return b;
}

int check_particle_call(const nebo_field_t* f, const double* psize, int64_t np, const nebo_particle_geom_t* geom,
                        const char* ctx)
{
  if (!f || !geom || (np > 0 && !psize)) return set_error(NEBO_ERR_INVALID, ctx, "null argument");
  if (np < 0) return set_error(NEBO_ERR_INVALID, ctx, "negative particle count");
  if (f->device < 0) return set_error(NEBO_ERR_DEVICE, ctx, "the cell field must be resident on a GPU");
  if ((long)f->glob[0] * f->glob[1] * f->glob[2] >= (1L << 31))
    return set_error(NEBO_ERR_TOO_LARGE, ctx, "field has 2^31 or more points");
  return NEBO_OK;
}

}  // namespace

struct PointMap {
  int device;
  int64_t n;              // points
  int64_t max_index;
  int64_t* gather;        // n indices (FieldToPoint)
  int64_t* scatter_src;   // m point positions (PointToField, last occurrence of each index)
  int64_t* scatter_dst;   // m field indices
  int64_t m;
};

}  // namespace nebo

struct nebo_point_map : nebo::PointMap {};

using namespace nebo;

extern "C" int nebo_cell_to_particle(double* dest, const nebo_field_t* src, const double* px, const double* py,
                                     const double* pz, const double* psize, int64_t np,
                                     const nebo_particle_geom_t* geom, int32_t* skipped, void* stream)
{
  static const char* ctx = "Nebo Particle Interpolation";
  clear_error();
  int rc = check_particle_call(src, psize, np, geom, ctx);
  if (rc) return rc;
  if (np == 0) return NEBO_OK;
  if (!dest) return set_error(NEBO_ERR_INVALID, ctx, "null argument");
  const CellGrid g = make_grid(src, *geom);
  const Coords pc{{px, py, pz}};
  const long blocks = (np + kBlock - 1) / kBlock;
  using Gather = void (*)(double*, const double*, CellGrid, Coords, const double*, long, int*);
  static const Gather gather[8] = {cell_to_particle_kernel<0>, cell_to_particle_kernel<1>, cell_to_particle_kernel<2>,
                                   cell_to_particle_kernel<3>, cell_to_particle_kernel<4>, cell_to_particle_kernel<5>,
                                   cell_to_particle_kernel<6>, cell_to_particle_kernel<7>};
  hipLaunchKernelGGL(gather[(px ? 1 : 0) | (py ? 2 : 0) | (pz ? 4 : 0)], dim3((unsigned)blocks), dim3(kBlock), 0, (hipStream_t)stream,
                     dest, static_cast<const double*>(src->values), g, pc, psize, (long)np, skipped);
  return check_hip(hipGetLastError(), ctx);
}

extern "C" int nebo_particle_to_cell(const nebo_field_t* dest, const double* src, const double* px,
                                     const double* py, const double* pz, const double* psize, int64_t np,
                                     const nebo_particle_geom_t* geom, int32_t* skipped, void* stream)
{
  static const char* ctx = "Nebo Particle Interpolation";
  clear_error();
  int rc = check_particle_call(dest, psize, np, geom, ctx);
  if (rc) return rc;
  if (np > 0 && !src) return set_error(NEBO_ERR_INVALID, ctx, "null argument");
  // dest <<= 0.0 (the reference's first step; same limits as any scalar assignment)
  {
    nebo_node_t zero;
    std::memset(&zero, 0, sizeof zero);
    zero.op = NEBO_SCALAR;
    zero.value = 0.0;
    const nebo_expr_t e{1, &zero, 0, nullptr, 0, nullptr, 0, nullptr};
    if ((rc = nebo_assign(dest, &e, 1, stream))) return rc;
    clear_error();
  }
  if (np == 0) return NEBO_OK;
  hipStream_t s = (hipStream_t)stream;
  const CellGrid g = make_grid(dest, *geom);
  const Coords pc{{px, py, pz}};
  {
    bool counted = false, done = false;
    rc = scatter_by_bricks(static_cast<double*>(dest->values), src, g, pc, psize, np, skipped, s, ctx, &counted, &done);
    if (rc || done) return rc;
    if (counted) skipped = nullptr;
  }
  const unsigned blocks = (unsigned)((np + kBlock - 1) / kBlock);
  long* counts = nullptr;
  long* offsets = nullptr;
  if ((rc = scratch_alloc((void**)&counts, sizeof(long) * 2 * np, s, ctx))) return rc;
  offsets = counts + np;
  hipLaunchKernelGGL(count_kernel, dim3(blocks), dim3(kBlock), 0, s, counts, g, pc, psize, (long)np, skipped);
  size_t tmp_bytes = 0;
  void* tmp = nullptr;
  rc = check_hip(rocprim::exclusive_scan(nullptr, tmp_bytes, counts, offsets, 0L, (size_t)np,
                                         rocprim::plus<long>(), s),
                 ctx);
  if (!rc) rc = scratch_alloc(&tmp, tmp_bytes, s, ctx);
  if (!rc)
    rc = check_hip(rocprim::exclusive_scan(tmp, tmp_bytes, counts, offsets, 0L, (size_t)np,
                                           rocprim::plus<long>(), s),
                   ctx);
  long last[2] = {0, 0};
  if (!rc) rc = check_hip(hipMemcpyAsync(&last[0], offsets + np - 1, sizeof(long), hipMemcpyDeviceToHost, s), ctx);
  if (!rc) rc = check_hip(hipMemcpyAsync(&last[1], counts + np - 1, sizeof(long), hipMemcpyDeviceToHost, s), ctx);
  if (!rc) rc = check_hip(hipStreamSynchronize(s), ctx);
  scratch_free(tmp, s);
  tmp = nullptr;
  const long total = last[0] + last[1];
  if (rc || total == 0) {
    scratch_free(counts, s);
    return rc;
  }
  // cells fit 32-bit keys (the field has fewer than 2^31 points, checked above)
  const long npts = (long)dest->glob[0] * dest->glob[1] * dest->glob[2];
  const int cbits = bits_for((uint64_t)npts);
  uint32_t* keys = nullptr;
  double* vals = nullptr;
  rc = scratch_alloc((void**)&keys, sizeof(uint32_t) * 2 * total, s, ctx);
  if (!rc) rc = scratch_alloc((void**)&vals, sizeof(double) * 2 * total, s, ctx);
  if (!rc) {
    hipLaunchKernelGGL(fill_kernel, dim3(blocks), dim3(kBlock), 0, s, keys, vals, offsets, src, g, pc, psize,
                       (long)np);
    rc = check_hip(hipGetLastError(), ctx);
  }
  // stable LSD radix sort on the cell alone: within a cell the entries keep
  // their serial order, so the run sums add in the serial loop's order
  uint32_t* skeys = keys ? keys + total : nullptr;
  double* svals = vals ? vals + total : nullptr;
  if (!rc)
    rc = check_hip(rocprim::radix_sort_pairs(nullptr, tmp_bytes, keys, skeys, vals, svals, (size_t)total, 0,
                                             (unsigned)cbits, s),
                   ctx);
  if (!rc) rc = scratch_alloc(&tmp, tmp_bytes, s, ctx);
  if (!rc)
    rc = check_hip(rocprim::radix_sort_pairs(tmp, tmp_bytes, keys, skeys, vals, svals, (size_t)total, 0,
                                             (unsigned)cbits, s),
                   ctx);
  if (!rc) {
    hipLaunchKernelGGL(run_sum_kernel, dim3((unsigned)((total + kBlock - 1) / kBlock)), dim3(kBlock), 0, s,
                       static_cast<double*>(dest->values), skeys, svals, total);
    rc = check_hip(hipGetLastError(), ctx);
  }
  scratch_free(tmp, s);
  scratch_free(vals, s);
  scratch_free(keys, s);
  scratch_free(counts, s);
  return rc;
}

namespace {

__global__ void gather_kernel(double* __restrict__ dest, const double* __restrict__ src,
                              const int64_t* __restrict__ idx, long n)
{
  const long i = (long)blockIdx.x * kBlock + threadIdx.x;
  if (i < n) dest[i] = src[idx[i]];
}

__global__ void scatter_kernel(double* __restrict__ dest, const double* __restrict__ src,
                               const int64_t* __restrict__ from, const int64_t* __restrict__ to, long m)
{
  const long i = (long)blockIdx.x * kBlock + threadIdx.x;
  if (i < m) dest[to[i]] = src[from[i]];
}

int check_map_field(const nebo_point_map* map, const nebo_field_t* f, const char* ctx)
{
  if (!map || !f) return set_error(NEBO_ERR_INVALID, ctx, "null argument");
  if (f->device != map->device) return set_error(NEBO_ERR_DEVICE, ctx, "field and index list are on different devices");
  const long npts = (long)f->glob[0] * f->glob[1] * f->glob[2];
  if (map->n > 0 && map->max_index >= npts)
    return set_error(NEBO_ERR_INVALID, ctx, "point index beyond the field's block");
  return NEBO_OK;
}

}  // namespace

extern "C" int nebo_point_map_create(const int64_t* indices, int64_t n, int device, nebo_point_map_t** out)
{
  static const char* ctx = "Nebo Point Field";
  clear_error();
  if (!out || (n > 0 && !indices)) return set_error(NEBO_ERR_INVALID, ctx, "null argument");
  if (n < 0) return set_error(NEBO_ERR_INVALID, ctx, "negative point count");
  *out = nullptr;
  std::vector<int64_t> from, to;
  std::unordered_map<int64_t, size_t> slot;   // field index -> position in from/to
  int64_t mx = -1;
  for (int64_t i = 0; i < n; ++i) {
    if (indices[i] < 0) return set_error(NEBO_ERR_INVALID, ctx, "negative point index");
    mx = indices[i] > mx ? indices[i] : mx;
    auto it = slot.find(indices[i]);
    if (it == slot.end()) {
      slot.emplace(indices[i], from.size());
      from.push_back(i);
      to.push_back(indices[i]);
    } else {
      from[it->second] = i;   // a later point overwrites the same field entry
    }
  }
  int prev = 0;
  int rc = check_hip(hipGetDevice(&prev), ctx);
  if (!rc) rc = check_hip(hipSetDevice(device), ctx);
  if (rc) return rc;
  nebo_point_map* m = new nebo_point_map();
  m->device = device;
  m->n = n;
  m->max_index = mx;
  m->m = (int64_t)from.size();
  m->gather = m->scatter_src = m->scatter_dst = nullptr;
  const size_t b1 = sizeof(int64_t) * (size_t)n, b2 = sizeof(int64_t) * from.size();
  if (n > 0) {
    rc = device_alloc((void**)&m->gather, b1 + 2 * b2, ctx);
    if (!rc) {
      m->scatter_src = m->gather + n;
      m->scatter_dst = m->scatter_src + m->m;
      rc = check_hip(hipMemcpy(m->gather, indices, b1, hipMemcpyHostToDevice), ctx);
    }
    if (!rc) rc = check_hip(hipMemcpy(m->scatter_src, from.data(), b2, hipMemcpyHostToDevice), ctx);
    if (!rc) rc = check_hip(hipMemcpy(m->scatter_dst, to.data(), b2, hipMemcpyHostToDevice), ctx);
  }
  (void)hipSetDevice(prev);
  if (rc) {
    if (m->gather) (void)hipFree(m->gather);
    delete m;
    return rc;
  }
  *out = m;
  return NEBO_OK;
}

extern "C" int nebo_point_map_destroy(nebo_point_map_t* map)
{
  clear_error();
  if (!map) return NEBO_OK;
  int rc = NEBO_OK;
  if (map->gather) {
    int prev = 0;
    rc = check_hip(hipGetDevice(&prev), "Nebo Point Field");
    if (!rc) rc = check_hip(hipSetDevice(map->device), "Nebo Point Field");
    if (!rc) rc = check_hip(hipFree(map->gather), "Nebo Point Field");
    (void)hipSetDevice(prev);
  }
  delete map;
  return rc;
}

extern "C" int nebo_point_to_field(const nebo_point_map_t* map, const nebo_field_t* dest, const double* src,
                                   void* stream)
{
  static const char* ctx = "Nebo Point Field";
  clear_error();
  int rc = check_map_field(map, dest, ctx);
  if (rc) return rc;
  if (map->m == 0) return NEBO_OK;
  if (!src) return set_error(NEBO_ERR_INVALID, ctx, "null argument");
  hipLaunchKernelGGL(scatter_kernel, dim3((unsigned)((map->m + kBlock - 1) / kBlock)), dim3(kBlock), 0,
                     (hipStream_t)stream, static_cast<double*>(dest->values), src, map->scatter_src,
                     map->scatter_dst, (long)map->m);
  return check_hip(hipGetLastError(), ctx);
}

extern "C" int nebo_field_to_point(const nebo_point_map_t* map, double* dest, const nebo_field_t* src,
                                   void* stream)
{
  static const char* ctx = "Nebo Point Field";
  clear_error();
  int rc = check_map_field(map, src, ctx);
  if (rc) return rc;
  if (map->n == 0) return NEBO_OK;
  if (!dest) return set_error(NEBO_ERR_INVALID, ctx, "null argument");
  hipLaunchKernelGGL(gather_kernel, dim3((unsigned)((map->n + kBlock - 1) / kBlock)), dim3(kBlock), 0,
                     (hipStream_t)stream, dest, static_cast<const double*>(src->values), map->gather,
                     (long)map->n);
  return check_hip(hipGetLastError(), ctx);
}
