// FP32-bulk form of the per-timestep parcel path on MI355X (pmpic_config.precision = 1).
//
// Reference path: components/rk4_integrator/src/rk4_integrator.F90:95-319,
// model_core/src/parcels/parcel_interpolation.F90:186-481, model_core/src/parcels/haloswap.F90,
// components/parcel_splitting/src/parcel_splitting.F90:47-168,
// components/parcel_mixing/src/parcel_mixing.F90:68-624.
//
// The algorithm is the plain FP64 form's, step for step (same RK4 stage formulas, split and
// mix rules, slot placement of children and new parcels, same deterministic cell-binned
// par2grid); the representation is what changes:
//  * a position is the index of the cell holding the parcel (int32, c = (k*ny + j)*nx + i) plus
//    three FP32 offsets in [0,1) inside the cell, so it carries 24 bits relative to the cell
//    rather than to the whole domain; vorticity, buoyancy, humidity, volume and stretch are
//    FP32, and interpolation and the par2grid sums run in FP32;
//  * the RK4 origin is the other of two sets of positions and vorticity, and the RK4 accumulator
//    dt/6 k1 + dt/3 k2 + dt/3 k3 + dt/6 k4 is kept in cells relative to it;
//  * the haloswap becomes index arithmetic: leaving through x or y wraps the cell index and the
//    z reflection mirrors (cell, offset) about the boundary, so parcels keep their slots (the
//    plain form reproduces the reference's send-to-self slot permutation instead);
//  * parcel tendencies dxdt..drdt are stored at stage 4 only (the values that survive a step).
// The spectral inversion, the timestep selection and the conservation sums stay FP64: the
// grids are a few percent of the parcel bytes.
#include "node_sum.h"

#include <algorithm>
#include <math.h>
#include <stdlib.h>
#include <string.h>

#include <memory>
#include <new>

// The FP32-bulk form is not held to the reference's operation order (its bar is the velocity
// error against the FP64 form), so multiply-adds may fuse here.
#pragma clang fp contract(fast)

namespace pmpic {

namespace {

constexpr int TPB = 256;

// A parcel's cell is stored packed as k << 20 | j << 10 | i (nx, ny <= 1024, nz < 2048), so
// unpacking is shifts and masks; the linear cell index (k*ny + j)*nx + i is formed only where
// buckets are indexed.
__device__ __forceinline__ int32_t pack_cell(int i, int j, int k) { return (k << 20) | (j << 10) | i; }
__device__ __forceinline__ void cell_ijk(const Geometry &, int32_t c, int &i, int &j, int &k) {
  i = c & 1023;
  j = (c >> 10) & 1023;
  k = c >> 20;
}
__device__ __forceinline__ int32_t linear_cell(const Geometry &g, int32_t c) {
  return ((c >> 20) * g.ny + ((c >> 10) & 1023)) * g.nx + (c & 1023);
}

// Loads and stores at a uniform base plus a 32-bit byte offset (the global_load/store form
// with a scalar base), valid while index * sizeof(T) < 2^32: capacities are checked at set-up.
template <typename T>
__device__ __forceinline__ T ld(const T *base, uint32_t i) {
  return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(base) +
                                      i * (uint32_t)sizeof(T));
}
template <typename T>
__device__ __forceinline__ void st(T *base, uint32_t i, T v) {
  *reinterpret_cast<T *>(reinterpret_cast<char *>(base) + i * (uint32_t)sizeof(T)) = v;
}
// streaming forms for parcel fields that one kernel reads or writes once: they bypass the
// caches' retention so the grids being gathered stay resident
template <typename T>
__device__ __forceinline__ T ldnt(const T *base, uint32_t i) {
  return __builtin_nontemporal_load(reinterpret_cast<const T *>(
      reinterpret_cast<const char *>(base) + i * (uint32_t)sizeof(T)));
}
template <typename T>
__device__ __forceinline__ void stnt(T *base, uint32_t i, T v) {
  __builtin_nontemporal_store(v, reinterpret_cast<T *>(reinterpret_cast<char *>(base) +
                                                       i * (uint32_t)sizeof(T)));
}

struct Float3 {
  float x, y, z;
};
__device__ __forceinline__ Float3 ld3(const float *base, int64_t i) {
  const float *a = base + 3 * i;
  return {__builtin_nontemporal_load(a), __builtin_nontemporal_load(a + 1),
          __builtin_nontemporal_load(a + 2)};
}
__device__ __forceinline__ void st3(float *base, int64_t i, float x, float y, float z) {
  float *a = base + 3 * i;
  __builtin_nontemporal_store(x, a);
  __builtin_nontemporal_store(y, a + 1);
  __builtin_nontemporal_store(z, a + 2);
}

// fold an offset outside [0,1) into the cell index
__device__ __forceinline__ void fold1(int &i, float &o) {
  const float f = floorf(o);
  i += (int)f;
  o = o - f;
  if (o >= 1.0f) {  // o was a tiny negative number
    o -= 1.0f;
    i += 1;
  }
}

// cell (i, j, k) + offsets (tx, ty, tz) in cells, offsets anywhere -> cell index and offsets in
// [0,1): periodic in x and y, z mirrored about 0 and nz (haloswap.F90:447-454 on the cell
// scale; a position exactly on the top boundary stays in the top cell with offset 1).  Returns
// false if the position is still outside in z.
__device__ __forceinline__ bool place(const Geometry &g, int i, int j, int k, float tx, float ty,
                                      float tz, int32_t &cell, float &ox, float &oy, float &oz) {
  fold1(i, tx);
  fold1(j, ty);
  fold1(k, tz);
  // a stage moves a parcel by far less than a period, so one correction is the common case
  if (i < 0 || i >= g.nx) {
    i %= g.nx;
    if (i < 0) i += g.nx;
  }
  if (j < 0 || j >= g.ny) {
    j %= g.ny;
    if (j < 0) j += g.ny;
  }
  const int nz = g.ncz;
  if (k < 0) {  // z' = -z
    if (tz == 0.0f) {
      k = -k;
    } else {
      k = -k - 1;
      tz = 1.0f - tz;
      if (tz >= 1.0f) { tz -= 1.0f; k += 1; }
    }
  } else if (k >= nz && !(k == nz && tz == 0.0f)) {  // z' = 2 nz - z
    if (tz == 0.0f) {
      k = 2 * nz - k;
    } else {
      k = 2 * nz - k - 1;
      tz = 1.0f - tz;
      if (tz >= 1.0f) { tz -= 1.0f; k += 1; }
    }
  }
  if (k == nz && tz == 0.0f) {
    k = nz - 1;
    tz = 1.0f;
  }
  if (k < 0 || k >= nz) return false;
  cell = pack_cell(i, j, k);
  ox = tx;
  oy = ty;
  oz = tz;
  return true;
}

// node offsets of the 8 corners of cell (i, j, k), corner bits z<<2 | y<<1 | x
__device__ __forceinline__ void corner_nodes(const Geometry &g, int i, int j, int k, int32_t o[8]) {
  const int i1 = (i + 1 == g.nx) ? 0 : i + 1;
  const int j1 = (j + 1 == g.ny) ? 0 : j + 1;
  const int32_t b00 = (k * g.ny + j) * g.nx, b01 = (k * g.ny + j1) * g.nx;
  const int32_t b10 = ((k + 1) * g.ny + j) * g.nx, b11 = ((k + 1) * g.ny + j1) * g.nx;
  o[0] = b00 + i; o[1] = b00 + i1; o[2] = b01 + i; o[3] = b01 + i1;
  o[4] = b10 + i; o[5] = b10 + i1; o[6] = b11 + i; o[7] = b11 + i1;
}

// trilinear interpolation of the eight corner values in the reference's order
// (parcel_interpolation.F90:309-321)
__device__ __forceinline__ float interp(const float c[8], float ox, float oy, float oz) {
  const float c00 = c[0] * (1 - oz) + c[4] * oz;
  const float c01 = c[1] * (1 - oz) + c[5] * oz;
  const float c10 = c[2] * (1 - oz) + c[6] * oz;
  const float c11 = c[3] * (1 - oz) + c[7] * oz;
  const float c0 = c00 * (1 - oy) + c10 * oy;
  const float c1 = c01 * (1 - oy) + c11 * oy;
  return c0 * (1 - ox) + c1 * ox;
}

// ---- host <-> device conversion of the parcel state ----
// axis a of the position: (x - bottom)/d -> cell index part and offset
__global__ void k32_pos_in(Geometry g, int axis, const double *__restrict__ x, int64_t n,
                           int32_t *__restrict__ cell, float *__restrict__ off, DevScalars *sc) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  const double bot = axis == 0 ? g.xbot : (axis == 1 ? g.ybot : g.zbot);
  const double d = axis == 0 ? g.dx : (axis == 1 ? g.dy : g.dz);
  const int ncells = axis == 0 ? g.nx : (axis == 1 ? g.ny : g.ncz);
  const double u = (x[p] - bot) / d;
  const double fu = floor(u);
  int i = (int)fu;
  float o = (float)(u - fu);
  if (o >= 1.0f) { o = 0.0f; i += 1; }
  if (axis < 2) {
    i %= ncells;
    if (i < 0) i += ncells;
  } else {
    if (i == ncells && o == 0.0f) { i = ncells - 1; o = 1.0f; }
    if (i < 0 || i >= ncells) {
      raise_status(sc, PMPIC_ERR_OUT_OF_BOX_Z);
      i = 0;
    }
  }
  off[3 * p + axis] = o;
  cell[p] = (axis == 0 ? 0 : cell[p]) | (i << (10 * axis));
}

__global__ void k32_pos_out(Geometry g, int axis, const int32_t *__restrict__ cell,
                            const float *__restrict__ off, int64_t n, double *__restrict__ x) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  int i, j, k;
  cell_ijk(g, cell[p], i, j, k);
  const int idx = axis == 0 ? i : (axis == 1 ? j : k);
  const double bot = axis == 0 ? g.xbot : (axis == 1 ? g.ybot : g.zbot);
  const double d = axis == 0 ? g.dx : (axis == 1 ? g.dy : g.dz);
  x[p] = bot + ((double)idx + (double)off[3 * p + axis]) * d;
}

__global__ void k32_from_f64(const double *__restrict__ a, int64_t n, float *__restrict__ b,
                             int stride) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p < n) b[p * stride] = (float)a[p];
}

__global__ void k32_to_f64(const float *__restrict__ a, int stride, int64_t n,
                           double *__restrict__ b) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p < n) b[p] = (double)a[p * stride];
}

// ---- tiles of eight cells of an x row ----
__host__ __device__ inline int tiles_x(const Geometry &g) { return (g.nx + 7) / 8; }
// tile of cell (i, j, k)
__device__ __forceinline__ int64_t tile_of(const Geometry &g, int i, int j, int k) {
  return ((int64_t)k * g.ny + j) * tiles_x(g) + (i >> 3);
}

// ---- cell binning ----
// A wavefront walks BIN_SEQ consecutive groups of 64 parcels in order and takes one atomic per
// run of equal cells, so a cell whose parcels are consecutive in slot order gets its ranks in
// ascending parcel order unless it straddles two wavefronts' ranges; the accumulation only has
// to reorder those cells.  A parcel of rank < capc is listed at slot[cell * capc + rank], so a
// typical cell needs no scatter pass.  A parcel of higher rank is appended, with
// its rank, to an overflow list; every cell holding more than capc parcels is then laid out
// densely, all its parcels in rank order, in `sorted` from ostart[cell] (room by
// bin_alloc).  capc = 0 lays out every cell that way.  capc is chosen per binning:
// CAPC_LOW while the mean is at most LOW_PPC parcels per cell, so a sparse grid does not read
// mostly empty entries, else CAPC.
constexpr int BIN_SEQ = 16;
constexpr int CAPC = 32;      // slot entries per cell of the table, and the full capacity
constexpr int CAPC_LOW = 16;
constexpr int LOW_PPC = 10;
constexpr int MIX_MOVES = 16;  // mixing's changes that the lists follow: up to 1 in so many parcels

__global__ void k32_bin_reset(int32_t *__restrict__ count, int64_t nc1, DevScalars *dsc) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < nc1) count[i] = 0;
  if (i == 0) dsc->novf = 0;
}

// capc = 0 (no slot table): every parcel's rank within its cell goes to rankv instead, and
// k32_dense_scatter lays all cells out densely after the scan
__global__ void k32_bin_slot(Geometry g, const int32_t *__restrict__ cellv, int64_t n, int capc,
                             int32_t *__restrict__ slot, int2 *__restrict__ ovf,
                             int32_t *__restrict__ ovfc, int32_t *__restrict__ where,
                             int32_t *__restrict__ rankv, int32_t *__restrict__ count,
                             DevScalars *dsc) {
  // parcel indices fit 32 bits (capacity < 2^30)
  const int lane = threadIdx.x & 63;
  const int32_t w0 = (int32_t)((blockIdx.x * blockDim.x + threadIdx.x) >> 6) * 64 * BIN_SEQ;
  // the parcel count from device memory: a graph replays this launch, sized for a bound on
  // the count, whatever the count is then (n is the launch's size only)
  (void)n;
  const int32_t n32 = (int32_t)dsc->n;
  if (n32 == 0 || w0 >= n32) return;
  // all count atomics of the wavefront are issued before any result is used, in group order;
  // run[it]: the cell and the head lane of the parcel's run (the cell is only used while the slot
  // table exists, whose grids have at most 2^26 cells)
  int base[BIN_SEQ];
  uint32_t run[BIN_SEQ];
  int32_t cv[BIN_SEQ];  // every load issued before the first is used (clamped index, n >= 1)
#pragma unroll
  for (int it = 0; it < BIN_SEQ; it++)
    cv[it] = ld(cellv, (uint32_t)min(w0 + it * 64 + lane, n32 - 1));
#pragma unroll
  for (int it = 0; it < BIN_SEQ; it++) {
    const int32_t p = w0 + it * 64 + lane;
    const int32_t c = (p < n32) ? linear_cell(g, cv[it]) : -1;
    const int32_t cprev = __shfl_up(c, 1);
    const bool head = (lane == 0) || (c != cprev);
    const unsigned long long hm = __ballot(head);
    const unsigned long long upto = hm & ((2ull << lane) - 1ull);
    const int hl = 63 - __clzll(upto);
    const unsigned long long above = hm & ~((2ull << hl) - 1ull);
    const int next = above ? (__ffsll(above) - 1) : 64;
    base[it] = (head && c >= 0) ? atomicAdd(&count[c], next - hl) : 0;
    run[it] = pack_run(c, hl);
  }
  if (capc == 0) {
#pragma unroll
    for (int it = 0; it < BIN_SEQ; it++) {
      const int32_t p = w0 + it * 64 + lane;
      const int hl = run_head(run[it]);
      const int32_t rk = __shfl(base[it], hl) + (lane - hl);
      if (p < n32) st(rankv, (uint32_t)p, rk);
    }
    return;
  }
  bool anyover = false;
#pragma unroll
  for (int it = 0; it < BIN_SEQ; it++) {
    const int32_t p = w0 + it * 64 + lane;
    const int hl = run_head(run[it]);
    const int32_t rk = __shfl(base[it], hl) + (lane - hl);
    if (p < n32) {
      if (rk < capc) st(slot, (uint32_t)(run_cell(run[it]) * capc + rk), p);
      else anyover = true;
    }
  }
  if (__ballot(anyover) == 0ull) return;
#pragma unroll
  for (int it = 0; it < BIN_SEQ; it++) {
    const int32_t p = w0 + it * 64 + lane;
    const int hl = run_head(run[it]);
    const int32_t rk = __shfl(base[it], hl) + (lane - hl);
    const bool over = (p < n32) && rk >= capc;
    const unsigned long long om = __ballot(over);
    if (om) {
      const int lead = __ffsll(om) - 1;
      int32_t ob = 0;
      if (lane == lead) ob = atomicAdd(&dsc->novf, (int32_t)__popcll(om));
      ob = __shfl(ob, lead);
      if (over) {
        const int32_t o = ob + __popcll(om & ((1ull << lane) - 1ull));
        ovf[o] = make_int2(p, rk);
        ovfc[o] = run_cell(run[it]);
        if (where) where[p] = o;
      }
    }
  }
}

// the overflow list into the dense region; the parcel of rank capc also copies its cell's
// capc slot entries there, so the region holds ranks 0 .. count-1.  Entries that have left
// are holes (-1).
__global__ void k32_ovf_scatter(const int2 *__restrict__ ovf, const int32_t *__restrict__ ovfc,
                                const DevScalars *dsc, const int32_t *__restrict__ ostart,
                                const int32_t *__restrict__ slot, int capc,
                                int32_t *__restrict__ sorted) {
  const int32_t no = dsc->novf;
  const int32_t stride = gridDim.x * blockDim.x;
  for (int32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < no; i += stride) {
    const int2 e = ovf[i];
    const int32_t c = ovfc[i];
    const int32_t b0 = ostart[c];
    sorted[b0 + e.y] = e.x;
    if (e.y == capc)
      for (int r = 0; r < capc; r++) sorted[b0 + r] = slot[c * capc + r];
  }
}

// the lists a binning fills
struct BinOut {
  int on;                // in an RK stage: 0 none, 1 all parcels, 2 the ones that change cell
  int capc;              // slot capacity of the binning, 0 for the dense ranks
  int32_t *count;        // per cell
  int32_t *slot;         // [cell * capc + rank]
  int2 *ovf;             // (parcel, rank) past the capacity; their number in DevScalars::novf
  int32_t *ovfc;         // ... their cells
  int32_t *where;        // ... a parcel's entry there (may be null)
  int32_t *rank;         // per parcel, when capc = 0
};

// Parcel p's entry in cell c's list becomes a hole (-1), which the accumulation leaves out.  rows:
// the slot entries to search.  Where appends run meanwhile that is all of them, and p has an entry:
// the first match is it, since entries past the count the list had before may hold anything, but
// there are none below the capacity where p's entry is not in the table.
__device__ __forceinline__ void remove_entry(int32_t p, int32_t c, int rows, const BinOut &bo,
                                             const DevScalars *sc) {
  int32_t *row = bo.slot + (int64_t)c * bo.capc;
  for (int r = 0; r < rows; r += 4) {
    const int4 e = *reinterpret_cast<const int4 *>(row + r);
    const int at = e.x == p ? 0 : e.y == p ? 1 : e.z == p ? 2 : e.w == p ? 3 : -1;
    if (at >= 0 && r + at < rows) {
      row[r + at] = -1;
      return;
    }
  }
  const int32_t o = bo.where[p];
  if ((uint32_t)o < (uint32_t)sc->novf && bo.ovf[o].x == p) bo.ovf[o].x = -1;
}
__device__ __forceinline__ void append_entry(int32_t p, int32_t c, const BinOut &bo,
                                             DevScalars *sc) {
  const int32_t rk = atomicAdd(&bo.count[c], 1);
  if (rk < bo.capc) {
    bo.slot[(int64_t)c * bo.capc + rk] = p;
  } else {
    const int32_t o = atomicAdd(&sc->novf, 1);
    bo.ovf[o] = make_int2(p, rk);
    bo.ovfc[o] = c;
    bo.where[p] = o;
  }
}

// the lists of n_old parcels in cells `was` brought to the n parcels in cells `is` (parcels past
// n_old are new): 8 bytes a parcel read, where building the lists again is bound by its scattered
// 4-byte writes and atomics (67 M parcels 0.75 -> 0.10 ms, 1.8 M well mixed ones 40 -> 5 us)
__global__ void k32_bin_move(Geometry g, const int32_t *__restrict__ was,
                             const int32_t *__restrict__ is, int64_t n_old, int64_t n, BinOut bo,
                             DevScalars *sc) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  const int32_t from = p < n_old ? was[p] : -1, to = is[p];
  if (from == to) return;
  if (p < n_old) remove_entry((int32_t)p, linear_cell(g, from), bo.capc, bo, sc);
  append_entry((int32_t)p, linear_cell(g, to), bo, sc);
}

// Parcels that leave the lists (bo.on) and the sums (dirty, may be null: their tiles): the n listed
// ones, or without a list those from `base` on.  Nothing is appended meanwhile, so a cell's list
// ends at its count, and a parcel without an entry finds none.
__global__ void k32_unlist(Geometry g, const int32_t *__restrict__ cellv,
                           const int32_t *__restrict__ list, int64_t base, int64_t n, BinOut bo,
                           uint8_t *__restrict__ dirty, DevScalars *sc) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const int32_t p = list ? list[t] : (int32_t)(base + t), cell = cellv[p];
  if (dirty) {
    int i, j, k;
    cell_ijk(g, cell, i, j, k);
    dirty[tile_of(g, i, j, k)] = 1;
    if (t == 0) sc->anydirty = 1;
  }
  if (bo.on) {
    const int32_t c = linear_cell(g, cell);
    remove_entry(p, c, min(bo.count[c], bo.capc), bo, sc);
  }
}

// without a slot table: parcel p at its cell's dense offset plus its rank
__global__ void k32_dense_scatter(Geometry g, const int32_t *__restrict__ cellv,
                                  const int32_t *__restrict__ rankv, const DevScalars *dsc,
                                  const int32_t *__restrict__ start, int32_t *__restrict__ sorted) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= dsc->n) return;
  const int32_t c = linear_cell(g, ld(cellv, (uint32_t)p));
  st(sorted, (uint32_t)(start[c] + ld(rankv, (uint32_t)p)), (int32_t)p);
}

// ---- corner sums ----
// One wavefront per tile of eight cells of one x row; lane = 8 q + cl is corner q (bits z<<2 |
// y<<1 | x) of cell cl, and the cell's parcels are taken eight at a time: lane (q, cl) stages
// parcel q of the eight in LDS row 8 q + cl, then every lane adds its corner's weight and weight *
// value over the cell's rows.  The next eight parcels' loads are in flight meanwhile, and no
// barrier ties wavefronts together, so the CU's 32 overlap each other's loads and sums.  It is
// bound by the latency of the gathers: three 12-byte records a parcel, and
// half by the issue of the sums.  67 M parcels that have moved a few cells: 1.39 ms with nine 4-byte
// gathers and a workgroup staging all parcels of 16 cells, 1.12 ms (2.6 TB/s); 1.8 M well mixed
// ones in 221 k cells: 87 -> 58 us.
//
// Within a cell the additions run in ascending parcel order, so the sums do not depend on the
// order in which the binning's atomics came: the lanes check their adjacent entries and rank them
// where a pair is not ascending (in LDS up to LIST entries a cell, else in memory).  Holes (-1:
// remove_entry) are left out there too.
//
// A cell of up to capc parcels lists them in the slot table, whose first 16 entries are loaded
// before the count is known; the others in the dense region.
//
// The corner sums are combined along x as they are written: node position i of corner pair
// bb = (by, bz) adds the bx = 1 corner of cell i - 1 and the bx = 0 corner of cell i.  Value f of
// entry (bb, row, position) sits at ((f 4 + bb) nrows + row) (nx + ntx) + 9 tx + position - 8 tx,
// ntx tiles a row; a tile's last position holds its last cell's bx = 1 corner alone, completed by
// the node sums.
//
// A32_P2G: weight, p, q, r, total buoyancy (vort2vel + vorticity_tendency).  A32_MIX: those and
// b, h, of the kept parcels and (partial2) the residual ones (parcel_mixing), so that its first
// five planes are the ones the next par2grid would write; the tiles without residual parcels
// (almost all) are marked so in tileres and write none.  A32_DUMP: weight, b, h, p, q, r
// (writebinary's grids).
enum Acc32 { A32_P2G = 0, A32_MIX = 1, A32_DUMP = 2 };
constexpr int LIST = 64;

struct Zmap {
  float zbot, dz;  // z of a parcel = zbot + (k + oz) dz
};

// A parcel's weight at corner (bx, by, bz) of its cell: the factor of an axis is |t - offset|,
// t = 1 for the lower corner (1 - offset) and 0 for the upper (the offset, which lies in [0, 1]);
// the weight is ((fz fy) vol) fx.  No contraction here or in add_parcel: the compiler would
// otherwise fuse the weight's last product into the first sum in some of the kernels that inline
// these and not in others, and a tile that mixing left unchanged must have the par2grid's bits.
__device__ __forceinline__ float corner_weight(float ox, float oy, float oz, float vol, float tx,
                                               float ty, float tz) {
#pragma clang fp contract(off)
  const float fy = fabsf(ty - oy);
  const float fz = fabsf(tz - oz);
  const float wv = (fz * fy) * vol;
  return wv * fabsf(tx - ox);
}

// acc[0] += w, acc[1 + f] += w * v[f], fused
template <int NV>
__device__ __forceinline__ void add_parcel(float *acc, float w, const float *v) {
#pragma clang fp contract(off)
  acc[0] += w;
#pragma unroll
  for (int f = 0; f < NV; f++) acc[f + 1] = fmaf(w, v[f], acc[f + 1]);
}

// The lanes' W entries 8 i + q of eight lists of up to nmax entries (key e of list cl at
// keys(e)): their ranks among the list's entries
template <int W, typename K>
__device__ __forceinline__ void rank_entries(const int32_t *v, int *r, int nmax, K keys) {
#pragma unroll
  for (int i = 0; i < W; i++) r[i] = 0;
  for (int e = 0; e < nmax; e++) {
    const int32_t key = keys(e);
#pragma unroll
    for (int i = 0; i < W; i++) r[i] += key < v[i] ? 1 : 0;
  }
}

// the list's entries among all its lanes' W (lanes cl, cl + 8, ...)
template <int W>
__device__ __forceinline__ int entries(const int32_t *v) {
  int k = 0;
#pragma unroll
  for (int i = 0; i < W; i++) k += v[i] != INT32_MAX ? 1 : 0;
#pragma unroll
  for (int d = 8; d < 64; d <<= 1) k += __shfl_xor(k, d);
  return k;
}

template <int MODE>
__global__ void __launch_bounds__(64) k32_cell_accum(
    Geometry g, Parcels32 P, Zmap zm, float vmin, int capc, const int32_t *__restrict__ slot,
    int32_t *__restrict__ count, const int32_t *__restrict__ start,
    const int32_t *__restrict__ sorted, int32_t *__restrict__ order, float *__restrict__ partial,
    float *__restrict__ partial2, int32_t *__restrict__ npercell, uint8_t *__restrict__ tileres,
    uint8_t *__restrict__ dirty, int32_t *__restrict__ cursor, DevScalars *sc, int zero) {
  constexpr bool MIX = MODE == A32_MIX;
  constexpr int NV = MODE == A32_P2G ? 4 : MODE == A32_MIX ? 6 : 5;
  constexpr int NF = NV + 1;
  __shared__ float4 sgeo[64];               // offsets, vol
  __shared__ float4 sval[64];               // the first four values
  __shared__ float2 sval2[NV > 4 ? 64 : 1];  // the others
  __shared__ int32_t slist[LIST * 8];       // entry e of cell cl at 8 e + cl
  const int lane = threadIdx.x, cl = lane & 7, q = lane >> 3;
  const int bx = q & 1, by = (q >> 1) & 1, bz = q >> 2;
  const float tx = bx ? 0.f : 1.f, ty = by ? 0.f : 1.f, tz = bz ? 0.f : 1.f;
  const uint32_t ntx = (uint32_t)tiles_x(g);
  const uint32_t tile = xcd_block(blockIdx.x, gridDim.x);
  const uint32_t xrow = tile / ntx, tile_x = tile - xrow * ntx;
  const int m = min(8, g.nx - 8 * (int)tile_x);  // cells here
  const bool live = cl < m;
  const int64_t c = (int64_t)xrow * g.nx + 8 * tile_x + (live ? cl : 0);
  const int32_t *own = slot + c * capc;
  int32_t pre[2] = {0, 0};
  if (capc) {
    pre[0] = own[q];
    pre[1] = own[8 + q];
  }
  int n = live ? count[c] : 0;
  if (zero) {
    if (live && q == 0) count[c] = 0;
    if (tile == 0 && lane == 0) sc->novf = 0;
  }
  if (tile == 0 && lane == 0) *cursor = 0;
  if constexpr (MODE == A32_P2G) {
    // a par2grid whose sums the last mixing left current: only the tiles it changed
    if (dirty && !dirty[tile]) return;
  }
  int nmax = n;
#pragma unroll
  for (int d = 1; d < 8; d <<= 1) nmax = max(nmax, __shfl_xor(nmax, d));
  nmax = __builtin_amdgcn_readfirstlane(nmax);
  const int nch = (nmax + 7) >> 3;  // chunks of eight parcels a cell
  const bool small = nmax <= LIST;
  const bool dense = n > capc;
  const int64_t b = dense ? start[c] : 0;
  const int32_t *list = dense ? sorted + b : own;
  // entries 8 i + q of the cell, ordered by parcel
  bool hole = false;
  if (small) {
    bool bad = false;
#pragma unroll
    for (int i = 0; i < LIST / 8; i++) {
      if (i >= nch) break;
      const int e = 8 * i + q;
      const int32_t v = e >= n ? INT32_MAX : i < 2 && !dense ? pre[i < 2 ? i : 0] : list[e];
      hole |= v < 0;
      slist[64 * i + lane] = v < 0 ? INT32_MAX : v;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < LIST / 8; i++) {
      if (i >= nch) break;
      if (8 * i + q + 1 < n) bad |= slist[64 * i + lane] > slist[64 * i + lane + 8];
    }
    if (__any(bad || hole)) {
      auto sort = [&](auto w) {
        constexpr int W = decltype(w)::value;
        int32_t v[W];
        int r[W];
#pragma unroll
        for (int i = 0; i < W; i++) v[i] = i < nch ? slist[64 * i + lane] : INT32_MAX;
        rank_entries<W>(v, r, nmax, [&](int e) { return slist[8 * e + cl]; });
        __syncthreads();
#pragma unroll
        for (int i = 0; i < W; i++)
          if (v[i] != INT32_MAX) slist[8 * r[i] + cl] = v[i];
        n = entries<W>(v);
      };
      if (nch <= 2) sort(std::integral_constant<int, 2>());
      else sort(std::integral_constant<int, LIST / 8>());
      __syncthreads();
    }
  } else {
    bool bad = false;
    for (int i = 0; i < nch; i++) {
      const int e = 8 * i + q;
      if (e < n) hole |= list[e] < 0;
      if (e + 1 < n) bad |= list[e] > list[e + 1];
    }
    if (__any(bad || hole)) {
      // a cell still in the slot table is ordered into LDS
      int32_t *out = dense ? order + b : nullptr;
      int valid = 0;
      auto key = [&](int e) {
        const int32_t k = e < n ? list[e] : INT32_MAX;
        return k < 0 ? INT32_MAX : k;
      };
      for (int i0 = 0; i0 < nch; i0 += 8) {
        int32_t v[8];
        int r[8];
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] = key(8 * (i0 + i) + q);
        rank_entries<8>(v, r, nmax, key);
        valid += entries<8>(v);
#pragma unroll
        for (int i = 0; i < 8; i++)
          if (v[i] != INT32_MAX) {
            if (out) out[r[i]] = v[i];
            else slist[8 * r[i] + cl] = v[i];  // at most capc <= LIST entries
          }
      }
      __threadfence_block();
      __syncthreads();
      if (out) list = out;
      n = valid;
    } else {
      for (int i = 0; i < LIST / 8; i++)
        if (!dense && 8 * i + q < n) slist[64 * i + lane] = list[8 * i + q];
      __syncthreads();
    }
  }
  const bool in_lds = small || !dense;
  const float kz = (float)(xrow / (uint32_t)g.ny);
  Float3 off{}, vor{}, vbh{};
  auto fetch = [&](int ch) {
    const int e = 8 * ch + q;
    if (e < n) {
      const int64_t p = in_lds ? slist[64 * ch + lane] : list[e];
      off = ld3(P.off, p);
      vor = ld3(P.vor, p);
      vbh = ld3(P.vbh, p);
    }
  };
  float acc[NF], res[MIX ? NF : 1];
#pragma unroll
  for (int f = 0; f < NF; f++) acc[f] = 0.f;
#pragma unroll
  for (int f = 0; f < (MIX ? NF : 1); f++) res[f] = 0.f;
  int kept = 0;
  bool anyres = false;
  if (nch > 0) fetch(0);
  for (int ch = 0; ch < nch; ch++) {
    if (8 * ch + q < n) {
      sgeo[lane] = make_float4(off.x, off.y, off.z, vbh.x);
      if constexpr (MODE == A32_DUMP) {
        sval[lane] = make_float4(vbh.y, vbh.z, vor.x, vor.y);
        sval2[lane] = make_float2(vor.z, 0.f);
      } else {
        // total buoyancy (vorticity_tendency.F90:121-126)
        const float z = fmaf(kz + off.z, zm.dz, zm.zbot);
        const float hl = vbh.z - expf(-z);
        sval[lane] = make_float4(vor.x, vor.y, vor.z, fmaf(12.5f, hl > 0.f ? hl : 0.f, vbh.y));
        if constexpr (MIX) sval2[lane] = make_float2(vbh.y, vbh.z);
      }
    } else if constexpr (!MIX) {
      sgeo[lane] = sval[lane] = make_float4(0.f, 0.f, 0.f, 0.f);
      if constexpr (NV > 4) sval2[lane] = make_float2(0.f, 0.f);
    }
    __syncthreads();
    if (ch + 1 < nch) fetch(ch + 1);
    const int rows = min(8, nmax - 8 * ch), mine = n - 8 * ch;
    // (without a test for each row: those past a cell's parcels hold zeros.  256x256x128: 20.11 ->
    // 19.93 ms a step; mixing can't, its zero volume would count as a parcel to remove)
#pragma unroll MIX ? 2 : 4
    for (int a = 0; a < (MIX ? rows : (rows + 3) / 4 * 4); a++) {
      const int r = 8 * a + cl;
      const float4 ge = sgeo[r], v4 = sval[r];
      float v[6] = {v4.x, v4.y, v4.z, v4.w, 0.f, 0.f};
      if constexpr (NV > 4) {
        v[4] = sval2[r].x;
        v[5] = sval2[r].y;
      }
      const float w = corner_weight(ge.x, ge.y, ge.z, ge.w, tx, ty, tz);
      if constexpr (!MIX) {
        add_parcel<NV>(acc, w, v);
      } else if (a < mine) {
        if (!(ge.w < vmin)) {
          add_parcel<NV>(acc, w, v);
          kept++;
        } else {
          anyres = true;
          add_parcel<NV>(res, w, v);
        }
      }
    }
    __syncthreads();
  }
  const int64_t nrows = (int64_t)g.ny * g.ncz, W = g.nx + (int64_t)ntx;
  auto write_x = [&](const float *v, float *out) {
    const int64_t o = ((int64_t)(q >> 1) * nrows + xrow) * W + 9 * tile_x + (bx ? 8 : cl);
    const bool mine = bx ? (cl == 7 && m == 8) : cl <= m;
#pragma unroll
    for (int f = 0; f < NF; f++) {
      const float left = __shfl(v[f], (lane + 7) & 63);  // corner q | 1 of cell cl - 1
      if (mine) out[f * 4 * nrows * W + o] = bx || cl == 0 ? v[f] : left + v[f];
    }
  };
  write_x(acc, partial);
  if constexpr (MIX) {
    const bool any = __any(anyres) != 0;
    if (lane == 0) {
      tileres[tile] = any ? 1 : 0;
      dirty[tile] = 0;
    }
    if (tile == 0 && lane == 0) sc->anydirty = 0;
    if (any) write_x(res, partial2);
    if (live && q == 0) npercell[c] = kept;
  }
}

__global__ void k32_grid_to_f64(const float *__restrict__ a, double *__restrict__ b, int64_t n) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) b[t] = (double)a[t];
}

// ---- RK4 stage: gather the six tendencies, update, place (wrap x, y; reflect z) ----
struct Scale32 {
  float idx, idy, idz;  // cells per unit length
};

// k32_bin_slot's binning of one parcel per lane (c: its cell as stored, or -1 for none): the
// lanes of a run of equal cells share one count atomic, issued by the run's first lane
__device__ __forceinline__ void bin_lane(const Geometry &g, int32_t cell, uint32_t p,
                                         const BinOut &bo, DevScalars *dsc) {
  const int lane = threadIdx.x & 63;
  const int32_t c = cell >= 0 ? linear_cell(g, cell) : -1;
  const int32_t cprev = __shfl_up(c, 1);
  const bool head = (lane == 0) || (c != cprev);
  const unsigned long long hm = __ballot(head);
  const unsigned long long upto = hm & ((2ull << lane) - 1ull);
  const int hl = 63 - __clzll(upto);
  const unsigned long long above = hm & ~((2ull << hl) - 1ull);
  const int next = above ? (__ffsll(above) - 1) : 64;
  const int base = (head && c >= 0) ? atomicAdd(&bo.count[c], next - hl) : 0;
  const int32_t rk = __shfl(base, hl) + (lane - hl);
  if (bo.capc == 0) {
    if (c >= 0) st(bo.rank, p, rk);
    return;
  }
  const bool over = c >= 0 && rk >= bo.capc;
  if (c >= 0 && !over) st(bo.slot, (uint32_t)(c * bo.capc + rk), (int32_t)p);
  const unsigned long long om = __ballot(over);
  if (om) {
    const int lead = __ffsll(om) - 1;
    int32_t ob = 0;
    if (lane == lead) ob = atomicAdd(&dsc->novf, (int32_t)__popcll(om));
    ob = __shfl(ob, lead);
    if (over) {
      const int32_t o = ob + __popcll(om & ((1ull << lane) - 1ull));
      bo.ovf[o] = make_int2((int32_t)p, rk);
      bo.ovfc[o] = c;
      if (bo.where) bo.where[p] = o;
    }
  }
}

// the sets a stage reads, takes as the RK4 origin and writes
struct RkSets {
  const int32_t *cell, *cello;
  const float *off, *offo, *vor, *voro;
  int32_t *cell_to;
  float *off_to, *vor_to;
};

// The RK stage of parcel p; returns its new cell, or -1 where it would leave the box (status raised).
// It then stays where it is, in the set that the stage writes too, but is not in the lists that the
// stage builds: b32_forget drops those.  The sets of a stage may be the same arrays: a thread reads its
// parcel before it writes it.
template <int STAGE>
__device__ __forceinline__ int32_t rk_update(const Geometry &g, const Bulk32 &b, const RkSets &rs,
                                             const float4 *__restrict__ rec,
                                             const Scale32 &sc3,
                                             int stretch, uint8_t *__restrict__ split_flag,
                                             DevScalars *sc, uint32_t p) {
  const int32_t cell = ldnt(rs.cell, p);
  const Float3 off = ld3(rs.off, p);
  const float ox = off.x, oy = off.y, oz = off.z;
  int32_t cello = cell;
  float oo[3] = {ox, oy, oz}, df[3] = {0.f, 0.f, 0.f}, vo[3] = {0.f, 0.f, 0.f},
        vf[3] = {0.f, 0.f, 0.f};
  auto take = [](float *a, const Float3 &v) {
    a[0] = v.x;
    a[1] = v.y;
    a[2] = v.z;
  };
  if (STAGE == 1) {
    take(vo, ld3(rs.vor, p));
  } else {
    cello = ldnt(rs.cello, p);
    take(oo, ld3(rs.offo, p));
    take(df, ld3(b.df, p));
    if (STAGE != 4) take(vo, ld3(rs.voro, p));
    take(vf, ld3(b.pf, p));
  }
  const float s_old = (STAGE == 4 && stretch) ? ldnt(b.stretch, p) : 0.f;
  int i, j, k;
  cell_ijk(g, cell, i, j, k);
  int32_t o[8];
  corner_nodes(g, i, j, k, o);
  float kv[6], cv[6][8];
#pragma unroll
  for (int q = 0; q < 8; q++) {  // 32-byte records: a 64-bit index, nodes times 32 may pass 2^32
    const float4 r0 = rec[2 * (int64_t)o[q]];
    const float2 r1 = *reinterpret_cast<const float2 *>(rec + 2 * (int64_t)o[q] + 1);
    cv[0][q] = r0.x; cv[1][q] = r0.y; cv[2][q] = r0.z;
    cv[3][q] = r0.w; cv[4][q] = r1.x; cv[5][q] = r1.y;
  }
#pragma unroll
  for (int f = 0; f < 6; f++) kv[f] = interp(cv[f], ox, oy, oz);
  const double dtd = sc->dtm;
  const float dt = (float)dtd, dt6 = (float)(dtd / 6), dt2 = (float)(dtd / 2),
              dt3 = (float)(dtd / 3);
  const float kp[3] = {kv[0] * sc3.idx, kv[1] * sc3.idy, kv[2] * sc3.idz};
  float tpos[3], dfn[3], vn[3], vfn[3];
#pragma unroll
  for (int a = 0; a < 3; a++) {
    if (STAGE == 1) {
      dfn[a] = dt6 * kp[a];
      tpos[a] = oo[a] + dt2 * kp[a];
      vfn[a] = vo[a] + dt6 * kv[3 + a];
      vn[a] = vo[a] + dt2 * kv[3 + a];
    } else if (STAGE == 2) {
      dfn[a] = df[a] + dt3 * kp[a];
      tpos[a] = oo[a] + dt2 * kp[a];
      vfn[a] = vf[a] + dt3 * kv[3 + a];
      vn[a] = vo[a] + dt2 * kv[3 + a];
    } else if (STAGE == 3) {
      dfn[a] = df[a] + dt3 * kp[a];
      tpos[a] = oo[a] + dt * kp[a];
      vfn[a] = vf[a] + dt3 * kv[3 + a];
      vn[a] = vo[a] + dt * kv[3 + a];
    } else {
      dfn[a] = df[a] + dt6 * kp[a];
      tpos[a] = oo[a] + dfn[a];
      vfn[a] = vf[a] + dt6 * kv[3 + a];
      vn[a] = vfn[a];
    }
  }
  int io, jo, ko;
  cell_ijk(g, cello, io, jo, ko);
  int32_t ncell_;
  float nox, noy, noz;
  if (!place(g, io, jo, ko, tpos[0], tpos[1], tpos[2], ncell_, nox, noy, noz)) {
    raise_status(sc, PMPIC_ERR_OUT_OF_BOX_Z);
    if (STAGE == 1 || STAGE == 4) {
      const Float3 at = ld3(rs.off, p), v = ld3(rs.vor, p);
      stnt(rs.cell_to, p, ldnt(rs.cell, p));
      st3(rs.off_to, p, at.x, at.y, at.z);
      st3(rs.vor_to, p, v.x, v.y, v.z);
    }
    return -1;
  }
  stnt(rs.cell_to, p, ncell_);
  st3(rs.off_to, p, nox, noy, noz);
  st3(rs.vor_to, p, vn[0], vn[1], vn[2]);
  if (STAGE != 4) {
    st3(b.df, p, dfn[0], dfn[1], dfn[2]);
    st3(b.pf, p, vfn[0], vfn[1], vfn[2]);
  } else {
    st3(b.dx, p, kv[0], kv[1], kv[2]);
    st3(b.dp, p, kv[3], kv[4], kv[5]);
    if (stretch) {
      const float third = 1.f / 3.f;
      float ds = vn[0] * kv[3] + vn[1] * kv[4] + vn[2] * kv[5];
      ds = powf(fabsf(ds), third);
      const float snew = s_old + ds * dt;
      stnt(b.stretch, p, snew);
      split_flag[p] = (snew > 4.f) ? 1 : 0;  // the test of parcel_splitting.F90:76
    }
  }
  return ncell_;
}

template <int STAGE>
__global__ void __launch_bounds__(TPB) k32_rk_stage(Geometry g, Bulk32 b, RkSets rs, int64_t n,
                                                    const float4 *__restrict__ rec, Scale32 sc3,
                                                    int stretch,
                                                    uint8_t *__restrict__ split_flag,
                                                    DevScalars *sc, BinOut bo) {
  const int64_t p64 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  (void)n;  // launch size only: the count comes from device memory (see k32_bin_slot)
  const bool valid = p64 < sc->n;
  const uint32_t p = (uint32_t)p64;
  // with bo.on = 1, the parcel's new cell is binned for the next stage's par2grid as k32_bin_slot
  // bins it; every lane of the wavefront then takes part, parcels past the count as empty
  if (bo.on == 1) {
    const int32_t nc = valid ? rk_update<STAGE>(g, b, rs, rec, sc3, stretch, split_flag, sc, p)
                             : -1;
    bin_lane(g, nc, p, bo, sc);
    return;
  }
  if (!valid) return;
  const int32_t was = STAGE == 2 && bo.on ? rs.cell[p] : -1;  // (the stage updates it in place)
  const int32_t nc = rk_update<STAGE>(g, b, rs, rec, sc3, stretch, split_flag, sc, p);
  // with bo.on = 2, the entries of the parcels that change cell move
  if (STAGE == 2 && bo.on && nc >= 0 && nc != was) {
    remove_entry((int32_t)p, linear_cell(g, was), bo.capc, bo, sc);
    append_entry((int32_t)p, linear_cell(g, nc), bo, sc);
  }
}

// ---- splitting (parcel_splitting.F90:76-131, then the haloswap's wrap and reflection) ----
__global__ void k32_split_apply(Geometry g, Parcels32 P, int64_t cap, int64_t n, Scale32 sc3,
                                const int32_t *__restrict__ parents, int64_t nsplit,
                                DevScalars *sc) {
  const int64_t m = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (m >= nsplit) return;
  const int64_t i = parents[m];
  const int64_t c = n + m;
  if (c >= cap) {
    raise_status(sc, PMPIC_ERR_MAXPARCELS);
    return;
  }
  const float third = 1.f / 3.f;
  const float pi = 3.14159265358979f;
  const Float3 w = ld3(P.vor, i), vbh = ld3(P.vbh, i), off = ld3(P.off, i);
  const float p = w.x, q = w.y, r = w.z;
  const float vol = vbh.x;
  const float rr = powf(vol / 4.f / pi, third);
  const float absw = sqrtf(p * p + q * q + r * r);
  const float d[3] = {rr * p / absw * sc3.idx, rr * q / absw * sc3.idy, rr * r / absw * sc3.idz};
  int ci, cj, ck;
  cell_ijk(g, P.cell[i], ci, cj, ck);
  const float ox = off.x, oy = off.y, oz = off.z;
  int32_t cc, cp;
  float cx, cy, cz, px, py, pz;
  const bool okc = place(g, ci, cj, ck, ox + d[0], oy + d[1], oz + d[2], cc, cx, cy, cz);
  const bool okp = place(g, ci, cj, ck, ox - d[0], oy - d[1], oz - d[2], cp, px, py, pz);
  if (!okc || !okp) {
    raise_status(sc, PMPIC_ERR_OUT_OF_BOX_Z);
    return;
  }
  P.cell[c] = cc;
  st3(P.off, c, cx, cy, cz);
  st3(P.vor, c, p, q, r);
  const Float3 dx = ld3(P.dx, i), dp = ld3(P.dp, i);
  st3(P.dx, c, dx.x, dx.y, dx.z);
  st3(P.dp, c, dp.x, dp.y, dp.z);
  st3(P.vbh, c, vol / 2, vbh.y, vbh.z);
  P.stretch[c] = 0.f;
  P.tag[c] = P.tag[i];
  P.cell[i] = cp;
  st3(P.off, i, px, py, pz);
  P.vbh[3 * i] = vol / 2;
  P.stretch[i] = 0.f;
}

// ---- mixing (parcel_mixing.F90:157-389) ----
struct Mix32 {
  const float *G[6];  // kept vol, b, h, p, q, r (folded, doubled)
  float *R[6];        // residual vol .. r; after k32_mix_residual, divided by the kept volume
};

__global__ void k32_mix_new(Geometry g, Parcels32 P, int64_t cap, int64_t norig,
                            const int32_t *__restrict__ newcells, int64_t nadd,
                            const int32_t *__restrict__ zlist, int64_t nz_,
                            uint8_t *__restrict__ keep, Mix32 mg, float vmin,
                            float *__restrict__ portion_cell, uint8_t *__restrict__ dirty,
                            DevScalars *sc) {
  const int64_t m = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (m >= nadd) return;
  const int64_t ord = newcells[m];
  const int k = (int)(ord % g.ncz);
  const int j = (int)((ord / g.ncz) % g.ny);
  const int i = (int)(ord / ((int64_t)g.ncz * g.ny));
  const int64_t s = (m < nz_) ? (int64_t)zlist[m] : norig + (m - nz_);
  if (s + 2 > cap) {
    raise_status(sc, PMPIC_ERR_MAXPARCELS);
    return;
  }
  const int i1 = (i + 1 == g.nx) ? 0 : i + 1;
  const int j1 = (j + 1 == g.ny) ? 0 : j + 1;
  // 2x2x2 block in Fortran array-element order (z fastest, then y, then x)
  const int64_t q[8] = {gidx(g, k, j, i),      gidx(g, k + 1, j, i),  gidx(g, k, j1, i),
                        gidx(g, k + 1, j1, i), gidx(g, k, j, i1),     gidx(g, k + 1, j, i1),
                        gidx(g, k, j1, i1),    gidx(g, k + 1, j1, i1)};
  float s6[6];
#pragma unroll
  for (int f = 0; f < 6; f++) {
    float a = 0.f;
#pragma unroll
    for (int c = 0; c < 8; c++) a += mg.G[f][q[c]];
    s6[f] = a;
  }
  const float v = s6[0];
  P.cell[s] = pack_cell(i, j, k);
  st3(P.off, s, 0.5f, 0.5f, 0.5f);  // the cell centre
  st3(P.vor, s, s6[3] / v, s6[4] / v, s6[5] / v);
  st3(P.vbh, s, 2 * vmin, s6[1] / v, s6[2] / v);
  P.stretch[s] = 0.f;
  if (s + 1 < norig) keep[s] = 2;
  const int32_t c = (k * g.ny + j) * g.nx + i;
  portion_cell[c] = 2 * vmin / v;
  if (dirty) {
    dirty[tile_of(g, i, j, k)] = 1;
    if (m == 0) sc->anydirty = 1;
  }
}

// the new parcels into the lists (after the absorption, which reads the lists as they were scattered)
__global__ void k32_list_new(Geometry g, const int32_t *__restrict__ cellv, int64_t norig,
                             int64_t nadd, const int32_t *__restrict__ zlist, int64_t nz_, BinOut bo,
                             DevScalars *sc) {
  const int64_t m = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (m >= nadd) return;
  const int32_t s = m < nz_ ? zlist[m] : (int32_t)(norig + (m - nz_));
  append_entry(s, linear_cell(g, cellv[s]), bo, sc);
}

// ... and marks the cells around a node with a residual
__global__ void k32_mix_residual(Geometry g, Mix32 mg, const int32_t *__restrict__ npercell,
                                 const float *__restrict__ portion_cell,
                                 uint8_t *__restrict__ ctouch) {
  const int64_t nnode = (int64_t)g.nzn * g.ny * g.nx;
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= nnode) return;
  const int i = (int)(t % g.nx);
  const int j = (int)((t / g.nx) % g.ny);
  const int k = (int)(t / ((int64_t)g.nx * g.ny));
  int ci[2], cj[2];
  if (i == 0) { ci[0] = 0; ci[1] = g.nx - 1; } else { ci[0] = i - 1; ci[1] = i; }
  if (j == 0) { cj[0] = 0; cj[1] = g.ny - 1; } else { cj[0] = j - 1; cj[1] = j; }
  float r[6], gv[6];
#pragma unroll
  for (int f = 0; f < 6; f++) { r[f] = mg.R[f][t]; gv[f] = mg.G[f][t]; }
  for (int a = 0; a < 2; a++)
    for (int bb = 0; bb < 2; bb++)
      for (int kc = k - 1; kc <= k; kc++) {
        if (kc < 0 || kc >= g.ncz) continue;
        // a cell that received a new parcel: the test of the new-cell flags (npercell < 3),
        // read in cell order so consecutive nodes read consecutive cells
        const int64_t cn = ((int64_t)kc * g.ny + cj[bb]) * g.nx + ci[a];
        if (npercell[cn] >= 3) continue;
        const float portion = portion_cell[cn];
#pragma unroll
        for (int f = 0; f < 6; f++) r[f] = r[f] - portion * gv[f];
      }
  const float mlt = (k == 0 || k == g.nzn - 1) ? 2.f : 1.f;
  // stored divided by the node's kept volume: the absorption weights each node's residual by
  // w / vol_g (parcel_mixing.F90:247-340), so the division is done once per node here
  bool any = false;
#pragma unroll
  for (int f = 0; f < 6; f++) {
    const float v = (r[f] * mlt) / gv[0];
    mg.R[f][t] = v;
    any = any || v != 0.f;  // a NaN counts as not zero
  }
  if (!any) return;
  for (int kc = k - 1; kc <= k; kc++) {
    if (kc < 0 || kc >= g.ncz) continue;
    for (int bb = 0; bb < 2; bb++)
      for (int a = 0; a < 2; a++) ctouch[((int64_t)kc * g.ny + cj[bb]) * g.nx + ci[a]] = 1;
  }
}

__global__ void k32_fill_u8(uint8_t *__restrict__ a, int64_t n, uint8_t v) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) a[t] = v;
}

// the absorption of parcel p in cell (i, j, k), corners at o
__device__ __forceinline__ void absorb(const Parcels32 &P, int64_t p, const int32_t o[8],
                                       const Mix32 &mg) {
  const Float3 off = ld3(P.off, p), vor = ld3(P.vor, p), vbh = ld3(P.vbh, p);
  const float ox = off.x, oy = off.y, oz = off.z, v = vbh.x;
  const float fv[5] = {vbh.y, vbh.z, vor.x, vor.y, vor.z};
  float w[8];
  w[0] = (1 - oz) * (1 - oy) * (1 - ox) * v;
  w[1] = (1 - oz) * (1 - oy) * (ox) * v;
  w[2] = (1 - oz) * (oy) * (1 - ox) * v;
  w[3] = (1 - oz) * (oy) * (ox) * v;
  w[4] = (oz) * (1 - oy) * (1 - ox) * v;
  w[5] = (oz) * (1 - oy) * (ox) * v;
  w[6] = (oz) * (oy) * (1 - ox) * v;
  w[7] = (oz) * (oy) * (ox) * v;
  // the residual grids already hold residual / vol_g; 1 / vol_new once per parcel
  float vn = v;
#pragma unroll
  for (int c = 0; c < 8; c++) vn = vn + w[c] * ld((const float *)mg.R[0], (uint32_t)o[c]);
  const float ivn = 1.f / vn;
  float out[5];
#pragma unroll
  for (int f = 0; f < 5; f++) {
    float acc = fv[f] * v;
#pragma unroll
    for (int c = 0; c < 8; c++) acc = acc + w[c] * ld((const float *)mg.R[f + 1], (uint32_t)o[c]);
    out[f] = acc * ivn;
  }
  st3(P.vbh, p, vn, out[0], out[1]);
  st3(P.vor, p, out[2], out[3], out[4]);
}

// Kept parcels absorb the residuals (parcel_mixing.F90:247-340): those in the lists of the cells
// that k32_mix_residual marked.  The parcels of the others (almost all: residuals arise only around
// removed parcels and the cells that received new ones) keep their values, which the arithmetic
// would return to within rounding, and are not read.  A wavefront looks at `per` tiles (up
// to eight) and takes those with marked cells one after another, a cell's parcels eight at a time:
// 67 M parcels in 8.4 M cells 0.40 ms from the parcels' flags and cells -> 0.15 ms.  zero: leaves
// the counts at zero.
__global__ void __launch_bounds__(64) k32_mix_absorb(
    Geometry g, Parcels32 P, int64_t norig, const uint8_t *__restrict__ keep, Mix32 mg, int capc,
    const int32_t *__restrict__ slot, int32_t *__restrict__ count,
    const int32_t *__restrict__ start, const int32_t *__restrict__ sorted,
    const uint8_t *__restrict__ ctouch, uint8_t *__restrict__ dirty, DevScalars *sc, int per,
    int zero) {
  const int lane = threadIdx.x, cl = lane & 7, q = lane >> 3;
  const uint32_t ntx = (uint32_t)tiles_x(g), ntile = ntx * (uint32_t)(g.ny * g.ncz);
  // a lane's cell among the wavefront's tiles
  const uint32_t t0 = per * xcd_block(blockIdx.x, gridDim.x), own = t0 + q;
  const uint32_t row = own / ntx;
  const int x = 8 * (int)(own - row * ntx) + cl;
  const bool live = q < per && own < ntile && x < g.nx;
  const bool touched = live && ctouch[(int64_t)row * g.nx + x] != 0;
  const int held = live ? count[(int64_t)row * g.nx + x] : 0;
  if (zero) {
    if (live) count[(int64_t)row * g.nx + x] = 0;
    if (t0 == 0 && lane == 0) sc->novf = 0;
  }
  uint64_t left = __ballot(touched);
  while (left) {
    const int t = (__ffsll((unsigned long long)left) - 1) >> 3;  // a tile with touched cells
    const bool mine = (left >> (8 * t + cl)) & 1ull;
    left &= ~(0xffull << (8 * t));
    const uint32_t tile = t0 + t, xrow = tile / ntx;
    if (dirty && lane == 0) {
      dirty[tile] = 1;
      sc->anydirty = 1;
    }
    const int n = __shfl(held, 8 * t + cl);
    if (!mine || n == 0) continue;
    const int i = 8 * (int)(tile - xrow * ntx) + cl;
    const int64_t c = (int64_t)xrow * g.nx + i;
    const int32_t *list = n > capc ? sorted + start[c] : slot + c * capc;
    const int k = (int)(xrow / (uint32_t)g.ny), j = (int)(xrow - (uint32_t)k * (uint32_t)g.ny);
    int32_t o[8];
    corner_nodes(g, i, j, k, o);
    for (int e = q; e < n; e += 8) {
      const int32_t p = list[e];
      if (p >= 0 && p < norig && keep[p] == 1) absorb(P, p, o, mg);
    }
  }
}

// backfill: the state fields of the j-th kept slot from the end into the j-th removed slot
// (the reference copies x, y, z, p, q, r, b, h, vol, tag and stretch)
__global__ void k32_mix_backfill(Geometry g, Parcels32 P, const int32_t *__restrict__ dst,
                                 int64_t R, const int32_t *__restrict__ k1, int64_t K1,
                                 int64_t n, BinOut bo, uint8_t *__restrict__ dirty,
                                 DevScalars *sc) {
  const int64_t jx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (jx >= R) return;
  const int64_t s = k1[K1 - 1 - jx], d = dst[jx];
  const int32_t cell = P.cell[s];
  // a moved parcel changes the parcel order of its cell's sums
  if (dirty) {
    int i, j, k;
    cell_ijk(g, cell, i, j, k);
    dirty[tile_of(g, i, j, k)] = 1;
    if (jx == 0) sc->anydirty = 1;
  }
  P.cell[d] = cell;
#pragma unroll
  for (int e = 0; e < 3; e++) {
    P.off[3 * d + e] = P.off[3 * s + e];
    P.vor[3 * d + e] = P.vor[3 * s + e];
    P.vbh[3 * d + e] = P.vbh[3 * s + e];
  }
  P.stretch[d] = P.stretch[s];
  P.tag[d] = P.tag[s];
  // n: the parcels there are from now on
  if (bo.on && d < n) append_entry((int32_t)d, linear_cell(g, cell), bo, sc);
}

Zmap zmap_of(const Geometry &g) { return Zmap{(float)g.zbot, (float)g.dz}; }
Scale32 scale_of(const Geometry &g) {
  return Scale32{(float)(1.0 / g.dx), (float)(1.0 / g.dy), (float)(1.0 / g.dz)};
}

template <typename T>
int dalloc32(T **p, int64_t n) {
  *p = nullptr;
  if (n <= 0) n = 1;
  if (hipMalloc((void **)p, sizeof(T) * (size_t)n) != hipSuccess) return PMPIC_ERR_NOMEM;
  return PMPIC_OK;
}

// the counts, the cursor behind them and the overflow list's length at zero (the accumulation that
// uses a binning leaves them so)
int zero_counts(Ctx *c) {
  c->b32.mix_moves = 0;
  if (c->b32.counts_zero) return PMPIC_OK;
  hipLaunchKernelGGL(k32_bin_reset, dim3(cdiv(c->ncell + 1, TPB)), dim3(TPB), 0, c->stream,
                     c->cell_count, c->ncell + 1, c->dsc);
  PMPIC_CHECK(hipGetLastError());
  c->b32.counts_zero = true;
  return PMPIC_OK;
}

BinOut bin_out(const Ctx *c, int on, int capc) {
  const Bulk32 &b = c->b32;
  return BinOut{on, capc, c->cell_count, b.slot, b.ovf, b.ovfc, b.where, c->rank};
}

// the lists built last no longer stand
void unbin(Ctx *c) { c->b32.binned = false; }

int bin32(Ctx *c, int64_t n) {
  Bulk32 &b = c->b32;
  const int32_t *cells = b.cell[b.cur];
  const int capc = b32_choose_capc(c, n);
  // the launches of a captured graph cover a parcel bound (the kernels read the count)
  const int64_t ln = c->graph_n ? c->graph_n : n;
  if (b.binned && b.capc == capc && b.binned_set == b.cur && b.binned_n == n) {
    // a stage binned the cells it wrote, or moved the entries of the last binning
  } else if (b.binned && b.moving && b.capc == capc && capc > 0 && b.binned_set != b.cur &&
             b.binned_n <= n && !c->graph_n) {
    // the other set still holds the cells that were binned
    if (n > 0)
      hipLaunchKernelGGL(k32_bin_move, dim3(cdiv(n, TPB)), dim3(TPB), 0, c->stream, c->g,
                         b.cell[b.binned_set], cells, b.binned_n, n, bin_out(c, 2, capc), c->dsc);
  } else {
    b.capc = capc;
    PMPIC_TRY(zero_counts(c));
    b.counts_zero = false;
    if (ln > 0)
      hipLaunchKernelGGL(k32_bin_slot, dim3(cdiv(ln, (int64_t)TPB * BIN_SEQ)), dim3(TPB), 0,
                         c->stream, c->g, cells, ln, b.capc, b.slot, b.ovf, b.ovfc, b.where, c->rank,
                         c->cell_count, c->dsc);
  }
  b.binned = true;
  b.binned_set = b.cur;
  b.binned_n = n;
  // the dense region's buckets, of the cells past the slot capacity
  bin_alloc(c, c->cell_count, b.capc, c->cell_start, c->cell_count + c->ncell);
  if (ln > 0 && b.capc == 0) {
    hipLaunchKernelGGL(k32_dense_scatter, dim3(cdiv(ln, TPB)), dim3(TPB), 0, c->stream, c->g,
                       cells, c->rank, c->dsc, c->cell_start, c->sorted);
  } else if (ln > 0) {
    const int64_t nb = std::min<int64_t>(cdiv(ln, TPB), 1024);
    hipLaunchKernelGGL(k32_ovf_scatter, dim3(nb), dim3(TPB), 0, c->stream, b.ovf, b.ovfc, c->dsc,
                       c->cell_start, b.slot, b.capc, c->sorted);
  }
  PMPIC_CHECK(hipGetLastError());
  return PMPIC_OK;
}

Parcels32 parcels32(const Bulk32 &b) {
  return Parcels32{b.cell[b.cur], b.off[b.cur], b.vor[b.cur], b.vbh, b.dx, b.dp, b.stretch, b.tag};
}

// one accumulation of the current binning; zero: the counts are left at zero, so the lists no
// longer stand
template <int MODE>
int accumulate(Ctx *c, float *partial, float *partial2, uint8_t *dirty, bool zero = true,
               bool timed = false) {
  Bulk32 &b = c->b32;
  const dim3 grid(tiles_x(c->g) * c->g.ny * c->g.ncz), blk(64);
  auto k = k32_cell_accum<MODE>;
  if (timed)
    PMPIC_TRY(launch_timed(c, T_ACCUM, k, grid, blk, 0, c->g, parcels32(b), zmap_of(c->g),
                           (float)c->g.vmin, b.capc, b.slot, c->cell_count, c->cell_start,
                           c->sorted, c->rank, partial, partial2, c->npercell, c->cellflag, dirty,
                           c->cell_count + c->ncell, c->dsc, zero ? 1 : 0));
  else
    hipLaunchKernelGGL(k, grid, blk, 0, c->stream, c->g, parcels32(b), zmap_of(c->g),
                       (float)c->g.vmin, b.capc, b.slot, c->cell_count, c->cell_start, c->sorted,
                       c->rank, partial, partial2, c->npercell, c->cellflag, dirty,
                       c->cell_count + c->ncell, c->dsc, zero ? 1 : 0);
  PMPIC_CHECK(hipGetLastError());
  b.counts_zero = zero;
  if (zero) unbin(c);
  return PMPIC_OK;
}

// FP32 corner partials live in the plain form's partial buffers (48 doubles per cell hold
// 96 floats)
float *partial32(Ctx *c) { return reinterpret_cast<float *>(c->partial); }
float *partial32b(Ctx *c) { return reinterpret_cast<float *>(c->partial2); }

}  // namespace

__global__ void k32_set_n(DevScalars *sc, int64_t n) {
  if (threadIdx.x == 0 && blockIdx.x == 0) sc->n = n;
}

int b32_publish_n(Ctx *c) {
  if (c->hsc.n == c->n) return PMPIC_OK;
  hipLaunchKernelGGL(k32_set_n, dim3(1), dim3(64), 0, c->stream, c->dsc, c->n);
  PMPIC_CHECK(hipGetLastError());
  c->hsc.n = c->n;
  return PMPIC_OK;
}

// 16 entries while the mean is at most LOW_PPC parcels per cell (fewer empty entries to read),
// else 32; a capacity fixed from the environment or picked by the tuning wins; never more than
// the table holds
int b32_mean_capc(const Ctx *c, int64_t n) {
  const int capc = (n <= (int64_t)LOW_PPC * c->ncell) ? CAPC_LOW : CAPC;
  return capc > c->b32.capmax ? c->b32.capmax : capc;
}

int b32_choose_capc(const Ctx *c, int64_t n) {
  const Bulk32 &b = c->b32;
  int capc;
  if (b.capmax == 0) capc = 0;
  else if (b.capfix) capc = b.capfix;
  else if (b.captuned) capc = b.captuned;
  else capc = (n <= (int64_t)LOW_PPC * c->ncell) ? CAPC_LOW : CAPC;
  return capc > b.capmax ? b.capmax : capc;
}

int b32_alloc(Ctx *c) {
  Bulk32 &b = c->b32;
  for (int f = 0; f < 6; f++) b.kept_pending[f] = false;
  PMPIC_TRY(dalloc32(&b.pool, (int64_t)PARCEL32_WORDS * c->cap));
  float *at = b.pool;
  auto take = [&](int words) {
    float *p = at;
    at += (int64_t)words * c->cap;
    return p;
  };
  for (int i = 0; i < 2; i++) {
    b.cell[i] = reinterpret_cast<int32_t *>(take(1));
    b.off[i] = take(3);
    b.vor[i] = take(3);
  }
  b.vbh = take(3);
  b.dx = take(3);
  b.dp = take(3);
  b.stretch = take(1);
  b.df = take(3);
  b.pf = take(3);
  b.cur = 0;
  PMPIC_TRY(dalloc32(&b.tag, c->cap));
  // a parcel created by mixing takes neither a tag nor tendencies (parcel_mixing.F90 copies
  // tags only when it backfills, :377, and never writes dxdt..drdt): a slot past every earlier
  // count reads 0 for them, as in the FP64 form's arrays, which are cleared at allocation too
  PMPIC_CHECK(hipMemset(b.pool, 0, sizeof(float) * PARCEL32_WORDS * (size_t)c->cap));
  PMPIC_CHECK(hipMemset(b.tag, 0, sizeof(double) * (size_t)c->cap));
  // (zero until the first vort2vel, as the FP64 form's grids are)
  for (int i = 0; i < 3; i++) {
    PMPIC_TRY(dalloc32(&b.grid[i], c->gsz));
    PMPIC_CHECK(hipMemset(b.grid[i], 0, sizeof(float) * (size_t)c->gsz));
  }
  for (int i = 0; i < 12; i++) PMPIC_TRY(dalloc32(&b.mgrid[i], c->gsz));
  PMPIC_TRY(dalloc32(&b.newcells, c->ncell));
  PMPIC_TRY(dalloc32(&b.dirty, (int64_t)tiles_x(c->g) * c->g.ny * c->g.ncz));
  b.counts_zero = false;
  b.p2g_reuse = false;
  b.dirty_seq = 0;
  const char *renv = getenv("PMPIC_P2G_REUSE");
  b.reuse_off = renv && renv[0] == '0';
  for (int i = 0; i < 4; i++) {
    PMPIC_TRY(dalloc32(&b.pgrid[i], c->gsz));
    PMPIC_CHECK(hipMemset(b.pgrid[i], 0, sizeof(float) * (size_t)c->gsz));
    b.p2g_pending[i] = false;
  }
  // 32-bit byte offsets into the slot table.  PMPIC_SLOT_CAPACITY in the environment: 0 drops
  // the table (every cell then binned through the dense region, as grids beyond that range
  // are); 16 or 32 fixes the capacity instead of choosing it by the mean parcels per cell;
  // "tune" lets the first par2grid time the accumulation at both and keep the faster
  // (a table of 16 entries per cell reaches 2^30 entries at 512 x 512 x 256 cells)
  b.capmax = (c->ncell * CAPC <= ((int64_t)1 << 30))       ? CAPC
             : (c->ncell * CAPC_LOW <= ((int64_t)1 << 30)) ? CAPC_LOW
                                                            : 0;
  b.capfix = 0;
  b.captune = false;
  b.captuned = 0;
  b.rk_tpb = TPB;
  // Binning fused into the RK stages (1 and 3; stage 2 moves entries): a pass of its own reads the
  // cells again and is one more launch a stage (ms a step, apart and fused: 16x12x12 0.232 and 0.220,
  // 48^3 0.474 and 0.462, a stirred 90x60x41 1.035 and 1.014, eight members together 9.73 and 9.68,
  // 128^3 3.97 and 3.86, 256x256x128 15.68 and 15.38).  PMPIC_FUSED_BINNING=0 forces the pass.
  const char *fenv = getenv("PMPIC_FUSED_BINNING");
  b.fused_bin = fenv ? fenv[0] == '1' : true;
  b.binned = false;
  b.moving = c->cap <= (int64_t)1 << 27;
  // every parcel past its cell's capacity, every one moved there, and what mixing adds (MIX_MOVES)
  b.room = b.moving ? 2 * c->cap + c->cap / MIX_MOVES + 64 : c->cap;
  const char *env = getenv("PMPIC_SLOT_CAPACITY");
  if (env && strcmp(env, "tune") == 0) {
    b.captune = b.capmax == CAPC;
  } else if (env) {
    const int v = atoi(env);
    if (v == 0) b.capmax = 0;
    else if (v == CAPC_LOW || v == CAPC) b.capfix = v;
  }
  b.capc = b.capmax;
  b.slot = nullptr;
  if (b.capmax > 0) PMPIC_TRY(dalloc32(&b.slot, c->ncell * b.capmax));
  PMPIC_TRY(dalloc32(&b.ovf, b.room));
  PMPIC_TRY(dalloc32(&b.ovfc, b.room));
  b.where = nullptr;
  if (b.moving) PMPIC_TRY(dalloc32(&b.where, c->cap));
  return PMPIC_OK;
}

void b32_free(Ctx *c) {
  Bulk32 &b = c->b32;
  hipFree(b.pool);
  hipFree(b.tag);
  for (int i = 0; i < 3; i++) hipFree(b.grid[i]);
  for (int i = 0; i < 12; i++) hipFree(b.mgrid[i]);
  hipFree(b.newcells);
  hipFree(b.dirty);
  for (int i = 0; i < 4; i++) hipFree(b.pgrid[i]);
  hipFree(b.slot);
  hipFree(b.ovf);
  hipFree(b.ovfc);
  hipFree(b.where);
}

// field f (FP..FSTRETCH) of the parcels
struct Column {
  float *p;
  int stride;
};
static Column column(const Bulk32 &b, int f) {
  if (f >= FP && f <= FR) return {b.vor[b.cur] + (f - FP), 3};
  if (f >= FDXDT && f <= FDZDT) return {b.dx + (f - FDXDT), 3};
  if (f >= FDPDT && f <= FDRDT) return {b.dp + (f - FDPDT), 3};
  if (f == FH) return {b.vbh + 2, 3};
  if (f == FB) return {b.vbh + 1, 3};
  if (f == FVOL) return {b.vbh, 3};
  return {b.stretch, 1};
}

static int put_field(Ctx *c, double *dev, const double *host, int64_t n) {
  const HostPart p{const_cast<double *>(host), dev, sizeof(double) * (size_t)n};
  return copy_to_device(c, &p, 1);
}
static int get_field(Ctx *c, double *host, double *dev, int64_t n) {
  const HostPart p{host, dev, sizeof(double) * (size_t)n};
  return copy_to_host(c, &p, 1, false);
}

void b32_forget(Ctx *c) {
  unbin(c);
  c->b32.p2g_reuse = false;
}

int b32_set_parcels(Ctx *c, int64_t n, const double *const *fields) {
  PMPIC_TRY(ensure_fbuf(c));
  Bulk32 &b = c->b32;
  b32_forget(c);
  const dim3 gb(cdiv(n > 0 ? n : 1, TPB)), tb(TPB);
  for (int a = 0; a < 3; a++) {
    if (n > 0) {
      PMPIC_TRY(put_field(c, c->fbuf, fields[a], n));
      hipLaunchKernelGGL(k32_pos_in, gb, tb, 0, c->stream, c->g, a, c->fbuf, n, b.cell[b.cur],
                         b.off[b.cur], c->dsc);
    }
  }
  for (int f = FP; f <= FSTRETCH; f++) {
    if (n > 0) {
      PMPIC_TRY(put_field(c, c->fbuf, fields[f], n));
      const Column col = column(b, f);
      hipLaunchKernelGGL(k32_from_f64, gb, tb, 0, c->stream, c->fbuf, n, col.p, col.stride);
    }
  }
  if (n > 0)
    PMPIC_TRY(put_field(c, b.tag, fields[FTAG], n));
  PMPIC_CHECK(hipGetLastError());
  PMPIC_CHECK(hipStreamSynchronize(c->stream));
  return PMPIC_OK;
}

int b32_get_parcels(Ctx *c, double *const *fields) {
  PMPIC_TRY(ensure_fbuf(c));
  Bulk32 &b = c->b32;
  const int64_t n = c->n;
  if (n == 0) return PMPIC_OK;
  const dim3 gb(cdiv(n, TPB)), tb(TPB);
  for (int f = 0; f < 17; f++) {
    if (!fields[f]) continue;
    if (f == FTAG) {
      PMPIC_TRY(get_field(c, fields[f], b.tag, n));
      continue;
    }
    if (f < 3)
      hipLaunchKernelGGL(k32_pos_out, gb, tb, 0, c->stream, c->g, f, b.cell[b.cur],
                         b.off[b.cur], n, c->fbuf);
    else {
      const Column col = column(b, f);
      hipLaunchKernelGGL(k32_to_f64, gb, tb, 0, c->stream, col.p, col.stride, n, c->fbuf);
    }
    PMPIC_TRY(get_field(c, fields[f], c->fbuf, n));
  }
  PMPIC_CHECK(hipGetLastError());
  PMPIC_CHECK(hipStreamSynchronize(c->stream));
  return PMPIC_OK;
}

// The last mixing's kept sums stand for the next par2grid on x rows of whole 16-cell pieces.  The
// tiles and their flags would serve every length; elsewhere every par2grid sums every tile, one full
// launch a stage, as the accumulation's timer counts them there.
static bool reuse_sums(const Ctx *c) { return c->g.nx % 16 == 0 && !c->b32.reuse_off; }

// A graph of stages 1-3 always captures stage 1's par2grid reading the dirty-tile flags (with the
// reuse on) and finding the counts at zero; where the last mixing's sums are not current, every
// tile is marked dirty first, so the captured par2grid sums them all.
int b32_graph_reuse(Ctx *c) {
  Bulk32 &b = c->b32;
  unbin(c);
  PMPIC_TRY(zero_counts(c));
  if (!reuse_sums(c)) return PMPIC_OK;
  if (!b.p2g_reuse) {
    const int64_t nt = (int64_t)tiles_x(c->g) * c->g.ny * c->g.ncz;
    hipLaunchKernelGGL(k32_fill_u8, dim3(cdiv(nt, TPB)), dim3(TPB), 0, c->stream, b.dirty, nt,
                       (uint8_t)1);
    PMPIC_CHECK(hipGetLastError());
  }
  b.p2g_reuse = true;
  return PMPIC_OK;
}

// the par2grid accumulation; with `dirty`, only the tiles it marks (the others keep the
// partials the last mixing summed): that launch is left out of the kernel timer, whose
// per-launch figures are those of full launches
static int p2g_accum(Ctx *c, uint8_t *dirty = nullptr, bool zero = true) {
  return accumulate<A32_P2G>(c, partial32(c), nullptr, dirty, zero, dirty == nullptr);
}

// The capacity tuning: bin at 16 and at 32 slots, time the accumulation of each (its second
// launch, after one to warm the caches) and keep the faster for every later binning of this
// context.  Both capacities sum each cell's parcels in ascending parcel order, so the choice
// changes no result; the partials of the last run are this par2grid's.
static int tune_capacity(Ctx *c, int64_t n) {
  Bulk32 &b = c->b32;
  const int caps[2] = {CAPC_LOW, CAPC};
  float ms[2] = {0.f, 0.f};
  hipEvent_t e0, e1;
  PMPIC_CHECK(hipEventCreate(&e0));
  if (hipEventCreate(&e1) != hipSuccess) {
    hipEventDestroy(e0);
    return PMPIC_ERR_HIP;
  }
  int rc = PMPIC_OK;
  for (int t = 0; t < 2 && rc == PMPIC_OK; t++) {
    b.capfix = caps[t];
    unbin(c);
    rc = bin32(c, n);
    if (rc == PMPIC_OK) rc = p2g_accum(c, nullptr, false);
    if (rc == PMPIC_OK && hipEventRecord(e0, c->stream) != hipSuccess) rc = PMPIC_ERR_HIP;
    if (rc == PMPIC_OK) rc = p2g_accum(c);
    if (rc == PMPIC_OK && (hipEventRecord(e1, c->stream) != hipSuccess ||
                           hipEventSynchronize(e1) != hipSuccess ||
                           hipEventElapsedTime(&ms[t], e0, e1) != hipSuccess))
      rc = PMPIC_ERR_HIP;
  }
  b.capfix = 0;
  hipEventDestroy(e0);
  hipEventDestroy(e1);
  if (rc != PMPIC_OK) return rc;
  b.captuned = (ms[0] < ms[1]) ? caps[0] : caps[1];
  b.captune = false;
  return PMPIC_OK;
}

int b32_par2grid(Ctx *c) {
  const int64_t n = c->n;
  // this par2grid writes the FP32 p, q, r and total-buoyancy grids, current for the exports of
  // GP..GR and GB: the kept p, q, r, b of the last mixing are superseded
  Bulk32 &b = c->b32;
  b.kept_pending[1] = b.kept_pending[3] = false;
  b.kept_pending[4] = b.kept_pending[5] = false;
  for (int i = 0; i < 4; i++) b.p2g_pending[i] = true;
  // the last mixing's kept sums, where it left them current, stand for this accumulation
  // except on the tiles it changed
  uint8_t *dirty = (b.p2g_reuse && !b.captune) ? b.dirty : nullptr;
  b.p2g_reuse = false;
  // a mixing that changed no tile (known to the host once it has read the device scalars back,
  // and not inside a graph capture): the partials are all current, so no binning or sums
  const bool none = dirty && c->graph_n == 0 && b.dirty_seq < c->sync_seq && c->hsc.anydirty == 0;
  if (c->b32.captune && n > 0) {
    PMPIC_TRY(tune_capacity(c, n));
  } else if (!none) {
    PMPIC_TRY(bin32(c, n));
    // the lists of stages 2 and 4 are kept for the RK stage that follows and what comes after it
    const bool keep = b.moving && b.capc > 0 && c->rkstep % 2 == 0;
    PMPIC_TRY(p2g_accum(c, dirty, !keep));
  }
  launch_node_sum<float, float, 5, true>(
      c, {partial32(c), {b.pgrid[0], b.pgrid[1], b.pgrid[2], b.pgrid[3]}, nullptr, 1.f});
  PMPIC_CHECK(hipGetLastError());
  return PMPIC_OK;
}

int b32_rk_stage(Ctx *c, int stage, int stretch) {
  const int64_t n = c->n;
  Bulk32 &b = c->b32;
  const int from = b.cur, to = stage < 4 ? 1 : 0;
  const RkSets rs = {b.cell[from], b.cell[0], b.off[from], b.off[0],  b.vor[from],
                     b.vor[0],     b.cell[to], b.off[to],  b.vor[to]};
  if (n > 0) PMPIC_TRY(records_current(c));
  b.cur = to;
  if (n == 0) return PMPIC_OK;
  const Scale32 s3 = scale_of(c->g);
  b.p2g_reuse = false;
  const dim3 gb(cdiv(c->graph_n ? c->graph_n : n, b.rk_tpb)), tb(b.rk_tpb);
  // Stage 2 moves the entries of the parcels that its better velocity takes to another cell (per
  // mille of them; 67 M parcels: 2.38 -> 1.62 ms against binning them all).  Otherwise stages 1-3
  // may bin the cells they write for the next stage's par2grid (not while the capacity is being
  // tuned).  Stage 4 is followed by splitting and mixing, whose
  // binning compares the cells of both sets.
  const int capc = b32_choose_capc(c, n);
  const bool stands = b.binned && b.binned_set == from && b.binned_n == n && b.capc == capc;
  int on = 0;
  if (stage == 2 && stands && b.moving && capc > 0 && !b.captune) on = 2;
  else if (stage < 4 && b.fused_bin && !b.captune) on = 1;
  if (on != 2 && !(stage == 4 && stands)) unbin(c);
  if (on == 1) {
    PMPIC_TRY(zero_counts(c));
    b.counts_zero = false;
  }
  const BinOut bo = bin_out(c, on, capc);
  switch (stage) {
    case 1:
      PMPIC_TRY(launch_timed(c, T_RK, k32_rk_stage<1>, gb, tb, 0, c->g, c->b32, rs, n,
                             c->rec32, s3, stretch, c->flag, c->dsc, bo));
      break;
    case 2:
      PMPIC_TRY(launch_timed(c, T_RK, k32_rk_stage<2>, gb, tb, 0, c->g, c->b32, rs, n,
                             c->rec32, s3, stretch, c->flag, c->dsc, bo));
      break;
    case 3:
      PMPIC_TRY(launch_timed(c, T_RK, k32_rk_stage<3>, gb, tb, 0, c->g, c->b32, rs, n,
                             c->rec32, s3, stretch, c->flag, c->dsc, bo));
      break;
    default:
      PMPIC_TRY(launch_timed(c, T_RK, k32_rk_stage<4>, gb, tb, 0, c->g, c->b32, rs, n,
                             c->rec32, s3, stretch, c->flag, c->dsc, bo));
      break;
  }
  PMPIC_CHECK(hipGetLastError());
  if (on) {
    b.binned = true;
    b.binned_set = to;
    b.binned_n = n;
    b.capc = capc;
  }
  c->split_flags_fresh = (stage == 4 && stretch) ? 1 : 0;
  return PMPIC_OK;
}

int b32_split(Ctx *c) {
  const int64_t n = c->n;
  if (c->b32.binned_set == c->b32.cur) unbin(c);  // parents move within this set
  c->b32.p2g_reuse = false;
  if (n > 0) {
    // the stage-4 RK kernel already flagged the parcels to split
    if (c->split_flags_fresh)
      PMPIC_TRY(compact_flags(c, c->flag, 1, n, c->list_b, &c->dsc->nsplit));
    else
      PMPIC_TRY(split_list(c, c->b32.stretch, n));
    c->split_flags_fresh = 0;
  } else {
    c->hsc.nsplit = 0;
    PMPIC_CHECK(hipMemcpyAsync(&c->dsc->nsplit, &c->hsc.nsplit, sizeof(int64_t),
                               hipMemcpyHostToDevice, c->stream));
  }
  PMPIC_TRY(sync_scalars(c));
  const int64_t ns = c->hsc.nsplit;
  if (ns > 0) {
    if (n + ns > c->cap) return PMPIC_ERR_MAXPARCELS;
    hipLaunchKernelGGL(k32_split_apply, dim3(cdiv(ns, TPB)), dim3(TPB), 0, c->stream, c->g,
                       parcels32(c->b32), c->cap, n, scale_of(c->g), c->list_b, ns, c->dsc);
    PMPIC_CHECK(hipGetLastError());
  }
  c->n = n + ns;
  return b32_publish_n(c);
}

int b32_mix(Ctx *c) {
  const Geometry &g = c->g;
  Bulk32 &b = c->b32;
  const int64_t norig = c->n;
  const float vmin = (float)g.vmin;
  // kept and residual grids (construct_grids, parcel_mixing.F90:440-624)
  PMPIC_TRY(bin32(c, norig));
  // the kept sums' first five planes (weight, p, q, r, total buoyancy) are what the next
  // par2grid would sum on every tile this mixing leaves unchanged; the tiles it changes
  // are marked below (removed, new, absorbing and moved parcels).  cellflag holds the tiles'
  // residual flags until the new-parcel flags reuse it.
  b.p2g_reuse = false;
  const bool reuse = reuse_sums(c);
  uint8_t *dirty = reuse ? b.dirty : nullptr;
  PMPIC_TRY(accumulate<A32_MIX>(c, partial32(c), partial32b(c), b.dirty, false));
  unbin(c);  // until mixing is through
  const Parcels32 P = parcels32(b);
  const int64_t nnode = (int64_t)g.nzn * g.ny * g.nx;
  // planes weight, p, q, r, total buoyancy (not kept), b, h
  const NodeSums<float, float> kept = {
      partial32(c),
      {b.mgrid[0], b.mgrid[3], b.mgrid[4], b.mgrid[5], nullptr, b.mgrid[1], b.mgrid[2]},
      nullptr, 2.f};
  const NodeSums<float, float> res = {
      partial32b(c),
      {b.mgrid[6], b.mgrid[9], b.mgrid[10], b.mgrid[11], nullptr, b.mgrid[7], b.mgrid[8]},
      c->cellflag, 1.f};
  launch_node_sum<float, float, 7, false>(c, kept, &res);
  // the reference builds the kept grids in the model's vol, b, hg, p, q, r grids
  // (parcel_mixing.F90:131), which is what a grid export shows after mixing; nothing in the
  // step reads them there, so b32_export_grid widens them when one is exported
  for (int f = 0; f < 6; f++) b.kept_pending[f] = true;
  for (int f = 0; f < 4; f++) b.p2g_pending[f] = false;
  PMPIC_TRY(mix_lists(c, (const float *)b.vbh, 3, vmin, norig, b.newcells));
  PMPIC_TRY(sync_scalars(c));
  const int64_t Z = c->hsc.nzero, nadd = c->hsc.nadd;
  Mix32 mg = {{b.mgrid[0], b.mgrid[1], b.mgrid[2], b.mgrid[3], b.mgrid[4], b.mgrid[5]},
              {b.mgrid[6], b.mgrid[7], b.mgrid[8], b.mgrid[9], b.mgrid[10], b.mgrid[11]}};
  float *portion = partial32b(c);  // the residual partials are consumed by now
  // The lists follow where few parcels change (a captured graph builds its own first ones).  The
  // removed parcels leave them before new ones take their slots.
  const bool none = reuse && Z + nadd == 0;  // the next par2grid wants no lists
  const bool lists = b.moving && b.capc > 0 && !c->graph_on && !none && norig + nadd < c->cap &&
                     b.mix_moves + Z + nadd <= norig / MIX_MOVES;
  if (lists) b.mix_moves += Z + nadd;
  const BinOut bo = bin_out(c, lists ? 2 : 0, b.capc);
  if (Z > 0 && (lists || reuse))
    hipLaunchKernelGGL(k32_unlist, dim3(cdiv(Z, TPB)), dim3(TPB), 0, c->stream, g, P.cell,
                       c->list_a, 0, Z, bo, dirty, c->dsc);
  if (nadd > 0)
    hipLaunchKernelGGL(k32_mix_new, dim3(cdiv(nadd, TPB)), dim3(TPB), 0, c->stream, g, P, c->cap,
                       norig, b.newcells, nadd, c->list_a, Z, c->flag, mg, vmin, portion, dirty,
                       c->dsc);
  hipLaunchKernelGGL(k32_mix_residual, dim3(cdiv(nnode, TPB)), dim3(TPB), 0, c->stream, g, mg,
                     c->npercell, portion, c->ctouch);
  // eight tiles a wavefront where that leaves the chip full of them (150 us against 271 with one in
  // 1.05 M tiles; but 27 against 22 in 29 k)
  const int64_t tiles = (int64_t)tiles_x(g) * g.ny * g.ncz;
  const int per = tiles >= (1 << 17) ? 8 : 1;
  hipLaunchKernelGGL(k32_mix_absorb, dim3(cdiv(tiles, per)), dim3(64), 0, c->stream, g, P,
                     norig, c->flag, mg, b.capc, b.slot, c->cell_count, c->cell_start, c->sorted,
                     c->ctouch, dirty, c->dsc, per, lists ? 0 : 1);
  b.counts_zero = !lists;
  if (lists && nadd > 0)
    hipLaunchKernelGGL(k32_list_new, dim3(cdiv(nadd, TPB)), dim3(TPB), 0, c->stream, g, P.cell,
                       norig, nadd, c->list_a, Z, bo, c->dsc);
  PMPIC_CHECK(hipGetLastError());
  // new count (parcel_mixing.F90:217), then the backfill of removed slots (:347-389)
  int64_t np = norig;
  if (nadd > 0) {
    int64_t slast;
    if (nadd - 1 < Z) {
      int32_t v;
      PMPIC_TRY(read_back(c, &v, c->list_a + (nadd - 1), sizeof(int32_t)));
      slast = v;
    } else {
      slast = norig + (nadd - 1 - Z);
    }
    if (slast + 1 > np) np = slast + 1;
  }
  // what k32_mix_new raised (nothing else since the last read-back raises anything)
  if (nadd > 0) PMPIC_TRY(sync_scalars(c));
  c->last_removed = Z;
  c->last_added = nadd;
  if (np == norig) {
    int64_t R = 0;
    const int32_t *dst = nullptr;
    if (nadd < Z) {
      R = Z - nadd;
      dst = c->list_a + nadd;
    } else if (nadd == Z && Z > 0) {
      int32_t v;
      PMPIC_TRY(read_back(c, &v, c->list_a + (Z - 1), sizeof(int32_t)));
      if (v == norig - 1) {
        R = 1;
        dst = c->list_a + (Z - 1);
      }
    }
    if (R > 0) {
      PMPIC_TRY(compact_flags(c, c->flag, 1, norig, c->list_b, &c->dsc->nkeep1));
      PMPIC_TRY(sync_scalars(c));
      const int64_t K1 = c->hsc.nkeep1;
      if (R > K1) return PMPIC_ERR_BACKFILL;
      np -= R;
      if (lists)  // the slots past the new count
        hipLaunchKernelGGL(k32_unlist, dim3(cdiv(R, TPB)), dim3(TPB), 0, c->stream, g, P.cell,
                           nullptr, np, R, bo, nullptr, c->dsc);
      hipLaunchKernelGGL(k32_mix_backfill, dim3(cdiv(R, TPB)), dim3(TPB), 0, c->stream, g, P,
                         dst, R, c->list_b, K1, np, bo, dirty, c->dsc);
      PMPIC_CHECK(hipGetLastError());
    }
  }
  c->n = np;
  b.binned = lists;
  b.binned_n = np;
  // whether any tile changed (anydirty) the host learns with the next read-back of the device
  // scalars (the status check that ends the component or the step)
  b.dirty_seq = c->sync_seq;
  b.p2g_reuse = reuse;
  return b32_publish_n(c);
}

// writebinary's grids (writebinary.F90:217-228): b, hg, p, q, r by par2grid of the FP32
// parcels' b, h, p, q, r, FP32 sums normalised into the FP64 grids
int b32_dump_grids(Ctx *c) {
  Bulk32 &b = c->b32;
  b.p2g_reuse = false;  // the dump's sums overwrite the partials
  PMPIC_TRY(bin32(c, c->n));
  PMPIC_TRY(accumulate<A32_DUMP>(c, partial32(c), nullptr, nullptr));
  launch_node_sum<float, double, 6, true>(
      c, {partial32(c), {c->grid[GB], c->grid[GHG], c->grid[GP], c->grid[GQ], c->grid[GR]}, nullptr,
          1.f});
  PMPIC_CHECK(hipGetLastError());
  // these grids now hold writebinary's values, not the kept grids of the last mixing or the
  // step's FP32 grids
  for (int f = 1; f < 6; f++) b.kept_pending[f] = false;
  for (int f = 0; f < 4; f++) b.p2g_pending[f] = false;
  return PMPIC_OK;
}

// the FP64 grid `id` as a grid export sees it in the FP32-bulk form: a kept grid of the last
// mixing still in mgrid, or the step's FP32 p, q, r or total buoyancy, is widened into it first
int b32_export_grid(Ctx *c, int id) {
  const GridId kept_ids[6] = {GVOL, GB, GHG, GP, GQ, GR};
  const GridId p2g_ids[4] = {GP, GQ, GR, GB};
  Bulk32 &b = c->b32;
  const int64_t nnode = (int64_t)c->g.nzn * c->g.ny * c->g.nx;
  for (int f = 0; f < 6; f++)
    if (kept_ids[f] == id && b.kept_pending[f]) {
      hipLaunchKernelGGL(k32_grid_to_f64, dim3(cdiv(nnode, TPB)), dim3(TPB), 0, c->stream,
                         b.mgrid[f], c->grid[id], nnode);
      PMPIC_CHECK(hipGetLastError());
      b.kept_pending[f] = false;
    }
  for (int f = 0; f < 4; f++)
    if (p2g_ids[f] == id && b.p2g_pending[f]) {
      hipLaunchKernelGGL(k32_grid_to_f64, dim3(cdiv(nnode, TPB)), dim3(TPB), 0, c->stream,
                         b.pgrid[f], c->grid[id], nnode);
      PMPIC_CHECK(hipGetLastError());
      b.p2g_pending[f] = false;
    }
  return PMPIC_OK;
}

// Six sums in one pass over the parcels on the host, whose chains of additions run beside each other,
// through buffers that stay in its caches: 0.88 and 8.4 M parcels 9.9 and 101 ms with a pass for each
// sum over all the records, 3.9 and 37 ms so.
int b32_conservation_sums(Ctx *c, double out6[6]) {
  constexpr int64_t PIECE = 1 << 16;
  const int64_t n = c->n, room = 3 * std::min(n, PIECE);
  // vol, b, h and p, q, r of each parcel
  std::unique_ptr<float[]> vbh(new (std::nothrow) float[room]), vor(new (std::nothrow) float[room]);
  if (!vbh || !vor) return PMPIC_ERR_NOMEM;
  double s[6] = {}, comp[6] = {};  // Neumaier summation in parcel order, FP64
  for (int64_t p0 = 0; p0 < n; p0 += PIECE) {
    const int64_t m = std::min(PIECE, n - p0);
    const size_t bytes = sizeof(float) * 3 * (size_t)m;
    PMPIC_CHECK(hipMemcpy(vbh.get(), c->b32.vbh + 3 * p0, bytes, hipMemcpyDeviceToHost));
    PMPIC_CHECK(hipMemcpy(vor.get(), c->b32.vor[c->b32.cur] + 3 * p0, bytes, hipMemcpyDeviceToHost));
    for (int64_t p = 0; p < m; p++) {
      const float *a = vbh.get() + 3 * p, *w = vor.get() + 3 * p;
      const double v = a[0];
      const double term[6] = {v, v * a[1], v * a[2], v * w[0], v * w[1], v * w[2]};
      for (int k = 0; k < 6; k++) {
        const double t = s[k] + term[k];
        if (fabs(s[k]) >= fabs(term[k])) comp[k] += (s[k] - t) + term[k];
        else comp[k] += (term[k] - t) + s[k];
        s[k] = t;
      }
    }
  }
  for (int k = 0; k < 6; k++) out6[k] = s[k] + comp[k];
  return PMPIC_OK;
}

}  // namespace pmpic
