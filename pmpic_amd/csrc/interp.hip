// Parcel <-> grid interpolation on MI355X: deterministic cell-binned par2grid, grid2par.
//
// Reference: model_core/src/parcels/parcel_interpolation.F90:186-481 (cache weights, grid2par,
// par2grid) and model_core/src/communication/MPIC_Haloswap.F90:95-307 (halo fold / fill, which
// on one GPU is periodic index arithmetic), components/parcel_mixing/src/parcel_mixing.F90:440-624
// (kept / residual grids).
//
// par2grid is a scatter; here it is a gather over a cell binning so that no floating-point
// atomics are used and every node sum has a fixed order:
//   1. bin:   each parcel finds its cell and takes a slot in the cell's bucket (integer atomics,
//             one per run of equal cells within a wavefront), the buckets are given room and the
//             parcel indices are scattered into them;
//   2. cell:  a wavefront takes eight cells of one x row; its 8 lanes a cell stage the cell's
//             parcels in LDS eight at a time, then lane q adds corner q's weight and weight *
//             value over them in ascending parcel order;
//   3. node:  one thread per node adds the matching corner sums of its adjacent cells (periodic
//             in x, y) in a fixed order and normalises by the summed weights.
// The result differs from the reference's sequential sum only by the order of additions.
#include "node_sum.h"

#include <hipcub/hipcub.hpp>

namespace pmpic {

namespace {

constexpr int TPB = 256;

// cell of every parcel and its slot in the cell's bucket.  Parcels that are neighbours in slot
// order usually share a cell, so lanes are grouped into runs of equal cell and one lane per run
// takes the whole run's slots with a single integer atomic.  Each wavefront walks BIN_SEQ
// consecutive groups of 64 parcels in order, so a cell whose parcels are consecutive in slot
// order gets ascending bucket slots unless it straddles two wavefronts' ranges.  16 groups where
// the parcels fill the chip with wavefronts that long (bin_seq); fewer below, down to one, where
// the walk is what takes the time (7,680 parcels: 13.3 us a call with 16 groups, 4 with one).
template <int BIN_SEQ>
__global__ void k_bin_count(Geometry g, const double *__restrict__ X, const double *__restrict__ Y,
                            const double *__restrict__ Z, int64_t n, int32_t *__restrict__ cell,
                            int32_t *__restrict__ rank, int32_t *__restrict__ count,
                            DevScalars *sc) {
  const int lane = threadIdx.x & 63;
  const int64_t w0 = (((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6) * 64 * BIN_SEQ;
  // all atomics of the wavefront are issued before any result is used, in group order
  int base[BIN_SEQ], hls[BIN_SEQ];
  // the positions of the next BIN_AHEAD groups are loaded before the current group is located
  // (clamped index, n >= 1), so the wavefront does not wait on memory once per group
  constexpr int BIN_AHEAD = BIN_SEQ < 4 ? BIN_SEQ : 4;
  double px[BIN_SEQ], py[BIN_SEQ], pz[BIN_SEQ];
  auto load_group = [&](int it) {
    const int64_t p = min(w0 + (int64_t)it * 64 + lane, n - 1);
    px[it] = X[p];
    py[it] = Y[p];
    pz[it] = Z[p];
  };
#pragma unroll
  for (int it = 0; it < BIN_AHEAD; it++) load_group(it);
#pragma unroll
  for (int it = 0; it < BIN_SEQ; it++) {
    if (it + BIN_AHEAD < BIN_SEQ) load_group(it + BIN_AHEAD);
    const int64_t p = w0 + (int64_t)it * 64 + lane;
    int32_t c = -1;
    if (p < n) {
      int i0, j0, k0;
      double dx_, dy_, dz_;
      const int st = locate(g, px[it], py[it], pz[it], i0, j0, k0, dx_, dy_, dz_);
      if (st != PMPIC_OK) raise_status(sc, st);
      else c = (int32_t)(((int64_t)k0 * g.ny + j0) * g.nx + i0);
      cell[p] = c;
    }
    const int32_t cprev = __shfl_up(c, 1);
    const bool head = (lane == 0) || (c != cprev);
    const unsigned long long hm = __ballot(head);
    const unsigned long long upto = hm & ((2ull << lane) - 1ull);
    const int hl = 63 - __clzll(upto);
    const unsigned long long above = hm & ~((2ull << hl) - 1ull);
    const int next = above ? (__ffsll(above) - 1) : 64;
    base[it] = (head && c >= 0) ? atomicAdd(&count[c], next - hl) : 0;
    hls[it] = hl;
  }
#pragma unroll
  for (int it = 0; it < BIN_SEQ; it++) {
    const int64_t p = w0 + (int64_t)it * 64 + lane;
    const int b = __shfl(base[it], hls[it]);
    if (p < n) rank[p] = b + (lane - hls[it]);
  }
}

// room for every bucket: start[c] from a running total.  The buckets' order does not matter to the
// sums, so each block takes its cells' total from the cursor with one atomic, and no scan of the
// whole array (two more launches) is needed.  A cell of up to `held` parcels takes none (its
// parcels are listed elsewhere).
constexpr int ALLOC_CELLS = 4;  // cells per thread
__global__ void __launch_bounds__(TPB) k_bin_alloc(const int32_t *__restrict__ count, int64_t ncell,
                                                   int held, int32_t *__restrict__ start,
                                                   int32_t *__restrict__ cursor) {
  __shared__ int32_t wave_sum[TPB / 64];
  __shared__ int32_t base;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t c0 = ((int64_t)blockIdx.x * TPB + threadIdx.x) * ALLOC_CELLS;
  int32_t k[ALLOC_CELLS], sum = 0;
#pragma unroll
  for (int i = 0; i < ALLOC_CELLS; i++) {
    k[i] = c0 + i < ncell ? count[c0 + i] : 0;
    if (k[i] <= held) k[i] = 0;
    sum += k[i];
  }
  int32_t incl = sum;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int32_t u = __shfl_up(incl, d);
    if (lane >= d) incl += u;
  }
  if (lane == 63) wave_sum[wave] = incl;
  __syncthreads();
  if (threadIdx.x == 0) {
    int32_t t = 0;
    for (int w = 0; w < TPB / 64; w++) {
      const int32_t v = wave_sum[w];
      wave_sum[w] = t;
      t += v;
    }
    base = t > 0 ? atomicAdd(cursor, t) : 0;
  }
  __syncthreads();
  int32_t o = base + wave_sum[wave] + incl - sum;
#pragma unroll
  for (int i = 0; i < ALLOC_CELLS; i++) {
    if (c0 + i < ncell && k[i]) start[c0 + i] = o;
    o += k[i];
  }
}

__global__ void k_bin_scatter(const int32_t *__restrict__ cell, const int32_t *__restrict__ rank,
                              const int32_t *__restrict__ start, int64_t n,
                              int32_t *__restrict__ sorted) {
  int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  int32_t c = cell[p];
  if (c < 0) return;
  sorted[start[c] + rank[p]] = (int32_t)p;
}

// value sources for the per-cell accumulation
enum AccMode { ACC_P2G = 0, ACC_SINGLE = 1, ACC_MIX = 2, ACC_DUMP = 4 };

// Per-cell corner sums.
//
// One wavefront per tile of 8 cells of one x row; lane = 8 q + cl is corner q (bits z<<2 | y<<1 |
// x) of cell cl.  A cell's parcels are taken eight at a time: lane (q, cl) loads and locates
// parcel q of the eight and stages (offsets, volume, values) in LDS row 8 q + cl; then every lane
// adds its corner's weight and weight * value over the cell's eight rows (the wavefront reads
// eight neighbouring 16-byte pairs at a time, each by eight lanes: no bank conflicts).  The next
// eight parcels' loads are in flight meanwhile.  With 2-5 KB of LDS and no barrier across
// wavefronts a CU holds 16 to 20 of them and the loads overlap the sums; the earlier form (a
// workgroup staging all parcels of 16 cells in 36 KB, 8 wavefronts a CU, its load and sum phases
// apart) took 2.18 ms for 57 M parcels in slot order and 224 us for 0.9 M well mixed ones, this one
// 1.78 ms (3.1 TB/s) and 115 us.  It is bound by the loads' latency.  The parcel loads are cached
// ones: a 128-byte line serves two chunks (streaming loads: 3.02 ms).
//
// Within a cell the additions run in ascending parcel order, the reference's: bucket slots come
// from atomics and may be out of order, so the lanes check their adjacent entries and rank the
// entries of the tile's cells where a pair is not ascending (in LDS up to LIST entries a cell, else
// in global memory through `order`).
//
// The corner sums are combined along x before they are written: node position i of corner pair
// bb = (by, bz) adds the bx = 1 corner of cell i - 1 and the bx = 0 corner of cell i.  Value f of
// entry (bb, row, position) sits at ((f 4 + bb) nrows + row) (nx + ntx) + 9 tx + position - 8 tx,
// ntx tiles a row; a tile's last position holds its last cell's bx = 1 corner alone, completed by
// k_node_sum.  180 bytes a cell for five values instead of 320.
//
// ACC_MIX sums the kept parcels into `partial` (and counts them) and the residual ones into
// `partial2`, whose tiles without residual parcels (almost all) are left unwritten and marked so in
// tileres.  Either output may be null.  `zero`: leaves count and the cursor at zero, as the next
// binning wants them.
constexpr int LIST = 64;

template <int MODE, int NV>
__device__ __forceinline__ void load_values(const double *__restrict__ par, int64_t cap,
                                            const double *__restrict__ var, int64_t p,
                                            double *val) {
  if constexpr (MODE == ACC_P2G) {
    val[0] = par[FP * cap + p];
    val[1] = par[FQ * cap + p];
    val[2] = par[FR * cap + p];
    val[3] = par[FB * cap + p];
    val[4] = par[FH * cap + p];
  } else if constexpr (MODE == ACC_SINGLE) {
    val[0] = var[p];
  } else {
    val[0] = par[FB * cap + p];
    val[1] = par[FH * cap + p];
    val[2] = par[FP * cap + p];
    val[3] = par[FQ * cap + p];
    val[4] = par[FR * cap + p];
  }
}

// one parcel's loads
template <int NL>
struct Row {
  double x, y, z, vol, val[NL];
};

template <int MODE, int NV>
__global__ void __launch_bounds__(64) k_cell_accum(Geometry g, const double *__restrict__ par,
                                                   int64_t cap, const double *__restrict__ var,
                                                   int32_t *__restrict__ count,
                                                   const int32_t *__restrict__ start,
                                                   const int32_t *__restrict__ sorted,
                                                   int32_t *__restrict__ order,
                                                   double *__restrict__ partial,
                                                   double *__restrict__ partial2,
                                                   int32_t *__restrict__ npercell,
                                                   uint8_t *__restrict__ tileres,
                                                   int32_t *__restrict__ cursor, int zero) {
  constexpr int NF = NV + 1;
  constexpr int NL = MODE == ACC_P2G ? 5 : NV;  // values loaded: p, q, r, b, h make four
  constexpr int NVS = (NV + 1) / 2;             // value pairs a row
  constexpr bool MIX = MODE == ACC_MIX;
  __shared__ double2 sgeo[2][64];    // (delx, dely), (delz, vol)
  __shared__ double2 sval[NVS][64];  // values, two per slot
  __shared__ int32_t slist[LIST * 8];  // entry e of cell cl at 8 e + cl
  const int lane = threadIdx.x, cl = lane & 7, q = lane >> 3;
  const int bx = q & 1, by = (q >> 1) & 1, bz = q >> 2;
  const int ntx = (g.nx + 7) / 8;
  const uint32_t tile = xcd_block(blockIdx.x, gridDim.x);
  const uint32_t xrow = tile / (uint32_t)ntx;
  const int tx = (int)(tile - xrow * (uint32_t)ntx), m = min(8, g.nx - 8 * tx);  // cells here
  const bool live = cl < m;
  const int64_t c = (int64_t)xrow * g.nx + 8 * tx + cl;
  const int n = live ? count[c] : 0;
  const int64_t b = live ? start[c] : 0;
  int nmax = n;
#pragma unroll
  for (int d = 1; d < 8; d <<= 1) nmax = max(nmax, __shfl_xor(nmax, d));
  nmax = __builtin_amdgcn_readfirstlane(nmax);
  const int nch = (nmax + 7) >> 3;  // chunks of eight parcels a cell
  const int32_t *list = sorted + b;
  const bool small = nmax <= LIST;
  // entries 8 (i0 + i) + q of the cell, i < 8, ordered by parcel
  bool bad = false;
  for (int i0 = 0; i0 < nch; i0 += 8) {
#pragma unroll
    for (int i = 0; i < 8; i++) {
      if (i0 + i >= nch) break;
      const int e = 8 * (i0 + i) + q;
      const int32_t v = e < n ? list[e] : INT32_MAX;
      if (small) slist[64 * i + lane] = v;
      bad |= e + 1 < n && v > list[e + 1];
    }
  }
  if (__any(bad)) {
    for (int i0 = 0; i0 < nch; i0 += 8) {
      int32_t v[8];
      int r[8];
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const int e = 8 * (i0 + i) + q;
        v[i] = e < n ? list[e] : INT32_MAX;
        r[i] = 0;
      }
      for (int e = 0; e < nmax; e++) {
        const int32_t key = small ? slist[8 * e + cl] : e < n ? list[e] : INT32_MAX;
#pragma unroll
        for (int i = 0; i < 8; i++) r[i] += key < v[i] ? 1 : 0;
      }
      __syncthreads();
#pragma unroll
      for (int i = 0; i < 8; i++)
        if (8 * (i0 + i) + q < n) {
          if (small) slist[8 * r[i] + cl] = v[i];
          else order[b + r[i]] = v[i];
        }
    }
    if (!small) {
      __threadfence_block();
      list = order + b;
    }
  }
  __syncthreads();
  const double *X = par + FX * cap, *Y = par + FY * cap, *Z = par + FZ * cap;
  const double *VOL = par + FVOL * cap;
  auto fetch = [&](int ch, Row<NL> &row) {
    const int e = 8 * ch + q;
    if (e < n) {
      const int64_t p = small ? slist[64 * ch + lane] : list[e];
      row.x = X[p];
      row.y = Y[p];
      row.z = Z[p];
      row.vol = VOL[p];
      load_values<MODE, NV>(par, cap, var, p, row.val);
    }
  };
  double acc[NF], res[MIX ? NF : 1];
#pragma unroll
  for (int f = 0; f < NF; f++) acc[f] = 0.0;
#pragma unroll
  for (int f = 0; f < (MIX ? NF : 1); f++) res[f] = 0.0;
  int kept = 0;
  bool anyres = false;
  Row<NL> row{};
  if (nch > 0) fetch(0, row);
  for (int ch = 0; ch < nch; ch++) {
    if (8 * ch + q < n) {
      int i0, j0, k0;
      double delx, dely, delz;
      locate(g, row.x, row.y, row.z, i0, j0, k0, delx, dely, delz);
      sgeo[0][lane] = make_double2(delx, dely);
      sgeo[1][lane] = make_double2(delz, row.vol);
      if constexpr (MODE == ACC_P2G) {
        // total buoyancy, vorticity_tendency.F90:121-126
        const double hl = row.val[4] - exp(-row.z);
        sval[0][lane] = make_double2(row.val[0], row.val[1]);
        sval[1][lane] = make_double2(row.val[2], row.val[3] + 12.5 * (hl > 0.0 ? hl : 0.0));
      } else {
#pragma unroll
        for (int f = 0; f < NVS; f++)
          sval[f][lane] = make_double2(row.val[2 * f], 2 * f + 1 < NL ? row.val[2 * f + 1 < NL ? 2 * f + 1 : 0] : 0.0);
      }
    }
    __syncthreads();
    if (ch + 1 < nch) fetch(ch + 1, row);
    const int rows = min(8, nmax - 8 * ch), mine = n - 8 * ch;
#pragma unroll 2
    for (int a = 0; a < rows; a++) {
      const int r = 8 * a + cl;
      const double2 g0 = sgeo[0][r], g1 = sgeo[1][r];
      double v[2 * NVS];
#pragma unroll
      for (int f = 0; f < NVS; f++) {
        const double2 t = sval[f][r];
        v[2 * f] = t.x;
        v[2 * f + 1] = t.y;
      }
      const double fx = bx ? g0.x : 1 - g0.x;
      const double fy = by ? g0.y : 1 - g0.y;
      const double fz = bz ? g1.x : 1 - g1.x;
      const double w = fz * fy * fx * g1.y;
      if (a < mine) {
        if (!MIX || !(g1.y < g.vmin)) {
          acc[0] += w;
#pragma unroll
          for (int f = 0; f < NV; f++) acc[f + 1] += w * v[f];
          kept++;
        } else if constexpr (MIX) {
          anyres = true;
          res[0] += w;
#pragma unroll
          for (int f = 0; f < NV; f++) res[f + 1] += w * v[f];
        }
      }
    }
    __syncthreads();
  }
  const int64_t nrows = (int64_t)g.ny * g.ncz, W = g.nx + ntx;
  auto write_x = [&](const double *v, double *out) {
    const int64_t o = ((int64_t)(q >> 1) * nrows + xrow) * W + 9 * tx + (bx ? 8 : cl);
    const bool mine = bx ? (cl == 7 && m == 8) : cl <= m;
#pragma unroll
    for (int f = 0; f < NF; f++) {
      const double left = __shfl(v[f], (lane + 7) & 63);  // corner q | 1 of cell cl - 1
      if (mine) out[f * 4 * nrows * W + o] = bx || cl == 0 ? v[f] : left + v[f];
    }
  };
  if (!MIX || partial) write_x(acc, partial);
  if constexpr (MIX) {
    const bool any = __any(anyres) != 0;
    if (tileres && lane == 0) tileres[tile] = any ? 1 : 0;
    if (partial2 && any) write_x(res, partial2);
    if (npercell && live && q == 0) npercell[c] = kept;
  }
  if (zero) {
    if (live && q == 0) count[c] = 0;
    if (tile == 0 && lane == 0) *cursor = 0;
  }
}

// grid2par of one field (parcel_interpolation.F90:287-327)
__global__ void k_grid2par(Geometry g, const double *__restrict__ par, int64_t cap, int64_t n,
                           const double *__restrict__ G, double *__restrict__ var,
                           DevScalars *sc) {
  int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  int i0, j0, k0;
  double delx, dely, delz;
  int st = locate(g, par[FX * cap + p], par[FY * cap + p], par[FZ * cap + p], i0, j0, k0, delx,
                  dely, delz);
  if (st != PMPIC_OK) {
    raise_status(sc, st);
    return;
  }
  const int i1 = (i0 + 1 == g.nx) ? 0 : i0 + 1;
  const int j1 = (j0 + 1 == g.ny) ? 0 : j0 + 1;
  const double c000 = G[gidx(g, k0, j0, i0)], c001 = G[gidx(g, k0, j0, i1)];
  const double c010 = G[gidx(g, k0, j1, i0)], c011 = G[gidx(g, k0, j1, i1)];
  const double c100 = G[gidx(g, k0 + 1, j0, i0)], c101 = G[gidx(g, k0 + 1, j0, i1)];
  const double c110 = G[gidx(g, k0 + 1, j1, i0)], c111 = G[gidx(g, k0 + 1, j1, i1)];
  const double c00 = c000 * (1 - delz) + c100 * delz;
  const double c01 = c001 * (1 - delz) + c101 * delz;
  const double c10 = c010 * (1 - delz) + c110 * delz;
  const double c11 = c011 * (1 - delz) + c111 * delz;
  const double c0 = c00 * (1 - dely) + c10 * dely;
  const double c1 = c01 * (1 - dely) + c11 * dely;
  var[p] = c0 * (1 - delx) + c1 * delx;
}

}  // namespace

int scan_exclusive_i32(Ctx *c, const int32_t *in, int32_t *out, int64_t n) {
  size_t need = 0;
  PMPIC_CHECK(hipcub::DeviceScan::ExclusiveSum(nullptr, need, in, out, (int)n, c->stream));
  if (need > c->scan_tmp_bytes) {
    if (c->scan_tmp) PMPIC_CHECK(hipFree(c->scan_tmp));
    c->scan_tmp = nullptr;
    PMPIC_CHECK(hipMalloc(&c->scan_tmp, need));
    c->scan_tmp_bytes = need;
  }
  size_t have = c->scan_tmp_bytes;
  PMPIC_CHECK(hipcub::DeviceScan::ExclusiveSum(c->scan_tmp, have, in, out, (int)n, c->stream));
  return PMPIC_OK;
}

// the context's own binning buffers
static BinWork ctx_work(Ctx *c) {
  BinWork w;
  w.cell = c->cell;
  w.rank = c->rank;
  w.count = c->cell_count;
  w.start = c->cell_start;
  w.sorted = c->sorted;
  w.cursor = c->cell_count + c->ncell;
  w.partial = c->partial;
  return w;
}

void bin_alloc(Ctx *c, const int32_t *count, int held, int32_t *start, int32_t *cursor) {
  hipLaunchKernelGGL(k_bin_alloc, dim3(cdiv(c->ncell, TPB * ALLOC_CELLS)), dim3(TPB), 0, c->stream,
                     count, c->ncell, held, start, cursor);
}

// bins n parcels; count and cursor must be zero, and the accumulation that follows zeroes them
int bin_parcels_ws(Ctx *c, int64_t n, const BinWork &w) {
  const Geometry &g = c->g;
  auto count = [&](auto kernel, int seq) {
    hipLaunchKernelGGL(kernel, dim3(cdiv(n, (int64_t)TPB * seq)), dim3(TPB), 0, c->stream, g,
                       c->par + FX * c->cap, c->par + FY * c->cap, c->par + FZ * c->cap, n,
                       w.cell, w.rank, w.count, c->dsc);
  };
  // wavefronts of 16 groups from 2^22 parcels (4,096 of them, four a SIMD), of four from 2^19
  if (n >= (int64_t)1 << 22) count(k_bin_count<16>, 16);
  else if (n >= (int64_t)1 << 19) count(k_bin_count<4>, 4);
  else if (n > 0) count(k_bin_count<1>, 1);
  bin_alloc(c, w.count, 0, w.start, w.cursor);
  if (n > 0)
    hipLaunchKernelGGL(k_bin_scatter, dim3(cdiv(n, TPB)), dim3(TPB), 0, c->stream, w.cell, w.rank,
                       w.start, n, w.sorted);
  PMPIC_CHECK(hipGetLastError());
  return PMPIC_OK;
}

__global__ void k_zero_i32(int32_t *__restrict__ a, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) a[i] = 0;
}

int zero_i32(Ctx *c, int32_t *a, int64_t n) {
  hipLaunchKernelGGL(k_zero_i32, dim3(cdiv(n, TPB)), dim3(TPB), 0, c->stream, a, n);
  PMPIC_CHECK(hipGetLastError());
  return PMPIC_OK;
}

// the context's binning no longer stands: counts and cursor at zero
int drop_bins(Ctx *c) {
  if (c->bins_n != BINS_NONE) PMPIC_TRY(zero_i32(c, c->cell_count, c->ncell + 1));
  c->bins_n = BINS_NONE;
  return PMPIC_OK;
}

int bin_parcels(Ctx *c, int64_t n) {
  if (c->bins_n == n) return PMPIC_OK;  // mixing's, which changed no parcel's cell or slot
  PMPIC_TRY(drop_bins(c));
  return bin_parcels_ws(c, n, ctx_work(c));
}

static dim3 accum_tiles(const Ctx *c) {
  return dim3((unsigned)(cdiv(c->g.nx, 8) * c->g.ny * c->g.ncz));
}

template <int MODE, int NV>
static void launch_accum(Ctx *c, const BinWork &w, const double *var, double *partial,
                         double *partial2, int32_t *npc, uint8_t *tileres, int zero) {
  if (w.count == c->cell_count) c->bins_n = zero ? BINS_NONE : BINS_STALE;
  hipLaunchKernelGGL((k_cell_accum<MODE, NV>), accum_tiles(c), dim3(64), 0, c->stream, c->g, c->par,
                     c->cap, var, w.count, w.start, w.sorted, w.rank, partial, partial2, npc,
                     tileres, w.cursor, zero);
}

template <int NF, bool NORM>
static void node_sums(Ctx *c, const NodeSums<double, double> &first,
                      const NodeSums<double, double> *second = nullptr) {
  launch_node_sum<double, double, NF, NORM>(c, first, second);
}

int par2grid_fused(Ctx *c, int64_t n) {
  PMPIC_TRY(bin_parcels(c, n));
  const BinWork w = ctx_work(c);
  c->bins_n = BINS_NONE;
  PMPIC_TRY(launch_timed(c, T_ACCUM, k_cell_accum<ACC_P2G, 4>, accum_tiles(c), dim3(64), 0, c->g,
                         c->par, c->cap, nullptr, w.count, w.start, w.sorted, w.rank, w.partial,
                         nullptr, nullptr, nullptr, w.cursor, 1));
  node_sums<5, true>(c, {w.partial, {c->grid[GP], c->grid[GQ], c->grid[GR], c->grid[GB]}, nullptr, 1.});
  PMPIC_CHECK(hipGetLastError());
  return PMPIC_OK;
}

int par2grid_single_ws(Ctx *c, int64_t n, const double *d_var, double *d_grid,
                       const BinWork &w) {
  if (w.count == c->cell_count) PMPIC_TRY(bin_parcels(c, n));
  else PMPIC_TRY(bin_parcels_ws(c, n, w));
  launch_accum<ACC_SINGLE, 1>(c, w, d_var, w.partial, nullptr, nullptr, nullptr, 1);
  node_sums<2, true>(c, {w.partial, {d_grid}, nullptr, 1.});
  PMPIC_CHECK(hipGetLastError());
  return PMPIC_OK;
}

int par2grid_single(Ctx *c, int64_t n, const double *d_var, double *d_grid) {
  return par2grid_single_ws(c, n, d_var, d_grid, ctx_work(c));
}

// writebinary's grids (writebinary.F90:217-233): b, hg, p, q, r by par2grid of the parcels'
// b, h, p, q, r (one binning, the five sums of each node in parcel order as five par2grid
// calls would take them), then hgliq = max(0, hg - exp(-z)) and b += 12.5 hgliq per node
__global__ void k_hgliq(Geometry g, double *__restrict__ B, const double *__restrict__ HG,
                        double *__restrict__ HGLIQ) {
  const int64_t nnode = (int64_t)g.nzn * g.ny * g.nx;
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= nnode) return;
  const int k = (int)(t / ((int64_t)g.nx * g.ny));
  const double z = g.zmin_h + (double)k * g.dz + g.zbot;  // z_coords(k+1), setup as in create
  const double hl = HG[t] - exp(-z);
  const double liq = hl > 0. ? hl : 0.;
  HGLIQ[t] = liq;
  B[t] = B[t] + 12.5 * liq;
}

int dump_grids_f64(Ctx *c, int64_t n) {
  PMPIC_TRY(bin_parcels(c, n));
  launch_accum<ACC_DUMP, 5>(c, ctx_work(c), nullptr, c->partial, nullptr, nullptr, nullptr, 1);
  node_sums<6, true>(
      c, {c->partial, {c->grid[GB], c->grid[GHG], c->grid[GP], c->grid[GQ], c->grid[GR]}, nullptr, 1.});
  PMPIC_CHECK(hipGetLastError());
  return PMPIC_OK;
}

int hgliq_grid(Ctx *c) {
  const int64_t nnode = (int64_t)c->g.nzn * c->g.ny * c->g.nx;
  hipLaunchKernelGGL(k_hgliq, dim3(cdiv(nnode, TPB)), dim3(TPB), 0, c->stream, c->g, c->grid[GB],
                     c->grid[GHG], c->grid[GHGLIQ]);
  PMPIC_CHECK(hipGetLastError());
  return PMPIC_OK;
}

int grid2par_single(Ctx *c, int64_t n, const double *d_grid, double *d_var) {
  if (n > 0)
    hipLaunchKernelGGL(k_grid2par, dim3(cdiv(n, TPB)), dim3(TPB), 0, c->stream, c->g, c->par,
                       c->cap, n, d_grid, d_var, c->dsc);
  PMPIC_CHECK(hipGetLastError());
  return PMPIC_OK;
}

// kept and residual grids of parcel_mixing (construct_grids, parcel_mixing.F90:440-624, then
// the fold/fill of :133-138): grid[GVOL], GB, GHG, GP, GQ, GR hold the kept grids with the
// z-boundary doubling of :141-152; kres[0..5] hold the residual grids before the new-parcel
// correction of :202-207 and before their own doubling (:229-240).
// Without a residual buffer (partial2 null: a context too large for both) the kept and the
// residual sums take one pass each over `partial`, with the same sums.  cellflag holds the
// residual flags of the tiles (at most one a cell).  Leaves the binning as it is.
int mixing_grids(Ctx *c, int64_t n) {
  PMPIC_TRY(bin_parcels(c, n));
  const BinWork w = ctx_work(c);
  uint8_t *flags = c->cellflag;
  const NodeSums<double, double> kept = {
      c->partial,
      {c->grid[GVOL], c->grid[GB], c->grid[GHG], c->grid[GP], c->grid[GQ], c->grid[GR]}, nullptr, 2.};
  NodeSums<double, double> res = {
      c->partial2, {c->kres[0], c->kres[1], c->kres[2], c->kres[3], c->kres[4], c->kres[5]}, flags, 1.};
  if (c->partial2) {
    launch_accum<ACC_MIX, 5>(c, w, nullptr, c->partial, c->partial2, c->npercell, flags, 0);
    node_sums<6, false>(c, kept, &res);
  } else {
    launch_accum<ACC_MIX, 5>(c, w, nullptr, c->partial, nullptr, c->npercell, flags, 0);
    node_sums<6, false>(c, kept);
    launch_accum<ACC_MIX, 5>(c, w, nullptr, nullptr, c->partial, nullptr, nullptr, 0);
    res.partial = c->partial;
    node_sums<6, false>(c, res);
  }
  PMPIC_CHECK(hipGetLastError());
  return PMPIC_OK;
}

}  // namespace pmpic
