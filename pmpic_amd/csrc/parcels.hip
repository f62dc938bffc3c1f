// Parcel dynamics on MI355X: fused grid2par + RK4 stage update, the one-GPU parcel haloswap,
// parcel splitting and parcel mixing.
//
// Reference: components/rk4_integrator/src/rk4_integrator.F90:95-319,
// model_core/src/parcels/parcel_interpolation.F90:267-332 (grid2par),
// model_core/src/parcels/haloswap.F90:109-289, 296-456, 489-607, 678-771 (parcel haloswap),
// components/parcel_splitting/src/parcel_splitting.F90:47-168,
// components/parcel_mixing/src/parcel_mixing.F90:68-431.
//
// Slot order is kept exactly as the reference's one-rank run leaves it, because later steps
// depend on it (split children are appended in parent order, new mixing parcels fill removed
// slots in ascending order, backfill moves parcels from the end):
//  * haloswap: on one rank every parcel leaving through x or y is sent to self in direction
//    order N, NE, E, SE, S, SW, W, NW, shifted by one period, and unpacked into the vacated
//    slots in ascending slot order.  Here the stage kernel tags each parcel with its direction,
//    block-level ballot ranks plus one exclusive scan give every crossing parcel its rank in
//    (direction, slot) order and the rank of its own slot among the vacated ones, and two
//    gather/scatter kernels move the crossing parcels (all 29 fields) to their new slots.
//  * ranks within a block always come from wavefront ballots in lane order, so every
//    compaction and permutation is deterministic.
#include "common.h"

#include <float.h>
#include <string.h>

#include <algorithm>

#include <hipcub/hipcub.hpp>
#include <math.h>

namespace pmpic {

namespace {

constexpr int TPB = 256;
constexpr int NWAVE = TPB / 64;

// haloswap direction of a parcel (haloswap.F90:296-437); 0 = stays
__device__ __forceinline__ int direction(const Geometry &g, double x, double y) {
  const double xmin = g.hs_xmin, xmax = g.hs_xmax, ymin = g.hs_ymin, ymax = g.hs_ymax;
  if ((y >= ymax) && (x >= xmin && x < xmax)) return 1;   // N
  if (x >= xmax && y >= ymax) return 2;                    // NE
  if ((x >= xmax) && (y >= ymin && y < ymax)) return 3;   // E
  if (x >= xmax && y < ymin) return 4;                     // SE
  if ((y < ymin) && (x >= xmin && x < xmax)) return 5;    // S
  if (x < xmin && y < ymin) return 6;                      // SW
  if ((x < xmin) && (y >= ymin && y < ymax)) return 7;    // W
  if (x < xmin && y >= ymax) return 8;                     // NW
  return 0;
}

// Direction counts of a block: rows 0..7 = directions 1..8, row 8 = all crossing parcels.  Each
// wavefront's counts, one barrier, nine threads' sums; a wavefront none of whose parcels cross
// (almost every one) writes zeros.
__device__ __forceinline__ void wave_dir_counts(int dir, int32_t (*lds)[NWAVE]) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int mine = 0;
  if (__any(dir != 0)) {
#pragma unroll
    for (int d = 1; d <= 8; d++) {
      const int k = __popcll(__ballot(dir == d));
      if (lane == d - 1) mine = k;
    }
    const int k = __popcll(__ballot(dir != 0));
    if (lane == 8) mine = k;
  }
  if (lane < 9) lds[lane][wave] = mine;
}

__device__ __forceinline__ void write_dir_counts(int dir, int32_t *blk, int64_t nblk,
                                                 int32_t (*lds)[NWAVE]) {
  wave_dir_counts(dir, lds);
  __syncthreads();
  if (threadIdx.x < 9) {
    int t = 0;
#pragma unroll
    for (int w = 0; w < NWAVE; w++) t += lds[threadIdx.x][w];
    blk[(int64_t)threadIdx.x * nblk + blockIdx.x] = t;
  }
}

// grid2par of the six tendencies (vort2vel.F90:325-327, vorticity_tendency.F90:273-275) at the
// current positions, then the RK4 stage update (rk4_integrator.F90:109-296), the vertical
// reflection (haloswap.F90:440-456) and the haloswap direction of each parcel.  At stage 4 the
// stretch increment of parcel_splitting.F90:64-73 is applied too (it only needs the updated
// vorticity and the stage-4 tendencies of the same parcel).
//
// Bound by the parcel arrays' traffic.  keep_k: the stage's tendencies are stored too.  Inside a
// whole step only stage 4's are, the ones a caller can see: 48 of stage 2's 265 bytes a parcel
// (57 M parcels: 2.93 -> 2.43 ms, 4.9 TB/s).
template <int STAGE>
__global__ void __launch_bounds__(TPB) k_rk_stage(Geometry g, double *__restrict__ par, int64_t cap,
                                                  int64_t n, const double2 *__restrict__ rec,
                                                  int stretch, int keep_k,
                                                  DevScalars *sc,
                                                  uint8_t *__restrict__ flag,
                                                  int32_t *__restrict__ blk, int64_t nblk) {
  __shared__ int32_t lds[9][NWAVE];
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const bool active = p < n;
  int dir = 0;
  if (active) {
    // every parcel value the stage reads is loaded up front, so the loads overlap each other
    // and the grid gathers instead of waiting behind the stores
    const double x = ld_stream(&par[FX * cap + p]), y = ld_stream(&par[FY * cap + p]), z0 = ld_stream(&par[FZ * cap + p]);
    double yo[6], yf[6];
    if (STAGE == 1) {
      yo[0] = x;
      yo[1] = y;
      yo[2] = z0;
#pragma unroll
      for (int f = 3; f < 6; f++) yo[f] = ld_stream(&par[(FX + f) * cap + p]);
    } else {
#pragma unroll
      for (int f = 0; f < 6; f++) {
        if (STAGE != 4) yo[f] = ld_stream(&par[(f < 3 ? FXO + f : FPO + f - 3) * cap + p]);
        yf[f] = ld_stream(&par[(f < 3 ? FXF + f : FPF + f - 3) * cap + p]);
      }
    }
    const double s_old = (STAGE == 4 && stretch) ? ld_stream(&par[FSTRETCH * cap + p]) : 0.0;
    int i0, j0, k0;
    double delx, dely, delz;
    const int st = locate(g, x, y, z0, i0, j0, k0, delx, dely, delz);
    if (st != PMPIC_OK) {
      raise_status(sc, st);
    } else {
      const int i1 = (i0 + 1 == g.nx) ? 0 : i0 + 1;
      const int j1 = (j0 + 1 == g.ny) ? 0 : j0 + 1;
      const int64_t o[8] = {gidx(g, k0, j0, i0),     gidx(g, k0, j0, i1),
                            gidx(g, k0, j1, i0),     gidx(g, k0, j1, i1),
                            gidx(g, k0 + 1, j0, i0), gidx(g, k0 + 1, j0, i1),
                            gidx(g, k0 + 1, j1, i0), gidx(g, k0 + 1, j1, i1)};
      double kv[6];
#pragma unroll
      for (int h = 0; h < 3; h++) {  // two values of every corner's record at a time
        double2 G[8];
#pragma unroll
        for (int q = 0; q < 8; q++) G[q] = rec[3 * o[q] + h];
        auto interp = [&](double a0, double a1, double a2, double a3, double a4, double a5,
                          double a6, double a7) {
          const double c00 = a0 * (1 - delz) + a4 * delz;
          const double c01 = a1 * (1 - delz) + a5 * delz;
          const double c10 = a2 * (1 - delz) + a6 * delz;
          const double c11 = a3 * (1 - delz) + a7 * delz;
          const double c0 = c00 * (1 - dely) + c10 * dely;
          const double c1 = c01 * (1 - dely) + c11 * dely;
          return c0 * (1 - delx) + c1 * delx;
        };
        kv[2 * h] = interp(G[0].x, G[1].x, G[2].x, G[3].x, G[4].x, G[5].x, G[6].x, G[7].x);
        kv[2 * h + 1] = interp(G[0].y, G[1].y, G[2].y, G[3].y, G[4].y, G[5].y, G[6].y, G[7].y);
      }
      const double dt = sc->dtm;
      const double dt6 = dt / 6, dt2 = dt / 2, dt3 = dt / 3;
      double yv[6], yfn[6];
#pragma unroll
      for (int f = 0; f < 6; f++) {
        if (STAGE == 1) {
          yfn[f] = yo[f] + dt6 * kv[f];
          yv[f] = yo[f] + dt2 * kv[f];
        } else if (STAGE == 2) {
          yfn[f] = yf[f] + dt3 * kv[f];
          yv[f] = yo[f] + dt2 * kv[f];
        } else if (STAGE == 3) {
          yfn[f] = yf[f] + dt3 * kv[f];
          yv[f] = yo[f] + dt * kv[f];
        } else {
          yfn[f] = yf[f] + dt6 * kv[f];
          yv[f] = yfn[f];
        }
      }
      // reflect the current z only (haloswap.F90:447-454)
      double z = yv[2];
      if (z < g.zmin_h) z = g.zmin_h + (g.zmin_h - z);
      else if (z > g.zmax_h) z = g.zmax_h - (z - g.zmax_h);
      yv[2] = z;
#pragma unroll
      for (int f = 0; f < 6; f++) {
        if (STAGE == 4 || keep_k) st_stream(&par[(FDXDT + f) * cap + p], kv[f]);
        if (STAGE == 1) st_stream(&par[(f < 3 ? FXO + f : FPO + f - 3) * cap + p], yo[f]);
        st_stream(&par[(f < 3 ? FXF + f : FPF + f - 3) * cap + p], yfn[f]);
        st_stream(&par[(FX + f) * cap + p], yv[f]);
      }
      if (STAGE == 4 && stretch) {
        const double third = (double)(1.f / 3.f);
        double ds = yv[3] * kv[3] + yv[4] * kv[4] + yv[5] * kv[5];
        ds = pow(fabs(ds), third);
        st_stream(&par[FSTRETCH * cap + p], s_old + ds * dt);
      }
      dir = direction(g, yv[0], yv[1]);
    }
    flag[p] = (uint8_t)dir;
  }
  write_dir_counts(dir, blk, nblk, lds);
}

// direction classification only (haloswap after splitting): reflect, then tag
__global__ void __launch_bounds__(TPB) k_reflect_classify(Geometry g, double *__restrict__ par,
                                                          int64_t cap, int64_t n,
                                                          uint8_t *__restrict__ flag,
                                                          int32_t *__restrict__ blk, int64_t nblk) {
  __shared__ int32_t lds[9][NWAVE];
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const bool active = p < n;
  int dir = 0;
  if (active) {
    const double z = par[FZ * cap + p];
    if (z < g.zmin_h) par[FZ * cap + p] = g.zmin_h + (g.zmin_h - z);
    else if (z > g.zmax_h) par[FZ * cap + p] = g.zmax_h - (z - g.zmax_h);
    dir = direction(g, par[FX * cap + p], par[FY * cap + p]);
    flag[p] = (uint8_t)dir;
  }
  write_dir_counts(dir, blk, nblk, lds);
}

// Exclusive prefix sums of each of the nine rows of block counts, and the rows' totals (row 8's
// is the number of crossing parcels), a workgroup a row: every load issued at once (16
// counts a thread, four side by side) and one barrier.  One launch, 4.0 us at 30 blocks and 4.6
// at 3,456, up to the blocks it holds; above them the device-wide scan of all nine rows as one
// (two launches, and one for the total: 8 us and the gaps between them).
constexpr int SCAN_TPB = 1024, SCAN_TILES = 4, SCAN_MAX = SCAN_TILES * 4 * SCAN_TPB;
__global__ void __launch_bounds__(SCAN_TPB) k_hs_scan(const int32_t *__restrict__ blk,
                                                      int32_t *__restrict__ pre, int nblk,
                                                      int32_t *__restrict__ tot, DevScalars *sc) {
  constexpr int NW = SCAN_TPB / 64;
  static_assert(SCAN_TILES * NW == 64, "a (tile, wavefront) pair a lane");
  __shared__ int32_t wsum[SCAN_TILES * NW];
  const int row = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  blk += (int64_t)row * nblk;
  pre += (int64_t)row * nblk;
  int32_t v[SCAN_TILES][4], incl[SCAN_TILES];
#pragma unroll
  for (int t = 0; t < SCAN_TILES; t++)
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const int i = 4 * (t * SCAN_TPB + (int)threadIdx.x) + k;
      v[t][k] = i < nblk ? blk[i] : 0;
    }
#pragma unroll
  for (int t = 0; t < SCAN_TILES; t++) {
    incl[t] = v[t][0] + v[t][1] + v[t][2] + v[t][3];
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int32_t u = __shfl_up(incl[t], d);
      if (lane >= d) incl[t] += u;
    }
    if (lane == 63) wsum[t * NW + wave] = incl[t];
  }
  __syncthreads();
  const int32_t own = wsum[lane];
  int32_t s = own;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int32_t u = __shfl_up(s, d);
    if (lane >= d) s += u;
  }
#pragma unroll
  for (int t = 0; t < SCAN_TILES; t++) {
    int32_t o = __shfl(s - own, t * NW + wave) + incl[t] -
                (v[t][0] + v[t][1] + v[t][2] + v[t][3]);
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const int i = 4 * (t * SCAN_TPB + (int)threadIdx.x) + k;
      if (i < nblk) pre[i] = o;
      o += v[t][k];
    }
  }
  if (threadIdx.x == 63) {
    tot[row] = s;
    if (row == 8) sc->cross = s;
  }
}

__global__ void k_cross_total(const int32_t *__restrict__ pre, const int32_t *__restrict__ blk,
                              int64_t nblk, DevScalars *sc) {
  if (threadIdx.x || blockIdx.x) return;
  const int64_t last = 9 * nblk - 1;
  const int64_t total9 = (int64_t)pre[last] + blk[last];
  const int64_t base8 = pre[8 * nblk];
  sc->cross = total9 - base8;  // sum of row 8 = number of crossing parcels
}

// crossing parcels: record their slot at its rank among vacated slots and copy their fields,
// shifted by one period, to the staging slot given by their (direction, slot) rank.  A block
// without any returns at once; the others list theirs in LDS and copy a field a thread.  pre:
// prefix sums within each row, with the rows' totals, or (tot null) over all nine rows as one.
__global__ void __launch_bounds__(TPB) k_hs_gather(Geometry g, const double *__restrict__ par,
                                                   int64_t cap, int64_t n,
                                                   const uint8_t *__restrict__ flag,
                                                   const int32_t *__restrict__ blk,
                                                   const int32_t *__restrict__ pre, int64_t nblk,
                                                   const int32_t *__restrict__ tot,
                                                   int32_t *__restrict__ vacated,
                                                   double *__restrict__ tmp, int64_t tcap) {
  __shared__ int32_t lds[9][NWAVE];
  __shared__ int2 who[TPB];  // (slot, staging slot) of the block's crossing parcels
  __shared__ uint8_t wdir[TPB];
  const int K = blk[8 * nblk + blockIdx.x];
  if (K == 0) return;
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int dir = p < n ? flag[p] : 0;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  wave_dir_counts(dir, lds);
  const unsigned long long below = (1ull << lane) - 1ull;
  int wr = 0, wc = 0;  // ranks within the wavefront
  for (int d = 1; d <= 8; d++) {
    const unsigned long long m = __ballot(dir == d);
    if (dir == d) wr = __popcll(m & below);
  }
  wc = __popcll(__ballot(dir != 0) & below);
  __syncthreads();
  if (dir != 0) {
    for (int w = 0; w < wave; w++) {
      wr += lds[dir - 1][w];
      wc += lds[8][w];
    }
    int32_t t = pre[(int64_t)(dir - 1) * nblk + blockIdx.x] + wr;
    int32_t v = pre[(int64_t)8 * nblk + blockIdx.x] + wc;
    if (tot)
      for (int d = 0; d < dir - 1; d++) t += tot[d];
    else
      v -= pre[(int64_t)8 * nblk];
    vacated[v] = (int32_t)p;
    who[wc] = make_int2((int32_t)p, t);
    wdir[wc] = (uint8_t)dir;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < K * NFIELDS; e += TPB) {
    const int f = e / K, m = e - f * K;
    const int d = wdir[m];
    double val = par[(int64_t)f * cap + who[m].x];
    if (f == FX || f == FXO || f == FXF) {
      if (d == 2 || d == 3 || d == 4) val = val + g.xshift_e;
      else if (d == 6 || d == 7 || d == 8) val = val + g.xshift_w;
    }
    if (f == FY || f == FYO || f == FYF) {
      if (d == 1 || d == 2 || d == 8) val = val + g.yshift_n;
      else if (d == 4 || d == 5 || d == 6) val = val + g.yshift_s;
    }
    tmp[(int64_t)f * tcap + who[m].y] = val;
  }
}

__global__ void k_hs_scatter(double *__restrict__ par, int64_t cap, const double *__restrict__ tmp,
                             int64_t tcap, const int32_t *__restrict__ vacated,
                             const DevScalars *sc) {
  const int64_t K = sc->cross;
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < K * NFIELDS;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t f = e / K, t = e - f * K;
    par[f * cap + vacated[t]] = tmp[f * tcap + t];
  }
}

// ---- generic compaction: ascending indices i < n with flags[i] == want ----
// A thread takes FPT consecutive flags (one 16-byte load when all are in range), so a block
// covers FPB flags; the flags arrays start at allocation boundaries, so the loads are aligned.
constexpr int FPT = 16;
constexpr int FPB = FPT * TPB;

// bit q set when flags[i0 + q] == want (i0 < n)
__device__ __forceinline__ uint32_t flag_bits(const uint8_t *__restrict__ flags, uint8_t want,
                                              int64_t i0, int64_t n) {
  uint32_t m = 0;
  if (i0 + FPT <= n) {
    const uint4 v = *reinterpret_cast<const uint4 *>(flags + i0);
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int k = 0; k < 4; k++)
#pragma unroll
      for (int b = 0; b < 4; b++)
        if (((w[k] >> (8 * b)) & 0xffu) == want) m |= 1u << (4 * k + b);
  } else {
    for (int q = 0; q < FPT && i0 + q < n; q++)
      if (flags[i0 + q] == want) m |= 1u << q;
  }
  return m;
}

// exclusive prefix sum of v over the block in thread order; total = the block's sum
__device__ __forceinline__ int block_excl_scan(int v, int &total, int *lds) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int incl = v;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int u = __shfl_up(incl, d);
    if (lane >= d) incl += u;
  }
  if (lane == 63) lds[wave] = incl;
  __syncthreads();
  int off = 0, tot = 0;
#pragma unroll
  for (int w = 0; w < NWAVE; w++) {
    const int sw = lds[w];
    if (w < wave) off += sw;
    tot += sw;
  }
  __syncthreads();
  total = tot;
  return off + incl - v;
}

// The flags `want` of a block counted, from flags that a kernel has made already (k_flag_count)
// or that the block makes and stores itself (the others: one pass over the parcels or cells
// instead of two, KPT loads a thread in flight and each pass of them coalesced).
__global__ void __launch_bounds__(TPB) k_flag_count(const uint8_t *__restrict__ flags,
                                                    uint8_t want, int64_t n,
                                                    int32_t *__restrict__ blk) {
  __shared__ int lds[NWAVE];
  const int64_t i0 = ((int64_t)blockIdx.x * TPB + threadIdx.x) * FPT;
  const uint32_t m = (i0 < n) ? flag_bits(flags, want, i0, n) : 0u;
  int t;
  block_excl_scan(__popc(m), t, lds);
  if (threadIdx.x == 0) blk[blockIdx.x] = t;
}

// flag(i) of the block's items stored and the ones equal to want counted
template <typename F>
__device__ __forceinline__ void make_flags(const F &flag, uint8_t want, int64_t n, int64_t block,
                                           uint8_t *__restrict__ flags, int32_t *__restrict__ blk,
                                           int *lds) {
  const int64_t i0 = block * FPB + threadIdx.x;
  int k = 0;
  uint8_t v[FPT];
#pragma unroll
  for (int q = 0; q < FPT; q++) v[q] = flag(min(i0 + q * TPB, n - 1));
#pragma unroll
  for (int q = 0; q < FPT; q++)
    if (i0 + q * TPB < n) {
      flags[i0 + q * TPB] = v[q];
      k += v[q] == want;
    }
  int t;
  block_excl_scan(k, t, lds);
  if (threadIdx.x == 0) blk[block] = t;
}

// splitting (parcel_splitting.F90:76)
template <typename T>
__global__ void __launch_bounds__(TPB) k_split_flags(const T *__restrict__ stretch, int64_t n,
                                                     uint8_t *__restrict__ flags,
                                                     int32_t *__restrict__ blk) {
  __shared__ int lds[NWAVE];
  make_flags([&](int64_t i) { return (uint8_t)(stretch[i] > (T)4 ? 1 : 0); }, 1, n, blockIdx.x,
             flags, blk, lds);
}

// mixing: the first nblk blocks flag the parcels below vmin with 0 and the kept ones with 1, the
// others flag the cells with fewer than three kept parcels, in the reference's loop order (i
// outer, j, k inner; parcel_mixing.F90:160-162), and clear ctouch
template <typename T>
__global__ void __launch_bounds__(TPB) k_mix_flags(const T *__restrict__ vol, int stride, int64_t n,
                                                   T vmin,
                                                   uint8_t *__restrict__ keep,
                                                   int32_t *__restrict__ blk, int64_t nblk,
                                                   Geometry g, const int32_t *__restrict__ npercell,
                                                   int64_t ncell, uint8_t *__restrict__ cellflag,
                                                   uint8_t *__restrict__ ctouch,
                                                   int32_t *__restrict__ cblk) {
  __shared__ int lds[NWAVE];
  if (blockIdx.x < nblk) {
    if (n > 0)
      make_flags([&](int64_t i) { return (uint8_t)(vol[i * stride] < vmin ? 0 : 1); }, 0, n, blockIdx.x,
                 keep, blk, lds);
    else if (threadIdx.x == 0) blk[blockIdx.x] = 0;
    return;
  }
  make_flags(
      [&](int64_t o) {
        const uint32_t ord = (uint32_t)o, col = ord / (uint32_t)g.ncz;  // cells are below 2^31
        const uint32_t k = ord - col * (uint32_t)g.ncz, i = col / (uint32_t)g.ny;
        const uint32_t j = col - i * (uint32_t)g.ny;
        ctouch[ord] = 0;
        return (uint8_t)(npercell[((int64_t)k * g.ny + j) * g.nx + i] < 3 ? 1 : 0);
      },
      1, ncell, blockIdx.x - nblk, cellflag, cblk, lds);
}

// one flag array's compaction: the ascending indices of its flags `want`
struct FlagList {
  const uint8_t *flags;
  int64_t n, nblk;
  const int32_t *blk, *pre;  // per block: flags counted, and their prefix sums
  int32_t *out;
  int64_t *count;
  uint8_t want;
};

// up to OWN_PREFIX blocks a block sums the counts before it itself (at most 8 a thread), which
// takes less than the two launches of a scan; pre is null then
constexpr int OWN_PREFIX = 8 * TPB;

// the lists of a (its first a.nblk blocks) and b
__global__ void __launch_bounds__(TPB) k_flag_scatter(FlagList a, FlagList b) {
  __shared__ int lds[NWAVE];
  const bool second = blockIdx.x >= a.nblk;
  const FlagList &l = second ? b : a;
  const int64_t block = blockIdx.x - (second ? a.nblk : 0);
  const int64_t i0 = (block * TPB + threadIdx.x) * FPT;
  uint32_t m = (i0 < l.n) ? flag_bits(l.flags, l.want, i0, l.n) : 0u;
  int before = 0;
  if (l.pre) {
    before = l.pre[block];
  } else {
    int own = 0;
    for (int64_t q = threadIdx.x; q < block; q += TPB) own += l.blk[q];
    block_excl_scan(own, before, lds);
  }
  int t;
  int64_t o = (int64_t)before + block_excl_scan(__popc(m), t, lds);
  while (m) {
    l.out[o++] = (int32_t)(i0 + (__ffs(m) - 1));
    m &= m - 1u;
  }
  if (block == l.nblk - 1 && threadIdx.x == 0) *l.count = (int64_t)before + t;
}

// ---- splitting (parcel_splitting.F90:76-131) ----
__global__ void k_split_apply(double *__restrict__ par, int64_t cap, int64_t n,
                              const int32_t *__restrict__ parents, int64_t nsplit,
                              DevScalars *sc) {
  const int64_t m = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (m >= nsplit) return;
  const int64_t i = parents[m];
  const int64_t c = n + m;  // child slot n+1+m (1-based)
  if (c >= cap) {
    raise_status(sc, PMPIC_ERR_MAXPARCELS);
    return;
  }
  const double third = (double)(1.f / 3.f);
  const double pi = 4. * atan(1.0);
  const double p = par[FP * cap + i], q = par[FQ * cap + i], r = par[FR * cap + i];
  const double vol = par[FVOL * cap + i];
  double rr = vol / 4. / pi;
  rr = pow(rr, third);
  double absw = p * p + q * q + r * r;
  absw = sqrt(absw);
  const double x = par[FX * cap + i], y = par[FY * cap + i], z = par[FZ * cap + i];
  par[FX * cap + c] = x + rr * p / absw;
  par[FY * cap + c] = y + rr * q / absw;
  par[FZ * cap + c] = z + rr * r / absw;
  par[FP * cap + c] = p;
  par[FQ * cap + c] = q;
  par[FR * cap + c] = r;
  for (int f = FDXDT; f <= FDRDT; f++) par[(int64_t)f * cap + c] = par[(int64_t)f * cap + i];
  par[FH * cap + c] = par[FH * cap + i];
  par[FB * cap + c] = par[FB * cap + i];
  par[FVOL * cap + c] = vol / 2;
  par[FSTRETCH * cap + c] = 0.;
  par[FTAG * cap + c] = par[FTAG * cap + i];
  par[FX * cap + i] = x - rr * p / absw;
  par[FY * cap + i] = y - rr * q / absw;
  par[FZ * cap + i] = z - rr * r / absw;
  par[FVOL * cap + i] = vol / 2;
  par[FSTRETCH * cap + i] = 0.;
}

// ---- mixing (parcel_mixing.F90:157-389) ----
struct MixGrids {
  const double *G[6];  // kept vol, b, hg, p, q, r (folded, doubled)
  double *R[6];        // residual vres..rres
};

struct Coords {
  const double *xc, *yc, *zc;  // x_coords, y_coords, z_coords (reference values)
};

// one new parcel per sparse cell (parcel_mixing.F90:163-207 minus the residual update, which
// k_mix_residual applies per node in the same order)
__global__ void k_mix_new(Geometry g, double *__restrict__ par, int64_t cap, int64_t norig,
                          const int32_t *__restrict__ newcells, int64_t nadd,
                          const int32_t *__restrict__ zlist, int64_t nz_,
                          uint8_t *__restrict__ keep, MixGrids mg, Coords cc,
                          double *__restrict__ portion_cell, DevScalars *sc) {
  const int64_t m = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (m >= nadd) return;
  const int64_t ord = newcells[m];
  const int k = (int)(ord % g.ncz);
  const int j = (int)((ord / g.ncz) % g.ny);
  const int i = (int)(ord / ((int64_t)g.ncz * g.ny));
  const int64_t s = (m < nz_) ? (int64_t)zlist[m] : norig + (m - nz_);
  if (s + 2 > cap) {  // n > maxparcels after placing (parcel_mixing.F90:196-199)
    raise_status(sc, PMPIC_ERR_MAXPARCELS);
    return;
  }
  const int i1 = (i + 1 == g.nx) ? 0 : i + 1;
  const int j1 = (j + 1 == g.ny) ? 0 : j + 1;
  // sum over the 2x2x2 block in Fortran array-element order (z fastest, then y, then x)
  const int64_t q[8] = {gidx(g, k, j, i),   gidx(g, k + 1, j, i),   gidx(g, k, j1, i),
                        gidx(g, k + 1, j1, i), gidx(g, k, j, i1),  gidx(g, k + 1, j, i1),
                        gidx(g, k, j1, i1),  gidx(g, k + 1, j1, i1)};
  double s6[6];
#pragma unroll
  for (int f = 0; f < 6; f++) {
    double a = 0;
#pragma unroll
    for (int c = 0; c < 8; c++) a += mg.G[f][q[c]];
    s6[f] = a;
  }
  const double v = s6[0];
  const double portion = 2 * g.vmin / v;
  par[FX * cap + s] = 0.5 * (cc.xc[i + 2] + cc.xc[i + 3]);
  par[FY * cap + s] = 0.5 * (cc.yc[j + 2] + cc.yc[j + 3]);
  par[FZ * cap + s] = 0.5 * (cc.zc[k] + cc.zc[k + 1]);
  par[FVOL * cap + s] = 2 * g.vmin;
  par[FSTRETCH * cap + s] = 0;
  par[FB * cap + s] = s6[1] / v;
  par[FH * cap + s] = s6[2] / v;
  par[FP * cap + s] = s6[3] / v;
  par[FQ * cap + s] = s6[4] / v;
  par[FR * cap + s] = s6[5] / v;
  if (s + 1 < norig) keep[s] = 2;
  portion_cell[((int64_t)k * g.ny + j) * g.nx + i] = portion;
}

// residual minus the share of every adjacent new parcel, visiting cells in the reference's
// loop order, then the z-boundary doubling (parcel_mixing.F90:202-207, 221-240)
// ... and marks the cells around a node whose residual changes a parcel's values: not zero, or at
// a node without a (finite) kept volume to divide by
__global__ void k_mix_residual(Geometry g, MixGrids mg, const int32_t *__restrict__ npercell,
                               const double *__restrict__ portion_cell,
                               uint8_t *__restrict__ ctouch) {
  const int64_t nnode = (int64_t)g.nzn * g.ny * g.nx;
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= nnode) return;
  const int i = (int)(t % g.nx);
  const int j = (int)((t / g.nx) % g.ny);
  const int k = (int)(t / ((int64_t)g.nx * g.ny));
  // candidate cells in ascending halo'd index: the wrapped neighbour of node 0 comes last
  int ci[2], cj[2];
  if (i == 0) { ci[0] = 0; ci[1] = g.nx - 1; } else { ci[0] = i - 1; ci[1] = i; }
  if (j == 0) { cj[0] = 0; cj[1] = g.ny - 1; } else { cj[0] = j - 1; cj[1] = j; }
  double r[6], gv[6];
#pragma unroll
  for (int f = 0; f < 6; f++) { r[f] = mg.R[f][t]; gv[f] = mg.G[f][t]; }
  for (int a = 0; a < 2; a++)
    for (int b = 0; b < 2; b++)
      for (int kc = k - 1; kc <= k; kc++) {
        if (kc < 0 || kc >= g.ncz) continue;
        // a cell that received a new parcel: the test of the new-cell flags (npercell < 3),
        // read in cell order so consecutive nodes read consecutive cells
        const int64_t cn = ((int64_t)kc * g.ny + cj[b]) * g.nx + ci[a];
        if (npercell[cn] >= 3) continue;
        const double portion = portion_cell[cn];
#pragma unroll
        for (int f = 0; f < 6; f++) r[f] = r[f] - portion * gv[f];
      }
  const double mlt = (k == 0 || k == g.nzn - 1) ? 2. : 1.;
  bool any = !(gv[0] > 0.0 && gv[0] <= DBL_MAX);
#pragma unroll
  for (int f = 0; f < 6; f++) {
    const double v = r[f] * mlt;
    mg.R[f][t] = v;
    any = any || !(v == 0.0);
  }
  if (!any) return;
  for (int a = 0; a < 2; a++)
    for (int b = 0; b < 2; b++)
      for (int kc = k - 1; kc <= k; kc++)
        if (kc >= 0 && kc < g.ncz) ctouch[((int64_t)kc * g.ny + cj[b]) * g.nx + ci[a]] = 1;
}

// Kept parcels absorb the residuals (parcel_mixing.F90:247-340).  A parcel of a cell that
// k_mix_residual has not marked (almost all of them: residuals arise only around removed parcels
// and the cells that received new ones) keeps its values, which the arithmetic would return to
// within rounding: 6 bytes of flags and cells a parcel instead of 73 and the gathers (57 M
// parcels, none marked: 2.62 -> 0.29 ms).  cell: the mixing's binning.
__global__ void k_mix_absorb(Geometry g, double *__restrict__ par, int64_t cap, int64_t norig,
                             const uint8_t *__restrict__ keep, const int32_t *__restrict__ cell,
                             const uint8_t *__restrict__ ctouch, MixGrids mg) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= norig || keep[p] != 1) return;
  const int32_t c = cell[p];
  if (c < 0 || !ctouch[c]) return;  // (a parcel without a cell has ended the mixing before this)
  // all loads first (parcel values, then the gathers), all stores last
  const int fld[5] = {FB, FH, FP, FQ, FR};
  const double x = ld_stream(&par[FX * cap + p]), y = ld_stream(&par[FY * cap + p]),
               z = ld_stream(&par[FZ * cap + p]);
  const double v = ld_stream(&par[FVOL * cap + p]);
  double fv[5];
#pragma unroll
  for (int f = 0; f < 5; f++) fv[f] = ld_stream(&par[(int64_t)fld[f] * cap + p]);
  int i0, j0, k0;
  double delx, dely, delz;
  locate(g, x, y, z, i0, j0, k0, delx, dely, delz);
  const int i1 = (i0 + 1 == g.nx) ? 0 : i0 + 1;
  const int j1 = (j0 + 1 == g.ny) ? 0 : j0 + 1;
  const int64_t q[8] = {gidx(g, k0, j0, i0),     gidx(g, k0, j0, i1),
                        gidx(g, k0, j1, i0),     gidx(g, k0, j1, i1),
                        gidx(g, k0 + 1, j0, i0), gidx(g, k0 + 1, j0, i1),
                        gidx(g, k0 + 1, j1, i0), gidx(g, k0 + 1, j1, i1)};
  double w[8], g0[8];
  corner_weights(delx, dely, delz, v, w);
#pragma unroll
  for (int c = 0; c < 8; c++) g0[c] = mg.G[0][q[c]];
  double vn = v;
#pragma unroll
  for (int c = 0; c < 8; c++) vn = vn + w[c] * mg.R[0][q[c]] / g0[c];
  double out[5];
#pragma unroll
  for (int f = 0; f < 5; f++) {
    double acc = fv[f] * v;
#pragma unroll
    for (int c = 0; c < 8; c++) acc = acc + w[c] / g0[c] * mg.R[f + 1][q[c]];
    out[f] = acc / vn;
  }
  st_stream(&par[FVOL * cap + p], vn);
#pragma unroll
  for (int f = 0; f < 5; f++) st_stream(&par[(int64_t)fld[f] * cap + p], out[f]);
}

// backfill (parcel_mixing.F90:347-389): j-th remaining removed slot <- j-th kept slot from the
// end; only x, y, z, p, q, r, b, h, vol, tag and stretch are copied
__global__ void k_mix_backfill(double *__restrict__ par, int64_t cap,
                               const int32_t *__restrict__ dst, int64_t R,
                               const int32_t *__restrict__ k1, int64_t K1) {
  const int64_t jx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (jx >= R) return;
  const int64_t s = k1[K1 - 1 - jx], d = dst[jx];
  const int fl[11] = {FX, FY, FZ, FP, FQ, FR, FB, FH, FVOL, FTAG, FSTRETCH};
#pragma unroll
  for (int c = 0; c < 11; c++) par[(int64_t)fl[c] * cap + d] = par[(int64_t)fl[c] * cap + s];
}

}  // namespace

// The step's small read-backs go through pinned staging and wait on an event without the
// blocking-sync flag, which the host spins on: a pageable copy plus a stream synchronisation
// costs several times the latency.
int read_back(Ctx *c, void *host, const void *dev, size_t bytes) {
  if (bytes > 256) return PMPIC_ERR_ARG;
  PMPIC_CHECK(hipMemcpyAsync(c->pin, dev, bytes, hipMemcpyDeviceToHost, c->stream));
  PMPIC_CHECK(hipEventRecord(c->sync_ev, c->stream));
  PMPIC_CHECK(hipEventSynchronize(c->sync_ev));
  memcpy(host, c->pin, bytes);
  return PMPIC_OK;
}

int sync_scalars(Ctx *c) {
  PMPIC_TRY(read_back(c, &c->hsc, c->dsc, sizeof(DevScalars)));
  c->sync_seq++;
  return c->hsc.status;
}

// blk and pre of a list's counts; the scan where its blocks do not sum them themselves
static int list_prefix(Ctx *c, FlagList &l, int32_t *blk) {
  l.blk = blk;
  l.pre = nullptr;
  if (l.nblk <= OWN_PREFIX) return PMPIC_OK;
  l.pre = blk + l.nblk;
  return scan_exclusive_i32(c, blk, blk + l.nblk, l.nblk);
}

int compact_flags(Ctx *c, const uint8_t *flags, uint8_t want, int64_t n, int32_t *out,
                  int64_t *d_count) {
  FlagList l = {flags, n, cdiv(n > 0 ? n : 1, FPB), nullptr, nullptr, out, d_count, want};
  if (l.nblk > c->nblk_max) return PMPIC_ERR_ARG;
  hipLaunchKernelGGL(k_flag_count, dim3(l.nblk), dim3(TPB), 0, c->stream, flags, want, n, c->blk);
  PMPIC_TRY(list_prefix(c, l, c->blk));
  hipLaunchKernelGGL(k_flag_scatter, dim3(l.nblk), dim3(TPB), 0, c->stream, l, l);
  PMPIC_CHECK(hipGetLastError());
  return PMPIC_OK;
}

template <typename T>
int split_list(Ctx *c, const T *stretch, int64_t n) {
  FlagList l = {c->flag, n, cdiv(n, FPB), nullptr, nullptr, c->list_b, &c->dsc->nsplit, 1};
  if (n <= 0 || l.nblk > c->nblk_max) return PMPIC_ERR_ARG;
  hipLaunchKernelGGL(k_split_flags<T>, dim3(l.nblk), dim3(TPB), 0, c->stream, stretch, n, c->flag,
                     c->blk);
  PMPIC_TRY(list_prefix(c, l, c->blk));
  hipLaunchKernelGGL(k_flag_scatter, dim3(l.nblk), dim3(TPB), 0, c->stream, l, l);
  PMPIC_CHECK(hipGetLastError());
  return PMPIC_OK;
}

template <typename T>
int mix_lists(Ctx *c, const T *vol, int stride, T vmin, int64_t n, int32_t *cells) {
  FlagList a = {c->flag, n, cdiv(n > 0 ? n : 1, FPB), nullptr, nullptr, c->list_a,
                &c->dsc->nzero, 0};
  FlagList b = {c->cellflag, c->ncell, cdiv(c->ncell, FPB), nullptr, nullptr, cells,
                &c->dsc->nadd, 1};
  if (a.nblk > c->nblk_max || b.nblk > c->nblk_max) return PMPIC_ERR_ARG;
  int32_t *blk_a = c->blk, *blk_b = c->blk + 2 * a.nblk;
  hipLaunchKernelGGL(k_mix_flags<T>, dim3(a.nblk + b.nblk), dim3(TPB), 0, c->stream, vol, stride, n,
                     vmin, c->flag, blk_a, a.nblk, c->g, c->npercell, c->ncell, c->cellflag,
                     c->ctouch, blk_b);
  PMPIC_TRY(list_prefix(c, a, blk_a));
  PMPIC_TRY(list_prefix(c, b, blk_b));
  hipLaunchKernelGGL(k_flag_scatter, dim3(a.nblk + b.nblk), dim3(TPB), 0, c->stream, a, b);
  PMPIC_CHECK(hipGetLastError());
  return PMPIC_OK;
}

template int split_list<double>(Ctx *, const double *, int64_t);
template int split_list<float>(Ctx *, const float *, int64_t);
template int mix_lists<double>(Ctx *, const double *, int, double, int64_t, int32_t *);
template int mix_lists<float>(Ctx *, const float *, int, float, int64_t, int32_t *);

static int ensure_tmp(Ctx *c, int64_t need) {
  if (need <= c->tmp_cap) return PMPIC_OK;
  int64_t cap = need + need / 2 + 1024;
  if (cap > c->cap) cap = c->cap;
  if (c->tmp) PMPIC_CHECK(hipFree(c->tmp));
  c->tmp = nullptr;
  PMPIC_CHECK(hipMalloc(&c->tmp, sizeof(double) * NFIELDS * cap));
  c->tmp_cap = cap;
  return PMPIC_OK;
}

// Permutation part of the haloswap; expects flag[] and the per-block direction counts.  The
// staging buffer must hold every crossing parcel: up to HS_STAGE parcels it is made to hold them
// all, so nothing need be read back, which takes the host longer than the two copies take the device
// where nothing crosses; above, the count is read, and at most that much staged.
constexpr int64_t HS_STAGE = (int64_t)1 << 20;  // 232 MB of staging
static int haloswap_permute(Ctx *c, int64_t n, int64_t nblk) {
  int32_t *blk = c->blk, *pre = c->blk + 9 * nblk, *tot = nullptr;
  int64_t most = n;
  if (nblk <= SCAN_MAX) {
    tot = c->blk + 18 * nblk;
    hipLaunchKernelGGL(k_hs_scan, dim3(9), dim3(SCAN_TPB), 0, c->stream, blk, pre, (int)nblk, tot,
                       c->dsc);
  } else {
    PMPIC_TRY(scan_exclusive_i32(c, blk, pre, 9 * nblk));
    hipLaunchKernelGGL(k_cross_total, dim3(1), dim3(1), 0, c->stream, pre, blk, nblk, c->dsc);
  }
  if (n > HS_STAGE) {
    PMPIC_TRY(read_back(c, &c->hsc.cross, &c->dsc->cross, sizeof(int64_t)));
    most = c->hsc.cross;
  }
  if (most == 0) return PMPIC_OK;
  PMPIC_TRY(ensure_tmp(c, most));
  hipLaunchKernelGGL(k_hs_gather, dim3(nblk), dim3(TPB), 0, c->stream, c->g, c->par, c->cap, n,
                     c->flag, blk, pre, nblk, tot, c->list_a, c->tmp, c->tmp_cap);
  // a grid-stride copy: the count is the device's
  const int64_t sb = std::min<int64_t>(cdiv(most * NFIELDS, TPB), n > HS_STAGE ? 4096 : 256);
  hipLaunchKernelGGL(k_hs_scatter, dim3(sb), dim3(TPB), 0, c->stream, c->par, c->cap, c->tmp,
                     c->tmp_cap, c->list_a, c->dsc);
  PMPIC_CHECK(hipGetLastError());
  return PMPIC_OK;
}

int rk_stage_update(Ctx *c, int stage, int64_t n, int stretch) {
  const int64_t nblk = cdiv(n > 0 ? n : 1, TPB);
  if (nblk > c->nblk_max) return PMPIC_ERR_ARG;
  PMPIC_TRY(records_current(c));
  PMPIC_TRY(drop_bins(c));
  const int keep_k = c->whole_step ? 0 : 1;
  switch (stage) {
    case 1:
      PMPIC_TRY(launch_timed(c, T_RK, k_rk_stage<1>, dim3(nblk), dim3(TPB), 0, c->g, c->par,
                             c->cap, n, c->rec, stretch, keep_k, c->dsc, c->flag, c->blk, nblk));
      break;
    case 2:
      PMPIC_TRY(launch_timed(c, T_RK, k_rk_stage<2>, dim3(nblk), dim3(TPB), 0, c->g, c->par,
                             c->cap, n, c->rec, stretch, keep_k, c->dsc, c->flag, c->blk, nblk));
      break;
    case 3:
      PMPIC_TRY(launch_timed(c, T_RK, k_rk_stage<3>, dim3(nblk), dim3(TPB), 0, c->g, c->par,
                             c->cap, n, c->rec, stretch, keep_k, c->dsc, c->flag, c->blk, nblk));
      break;
    default:
      PMPIC_TRY(launch_timed(c, T_RK, k_rk_stage<4>, dim3(nblk), dim3(TPB), 0, c->g, c->par,
                             c->cap, n, c->rec, stretch, keep_k, c->dsc, c->flag, c->blk, nblk));
      break;
  }
  PMPIC_CHECK(hipGetLastError());
  return haloswap_permute(c, n, nblk);
}

int parcel_haloswap(Ctx *c, int64_t n, int reflect) {
  (void)reflect;
  PMPIC_TRY(drop_bins(c));
  const int64_t nblk = cdiv(n > 0 ? n : 1, TPB);
  if (nblk > c->nblk_max) return PMPIC_ERR_ARG;
  hipLaunchKernelGGL(k_reflect_classify, dim3(nblk), dim3(TPB), 0, c->stream, c->g, c->par, c->cap,
                     n, c->flag, c->blk, nblk);
  PMPIC_CHECK(hipGetLastError());
  return haloswap_permute(c, n, nblk);
}

// stage-4 splitting after the stretch update; then the second haloswap.  Updates c->n.
int parcel_split(Ctx *c) {
  const int64_t n = c->n;
  if (n > 0) {
    PMPIC_TRY(split_list(c, c->par + FSTRETCH * c->cap, n));
  } else {
    c->hsc.nsplit = 0;
    PMPIC_CHECK(hipMemcpyAsync(&c->dsc->nsplit, &c->hsc.nsplit, sizeof(int64_t),
                               hipMemcpyHostToDevice, c->stream));
  }
  PMPIC_TRY(sync_scalars(c));
  const int64_t ns = c->hsc.nsplit;
  if (ns > 0) {
    if (n + ns > c->cap) return PMPIC_ERR_MAXPARCELS;
    hipLaunchKernelGGL(k_split_apply, dim3(cdiv(ns, TPB)), dim3(TPB), 0, c->stream, c->par, c->cap,
                       n, c->list_b, ns, c->dsc);
    PMPIC_CHECK(hipGetLastError());
  }
  c->n = n + ns;
  return parcel_haloswap(c, c->n, 1);
}

// stage-4 mixing; updates c->n
int parcel_mix(Ctx *c) {
  const Geometry &g = c->g;
  const int64_t norig = c->n;
  PMPIC_TRY(mixing_grids(c, norig));
  // removed slots, ascending, and sparse cells in the reference's loop order
  PMPIC_TRY(mix_lists(c, c->par + FVOL * c->cap, 1, g.vmin, norig, c->sorted));
  PMPIC_TRY(sync_scalars(c));
  const int64_t Z = c->hsc.nzero, nadd = c->hsc.nadd;
  MixGrids mg = {{c->grid[GVOL], c->grid[GB], c->grid[GHG], c->grid[GP], c->grid[GQ], c->grid[GR]},
                 {c->kres[0], c->kres[1], c->kres[2], c->kres[3], c->kres[4], c->kres[5]}};
  Coords cc = {c->coords, c->coords + (g.nx + 4), c->coords + (g.nx + 4) + (g.ny + 4)};
  double *portion = c->partial;
  if (nadd > 0)
    hipLaunchKernelGGL(k_mix_new, dim3(cdiv(nadd, TPB)), dim3(TPB), 0, c->stream, g, c->par,
                       c->cap, norig, c->sorted, nadd, c->list_a, Z, c->flag, mg, cc, portion,
                       c->dsc);
  const int64_t nnode = (int64_t)g.nzn * g.ny * g.nx;
  hipLaunchKernelGGL(k_mix_residual, dim3(cdiv(nnode, TPB)), dim3(TPB), 0, c->stream, g, mg,
                     c->npercell, portion, c->ctouch);
  if (norig > 0)
    hipLaunchKernelGGL(k_mix_absorb, dim3(cdiv(norig, TPB)), dim3(TPB), 0, c->stream, g, c->par,
                       c->cap, norig, c->flag, c->cell, c->ctouch, mg);
  PMPIC_CHECK(hipGetLastError());
  // new count (parcel_mixing.F90:217)
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
  // what k_mix_new raised (nothing else since the last read-back raises anything)
  if (nadd > 0) PMPIC_TRY(sync_scalars(c));
  c->last_removed = Z;
  c->last_added = nadd;
  if (np == norig) {
    // removed slots still marked 0 after placement
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
      hipLaunchKernelGGL(k_mix_backfill, dim3(cdiv(R, TPB)), dim3(TPB), 0, c->stream, c->par,
                         c->cap, dst, R, c->list_b, K1);
      PMPIC_CHECK(hipGetLastError());
      np -= R;
    }
  }
  c->n = np;
  // no parcel removed or added: the binning stands for the next par2grid (else c->sorted holds the
  // sparse cells now)
  if (Z == 0 && nadd == 0) c->bins_n = np;
  return PMPIC_OK;
}

}  // namespace pmpic
