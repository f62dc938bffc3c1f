// Semi-spectral operators and the vort2vel / vorticity_tendency compositions on MI355X.
//
// Reference: model_core/src/fft/fft_ops.F90 (fftops_init :48-168, spectral_filter :176-197,
// diffx :204-302, diffy :305-401, diffz :419-483, laplinv :505-601, tridiagonal :620-656),
// components/vort2vel/src/vort2vel.F90:98-400 and
// components/vorticity_tendency/src/vorticity_tendency.F90:107-334.
//
// The standalone operators (pmpic_diffx ... pmpic_laplinv), the composition of vort2vel and
// vorticity_tendency from the transforms (fft.hip) and the fused column kernel (columns.hip), and
// the grid kernels of vorticity_tendency.  The standalone column solvers walk z with one thread or
// lane group per (kx,ky) column (z slowest in memory, so the walk is coalesced) and keep the
// reference's Thomas recurrence operation for operation (FP32-rounded literal coefficients,
// skipped k^2 = 0 columns).
#include "common.h"

#include <math.h>
#include <type_traits>
#include <vector>

namespace pmpic {

namespace {

constexpr int TPB = 256;

// diffx of element q (fft_ops.F90:266-269, :295): pair swap along x, times kx
__device__ __forceinline__ double dx_at(const double *in, const double *kx, int64_t q, int ii,
                                        int64_t col) {
  return ((ii & 1) == 0 ? (-1. * in[q + 1]) : in[q - 1]) * kx[col];
}
// diffy of element q (fft_ops.F90:366-369, :394)
__device__ __forceinline__ double dy_at(const double *in, const double *ky, int64_t q, int jj,
                                        int sx, int64_t col) {
  return ((jj & 1) == 0 ? (-1. * in[q + sx]) : in[q - sx]) * ky[col];
}

__global__ void k_diffx(Geometry g, const double *__restrict__ in, double *__restrict__ out,
                        const double *__restrict__ kx) {
  const int64_t ssz = (int64_t)g.nzn * g.sy * g.sx;
  int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= ssz) return;
  const int64_t col = q % ((int64_t)g.sy * g.sx);
  const int ii = (int)(q % g.sx);
  out[q] = dx_at(in, kx, q, ii, col);
}

__global__ void k_diffy(Geometry g, const double *__restrict__ in, double *__restrict__ out,
                        const double *__restrict__ ky) {
  const int64_t ssz = (int64_t)g.nzn * g.sy * g.sx;
  int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= ssz) return;
  const int64_t col = q % ((int64_t)g.sy * g.sx);
  const int jj = (int)(col / g.sx);
  out[q] = dy_at(in, ky, q, jj, g.sx, col);
}

// spectral_filter (fft_ops.F90:176-197)
__global__ void k_filter(Geometry g, const double *__restrict__ in, double *__restrict__ out,
                         const double *__restrict__ filt) {
  const int64_t ssz = (int64_t)g.nzn * g.sy * g.sx;
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= ssz) return;
  out[q] = in[q] * filt[q % ((int64_t)g.sy * g.sx)];
}

// Column stage-in with many loads in flight: a chunk of LVL levels is read into registers
// (independent loads, issued back to back) before any is written to the LDS slice.
constexpr int LVL = 16;
__device__ __forceinline__ void column_to_lds(const double *__restrict__ f, int64_t plane, int nz,
                                              double *F, int nc) {
  for (int k0 = 0; k0 < nz; k0 += LVL) {
    double t[LVL];
#pragma unroll
    for (int u = 0; u < LVL; u++)
      if (k0 + u < nz) t[u] = f[(int64_t)(k0 + u) * plane];
#pragma unroll
    for (int u = 0; u < LVL; u++)
      if (k0 + u < nz) F[(k0 + u) * nc] = t[u];
  }
}

// Column solvers.  One thread owns one (kx,ky) column and runs the reference's Thomas
// recurrence on it.  The column (and the elimination coefficients cp) sit either in HBM
// (stride = one spectral plane) or, when they fit, in an LDS slice private to the thread
// (stride = threads per block): the whole column is loaded with independent coalesced reads,
// solved in LDS, and stored back, so the level-by-level recurrence never waits on HBM.  Both
// forms run the same arithmetic.
template <typename T>
struct Col {
  T *p;
  int64_t s;
  __device__ __forceinline__ T &operator[](int k) const { return p[(int64_t)k * s]; }
};

// laplinv (fft_ops.F90:505-601) of one column, in place.  The right-hand side of row k reads
// the original f(k-1), f(k), f(k+1); a sliding window keeps the originals while the forward
// sweep overwrites f with d'.  Returns PMPIC_ERR_ZERO_PIVOT on a zero pivot.
template <typename CF, typename CC>
__device__ __forceinline__ int laplinv_column(const Geometry &g, CF F, CC CP, double k2, int df0) {
  const int nz = g.nzn;
  const double f16 = (double)(1.f / 6.f), f13 = (double)(1.f / 3.f);
  const double f112 = (double)(1.f / 12.f), f56 = (double)(5.f / 6.f);
  const double dz = g.dz;
  const double i2dz2 = 2. / dz / dz, idz2 = 1. / dz / dz;
  // interior coefficients (constant along the column)
  const double ai = idz2 - f112 * k2, bi = -i2dz2 - f56 * k2, ci = idz2 - f112 * k2;
  double fm = 0.0, f0 = F[0], fp = F[1];  // originals f(k-1), f(k), f(k+1)
  // row 1
  double b1, c1, d1;
  if (!df0) { b1 = 1.; c1 = 0.; d1 = 0.; }
  else { b1 = -idz2 - f13 * k2; c1 = idz2 - f16 * k2; d1 = f13 * f0 + f16 * fp; }
  double denominator = b1;
  double fprev = d1 / denominator;
  F[0] = fprev;
  double cprev = c1;  // c(i-1)
#pragma unroll 4
  for (int k = 2; k <= nz; k++) {
    fm = f0;
    f0 = fp;
    fp = (k < nz) ? F[k] : 0.0;
    double a, b, c, d;
    if (k < nz) {
      a = ai; b = bi; c = ci;
      d = f112 * fm + f56 * f0 + f112 * fp;
    } else if (!df0) {
      a = 0.; b = 1.; c = 0.; d = 0.;
    } else {
      a = idz2 - f16 * k2; b = -idz2 - f13 * k2; c = 0.;
      d = f13 * f0 + f16 * fm;
    }
    const double cpk = cprev / denominator;
    CP[k - 1] = cpk;
    denominator = b - a * cpk;
    if (denominator == 0) return PMPIC_ERR_ZERO_PIVOT;
    fprev = (d - a * fprev) / (denominator);
    F[k - 1] = fprev;
    cprev = c;
  }
  double fnext = fprev;
#pragma unroll 4
  for (int k = nz - 1; k >= 1; k--) {
    const double v = F[k - 1] - CP[k] * fnext;
    F[k - 1] = v;
    fnext = v;
  }
  return PMPIC_OK;
}

// diffz (fft_ops.F90:419-483) of one column; O may alias F (the original f(k-2), f(k-1) are
// kept in registers, and f(k) is read before d'(k-1) is written).
template <typename CI, typename CO, typename CC>
__device__ __forceinline__ int diffz_column(const Geometry &g, CI F, CO O, CC CP, bool bt,
                                            double bot, double top) {
  const int nz = g.nzn;
  const double a1 = (double)(1.f / 6.f), b1 = (double)(2.f / 3.f), c1 = (double)(1.f / 6.f);
  const double al = (double)(1.f / 3.f), cl = (double)(1.f / 3.f);
  const double dz = g.dz;
  double fkm2 = F[0], fkm1 = F[1];  // f(k-2), f(k-1) of the next row
  // row 1
  double d = bt ? fkm1 / dz - a1 * bot * dz : 0.0;
  double denominator = 1.;  // b(1) = b0
  double fprev = d / denominator;
  O[0] = fprev;
  double cprev = bt ? cl : 0.;  // c(1)
#pragma unroll 4
  for (int k = 2; k <= nz; k++) {
    double a, b, c, fk = 0.0;
    if (k < nz) {
      a = a1; b = b1; c = c1;
      fk = F[k];
      d = (fk - fkm2) / 2. / dz;
    } else {
      a = bt ? al : 0.; b = 1.; c = 0.;
      d = bt ? -fkm2 / dz + a1 * top * dz : 0.0;
    }
    const double cpk = cprev / denominator;
    CP[k - 1] = cpk;
    denominator = b - a * cpk;
    if (denominator == 0) return PMPIC_ERR_ZERO_PIVOT;
    fprev = (d - a * fprev) / (denominator);
    O[k - 1] = fprev;
    cprev = c;
    fkm2 = fkm1;
    fkm1 = fk;
  }
  double fnext = fprev;
#pragma unroll 4
  for (int k = nz - 1; k >= 1; k--) {
    const double v = O[k - 1] - CP[k] * fnext;
    O[k - 1] = v;
    fnext = v;
  }
  return PMPIC_OK;
}

struct ColField {
  const double *in;
  double *out;
  const double *bot, *top;
  int df0;
};

__global__ void k_laplinv(Geometry g, ColField cf, double *__restrict__ cp,
                          const double *__restrict__ k2a, DevScalars *sc) {
  const int64_t plane = (int64_t)g.sy * g.sx;
  const int64_t col = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (col >= plane) return;
  const double k2 = k2a[col];
  if (k2 == 0) return;
  Col<double> F{cf.out + col, plane};
  Col<double> CP{cp + col, plane};
  const int st = laplinv_column(g, F, CP, k2, cf.df0);
  if (st != PMPIC_OK) raise_status(sc, st);
}

__global__ void __launch_bounds__(64) k_laplinv_lds(Geometry g, ColField cf,
                                                    const double *__restrict__ k2a,
                                                    DevScalars *sc) {
  extern __shared__ double sh[];
  const int nc = blockDim.x, t = threadIdx.x, nz = g.nzn;
  const int64_t plane = (int64_t)g.sy * g.sx;
  const int64_t col = (int64_t)blockIdx.x * nc + t;
  if (col >= plane) return;  // no barriers below: each thread touches only its own slice
  const double k2 = k2a[col];
  if (k2 == 0) return;
  double *f = cf.out + col;
  Col<double> F{sh + t, nc}, CP{sh + (int64_t)nz * nc + t, nc};
  column_to_lds(f, plane, nz, sh + t, nc);
  const int st = laplinv_column(g, F, CP, k2, cf.df0);
  if (st != PMPIC_OK) {
    raise_status(sc, st);
    return;
  }
#pragma unroll 8
  for (int k = 0; k < nz; k++) f[(int64_t)k * plane] = F[k];
}

__global__ void k_diffz(Geometry g, ColField cf, double *__restrict__ cp, DevScalars *sc) {
  const int64_t plane = (int64_t)g.sy * g.sx;
  const int64_t col = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (col >= plane) return;
  const bool bt = cf.bot != nullptr && cf.top != nullptr;
  Col<const double> F{cf.in + col, plane};
  Col<double> O{cf.out + col, plane};
  Col<double> CP{cp + col, plane};
  const int st = diffz_column(g, F, O, CP, bt, bt ? cf.bot[col] : 0.0,
                              bt ? cf.top[col] : 0.0);
  if (st != PMPIC_OK) raise_status(sc, st);
}

__global__ void __launch_bounds__(64) k_diffz_lds(Geometry g, ColField cf, DevScalars *sc) {
  extern __shared__ double sh[];
  const int nc = blockDim.x, t = threadIdx.x, nz = g.nzn;
  const int64_t plane = (int64_t)g.sy * g.sx;
  const int64_t col = (int64_t)blockIdx.x * nc + t;
  if (col >= plane) return;  // no barriers below: each thread touches only its own slice
  const bool bt = cf.bot != nullptr && cf.top != nullptr;
  const double *f = cf.in + col;
  double *o = cf.out + col;
  Col<double> F{sh + t, nc}, CP{sh + (int64_t)nz * nc + t, nc};
  column_to_lds(f, plane, nz, sh + t, nc);
  const int st = diffz_column(g, F, F, CP, bt, bt ? cf.bot[col] : 0.0,
                              bt ? cf.top[col] : 0.0);
  if (st != PMPIC_OK) {
    raise_status(sc, st);
    return;
  }
#pragma unroll 8
  for (int k = 0; k < nz; k++) o[(int64_t)k * plane] = F[k];
}

// Register-resident column solvers: the column stays in registers (NZ levels, unrolled) and
// the level-by-level recurrence never waits on memory.  diffz's Thomas denominators and c' are
// the same for every column, so they are built once (k_dz_tables, with the same operations as
// diffz_column) and each call runs only the data recurrence.  laplinv's depend on the column's
// k^2: they are computed alongside the data recurrence (an independent chain).  Results are
// bit-identical to the LDS and HBM forms.
__global__ void k_dz_tables(Geometry g, double *__restrict__ den, double *__restrict__ cp) {
  if (threadIdx.x || blockIdx.x) return;
  const int nz = g.nzn;
  const double a1 = (double)(1.f / 6.f), b1 = (double)(2.f / 3.f), c1 = (double)(1.f / 6.f);
  const double al = (double)(1.f / 3.f), cl = (double)(1.f / 3.f);
  for (int bt = 0; bt < 2; bt++) {
    double *D = den + bt * nz, *C = cp + bt * nz;
    double denominator = 1.;
    D[0] = denominator;
    C[0] = 0.;
    double cprev = bt ? cl : 0.;
    for (int k = 2; k <= nz; k++) {
      double a, b, c;
      if (k < nz) { a = a1; b = b1; c = c1; }
      else { a = bt ? al : 0.; b = 1.; c = 0.; }
      const double cpk = cprev / denominator;
      C[k - 1] = cpk;
      denominator = b - a * cpk;
      D[k - 1] = denominator;
      cprev = c;
    }
  }
}

// laplinv with Q lanes per column (1, 2 or 4): lane q * CPW + c holds levels [q L, q L + L) of
// column c of the wavefront's CPW = 64 / Q, both the column values and the forward sweep's c',
// in registers.  The sweeps run lane group after lane group (the others masked), the recurrence
// state crossing to the next group by a lane shuffle, so no level waits on memory and every
// operation is the one of laplinv_column in the same order: results are bit-identical.  A zero
// pivot is flagged and raised after the sweeps (the reference stops there; the column's values
// are then moot).
template <int Q, int NZ>
__global__ void __launch_bounds__(64) k_laplinv_reg(Geometry g, ColField cf,
                                                    const double *__restrict__ k2a,
                                                    DevScalars *sc) {
  static_assert(Q == 1 || Q == 2 || Q == 4, "one, two or four lanes per column");
  constexpr int CPW = 64 / Q;  // columns per wavefront
  constexpr int L = (NZ + Q - 1) / Q;
  const int lane = threadIdx.x;
  const int q = lane / CPW;
  const int64_t plane = (int64_t)g.sy * g.sx;
  const int64_t col = (int64_t)blockIdx.x * CPW + (lane % CPW);
  if (col >= plane) return;
  const double k2 = k2a[col];
  if (k2 == 0) return;
  const int df0 = cf.df0;
  double *f = cf.out + col;
  double F[L], CPl[L];
#pragma unroll
  for (int i = 0; i < L; i++) {
    F[i] = 0.0;
    CPl[i] = 0.0;
  }
#pragma unroll
  for (int i = 0; i < L; i++)
    if (q * L + i < NZ) F[i] = f[(int64_t)(q * L + i) * plane];
  const double f16 = (double)(1.f / 6.f), f13 = (double)(1.f / 3.f);
  const double f112 = (double)(1.f / 12.f), f56 = (double)(5.f / 6.f);
  const double dz = g.dz;
  const double i2dz2 = 2. / dz / dz, idz2 = 1. / dz / dz;
  const double ai = idz2 - f112 * k2, bi = -i2dz2 - f56 * k2, ci = idz2 - f112 * k2;
  // the original of level q L + L, the next group's first (unused with one lane per column)
  const double nxt0 = __shfl(F[0], (lane + CPW) & 63);
  constexpr int PTOP = (NZ - 1) / L;  // group holding level NZ - 1
  double denominator = 0.0, fprev = 0.0, cprev = 0.0, f0 = 0.0, fp = 0.0;
  bool bad = false;
#pragma unroll
  for (int p = 0; p <= PTOP; p++) {
    if (p > 0) {
      denominator = __shfl(denominator, lane - CPW);
      fprev = __shfl(fprev, lane - CPW);
      cprev = __shfl(cprev, lane - CPW);
      f0 = __shfl(f0, lane - CPW);
      fp = __shfl(fp, lane - CPW);
    }
    if (q == p) {
#pragma unroll
      for (int i = 0; i < L; i++) {
        const int j = p * L + i;  // level (0-based); row j + 1 of the reference
        if (j >= NZ) break;
        const double onext = (i + 1 < L) ? F[i + 1 < L ? i + 1 : 0] : nxt0;  // original j + 1
        if (j == 0) {
          f0 = F[0];
          fp = onext;
          double b1, c1, d1;
          if (!df0) { b1 = 1.; c1 = 0.; d1 = 0.; }
          else { b1 = -idz2 - f13 * k2; c1 = idz2 - f16 * k2; d1 = f13 * f0 + f16 * fp; }
          denominator = b1;
          fprev = d1 / denominator;
          F[0] = fprev;
          cprev = c1;
          continue;
        }
        const double fm = f0;
        f0 = fp;
        fp = (j + 1 < NZ) ? onext : 0.0;
        double a, b, c, d;
        if (j + 1 < NZ) {
          a = ai; b = bi; c = ci;
          d = f112 * fm + f56 * f0 + f112 * fp;
        } else if (!df0) {
          a = 0.; b = 1.; c = 0.; d = 0.;
        } else {
          a = idz2 - f16 * k2; b = -idz2 - f13 * k2; c = 0.;
          d = f13 * f0 + f16 * fm;
        }
        const double cpk = cprev / denominator;
        CPl[i] = cpk;
        denominator = b - a * cpk;
        bad |= (denominator == 0);
        fprev = (d - a * fprev) / (denominator);
        F[i] = fprev;
        cprev = c;
      }
    }
  }
  // backward sweep from the top group down: level j takes c' of level j + 1
  const double cpn = __shfl(CPl[0], (lane + CPW) & 63);
  double fnext = fprev;
#pragma unroll
  for (int p = PTOP; p >= 0; p--) {
    if (p < PTOP) fnext = __shfl(fnext, lane + CPW);
    if (q == p) {
#pragma unroll
      for (int i = L - 1; i >= 0; i--) {
        const int j = p * L + i;
        if (j >= NZ - 1) continue;
        const double cpj1 = (i + 1 < L) ? CPl[i + 1 < L ? i + 1 : 0] : cpn;
        const double v = F[i] - cpj1 * fnext;
        F[i] = v;
        fnext = v;
      }
    }
  }
  if (bad) raise_status(sc, PMPIC_ERR_ZERO_PIVOT);
#pragma unroll
  for (int i = 0; i < L; i++)
    if (q * L + i < NZ) f[(int64_t)(q * L + i) * plane] = F[i];
}

template <int NZ>
__global__ void __launch_bounds__(64) k_diffz_reg(Geometry g, ColField cf,
                                                  const double *__restrict__ tden,
                                                  const double *__restrict__ tcp,
                                                  DevScalars *sc) {
  // the Thomas tables are the same for every column: staged once per block in LDS, so the
  // recurrence reads them without a memory round trip per level
  __shared__ double den[NZ], cpt[NZ];
  const int64_t plane = (int64_t)g.sy * g.sx;
  const int64_t col = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const bool bt = cf.bot != nullptr && cf.top != nullptr;
  for (int k = threadIdx.x; k < NZ; k += blockDim.x) {
    const double dn = tden[(bt ? NZ : 0) + k];
    den[k] = dn;
    cpt[k] = tcp[(bt ? NZ : 0) + k];
  }
  __syncthreads();
  if (col >= plane) return;
  const double *fin = cf.in + col;
  double *o = cf.out + col;
  double F[NZ];
#pragma unroll
  for (int k = 0; k < NZ; k++) F[k] = fin[(int64_t)k * plane];
  const double bot = bt ? cf.bot[col] : 0.0, top = bt ? cf.top[col] : 0.0;
  const double a1 = (double)(1.f / 6.f), al = (double)(1.f / 3.f);
  const double dz = g.dz;
  double fkm2 = F[0], fkm1 = F[1];  // originals f(k-2), f(k-1) of the next row
  const double d0 = bt ? (fkm1 / dz) - a1 * bot * dz : 0.0;
  double fprev = d0 / den[0];
  F[0] = fprev;
#pragma unroll
  for (int k = 2; k <= NZ; k++) {
    double a, d, fk = 0.0;
    if (k < NZ) {
      a = a1;
      fk = F[k < NZ ? k : 0];
      d = (fk - fkm2) / 2. / dz;
    } else {
      a = bt ? al : 0.;
      d = bt ? (-fkm2 / dz) + a1 * top * dz : 0.0;
    }
    const double dn = den[k - 1];
    if (dn == 0) { raise_status(sc, PMPIC_ERR_ZERO_PIVOT); return; }
    fprev = (d - a * fprev) / (dn);
    F[k - 1] = fprev;
    fkm2 = fkm1;
    fkm1 = fk;
  }
  double fnext = fprev;
#pragma unroll
  for (int k = NZ - 1; k >= 1; k--) {
    const double v = F[k - 1] - cpt[k] * fnext;
    F[k - 1] = v;
    fnext = v;
  }
#pragma unroll
  for (int k = 0; k < NZ; k++) o[(int64_t)k * plane] = F[k];
}

// Long columns (more z nodes than the instances above): Q lanes per column, lane q holding
// levels [q L, q L + L) of the column in registers, for any column length nz <= Q L chosen at
// run time.  The sweeps run lane group after lane group as in k_laplinv_reg, the recurrence
// state crossing by lane shuffles, every operation the one of laplinv_column / k_diffz_reg in
// the same order, so results are bit-identical to them.
template <int Q, int L>
__global__ void __launch_bounds__(64) k_laplinv_qn(Geometry g, ColField cf,
                                                   const double *__restrict__ k2a,
                                                   DevScalars *sc) {
  constexpr int CPW = 64 / Q;  // columns per wavefront
  const int NZ = g.nzn;
  const int lane = threadIdx.x;
  const int q = lane / CPW;
  const int64_t plane = (int64_t)g.sy * g.sx;
  const int64_t col = (int64_t)blockIdx.x * CPW + (lane % CPW);
  if (col >= plane) return;  // all Q lanes of a column leave together
  const double k2 = k2a[col];
  if (k2 == 0) return;
  const int df0 = cf.df0;
  double *f = cf.out + col;
  double F[L], CPl[L];
#pragma unroll
  for (int i = 0; i < L; i++) {
    F[i] = 0.0;
    CPl[i] = 0.0;
  }
#pragma unroll
  for (int i = 0; i < L; i++)
    if (q * L + i < NZ) F[i] = f[(int64_t)(q * L + i) * plane];
  const double f16 = (double)(1.f / 6.f), f13 = (double)(1.f / 3.f);
  const double f112 = (double)(1.f / 12.f), f56 = (double)(5.f / 6.f);
  const double dz = g.dz;
  const double i2dz2 = 2. / dz / dz, idz2 = 1. / dz / dz;
  const double ai = idz2 - f112 * k2, bi = -i2dz2 - f56 * k2, ci = idz2 - f112 * k2;
  const double nxt0 = __shfl(F[0], lane + CPW);  // the next group's first original
  const int PTOP = (NZ - 1) / L;                         // group holding level NZ - 1
  double denominator = 0.0, fprev = 0.0, cprev = 0.0, f0 = 0.0, fp = 0.0;
  bool bad = false;
  for (int p = 0; p <= PTOP; p++) {
    if (p > 0) {
      denominator = __shfl(denominator, lane - CPW);
      fprev = __shfl(fprev, lane - CPW);
      cprev = __shfl(cprev, lane - CPW);
      f0 = __shfl(f0, lane - CPW);
      fp = __shfl(fp, lane - CPW);
    }
    if (q == p) {
#pragma unroll
      for (int i = 0; i < L; i++) {
        const int j = p * L + i;
        if (j >= NZ) break;
        const double onext = (i + 1 < L) ? F[i + 1 < L ? i + 1 : 0] : nxt0;
        if (j == 0) {
          f0 = F[0];
          fp = onext;
          double b1, c1, d1;
          if (!df0) { b1 = 1.; c1 = 0.; d1 = 0.; }
          else { b1 = -idz2 - f13 * k2; c1 = idz2 - f16 * k2; d1 = f13 * f0 + f16 * fp; }
          denominator = b1;
          fprev = d1 / denominator;
          F[0] = fprev;
          cprev = c1;
          continue;
        }
        const double fm = f0;
        f0 = fp;
        fp = (j + 1 < NZ) ? onext : 0.0;
        double a, b, c, d;
        if (j + 1 < NZ) {
          a = ai; b = bi; c = ci;
          d = f112 * fm + f56 * f0 + f112 * fp;
        } else if (!df0) {
          a = 0.; b = 1.; c = 0.; d = 0.;
        } else {
          a = idz2 - f16 * k2; b = -idz2 - f13 * k2; c = 0.;
          d = f13 * f0 + f16 * fm;
        }
        const double cpk = cprev / denominator;
        CPl[i] = cpk;
        denominator = b - a * cpk;
        bad |= (denominator == 0);
        fprev = (d - a * fprev) / (denominator);
        F[i] = fprev;
        cprev = c;
      }
    }
  }
  const double cpn = __shfl(CPl[0], lane + CPW);
  double fnext = fprev;
  for (int p = PTOP; p >= 0; p--) {
    if (p < PTOP) fnext = __shfl(fnext, lane + CPW);
    if (q == p) {
#pragma unroll
      for (int i = L - 1; i >= 0; i--) {
        const int j = p * L + i;
        if (j >= NZ - 1) continue;
        const double cpj1 = (i + 1 < L) ? CPl[i + 1 < L ? i + 1 : 0] : cpn;
        const double v = F[i] - cpj1 * fnext;
        F[i] = v;
        fnext = v;
      }
    }
  }
  if (bad) raise_status(sc, PMPIC_ERR_ZERO_PIVOT);
#pragma unroll
  for (int i = 0; i < L; i++)
    if (q * L + i < NZ) f[(int64_t)(q * L + i) * plane] = F[i];
}

template <int Q, int L>
__global__ void __launch_bounds__(64) k_diffz_qn(Geometry g, ColField cf,
                                                 const double *__restrict__ tden,
                                                 const double *__restrict__ tcp,
                                                 DevScalars *sc) {
  constexpr int CPW = 64 / Q;
  __shared__ double den[Q * L], cpt[Q * L];
  const int NZ = g.nzn;
  const int lane = threadIdx.x;
  const int q = lane / CPW;
  const int64_t plane = (int64_t)g.sy * g.sx;
  const int64_t col = (int64_t)blockIdx.x * CPW + (lane % CPW);
  const bool bt = cf.bot != nullptr && cf.top != nullptr;
  for (int k = threadIdx.x; k < NZ; k += blockDim.x) {
    const double dn = tden[(bt ? NZ : 0) + k];
    den[k] = dn;
    cpt[k] = tcp[(bt ? NZ : 0) + k];
  }
  __syncthreads();
  if (col >= plane) return;  // all Q lanes of a column leave together
  const double *fin = cf.in + col;
  double *o = cf.out + col;
  double F[L];
#pragma unroll
  for (int i = 0; i < L; i++) F[i] = (q * L + i < NZ) ? fin[(int64_t)(q * L + i) * plane] : 0.0;
  const double bot = bt ? cf.bot[col] : 0.0, top = bt ? cf.top[col] : 0.0;
  const double a1 = (double)(1.f / 6.f), al = (double)(1.f / 3.f);
  const double dz = g.dz;
  const double nxt0 = __shfl(F[0], lane + CPW);  // the original of the next group's first level
  const int PTOP = (NZ - 1) / L;
  double fprev = 0.0, fkm2 = 0.0, fkm1 = 0.0;  // originals f(k-2), f(k-1) of the next row
  bool bad = false;
  for (int p = 0; p <= PTOP; p++) {
    if (p > 0) {
      fprev = __shfl(fprev, lane - CPW);
      fkm2 = __shfl(fkm2, lane - CPW);
      fkm1 = __shfl(fkm1, lane - CPW);
    }
    if (q == p) {
#pragma unroll
      for (int i = 0; i < L; i++) {
        const int j = p * L + i;  // level written: row j + 1 of the reference
        if (j >= NZ) break;
        const double onext = (i + 1 < L) ? F[i + 1 < L ? i + 1 : 0] : nxt0;  // original j + 1
        if (j == 0) {
          fkm2 = F[0];
          fkm1 = onext;
          const double d0 = bt ? (fkm1 / dz) - a1 * bot * dz : 0.0;
          bad |= (den[0] == 0);
          fprev = d0 / den[0];
          F[0] = fprev;
          continue;
        }
        double a, d, fk = 0.0;
        if (j + 1 < NZ) {
          a = a1;
          fk = onext;
          d = (fk - fkm2) / 2. / dz;
        } else {
          a = bt ? al : 0.;
          d = bt ? (-fkm2 / dz) + a1 * top * dz : 0.0;
        }
        const double dn = den[j];
        bad |= (dn == 0);
        fprev = (d - a * fprev) / (dn);
        F[i] = fprev;
        fkm2 = fkm1;
        fkm1 = fk;
      }
    }
  }
  double fnext = fprev;
  for (int p = PTOP; p >= 0; p--) {
    if (p < PTOP) fnext = __shfl(fnext, lane + CPW);
    if (q == p) {
#pragma unroll
      for (int i = L - 1; i >= 0; i--) {
        const int j = p * L + i;
        if (j >= NZ - 1) continue;
        const double v = F[i] - cpt[j + 1] * fnext;
        F[i] = v;
        fnext = v;
      }
    }
  }
  if (bad) raise_status(sc, PMPIC_ERR_ZERO_PIVOT);
#pragma unroll
  for (int i = 0; i < L; i++)
    if (q * L + i < NZ) o[(int64_t)(q * L + i) * plane] = F[i];
}

// a node's record (common.h)
__device__ __forceinline__ void put_record(double2 *rec, int64_t t, double u, double v, double w,
                                           double dp, double dq, double dr) {
  rec[3 * t] = make_double2(u, v);
  rec[3 * t + 1] = make_double2(w, dp);
  rec[3 * t + 2] = make_double2(dq, dr);
}
__device__ __forceinline__ void put_record(float4 *rec, int64_t t, float u, float v, float w,
                                           double dp, double dq, double dr) {
  rec[2 * t] = make_float4(u, v, w, (float)dp);
  rec[2 * t + 1] = make_float4((float)dq, (float)dr, 0.f, 0.f);
}

// the block's maxima, one value per block and quantity; k_max4_final reduces them (no contended
// atomics)
__device__ __forceinline__ void block_max4(const double m[4], double *__restrict__ blkmax) {
  __shared__ double sm[4][TPB];
  for (int f = 0; f < 4; f++) sm[f][threadIdx.x] = m[f];
  __syncthreads();
  for (int s = blockDim.x / 2; s > 0; s >>= 1) {
    if (threadIdx.x < s)
      for (int f = 0; f < 4; f++) sm[f][threadIdx.x] = fmax(sm[f][threadIdx.x], sm[f][threadIdx.x + s]);
    __syncthreads();
  }
  if (threadIdx.x == 0)
    for (int f = 0; f < 4; f++) blkmax[(int64_t)f * gridDim.x + blockIdx.x] = sm[f][0];
}

// vorticity_tendency.F90:169-265, physical interior, accumulation order as written, and the node
// records of the RK stage's gathers.
// T: the type of the grids (FP64, or FP32 in the FP32-bulk form, widened exactly); the products
// are formed in FP64 in both forms.  Bound by memory (14 grids read, a record written).
// blkmax (may be null): the block's maxima for the timestep as well, of the grids that it reads.
template <typename T, typename REC>
__global__ void k_tendency(int64_t nnode, const T *__restrict__ P, const T *__restrict__ Q,
                           const T *__restrict__ R, const T *__restrict__ dbdy,
                           const T *__restrict__ dudx, const T *__restrict__ dudy,
                           const T *__restrict__ dwdx, const T *__restrict__ dbdx,
                           const T *__restrict__ dvdx, const T *__restrict__ dvdy,
                           const T *__restrict__ dwdy, const T *__restrict__ U,
                           const T *__restrict__ V, const T *__restrict__ W,
                           REC *__restrict__ rec, double *__restrict__ blkmax) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= nnode && !blkmax) return;
  const int64_t q = min(t, nnode - 1);  // past the end the last node again: the same record
  const double p = P[q], qq = Q[q], r = R[q];
  double dp = dbdy[q];
  dp = dp + p * (double)dudx[q];
  dp = dp + qq * (double)dudy[q];
  dp = dp + r * (qq + (double)dwdx[q]);
  double dq = dbdx[q];
  dq = -dq + p * (double)dvdx[q];
  dq = dq + qq * (double)dvdy[q];
  dq = dq + r * (-p + (double)dwdy[q]);
  double dr = p * (double)dwdx[q];
  dr = dr + qq * (double)dwdy[q];
  dr = dr + r * (-(double)dudx[q]);
  dr = dr + r * (-(double)dvdy[q]);
  const double u = U[q], v = V[q], w = W[q];
  put_record(rec, q, u, v, w, dp, dq, dr);
  if (blkmax) {
    const double m[4] = {u * u, v * v, w * w, p * p + qq * qq + r * r};
    block_max4(m, blkmax);
  }
}

// newer velocities into the records (vort2vel called again without vorticity_tendency)
__global__ void k_record_velocity(int64_t nnode, const double *__restrict__ U,
                                  const double *__restrict__ V, const double *__restrict__ W,
                                  double2 *__restrict__ rec) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= nnode) return;
  rec[3 * q] = make_double2(U[q], V[q]);
  rec[3 * q + 1].x = W[q];
}
__global__ void k_record_velocity32(int64_t nnode, const float *__restrict__ U,
                                    const float *__restrict__ V, const float *__restrict__ W,
                                    float4 *__restrict__ rec) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= nnode) return;
  rec[2 * q] = make_float4(U[q], V[q], W[q], rec[2 * q].w);
}

// maxima of u^2, v^2, w^2 and p^2+q^2+r^2 over the interior (vort2vel.F90:331-337,
// vorticity_tendency.F90:279-282), per block; a maximum is exact in any order, so the result
// is deterministic.
// TU: the grids' type (double, or float for the FP32-bulk form's grids)
template <typename TU>
__global__ void k_max4(int64_t nnode, const TU *__restrict__ U, const TU *__restrict__ V,
                       const TU *__restrict__ W, const TU *__restrict__ P,
                       const TU *__restrict__ Q, const TU *__restrict__ R,
                       double *__restrict__ blkmax) {
  double m[4] = {0, 0, 0, 0};
  // MPT nodes per pass, their loads issued together; an index past the end is clamped to the
  // last node, which the maximum tolerates
  constexpr int MPT = 4;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t q0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q0 < nnode;
       q0 += MPT * stride) {
    double u[MPT], v[MPT], w[MPT], pp[MPT], qq[MPT], rr[MPT];  // velocities widened exactly
#pragma unroll
    for (int k = 0; k < MPT; k++) {
      const int64_t q = min(q0 + k * stride, nnode - 1);
      u[k] = U[q]; v[k] = V[q]; w[k] = W[q];
      pp[k] = P[q]; qq[k] = Q[q]; rr[k] = R[q];
    }
#pragma unroll
    for (int k = 0; k < MPT; k++) {
      const double o = pp[k] * pp[k] + qq[k] * qq[k] + rr[k] * rr[k];
      m[0] = fmax(m[0], u[k] * u[k]);
      m[1] = fmax(m[1], v[k] * v[k]);
      m[2] = fmax(m[2], w[k] * w[k]);
      m[3] = fmax(m[3], o);
    }
  }
  block_max4(m, blkmax);
}

// timestep selection at RK stage 1: vort2vel.F90:329-381 then vorticity_tendency.F90:277-321
__device__ __forceinline__ void select_dt(const Geometry &g, DevScalars *sc) {
  double umax = sqrt(sc->umax2), vmax = sqrt(sc->vmax2), wmax = sqrt(sc->wmax2);
  const double tiny = (double)1.E-15f;
  if (umax == 0) umax = tiny;
  if (vmax == 0) vmax = tiny;
  if (wmax == 0) wmax = tiny;
  const double t1 = g.lx_cfl / umax, t2 = g.ly_cfl / vmax, t3 = g.lz_cfl / wmax;
  double dtmaxg = t1;
  if (t2 < dtmaxg) dtmaxg = t2;
  if (t3 < dtmaxg) dtmaxg = t3;
  double dtm = (sc->dtmax > dtmaxg) ? dtmaxg : sc->dtmax;
  const double omax = sqrt(sc->omax2);
  double dtv;
  if (omax > 0.) dtv = sc->prefactor / omax;
  else dtv = sc->dtmax;
  if (dtm > dtv) dtm = dtv;
  sc->dtm = dtm;
}

// the maxima over the nb blocks (one workgroup), a maximum being exact in any order, and the
// timestep from them
__global__ void k_max4_final(Geometry g, int nb, const double *__restrict__ blkmax,
                             DevScalars *sc) {
  __shared__ double sm[4][TPB];
  double m[4] = {0, 0, 0, 0};
  for (int i = threadIdx.x; i < nb; i += blockDim.x)
#pragma unroll
    for (int f = 0; f < 4; f++) m[f] = fmax(m[f], blkmax[(int64_t)f * nb + i]);
  for (int f = 0; f < 4; f++) sm[f][threadIdx.x] = m[f];
  __syncthreads();
  for (int s = blockDim.x / 2; s > 0; s >>= 1) {
    if (threadIdx.x < s)
      for (int f = 0; f < 4; f++) sm[f][threadIdx.x] = fmax(sm[f][threadIdx.x], sm[f][threadIdx.x + s]);
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    sc->umax2 = sm[0][0];
    sc->vmax2 = sm[1][0];
    sc->wmax2 = sm[2][0];
    sc->omax2 = sm[3][0];
    select_dt(g, sc);
  }
}

inline int64_t ssz_of(const Geometry &g) { return (int64_t)g.nzn * g.sy * g.sx; }
inline int64_t plane_of(const Geometry &g) { return (int64_t)g.sy * g.sx; }

}  // namespace

// wavenumbers and 2/3-rule filter, fft_ops.F90:111-139 on one rank (x_start = y_start = 1)
int spectral_setup(Ctx *c) {
  const Geometry &g = c->g;
  const int sx = g.sx, sy = g.sy;
  std::vector<double> kx(sx * sy), ky(sx * sy), k2(sx * sy), fl(sx * sy);
  const double twopi = 8.0 * atan(1.0);
  const double lx = g.dx * (double)g.nx, ly = g.dy * (double)g.ny;
  const double hx = (double)((float)g.nx / 2.0f), hy = (double)((float)g.ny / 2.0f);
  double ksqmax = (hx / lx) * (hx / lx) + (hy / ly) * (hy / ly);
  ksqmax = ksqmax * 2. / 9.;
  for (int jj = 0; jj < sy; jj++)
    for (int ii = 0; ii < sx; ii++) {
      const double xval = (double)(ii / 2) / lx;
      const double yval = (double)(jj / 2) / ly;
      const double kk = xval * xval + yval * yval;
      const int q = jj * sx + ii;
      fl[q] = (kk > ksqmax) ? 0. : 1.;
      kx[q] = xval * twopi;
      ky[q] = yval * twopi;
      k2[q] = kk * twopi * twopi;
    }
  const size_t b = sizeof(double) * sx * sy;
  PMPIC_CHECK(hipMemcpy(c->kx, kx.data(), b, hipMemcpyHostToDevice));
  PMPIC_CHECK(hipMemcpy(c->ky, ky.data(), b, hipMemcpyHostToDevice));
  PMPIC_CHECK(hipMemcpy(c->k2, k2.data(), b, hipMemcpyHostToDevice));
  PMPIC_CHECK(hipMemcpy(c->filt, fl.data(), b, hipMemcpyHostToDevice));
  std::vector<int> lcut(sy / 2, 0);
  c->mcut = 0;
  for (int m = 0; m < sy / 2; m++)
    for (int l = 0; l < sx / 2; l++)
      if (fl[(2 * m) * sx + 2 * l] != 0.) {
        lcut[m] = l + 1;
        c->mcut = m + 1;
      }
  PMPIC_CHECK(hipMemcpy(c->lcut, lcut.data(), sizeof(int) * lcut.size(), hipMemcpyHostToDevice));
  hipLaunchKernelGGL(k_dz_tables, dim3(1), dim3(1), 0, c->stream, g, c->dz_den, c->dz_cp);
  PMPIC_CHECK(hipGetLastError());
  PMPIC_CHECK(hipStreamSynchronize(c->stream));
  return PMPIC_OK;
}

int op_diffx(Ctx *c, const double *in, double *out) {
  hipLaunchKernelGGL(k_diffx, dim3(cdiv(ssz_of(c->g), TPB)), dim3(TPB), 0, c->stream, c->g, in,
                     out, c->kx);
  PMPIC_CHECK(hipGetLastError());
  return PMPIC_OK;
}
int op_diffy(Ctx *c, const double *in, double *out) {
  hipLaunchKernelGGL(k_diffy, dim3(cdiv(ssz_of(c->g), TPB)), dim3(TPB), 0, c->stream, c->g, in,
                     out, c->ky);
  PMPIC_CHECK(hipGetLastError());
  return PMPIC_OK;
}
// threads per block of the LDS column kernels: the most columns (64 down to 8) whose two
// slices (f and cp) fit in 64 KiB of LDS; 0 = columns too long, solve straight from HBM
static int lds_cols(const Geometry &g) {
  for (int nc = 64; nc >= 8; nc /= 2)
    if (2 * (int64_t)nc * g.nzn * (int64_t)sizeof(double) <= 65536) return nc;
  return 0;
}

// column lengths (z nodes) with a register-resident solver instance
#define PMPIC_REG_COLUMNS(X) X(9) X(17) X(33) X(65) X(129)
// lanes per column of the register-resident laplinv
constexpr int LAP_Q = 4;
// longer columns, up to LONG_Q * LONG_L z nodes: LONG_Q lanes per column, LONG_L levels each
constexpr int LONG_Q = 8, LONG_L = 33;
// other lengths up to 129 z nodes (48^3 and 96^3 grids, say) in the same lane-group form: four
// lanes per column with 13 levels each up to 52 nodes, 33 each up to 129
constexpr int MID_Q = 4, MID_L_SHORT = 13, MID_L = 33;

int op_filter(Ctx *c, const double *in, double *out) {
  hipLaunchKernelGGL(k_filter, dim3(cdiv(ssz_of(c->g), TPB)), dim3(TPB), 0, c->stream, c->g, in,
                     out, c->filt);
  PMPIC_CHECK(hipGetLastError());
  return PMPIC_OK;
}

int op_diffz(Ctx *c, const double *in, double *out, const double *bot, const double *top) {
  const int64_t plane = plane_of(c->g);
  const int nzn = c->g.nzn, nc = lds_cols(c->g);
  const ColField f{in, out, bot, top, 0};
  auto run = [&](auto kernel, int columns) {
    hipLaunchKernelGGL(kernel, dim3(cdiv(plane, columns)), dim3(64), 0, c->stream, c->g, f,
                       c->dz_den, c->dz_cp, c->dsc);
  };
  switch (nzn) {
#define PMPIC_DZ_CASE(NZ) case NZ: run(k_diffz_reg<NZ>, 64); break;
    PMPIC_REG_COLUMNS(PMPIC_DZ_CASE)
#undef PMPIC_DZ_CASE
    default:
      if (nzn <= MID_Q * MID_L_SHORT) run(k_diffz_qn<MID_Q, MID_L_SHORT>, 64 / MID_Q);
      else if (nzn <= 129) run(k_diffz_qn<MID_Q, MID_L>, 64 / MID_Q);
      else if (nzn <= LONG_Q * LONG_L) run(k_diffz_qn<LONG_Q, LONG_L>, 64 / LONG_Q);
      else if (nc > 0)
        hipLaunchKernelGGL(k_diffz_lds, dim3(cdiv(plane, nc)), dim3(nc),
                           (size_t)2 * nc * nzn * sizeof(double), c->stream, c->g, f, c->dsc);
      else
        hipLaunchKernelGGL(k_diffz, dim3(cdiv(plane, 64)), dim3(64), 0, c->stream, c->g, f,
                           c->sder[5], c->dsc);
  }
  PMPIC_CHECK(hipGetLastError());
  return PMPIC_OK;
}

int op_laplinv(Ctx *c, double *data, int df0) {
  const int64_t plane = plane_of(c->g);
  const int nzn = c->g.nzn, nc = lds_cols(c->g);
  const ColField f{nullptr, data, nullptr, nullptr, df0 ? 1 : 0};
  auto run = [&](auto kernel, int columns) {
    hipLaunchKernelGGL(kernel, dim3(cdiv(plane, columns)), dim3(64), 0, c->stream, c->g, f, c->k2,
                       c->dsc);
  };
  switch (nzn) {
#define PMPIC_LAP_CASE(NZ) case NZ: run(k_laplinv_reg<LAP_Q, NZ>, 64 / LAP_Q); break;
    PMPIC_REG_COLUMNS(PMPIC_LAP_CASE)
#undef PMPIC_LAP_CASE
    default:
      if (nzn <= MID_Q * MID_L_SHORT) run(k_laplinv_qn<MID_Q, MID_L_SHORT>, 64 / MID_Q);
      else if (nzn <= 129) run(k_laplinv_qn<MID_Q, MID_L>, 64 / MID_Q);
      else if (nzn <= LONG_Q * LONG_L) run(k_laplinv_qn<LONG_Q, LONG_L>, 64 / LONG_Q);
      else if (nc > 0)
        hipLaunchKernelGGL(k_laplinv_lds, dim3(cdiv(plane, nc)), dim3(nc),
                           (size_t)2 * nc * nzn * sizeof(double), c->stream, c->g, f, c->k2,
                           c->dsc);
      else
        hipLaunchKernelGGL(k_laplinv, dim3(cdiv(plane, 64)), dim3(64), 0, c->stream, c->g, f,
                           c->sder[5], c->k2, c->dsc);
  }
  PMPIC_CHECK(hipGetLastError());
  return PMPIC_OK;
}

namespace {
// the spectral scratch arrays as arrays of the form's spectral type (the FP32-bulk form uses
// the first half of each FP64 allocation)
template <typename S> S *sp(double *a) { return reinterpret_cast<S *>(a); }
}  // namespace

// the physical p, q, r and total-buoyancy grids (k = 0..3) in the transforms' precision: the
// FP64 grids GP, GQ, GR, GB, or the FP32-bulk form's FP32 grids
static_assert(GQ == GP + 1 && GR == GP + 2 && GB == GP + 3, "grid ids p, q, r, b in sequence");
template <typename S> S *pqrb(Ctx *c, int k);
template <> double *pqrb<double>(Ctx *c, int k) { return c->grid[GP + k]; }
template <> float *pqrb<float>(Ctx *c, int k) { return c->b32.pgrid[k]; }

// vort2vel timestep_callback (vort2vel.F90:134-320) after par2grid of p, q, r (and the total
// buoyancy) into the grids: corrected and filtered vorticity back into grid[GP..GR], velocities
// into grid[GU..GW], the filtered velocity spectra into su, sv, sw.  Also what
// vorticity_tendency.F90:147-232 takes from the same spectra: the transform of the total buoyancy
// and the eight derivative grids of the tendency (db/dy, du/dx, du/dy, dw/dx, db/dx, dv/dx, dv/dy,
// dw/dy) into gtmp, each derivative taken while its inverse transform reads the spectrum, so that
// the two components share one forward and one inverse transform call.  S: the spectral arrays'
// type (FP32 in the FP32-bulk form, which keeps every grid here in FP32 only).
template <typename S>
static int vort2vel_spectral_t(Ctx *c) {
  S *sbs = sp<S>(c->sbs);
  {
    const S *src[4] = {pqrb<S>(c, 0), pqrb<S>(c, 1), pqrb<S>(c, 2), pqrb<S>(c, 3)};
    S *dst[4] = {sp<S>(c->sa), sp<S>(c->sb), sp<S>(c->sc), sbs};
    PMPIC_TRY(fft_forward_t<S>(c, 4, src, dst));
  }
  PMPIC_TRY(vort2vel_columns<S>(c));
  S *su = sp<S>(c->su), *sv = sp<S>(c->sv), *sw = sp<S>(c->sw);
  const S *src[14] = {sp<S>(c->sd), sp<S>(c->se), sp<S>(c->sf), sp<S>(c->sder[2]),
                      sp<S>(c->sder[3]), sp<S>(c->sder[4]), sbs, su, su, sw, sbs, sv, sv, sw};
  constexpr int F = SPEC_FILTERED;
  const int op[14] = {SPEC_PLAIN | F, SPEC_PLAIN | F, SPEC_PLAIN | F, SPEC_PLAIN,  SPEC_PLAIN,
                      SPEC_PLAIN,     SPEC_DY,        SPEC_DX | F,    SPEC_DY | F, SPEC_DX | F,
                      SPEC_DX,        SPEC_DX | F,    SPEC_DY | F,    SPEC_DY | F};
  double *dst[14] = {c->grid[GP], c->grid[GQ], c->grid[GR], c->grid[GU], c->grid[GV], c->grid[GW]};
  float *dst32[14] = {};
  for (int f = 0; f < 8; f++) dst[6 + f] = c->gtmp[f];
  if (c->precision == 1)
    for (int f = 0; f < 14; f++) {
      // the derivative grids in the first half of each FP64 scratch grid
      dst32[f] = f < 3 ? c->b32.pgrid[f] : f < 6 ? c->b32.grid[f - 3]
                                                 : reinterpret_cast<float *>(c->gtmp[f - 6]);
      dst[f] = nullptr;
    }
  c->rec_stale = true;
  return fft_backward_t<S>(c, 14, src, dst, dst32, op);
}

int vort2vel_spectral(Ctx *c) {
  return c->precision == 1 ? vort2vel_spectral_t<float>(c) : vort2vel_spectral_t<double>(c);
}

// the timestep from the grids' maxima: those of nb blocks in maxblk, or with nb = 0 taken here
static int grid_max_reduce(Ctx *c, int nb) {
  const Geometry &g = c->g;
  const int64_t nnode = (int64_t)g.nzn * g.ny * g.nx;
  if (nb == 0) {
    nb = (int)std::min<int64_t>(cdiv(nnode, TPB), MAXBLK);
    if (c->precision == 1)  // the FP32-bulk form's grids are FP32
      hipLaunchKernelGGL(k_max4<float>, dim3(nb), dim3(TPB), 0, c->stream, nnode, c->b32.grid[0],
                         c->b32.grid[1], c->b32.grid[2], c->b32.pgrid[0], c->b32.pgrid[1],
                         c->b32.pgrid[2], c->maxblk);
    else
      hipLaunchKernelGGL(k_max4<double>, dim3(nb), dim3(TPB), 0, c->stream, nnode, c->grid[GU],
                         c->grid[GV], c->grid[GW], c->grid[GP], c->grid[GQ], c->grid[GR],
                         c->maxblk);
  }
  hipLaunchKernelGGL(k_max4_final, dim3(1), dim3(TPB), 0, c->stream, g, nb, c->maxblk, c->dsc);
  PMPIC_CHECK(hipGetLastError());
  return PMPIC_OK;
}

// vorticity_tendency timestep_callback (vorticity_tendency.F90:169-265) from the grids of
// vort2vel: the tendencies, with the velocities, into the node records
int vorticity_tendency_grids(Ctx *c, bool maxima) {
  const Geometry &g = c->g;
  const int64_t nnode = (int64_t)g.nzn * g.ny * g.nx;
  const dim3 gb(cdiv(nnode, TPB)), tb(TPB);
  // up to MAXBLK blocks the tendency takes the maxima for the timestep along (a launch of 4 us
  // less); the blocks of a larger grid would be too many for the final reduction
  double *blkmax = maxima && gb.x <= MAXBLK ? c->maxblk : nullptr;
  if (c->precision == 1) {
    const Bulk32 &b = c->b32;
    const float *d[8];
    for (int f = 0; f < 8; f++) d[f] = reinterpret_cast<const float *>(c->gtmp[f]);
    hipLaunchKernelGGL((k_tendency<float, float4>), gb, tb, 0, c->stream, nnode, b.pgrid[0],
                       b.pgrid[1], b.pgrid[2], d[0], d[1], d[2], d[3], d[4], d[5], d[6], d[7],
                       b.grid[0], b.grid[1], b.grid[2], c->rec32, blkmax);
  } else {
    double *const *d = c->gtmp;
    hipLaunchKernelGGL((k_tendency<double, double2>), gb, tb, 0, c->stream, nnode, c->grid[GP],
                       c->grid[GQ], c->grid[GR], d[0], d[1], d[2], d[3], d[4], d[5], d[6], d[7],
                       c->grid[GU], c->grid[GV], c->grid[GW], c->rec, blkmax);
  }
  c->rec_stale = false;
  PMPIC_CHECK(hipGetLastError());
  if (maxima) PMPIC_TRY(grid_max_reduce(c, blkmax ? (int)gb.x : 0));
  return PMPIC_OK;
}

int records_current(Ctx *c) {
  if (!c->rec_stale) return PMPIC_OK;
  const int64_t nnode = c->gsz;
  const dim3 gb(cdiv(nnode, TPB)), tb(TPB);
  if (c->precision == 1)
    hipLaunchKernelGGL(k_record_velocity32, gb, tb, 0, c->stream, nnode, c->b32.grid[0],
                       c->b32.grid[1], c->b32.grid[2], c->rec32);
  else
    hipLaunchKernelGGL(k_record_velocity, gb, tb, 0, c->stream, nnode, c->grid[GU], c->grid[GV],
                       c->grid[GW], c->rec);
  c->rec_stale = false;
  PMPIC_CHECK(hipGetLastError());
  return PMPIC_OK;
}

}  // namespace pmpic
