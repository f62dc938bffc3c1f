// The spectral part of vort2vel between its transforms as one kernel on MI355X.
//
// Reference: components/vort2vel/src/vort2vel.F90:158-320 over model_core/src/fft/fft_ops.F90
// (diffx :204-302, diffy :305-401, diffz :419-483, laplinv :505-601, tridiagonal :620-656).
//
// diffx pairs the columns 2l, 2l+1 and diffy the rows 2m, 2m+1, so the four columns of a (m, l)
// block are closed under everything vort2vel does between the forward and the inverse
// transforms: divergence, inverse Laplacian, filter, correction, z derivative, three inverse
// Laplacians, two z derivatives and the velocity spectra.  One lane takes one column, the four
// lanes of a quad one block, so the pair values cross by quad permutes.
//
// The solves are Thomas recurrences along z.  Both matrices (the inverse Laplacian's and the
// compact z derivative's) are the same read from the bottom and from the top, so an elimination
// may run either way with the same pivots, and the back-substitution of one solve runs in the
// same pass over z as the eliminations of the next: four passes up, down, up, down instead of
// two for each of the seven solves and one for each element-wise operator.
//
//   up    divergence of (a, b, c); elimination of the divergence's solve              -> f
//   down  its solution, filtered, off a and b; eliminations of dz(f), a, b            -> f, a, b
//   up    dz(f) off c; a and b solved, w = dy(a) - dx(b); eliminations of c, dz(a), dz(b)
//   down  c, dz(a), dz(b) solved; u = dz(b) - dy(c), v = dx(c) - dz(a)
//
// The pivots depend on the column's k^2 only: they are tabled once per context, four columns
// sharing an entry, and no pass divides.  The FP64 form gets its quotients from the tabled
// reciprocal with one residual correction (div_by), which rounds as the division does for finite
// values; the FP32-bulk form multiplies by the FP64 reciprocal.  All arithmetic is FP64 in both forms;
// the arrays between the passes are of the spectral type S.
//
// Bound by memory on large grids (26 passes over a spectral array where the separate kernels took
// 41) and by the instruction latency of one wavefront on small ones.  A call, against the sum of
// the ten kernels it stands for: 170 / 540 us at 256x256x128 FP32, 125 / 280 us at
// 128x128x128 FP64 (197 and 143 before the tiles that the filter clears left its zeros alone), 22 / 91 us at 48x48x48 FP32, 9 / 26 us at 12x10x8 FP64.
#include "common.h"

#include <type_traits>

namespace pmpic {

namespace {

// the value of the quad's other column (lane ^ 1) or other row (lane ^ 2)
template <int CTRL>
__device__ __forceinline__ float quad_perm(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xf, 0xf, true));
}
template <int CTRL>
__device__ __forceinline__ double quad_perm(double v) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}
template <typename S>
__device__ __forceinline__ double other_x(S v) { return (double)quad_perm<0xB1>(v); }  // 1,0,3,2
template <typename S>
__device__ __forceinline__ double other_y(S v) { return (double)quad_perm<0x4E>(v); }  // 2,3,0,1

// n / den, with r = 1 / den rounded to nearest
template <typename S>
__device__ __forceinline__ double quot(double n, double den, double r) {
  if constexpr (std::is_same<S, float>::value) return n * r;
  return div_by(n, den, r);
}

// Pivots of the compact inverse Laplacian for both boundary conditions (bc 0: zero value, 1: zero
// derivative) of every (m, l) block, and of the compact z derivative (bt 0, 1), step by step of
// the elimination.  The k^2 = 0 block is left alone by laplinv: pivots 1, no coupling.
__global__ void k_lap_tables(Geometry g, const double *__restrict__ k2a, double *__restrict__ rcp,
                             double *__restrict__ den, double *__restrict__ cp, int *bad) {
  const int nl = g.sx / 2, nblk = nl * (g.sy / 2), nz = g.nzn, ntile = spec_tiles(g);
  const int b = blockIdx.x * blockDim.x + threadIdx.x, bc = blockIdx.y;
  if (b >= ntile * 16) return;
  const int blk = min(b, nblk - 1);  // the blocks past the last one hold zeros: any pivots do
  const double k2 = k2a[(int64_t)(2 * (blk / nl)) * g.sx + 2 * (blk % nl)];
  const double f16 = (double)(1.f / 6.f), f13 = (double)(1.f / 3.f);
  const double f112 = (double)(1.f / 12.f), f56 = (double)(5.f / 6.f);
  const double idz2 = 1. / g.dz / g.dz, i2dz2 = 2. / g.dz / g.dz;
  const bool skip = k2 == 0;
  const double off = skip ? 0. : idz2 - f112 * k2, mid = skip ? 1. : -i2dz2 - f56 * k2;
  const double bend = skip || !bc ? 1. : -idz2 - f13 * k2;
  const double cend = skip || !bc ? 0. : idz2 - f16 * k2;
  double d = bend, c = cend;
  for (int s = 0; s < nz; s++) {
    const int64_t at = (((int64_t)bc * ntile + (b >> 4)) * nz + s) * 16 + (b & 15);
    double cps = 0.;
    if (s > 0) {
      cps = c / d;
      d = (s < nz - 1 ? mid : bend) - (s < nz - 1 ? off : cend) * cps;
      c = off;
    }
    if (d == 0) *bad = 1;
    rcp[at] = 1. / d;
    if (den) den[at] = d;
    if (cp) cp[at] = cps;
  }
}

__global__ void k_dz_rcp(Geometry g, const double *__restrict__ den, double *__restrict__ rcp,
                         int *bad) {
  for (int k = threadIdx.x; k < 2 * g.nzn; k += blockDim.x) {
    if (den[k] == 0) *bad = 1;
    rcp[k] = 1. / den[k];
  }
}

template <typename S>
struct ColumnArrays {
  S *a, *b, *c;        // in: vorticity spectra; overwritten by the intermediates
  S *f;                // scratch; a, b, c, f, fc, us and vs are padded (COLUMN_PAD)
  S *fa, *fb, *fc;     // out: filtered corrected vorticity
  S *u, *v, *w;        // out: velocity spectra
  S *us, *vs, *ws;     // out: filtered velocity spectra
  const double *kx, *ky, *k2, *filt;
  const double *lrcp, *lden, *lcp;       // k_lap_tables (lden, lcp: FP64 form)
  const double *zrcp, *zden, *zcp;       // compact z derivative, [bt][step]
  double *ubar, *vbar;
  const int *bad;      // a zero pivot was tabled
};

// Mean flow (vort2vel.F90:230-241) by one wavefront: the sums over z run in the reference's order,
// each lane keeping the levels it loads; u and v of the column (0, 0).  Runs beside the column
// waves: the correction leaves that column of a and b as it is (its wavenumbers are zero).
template <typename S>
__device__ void mean_flow(const Geometry &g, const ColumnArrays<S> &ca) {
  const int lane = threadIdx.x, nz = g.nzn;
  const double hdz = g.dz / 2.;  // column (0, 0): element 0 of each of the first tile's levels
  double ub = 0., vb = 0., a0 = 0., b0 = 0.;  // running integrals and the level below's values
  for (int k0 = 0; k0 < nz; k0 += 64) {
    const int k = min(k0 + lane, nz - 1);
    const double a = ca.a[(int64_t)k * 64], b = ca.b[(int64_t)k * 64];
    double mu = 0., mv = 0.;
    const int m = min(64, nz - k0);
    for (int i = 0; i < m; i++) {
      const double ak = __shfl(a, i), bk = __shfl(b, i);
      if (k0 + i > 0) {
        ub = ub + hdz * (b0 + bk);
        vb = vb - hdz * (a0 + ak);
      }
      a0 = ak;
      b0 = bk;
      if (lane == i) { mu = ub; mv = vb; }
    }
    if (lane < m) { ca.ubar[k0 + lane] = mu; ca.vbar[k0 + lane] = mv; }
  }
  // ub, vb: the top level's integrals
  double su = 0., sv = 0.;
  for (int k0 = 0; k0 < nz - 1; k0 += 64) {
    const int m = min(64, nz - 1 - k0);
    const double u = lane < m ? ca.ubar[k0 + lane] : 0., v = lane < m ? ca.vbar[k0 + lane] : 0.;
    for (int i = 0; i < m; i++) {
      su += __shfl(u, i) + 0.5 * ub;
      sv += __shfl(v, i) + 0.5 * vb;
    }
  }
  const double rnz = (double)(1.f / (float)nz), fl = ca.filt[0];
  const double au = rnz * su, av = rnz * sv;
  for (int k = lane; k < nz; k += 64) {
    const double u = ca.ubar[k] - au, v = ca.vbar[k] - av;
    const int64_t q = (int64_t)k * 64;
    ca.ubar[k] = u;
    ca.vbar[k] = v;
    ca.u[q] = (S)u;
    ca.v[q] = (S)v;
    ca.us[q] = (S)(u * fl);
    ca.vs[q] = (S)(v * fl);
  }
}

// Runs body(s, loaded values of step s) for steps s0 .. n - 1 with the loads LV steps ahead: load(c, i)
// gives the values of step c + i, c the chunk's first step (uniform).  It is called for up to LV
// - 1 + LV steps past the end (the neighbouring tile's, or the COLUMN_PAD levels of padding at
// both ends of the arrays and tables), so the loop has no bounds, branches or clamps on its memory
// accesses: loads and stores retire in a known order, and no wait for a load covers the stores
// behind it.  LV = 8 against 4: 201 / 212 us at 256x256x128 FP32, 143 / 160 us at 128x128x128 FP64.
//
// before(): the steps below s0, whose values the caller has loaded.  EARLY: after the first loads
// are issued, so that a pass waits on memory once at its start and not twice (the values past its
// end are then loaded at its start too); the registers for it are there where a wavefront has a
// SIMD to itself.
constexpr int LV = 8;
static_assert(COLUMN_PAD >= 2 * LV, "padding of the arrays the sweeps read");
template <class T, bool EARLY, class Load, class Body, class Before>
__device__ __forceinline__ void sweep(int s0, int n, Load load, Body body, Before before) {
  T v[LV];
  if constexpr (!EARLY) before();
#pragma unroll
  for (int i = 0; i < LV; i++) v[i] = load(s0, i);
  if constexpr (EARLY) {
    __builtin_amdgcn_sched_barrier(0x7);
    before();
  }
  int s = s0;
  for (; s + LV <= n; s += LV) {
#pragma unroll
    for (int i = 0; i < LV; i++) {
      body(s, i, v[i]);
      v[i] = load(s + LV, i);
      // keep the loads here, LV - 1 levels ahead of their use (arithmetic may move)
      __builtin_amdgcn_sched_barrier(0x7);
    }
  }
#pragma unroll
  for (int i = 0; i < LV - 1; i++)
    if (s + i < n) body(s, i, v[i]);
}

// a tabled pivot: reciprocal, and for the FP64 form the pivot itself
struct Piv {
  double r, d;
};

// The column work of a tile.  KEEP: some of its columns pass the filter (where none does, the
// correction of the vorticity is zero).  FIRST: it holds the k^2 = 0 columns, which laplinv leaves
// alone, and of them the column (0, 0), whose u and v belong to the mean flow.
//
// SPLIT: four wavefronts share the tile instead of one.  One wavefront issues an instruction every
// four cycles or so, and a small grid has fewer tiles than the chip has CUs, so its time is the
// instructions of one wavefront (8,000 at 49 levels), and the loads of its unrolled code from cold
// caches.  The divergence is taken level by level by
// all four, into LDS; then the recurrences of a pass that do not depend on each other go to
// different wavefronts, those that several need (f's solution, a's and b's) computed by each of
// them; a barrier between the passes.  No pass may then overwrite what another wavefront still
// reads: the intermediates of dz(f), dz(a) and dz(b) lie in fc, vs and us, read last by the
// wavefront that writes the results there (and padded, like a, b, c and f, for its read-ahead).
// A call: 31 -> 22.5 us at 48^3 FP32, 29 -> 21 at 32^3 FP64, 12.9 -> 9.4 at 12x10x8 FP64.  With
// four or six levels ahead instead of eight 28 and 24 us at 48^3, with 16 (twice the code) 44; with
// the whole tile in LDS and rolled loops 25 to 27.
template <bool KEEP, bool FIRST, bool SPLIT, typename S>
__device__ __forceinline__ void columns(const Geometry &g, const ColumnArrays<S> &ca,
                                        double *lds) {
  // fused multiply-adds: fewer instructions and roundings in the recurrences
#pragma clang fp contract(fast)
  constexpr bool F32 = std::is_same<S, float>::value;
  constexpr std::true_type yes{};
  constexpr std::false_type no{};
  // a lane takes one of the 64 columns of a tile (16 blocks) of the spectral layout: lane bits 0
  // the column of the pair, 1 the row of the pair, 2-5 the block
  const int lane = threadIdx.x & 63, tile = blockIdx.x, ntile = spec_tiles(g), nz = g.nzn;
  const int role = SPLIT ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0;
  const int nl = g.sx / 2, blk = min(tile * 16 + (lane >> 2), nl * (g.sy / 2) - 1);
  const int m = blk / nl, l = blk - m * nl;
  const int col = (2 * m + ((lane >> 1) & 1)) * g.sx + 2 * l + (lane & 1);  // in the planes of k, filt
  const double k2 = ca.k2[col];
  const bool pass = KEEP && ca.filt[col] != 0.;  // the filter is 0 or 1
  S *const ef = SPLIT ? ca.fc : ca.f, *const za = SPLIT ? ca.vs : ca.a, *const zb = SPLIT ? ca.us : ca.b;
  // level k + i of an array, k uniform and 0 <= i < LV an immediate
  auto at = [&](S *p, int k, int i) { return p + ((int64_t)tile * nz + k) * 64 + (lane + i * 64); };
  auto get = [&](S *p, int k, int i) { return *at(p, k, i); };
  auto put = [&](S *p, int k, int i, double v) { *at(p, k, i) = (S)v; };
  // (where none of the tile's columns passes, the zeros are there since the arrays were allocated)
  auto put_filtered = [&](S *p, int k, int i, S v) {
    if (KEEP || SPLIT) *at(p, k, i) = pass ? v : (S)0;
  };
  auto tab = [&](const double *t, int bc, int s, int i) {
    return (t + (((int64_t)bc * ntile + tile) * nz + s) * 16)[(lane >> 2) + i * 16];
  };
  auto piv = [&](int bc, int s, int i) {
    return Piv{tab(ca.lrcp, bc, s, i), F32 ? 0. : tab(ca.lden, bc, s, i)};
  };
  // for the back-substitution at step s: the c' of step s + 1 (FP64), or the reciprocal pivot of
  // step s that it comes from (FP32)
  auto back = [&](int bc, int s, int i) {
    return F32 ? tab(ca.lrcp, bc, s, i) : tab(ca.lcp, bc, s + 1, i);
  };
  // signed wavenumbers: diffx of a column is kx times its pair's other column, negated for the
  // real one
  const double kx = (lane & 1) ? ca.kx[col] : -1. * ca.kx[col];
  const double ky = (lane & 2) ? ca.ky[col] : -1. * ca.ky[col];
  const bool skip = FIRST && k2 == 0;
  const double dz = g.dz, idz = 1. / dz, idz2 = 1. / dz / dz;
  const double f112 = (double)(1.f / 12.f), f56 = (double)(5.f / 6.f);
  const double f13 = (double)(1.f / 3.f), f16 = (double)(1.f / 6.f);
  const double off = skip ? 0. : idz2 - f112 * k2;
  const double cend = skip ? 0. : idz2 - f16 * k2;  // bc 1's first and last rows (bc 0: zero)
  // constant tables the same for every lane: scalar loads, which the stores do not hold up
  typedef const __attribute__((address_space(4))) double *ConstTab;
  const ConstTab zr0 = (ConstTab)ca.zrcp, zr1 = zr0 + nz, zd0 = (ConstTab)ca.zden, zd1 = zd0 + nz;
  const ConstTab zc0 = (ConstTab)ca.zcp, zc1 = zc0 + nz;
  auto half_dz = [&](double x) { return F32 ? x * (0.5 * idz) : quot<S>(x * 0.5, dz, idz); };
  auto per_dz = [&](double x) { return quot<S>(x, dz, idz); };
  // the c' of step s + 1 of an inverse Laplacian from back(bc, s); cf: step s's own c
  auto cp_of = [&](double cf, double t) { return F32 ? cf * t : t; };
  // rows of an inverse Laplacian's elimination: fm, f0, fp the right-hand side's values below,
  // at and above the row
  auto row = [&](double fm, double f0, double fp, double prev, const Piv &p) {
    const double q = quot<S>(f112 * (fm + fp) + f56 * f0 - off * prev, p.d, p.r);
    return skip ? f0 : q;
  };
  auto row_first = [&](double f0, double fp, const Piv &p) {  // bc 1
    const double q = quot<S>(f13 * f0 + f16 * fp, p.d, p.r);
    return skip ? f0 : q;
  };
  auto row_last = [&](double fm, double f0, double prev, const Piv &p) {  // bc 1
    const double q = quot<S>(f13 * f0 + f16 * fm - cend * prev, p.d, p.r);
    return skip ? f0 : q;
  };
  auto row_end = [&](double f0) { return skip ? f0 : 0.; };  // bc 0, first and last

  // ---- up: divergence (vort2vel.F90:158-174) and its elimination ----
  if constexpr (KEEP) {
    const double h = 1. / 2. / dz;
    auto horizontal = [&](S a, S b) { return other_x(a) * kx + other_y(b) * ky; };
    if constexpr (SPLIT) {
      constexpr int DB = 4;  // levels of a wavefront in flight
      for (int k0 = role; k0 < nz; k0 += 4 * DB) {
        S a[DB], b[DB], cl[DB], ch[DB];
#pragma unroll
        for (int i = 0; i < DB; i++) {
          const int k = min(k0 + 4 * i, nz - 1);
          a[i] = get(ca.a, k, 0);
          b[i] = get(ca.b, k, 0);
          cl[i] = get(ca.c, max(k - 1, 0), 0);
          ch[i] = get(ca.c, min(k + 1, nz - 1), 0);
        }
#pragma unroll
        for (int i = 0; i < DB; i++) {
          const int k = k0 + 4 * i;
          if (k >= nz) break;
          double fz = ((double)ch[i] - (double)cl[i]) * h;
          if (k == 0)  // cl: level 0, ch: level 1
            fz = h * (4. * (double)ch[i] - (double)get(ca.c, 2, 0) - 3. * (double)cl[i]);
          if (k == nz - 1)
            fz = h * ((double)get(ca.c, nz - 3, 0) + 3. * (double)ch[i] - 4. * (double)cl[i]);
          const double d = horizontal(a[i], b[i]) + fz;
          lds[k * 64 + lane] = FIRST && lane == 0 ? 0. : d;
        }
      }
      __syncthreads();
      if (role == 0) {
        struct T { double d; Piv p; };
        double dm = lds[lane], d0 = lds[64 + lane], fp = 0.;
        const Piv first = piv(1, 0, 0), end = piv(1, nz - 1, 0);
        auto step = [&](int k, int i, const T &t) {
          fp = row(dm, d0, t.d, fp, t.p);  // row k + i - 1
          put(ca.f, k - 1, i, fp);
          dm = d0; d0 = t.d;
        };
        auto load = [&](int k, int i) { return T{lds[(k + i) * 64 + lane], piv(1, k - 1, i)}; };
        sweep<T, SPLIT>(2, nz, load, step, [&]() {
          fp = row_first(dm, d0, first);
          put(ca.f, 0, 0, fp);
        });
        put(ca.f, nz - 1, 0, row_last(dm, d0, fp, end));
      }
      __syncthreads();
    } else {
      struct T { S a, b, c1; Piv p; };
      const S a0 = get(ca.a, 0, 0), a1 = get(ca.a, 1, 0), b0 = get(ca.b, 0, 0),
              b1 = get(ca.b, 1, 0);
      const double cA = (double)get(ca.c, 0, 0), cB = (double)get(ca.c, 1, 0),
                   cC = (double)get(ca.c, 2, 0);
      const Piv first = piv(1, 0, 0);
      double dm = 0., d0 = 0., fp = 0.;
      double cmm = cA, cm = cB, c0 = cC;  // c at levels k - 2, k - 1, k
      auto step = [&](int k, int i, double fz, S a, S b, const Piv &p) {
        double d1 = horizontal(a, b) + fz;
        if (FIRST && lane == 0) d1 = 0.;
        fp = row(dm, d0, d1, fp, p);  // row k + i - 1
        put(ca.f, k - 1, i, fp);
        dm = d0; d0 = d1;
      };
      sweep<T, SPLIT>(2, nz - 1,
          [&](int k, int i) {
            return T{get(ca.a, k, i), get(ca.b, k, i), get(ca.c, k + 1, i), piv(1, k - 1, i)};
          },
          [&](int k, int i, const T &t) {
            const double c1 = (double)t.c1;
            step(k, i, (c1 - cm) * h, t.a, t.b, t.p);
            cmm = cm; cm = c0; c0 = c1;
          },
          [&]() {
            dm = horizontal(a0, b0) + h * (4. * cB - cC - 3. * cA);
            d0 = horizontal(a1, b1) + (cC - cA) * h;
            if (FIRST && lane == 0) dm = d0 = 0.;
            fp = row_first(dm, d0, first);
            put(ca.f, 0, 0, fp);
          });
      step(nz - 1, 0, h * (cmm + 3. * c0 - 4. * cm), get(ca.a, nz - 1, 0), get(ca.b, nz - 1, 0),
           piv(1, nz - 2, 0));
      put(ca.f, nz - 1, 0, row_last(dm, d0, fp, piv(1, nz - 1, 0)));
    }
  }

  // ---- down: the correction of a and b (vort2vel.F90:176-194), eliminations of dz(f), a, b ----
  double atop = 0., abot = 0., btop = 0., bbot = 0.;
  auto down = [&](auto do_a, auto do_b, auto do_e) {
    constexpr bool A = decltype(do_a)::value, B = decltype(do_b)::value,
                   E = KEEP && decltype(do_e)::value;
    struct T { S f, a, b; double cp; Piv p; };
    double fn = 0., f0 = 0., f1 = 0., f2 = 0.;   // unfiltered; filtered at this level, +1, +2
    double a0 = 0., a1 = 0., a2 = 0., b0 = 0., b1 = 0., b2 = 0.;  // corrected
    double ep = 0., ap = 0., bp = 0.;            // eliminated values of the previous row
    // level k + i; cf: the c of its row (for the back-substitution), sub: below the top
    auto level = [&](int k, int i, const T &t, double cf, bool sub) {
      f2 = f1; f1 = f0;
      a2 = a1; b2 = b1;
      a0 = (double)t.a;
      b0 = (double)t.b;
      if constexpr (KEEP) {
        fn = sub ? (double)t.f - cp_of(cf, t.cp) * fn : (double)t.f;
        const S ff = pass ? (S)fn : (S)0;
        f0 = (double)ff;
        if constexpr (A) a0 = (double)(S)(a0 - other_x(ff) * kx);
        if constexpr (B) b0 = (double)(S)(b0 - other_y(ff) * ky);
      }
      if constexpr (A) put_filtered(ca.fa, k, i, (S)a0);
      if constexpr (B) put_filtered(ca.fb, k, i, (S)b0);
    };
    auto load = [&](int s, int k, int i, int r) {  // level k + r, elimination step s - 1 + i
      T t{};
      if constexpr (A) t.a = get(ca.a, k, r);
      if constexpr (B) t.b = get(ca.b, k, r);
      if constexpr (A || B) t.p = piv(0, s - 1, i);
      if constexpr (KEEP) {
        t.f = get(ca.f, k, r);
        t.cp = back(1, k, r);
      }
      return t;
    };
    const T top = load(1, nz - 1, 0, 0), next = load(1, nz - 2, 0, 0);
    T bottom{};
    if constexpr (SPLIT) bottom = load(nz - 1, 0, 0, 0);
    auto rows = [&](int s, int k, int i, int r, const T &t, double cf) {  // row above level k + r
      const double aa = a1, ab = a2, ba = b1, bb = b2;
      level(k, r, t, cf, true);
      if constexpr (E) {
        ep = quot<S>(half_dz(f2 - f0) - f16 * ep, zd0[s + i - 1], zr0[s + i - 1]);
        put(ef, k + 1, r, ep);
      }
      if constexpr (A) {
        ap = row(a0, aa, ab, ap, t.p);
        put(ca.a, k + 1, r, ap);
      }
      if constexpr (B) {
        bp = row(b0, ba, bb, bp, t.p);
        put(ca.b, k + 1, r, bp);
      }
      a2 = aa; a1 = a0;
      b2 = ba; b1 = b0;
    };
    // steps 2 .. nz - 2 are levels nz - 3 .. 1; a chunk's lowest level is k
    sweep<T, SPLIT>(2, nz - 1,
        [&](int s, int i) { return load(s, nz - s - LV, i, LV - 1 - i); },
        [&](int s, int i, const T &t) { rows(s, nz - s - LV, i, LV - 1 - i, t, off); },
        [&]() {
          level(nz - 1, 0, top, 0., false);
          atop = a0; btop = b0;
          a1 = a0; b1 = b0;
          level(nz - 2, 0, next, off, true);
          ap = row_end(a1);
          bp = row_end(b1);
          if constexpr (E) put(ef, nz - 1, 0, 0.);
          if constexpr (A) put(ca.a, nz - 1, 0, ap);
          if constexpr (B) put(ca.b, nz - 1, 0, bp);
          a2 = a1; a1 = a0;
          b2 = b1; b1 = b0;
        });
    if constexpr (!SPLIT) bottom = load(nz - 1, 0, 0, 0);
    rows(nz - 1, 0, 0, 0, bottom, cend);
    abot = a0;
    bbot = b0;
    if constexpr (E) put(ef, 0, 0, 0.);
    if constexpr (A) put(ca.a, 0, 0, row_end(a0));
    if constexpr (B) put(ca.b, 0, 0, row_end(b0));
  };
  if constexpr (SPLIT) {
    if (role == 0) down(yes, no, no);
    if (role == 1) down(no, yes, no);
    if (KEEP && role == 2) down(no, no, yes);
    __syncthreads();
  } else {
    down(yes, yes, yes);
  }

  // ---- up: the correction of c (vort2vel.F90:197-218), a and b solved, w; eliminations ----
  auto up = [&](auto do_a, auto do_b, auto do_c, auto do_w) {
    constexpr bool A = decltype(do_a)::value, B = decltype(do_b)::value;
    constexpr bool C = decltype(do_c)::value, W = decltype(do_w)::value;
    struct T { S f, c, a, b; double cp; Piv p; };
    double fn = 0., an = 0., bn = 0.;                       // solved values
    double cm = 0., c0 = 0., c1 = 0., cp1 = 0.;             // corrected c below, at row; eliminated
    double am = 0., a0 = 0., a1 = 0., bm = 0., b0 = 0., b1 = 0.;
    double zap = 0., zbp = 0.;
    // level k + i; zc: the dz solve's c' (unused at the bottom)
    auto level = [&](int k, int i, const T &t, double cf, double zc, bool sub) {
      if constexpr (C) {
        cm = c0; c0 = c1;
        c1 = (double)t.c;
        if constexpr (KEEP) {
          fn = sub ? (double)t.f - zc * fn : (double)t.f;
          c1 = (double)(S)(c1 - (double)(S)fn);
        }
        if (!sub) c1 = 0.;
        put_filtered(ca.fc, k, i, (S)c1);
      }
      const double cp = cp_of(cf, t.cp);
      if constexpr (A || W) {
        am = a0; a0 = a1;
        an = sub ? (double)t.a - cp * an : (double)t.a;
        a1 = (double)(S)an;
      }
      if constexpr (B || W) {
        bm = b0; b0 = b1;
        bn = sub ? (double)t.b - cp * bn : (double)t.b;
        b1 = (double)(S)bn;
      }
      if constexpr (W) {
        const double w = other_y((S)an) * ky - other_x((S)bn) * kx;
        put(ca.w, k, i, w);
        put_filtered(ca.ws, k, i, (S)w);
      }
    };
    auto store = [&](int k, int i, int z, double ra, double rb) {  // row k + i
      if constexpr (C) put(ca.c, k, i, cp1);
      if constexpr (A) zap = quot<S>(ra, zd1[z], zr1[z]);
      if constexpr (B) zbp = quot<S>(rb, zd1[z], zr1[z]);
      if (FIRST && lane == 0) return;  // column (0, 0) of a and b stays: the mean flow's input
      if constexpr (A) put(za, k, i, zap);
      if constexpr (B) put(zb, k, i, zbp);
    };
    auto load = [&](int k, int i, int s, int r, int q) {  // level k + i, its step s + r; row q + i
      T t{};
      if constexpr (A || W) t.a = get(ca.a, k, i);
      if constexpr (B || W) t.b = get(ca.b, k, i);
      if constexpr (A || B || W) t.cp = back(0, s, r);
      if constexpr (C) {
        t.c = get(ca.c, k, i);
        t.p = piv(1, q, i);
        if constexpr (KEEP) t.f = get(ef, k, i);
      }
      return t;
    };
    const T bottom = load(0, 0, nz - 2, 0, 0), next = load(1, 0, nz - 2, 0, 0);
    T top{};
    Piv end{};
    auto load_end = [&]() {
      top = load(nz - 1, 0, 0, 0, nz - 2);
      if constexpr (C) end = piv(1, nz - 1, 0);
    };
    if constexpr (SPLIT) load_end();
    auto rows = [&](int k, int i, const T &t, double cf, double zc) {
      level(k, i, t, cf, zc, true);
      if constexpr (C) cp1 = row(cm, c0, c1, cp1, t.p);
      store(k - 1, i, k + i - 1, half_dz(a1 - am) - f16 * zap, half_dz(b1 - bm) - f16 * zbp);
    };
    // levels 2 .. nz - 2; a chunk's levels k .. k + LV - 1 are steps nz - 1 - k downwards
    sweep<T, SPLIT>(2, nz - 1,
        [&](int k, int i) { return load(k, i, nz - k - LV, LV - 1 - i, k - 1); },
        [&](int k, int i, const T &t) { rows(k, i, t, off, zc0[nz - k - i]); },
        [&]() {
          level(0, 0, bottom, 0., 0., false);
          level(1, 0, next, off, zc0[nz - 1], true);
          if constexpr (C) cp1 = row_first(c0, c1, next.p);
          store(0, 0, 0, per_dz(a1) - f16 * abot * dz, per_dz(b1) - f16 * bbot * dz);
        });
    if constexpr (!SPLIT) load_end();
    // the top level's c' is that of the first step: no coupling with a zero value
    rows(nz - 1, 0, top, 0., zc0[1]);
    if constexpr (C) cp1 = row_last(c0, c1, cp1, end);
    store(nz - 1, 0, nz - 1, -per_dz(a0) + f16 * atop * dz - f13 * zap,
          -per_dz(b0) + f16 * btop * dz - f13 * zbp);
  };
  if constexpr (SPLIT) {
    if (role == 0) up(yes, no, no, no);
    if (role == 1) up(no, yes, no, no);
    if (role == 2) up(no, no, yes, no);
    if (role == 3) up(no, no, no, yes);
    __syncthreads();
  } else {
    up(yes, yes, yes, yes);
  }

  // ---- down: c, dz(a), dz(b) solved; u and v (vort2vel.F90:251-320) ----
  auto last = [&](auto do_u, auto do_v) {
    constexpr bool U = decltype(do_u)::value, V = decltype(do_v)::value;
    struct T { S c, a, b; double cp; };
    double cn = 0., zan = 0., zbn = 0.;
    auto level = [&](int k, int i, const T &t, double cf, double zc, bool sub) {
      cn = sub ? (double)t.c - cp_of(cf, t.cp) * cn : (double)t.c;
      const S cs = (S)cn;
      if constexpr (V) zan = sub ? (double)t.a - zc * zan : (double)t.a;
      if constexpr (U) zbn = sub ? (double)t.b - zc * zbn : (double)t.b;
      const double u = (double)(S)zbn - other_y(cs) * ky;
      const double v = other_x(cs) * kx - (double)(S)zan;
      if (FIRST && lane == 0) return;
      if constexpr (U) {
        put(ca.u, k, i, u);
        put_filtered(ca.us, k, i, (S)u);
      }
      if constexpr (V) {
        put(ca.v, k, i, v);
        put_filtered(ca.vs, k, i, (S)v);
      }
    };
    auto load = [&](int k, int i) {
      T t{get(ca.c, k, i), (S)0, (S)0, back(1, k, i)};
      if constexpr (V) t.a = get(za, k, i);
      if constexpr (U) t.b = get(zb, k, i);
      return t;
    };
    const T top = load(nz - 1, 0);
    T bottom{};
    if constexpr (SPLIT) bottom = load(0, 0);
    sweep<T, SPLIT>(1, nz - 1,
        [&](int s, int i) { return load(nz - s - LV, LV - 1 - i); },
        [&](int s, int i, const T &t) {
          level(nz - s - LV, LV - 1 - i, t, off, zc1[nz - s - i], true);
        },
        [&]() { level(nz - 1, 0, top, 0., 0., false); });
    if constexpr (!SPLIT) bottom = load(0, 0);
    level(0, 0, bottom, cend, zc1[1], true);
  };
  if constexpr (SPLIT) {
    if (role == 0) last(yes, no);
    if (role == 1) last(no, yes);
  } else {
    last(yes, yes);
  }
}

template <typename S, bool SPLIT>
__global__ void __launch_bounds__(SPLIT ? 256 : 64) k_vort2vel_columns(Geometry g,
                                                                       ColumnArrays<S> ca,
                                                                       DevScalars *sc) {
  extern __shared__ double columns_lds[];
  const int ntile = spec_tiles(g);
  if ((int)blockIdx.x == ntile) {
    if (threadIdx.x == 0 && *ca.bad) raise_status(sc, PMPIC_ERR_ZERO_PIVOT);
    if (threadIdx.x < 64) mean_flow(g, ca);
    return;
  }
  const int nl = g.sx / 2, blk = min((int)blockIdx.x * 16 + ((int)(threadIdx.x & 63) >> 2),
                                     nl * (g.sy / 2) - 1);
  const bool kept = ca.filt[(int64_t)(2 * (blk / nl)) * g.sx + 2 * (blk % nl)] != 0.;
  if (blockIdx.x == 0) columns<true, true, SPLIT, S>(g, ca, columns_lds);
  else if (__any(kept)) columns<true, false, SPLIT, S>(g, ca, columns_lds);
  else columns<false, false, SPLIT, S>(g, ca, columns_lds);
}

}  // namespace

// the pivot tables (once per context, after the wavenumbers and dz_den are set up)
int columns_setup(Ctx *c) {
  const Geometry &g = c->g;
  hipLaunchKernelGGL(k_lap_tables, dim3(cdiv(spec_tiles(g) * 16, 64), 2), dim3(64), 0, c->stream, g, c->k2,
                     c->lap_rcp, c->lap_den, c->lap_cp, c->lap_bad);
  hipLaunchKernelGGL(k_dz_rcp, dim3(1), dim3(256), 0, c->stream, g, c->dz_den, c->dz_rcp,
                     c->lap_bad);
  PMPIC_CHECK(hipGetLastError());
  PMPIC_CHECK(hipStreamSynchronize(c->stream));
  return PMPIC_OK;
}

// Four wavefronts a tile while there are at most as many tiles as CUs: above, one wavefront a SIMD
// fills the chip and shares no work (a step of 128x128x96 FP64, 265 tiles: 6.67 ms split, 6.65 not;
// 96x96x64, 150 tiles: 2.72, 2.77).
constexpr int SPLIT_TILES = 256;

template <typename S>
int vort2vel_columns(Ctx *c) {
  const Geometry &g = c->g;
  auto sp = [](double *a) { return reinterpret_cast<S *>(a); };
  const ColumnArrays<S> ca{sp(c->sa), sp(c->sb), sp(c->sc), sp(c->sder[0]), sp(c->sd), sp(c->se),
                           sp(c->sf), sp(c->sder[2]), sp(c->sder[3]), sp(c->sder[4]), sp(c->su),
                           sp(c->sv), sp(c->sw), c->kx, c->ky, c->k2, c->filt, c->lap_rcp,
                           c->lap_den, c->lap_cp, c->dz_rcp, c->dz_den, c->dz_cp, c->ubar, c->vbar,
                           c->lap_bad};
  const int tiles = spec_tiles(g);
  // the divergence of a tile's levels, with those the sweep reads past the last
  const size_t lds = sizeof(double) * 64 * (g.nzn + 2 * LV);
  if (tiles <= SPLIT_TILES && lds <= 64 * 1024)
    hipLaunchKernelGGL((k_vort2vel_columns<S, true>), dim3(tiles + 1), dim3(256), lds, c->stream, g,
                       ca, c->dsc);
  else
    hipLaunchKernelGGL((k_vort2vel_columns<S, false>), dim3(tiles + 1), dim3(64), 0, c->stream, g,
                       ca, c->dsc);
  PMPIC_CHECK(hipGetLastError());
  return PMPIC_OK;
}
template int vort2vel_columns<float>(Ctx *);
template int vort2vel_columns<double>(Ctx *);

}  // namespace pmpic
