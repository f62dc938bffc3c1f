// Semi-spectral 2-D transforms on MI355X (periodic x, y; z stays physical).
//
// Reference: model_core/src/fft/pencilfft.F90:151-212 (forward: r2c along y, (Re,Im) pairs
// interleaved, then r2c along x of each real y-row; backward: the reverse), over FFTE's 1-D
// transforms wrapped by model_core/src/fft/ffte_mod.F90:66-124 (forward sum x_j e^{-2 pi i jk/N},
// unnormalised; inverse = conj . forward . conj, scaled by 1/N, real part kept, so the imaginary
// parts of the DC and Nyquist bins are dropped).
//
// The spectral element S[k][2m+a][2l+b] is component b (Re/Im) at x-wavenumber l of the x-DFT
// of component a of the y-DFT at y-wavenumber m.  With F(m,l) the full 2-D DFT,
//   x-DFT of Re Y_m = (F(m,l) + F(-m,l))/2,   x-DFT of Im Y_m = (F(m,l) - F(-m,l))/(2i),
// so the layout follows from one real-to-complex pass along the contiguous x rows and one
// complex pass along y.  Each pass is one kernel: a workgroup stages a batch of rows (or of
// adjacent columns, for coalesced strided access) in LDS and runs a mixed radix-4/2/3/5
// Stockham FFT there, so each pass reads and writes HBM once.  A plane that fits the LDS takes both
// passes in one kernel.  The inverse builds, per (z, m),
// the complex row H = A_m + i B_m of the two real x-spectra, transforms it along x, and finishes
// with a complex-to-real pass along y.
#include "common.h"

#include <math.h>
#include <algorithm>
#include <type_traits>
#include <vector>

namespace pmpic {

namespace {

// radix schedule: radix of stage s in bits [4 s, 4 s + 4) of `code` (held in registers; no
// per-stage memory read)
struct Plan {
  int n;
  int nrad;
  uint64_t code;
};

// radix 4 stages first, then 2, 3, 5; nrad = -1 when n has another prime factor
__host__ __device__ constexpr Plan make_plan(int n) {
  Plan p{n, 0, 0};
  int m = n;
  const int radix[4] = {4, 2, 3, 5};
  for (int a = 0; a < 4; a++)
    while (m % radix[a] == 0 && p.nrad < 16) {
      p.code |= (uint64_t)radix[a] << (4 * p.nrad);
      p.nrad++;
      m /= radix[a];
    }
  if (m != 1) p.nrad = -1;
  return p;
}

// Transform lengths with kernels compiled for them (every index computation then divides by
// constants); other lengths run the same kernels with the length read at run time (NT = 0).
constexpr int FIXED_N[] = {16, 32, 48, 64, 96, 128, 256, 512};

constexpr int FFT_TPB = 256;
constexpr int MAXF = FFT_FIELDS;

// The transforms run in the precision S of the spectral arrays: FP64 (double2 complex
// elements), or FP32 (float2) in the FP32-bulk form, whose LDS buffers then hold twice as many
// elements, so a column pass covers twice as many adjacent columns.  The forward transform
// reads physical grids of the same precision; the inverse writes FP64 grids, FP32 grids or
// both.
template <typename S> struct Cx;
template <> struct Cx<double> { using T = double2; };
template <> struct Cx<float> { using T = float2; };
template <typename S> using cx_t = typename Cx<S>::T;
template <typename C> struct Re;
template <> struct Re<double2> { using T = double; };
template <> struct Re<float2> { using T = float; };
template <typename S>
__host__ __device__ constexpr int lds_cplx() { return 16384 / (int)sizeof(cx_t<S>); }  // 16 KiB

template <typename C, typename S>
__device__ __forceinline__ C mkc(S a, S b) {
  C r;
  r.x = a;
  r.y = b;
  return r;
}

struct FieldPtrs {
  const void *in[MAXF];  // forward: physical grids of type S; inverse: spectral arrays of type S
  void *out[MAXF];       // forward: spectral arrays of type S; inverse: FP64 physical grids
  float *out32[MAXF];    // optional FP32 copy of a real output (the FP32-bulk form's gathers)
  int op[MAXF];          // SpecOp applied to the input of the inverse; SPEC_FILTERED: it is zero
                         // where the filter is, which is then not read
  const int *lcut;       // the filter's extent (Ctx)
  int mcut;
  const double *kx, *ky;  // wavenumber planes for SPEC_DX / SPEC_DY
};

template <typename C>
__device__ __forceinline__ C cmul(C a, C b) {
  C r;
  r.x = a.x * b.x - a.y * b.y;
  r.y = a.x * b.y + a.y * b.x;
  return r;
}

// DFT of length R on registers: v[o] <- sum_q v[q] W^(o q), W = exp(-2 pi i / R) for the
// forward transform and its conjugate for the inverse (INV); products with +-1 and +-i are
// exact swaps and sign changes.  C is the complex type, S its real type.
template <int R, bool INV, typename C>
__device__ __forceinline__ void dft(C *v) {
  using S = typename Re<C>::T;
  if constexpr (R == 2) {
    const C a = v[0], b = v[1];
    v[0] = mkc<C, S>(a.x + b.x, a.y + b.y);
    v[1] = mkc<C, S>(a.x - b.x, a.y - b.y);
  } else if constexpr (R == 4) {
    const C s02 = mkc<C, S>(v[0].x + v[2].x, v[0].y + v[2].y);
    const C d02 = mkc<C, S>(v[0].x - v[2].x, v[0].y - v[2].y);
    const C s13 = mkc<C, S>(v[1].x + v[3].x, v[1].y + v[3].y);
    const C d13 = mkc<C, S>(v[1].x - v[3].x, v[1].y - v[3].y);
    // forward: y1 = d02 - i d13, y3 = d02 + i d13 (inverse swaps them)
    const C mi = mkc<C, S>(d13.y, -d13.x);  // -i * d13
    v[0] = mkc<C, S>(s02.x + s13.x, s02.y + s13.y);
    v[2] = mkc<C, S>(s02.x - s13.x, s02.y - s13.y);
    if (!INV) {
      v[1] = mkc<C, S>(d02.x + mi.x, d02.y + mi.y);
      v[3] = mkc<C, S>(d02.x - mi.x, d02.y - mi.y);
    } else {
      v[1] = mkc<C, S>(d02.x - mi.x, d02.y - mi.y);
      v[3] = mkc<C, S>(d02.x + mi.x, d02.y + mi.y);
    }
  } else if constexpr (R == 3) {
    constexpr S c = (S)-0.5;
    constexpr S s = INV ? (S)-0.86602540378443864676 : (S)0.86602540378443864676;
    const C t = mkc<C, S>(v[1].x + v[2].x, v[1].y + v[2].y);
    const C d = mkc<C, S>(v[1].x - v[2].x, v[1].y - v[2].y);
    const C a = mkc<C, S>(v[0].x + c * t.x, v[0].y + c * t.y);
    v[0] = mkc<C, S>(v[0].x + t.x, v[0].y + t.y);
    // y1 = a - i s d, y2 = a + i s d;  -i (x + i y) = y - i x
    v[1] = mkc<C, S>(a.x + s * d.y, a.y - s * d.x);
    v[2] = mkc<C, S>(a.x - s * d.y, a.y + s * d.x);
  } else {
    static_assert(R == 5, "radix 2, 3, 4 or 5");
    constexpr S c1 = (S)0.30901699437494742410, c2 = (S)-0.80901699437494742410;
    constexpr S s1 = INV ? (S)-0.95105651629515357212 : (S)0.95105651629515357212;
    constexpr S s2 = INV ? (S)-0.58778525229247312917 : (S)0.58778525229247312917;
    const C t1 = mkc<C, S>(v[1].x + v[4].x, v[1].y + v[4].y);
    const C t2 = mkc<C, S>(v[2].x + v[3].x, v[2].y + v[3].y);
    const C t3 = mkc<C, S>(v[1].x - v[4].x, v[1].y - v[4].y);
    const C t4 = mkc<C, S>(v[2].x - v[3].x, v[2].y - v[3].y);
    const C a1 = mkc<C, S>(v[0].x + c1 * t1.x + c2 * t2.x, v[0].y + c1 * t1.y + c2 * t2.y);
    const C a2 = mkc<C, S>(v[0].x + c2 * t1.x + c1 * t2.x, v[0].y + c2 * t1.y + c1 * t2.y);
    const C b1 = mkc<C, S>(s1 * t3.x + s2 * t4.x, s1 * t3.y + s2 * t4.y);
    const C b2 = mkc<C, S>(s2 * t3.x - s1 * t4.x, s2 * t3.y - s1 * t4.y);
    v[0] = mkc<C, S>(v[0].x + t1.x + t2.x, v[0].y + t1.y + t2.y);
    // y1 = a1 - i b1, y4 = a1 + i b1, y2 = a2 - i b2, y3 = a2 + i b2
    v[1] = mkc<C, S>(a1.x + b1.y, a1.y - b1.x);
    v[4] = mkc<C, S>(a1.x - b1.y, a1.y + b1.x);
    v[2] = mkc<C, S>(a2.x + b2.y, a2.y - b2.x);
    v[3] = mkc<C, S>(a2.x - b2.y, a2.y + b2.x);
  }
}

// One Stockham stage of radix R over nb transforms of length n (t-major in x), Ns = product of
// the radices already applied: item (t, i) takes x[i + q n/R], q < R, twiddled by
// W_n^(q k n/(Ns R)) with k = i mod Ns, and writes the R-point DFT to
// y[(i / Ns) Ns R + k + o Ns].  tw[e] = W_n^e staged in LDS (conjugated for the inverse).
template <int R, bool INV, typename C>
__device__ __forceinline__ void stockham_stage(const C *x, C *y, const C *tw, int n, int Ns,
                                               int nb) {
  const int nq = n / R;
  const int tstep = n / (Ns * R);
  const int tot = nb * nq;
  for (int bi = threadIdx.x; bi < tot; bi += FFT_TPB) {
    const int t = bi / nq, i = bi - t * nq;
    const int j = i / Ns, k = i - j * Ns;
    const C *xs = x + t * n + i;
    C v[R];
#pragma unroll
    for (int q = 0; q < R; q++) {
      const C e = xs[q * nq];
      v[q] = (q == 0 || k == 0) ? e : cmul(e, tw[q * k * tstep]);
    }
    dft<R, INV>(v);
    C *ys = y + t * n + j * Ns * R + k;
#pragma unroll
    for (int o = 0; o < R; o++) ys[o * Ns] = v[o];
  }
}

// the stages from stage ST of a fixed length N (NS = product of the earlier radices)
template <bool INV, int N, int ST, int NS, typename C>
__device__ __forceinline__ C *fixed_stages(C *a, C *b, const C *tw, int nb) {
  constexpr Plan P = make_plan(N);
  static_assert(P.nrad > 0, "a fixed length has a radix schedule");
  if constexpr (ST == P.nrad) {
    return a;
  } else {
    constexpr int R = (int)((P.code >> (4 * ST)) & 15u);
    stockham_stage<R, INV>(a, b, tw, N, NS, nb);
    __syncthreads();
    return fixed_stages<INV, N, ST + 1, NS * R>(b, a, tw, nb);
  }
}

// nb transforms of length p.n (NT when NT > 0) stored t-major in `a`; result in the returned
// buffer.
template <bool INV, int NT, typename C>
__device__ C *lds_fft(C *a, C *b, const C *tw, const Plan &p, int nb) {
  if constexpr (NT > 0) return fixed_stages<INV, NT, 0, 1>(a, b, tw, nb);
  int Ns = 1;
  for (int s = 0; s < p.nrad; s++) {
    const int r = (int)((p.code >> (4 * s)) & 15u);
    if (r == 4) stockham_stage<4, INV>(a, b, tw, p.n, Ns, nb);
    else if (r == 2) stockham_stage<2, INV>(a, b, tw, p.n, Ns, nb);
    else if (r == 3) stockham_stage<3, INV>(a, b, tw, p.n, Ns, nb);
    else stockham_stage<5, INV>(a, b, tw, p.n, Ns, nb);
    __syncthreads();
    C *sw = a;
    a = b;
    b = sw;
    Ns *= r;
  }
  return a;
}

// Loads into LDS are issued as a batch (each thread's elements loaded into registers, then
// stored), so a workgroup waits on memory once per pass rather than once per element.
template <typename S>
__host__ __device__ constexpr int ept() { return lds_cplx<S>() / FFT_TPB; }  // per thread
// The row passes read contiguous rows, so a smaller batch costs them no coalescing: in FP32
// they stage half as many elements (8 KiB per buffer), so twice the workgroups fit a CU's LDS
template <typename S>
__host__ __device__ constexpr int lds_rows() {
  return sizeof(S) == 4 ? lds_cplx<S>() / 2 : lds_cplx<S>();
}
template <typename S>
__host__ __device__ constexpr int ept_rows() { return lds_rows<S>() / FFT_TPB; }
constexpr int TPT = 512 / FFT_TPB;  // twiddles per thread (n <= 512)

// The column passes of FP32 columns of at most 128 points stage half the batch (8 KiB per
// buffer), so twice the workgroups fit a CU; that still takes at least 8 adjacent columns, 64
// bytes of each row.  Longer columns keep the full batch (fewer columns would cut the rows' runs
// to 32 bytes: 256-point columns measured 160 -> 264 us per inverse pass), and the inverse pass
// of 512-point FP32 columns takes twice the batch (eight column pairs, 64-byte runs: 1.97 ->
// 1.64 ms at 512 x 512 x 257 nodes, with half the workgroups per CU; the forward pass, whose
// registers then hold twice the elements, measured slower that way).  n = 0: a length known
// only at run time; inv: the inverse (complex-to-real) pass.
template <typename S>
__host__ __device__ constexpr int lds_cols(int n, bool inv) {
  return (sizeof(S) == 4 && n > 0 && n <= 128)   ? lds_cplx<S>() / 2
         : (sizeof(S) == 4 && inv && n == 512)   ? lds_cplx<S>() * 2
                                                 : lds_cplx<S>();
}

// adjacent columns (column pairs for the inverse) a column pass takes per workgroup
template <typename S>
__host__ __device__ constexpr int col_batch(int n, bool inv) {
  return lds_cols<S>(n, inv) / n > 32 ? 32 : lds_cols<S>(n, inv) / n;
}

// q = a / d and r = a - q d for 0 <= a < 2^22, 0 < d, with rd = 1/d rounded to FP32: the
// product's relative error is below 2^-23, so the truncated estimate is off by at most one
__device__ __forceinline__ int div_small(int a, int d, float rd, int &r) {
  int q = (int)((float)a * rd);
  r = a - q * d;
  if (r < 0) {
    q--;
    r += d;
  } else if (r >= d) {
    q++;
    r -= d;
  }
  return q;
}

template <typename C>
__device__ __forceinline__ void load_twiddles(C (&w)[TPT], const C *tw, int n) {
#pragma unroll
  for (int i = 0; i < TPT; i++) {
    const int e = threadIdx.x + i * FFT_TPB;
    if (e < n) w[i] = tw[e];
  }
}
template <typename C>
__device__ __forceinline__ void put_twiddles(C *tws, const C (&w)[TPT], int n, bool conj_) {
#pragma unroll
  for (int i = 0; i < TPT; i++) {
    const int e = threadIdx.x + i * FFT_TPB;
    if (e < n) tws[e] = conj_ ? mkc<C>(w[i].x, -w[i].y) : w[i];
  }
}

// forward pass 1: r2c along x of every row (k, y) -> C1[k][y][l], l <= nx/2.  Two real rows
// a, b share one complex transform Z = FFT(a + i b): A[l] = (Z[l] + conj Z[n-l]) / 2 and
// B[l] = (Z[l] - conj Z[n-l]) / (2i).
template <typename S, int NT>
__global__ void __launch_bounds__(FFT_TPB) k_rows_r2c(Plan p, const cx_t<S> *__restrict__ tw,
                                                      FieldPtrs fp, cx_t<S> *__restrict__ c1,
                                                      int64_t c1_field, int nrows, int nb) {
  using C = cx_t<S>;
  constexpr int EPT = ept_rows<S>();
  __shared__ C A[lds_rows<S>()], B[lds_rows<S>()], T[512];
  const int f = blockIdx.y;
  const S *src = static_cast<const S *>(fp.in[f]);
  C *dst = c1 + (int64_t)f * c1_field;
  const int n = NT ? NT : p.n, nl = n / 2 + 1;
  const int r0 = blockIdx.x * 2 * nb;                  // first row of this workgroup
  const int nbb = min(nb, (nrows - r0 + 1) / 2);       // transforms (row pairs)
  C w[TPT], v[EPT];
  load_twiddles(w, tw, n);
#pragma unroll
  for (int i = 0; i < EPT; i++) {
    const int e = threadIdx.x + i * FFT_TPB;
    if (e < nbb * n) {
      const int t = e / n, x = e - t * n;
      const int ra = r0 + 2 * t, rb = ra + 1;
      v[i].x = src[(int64_t)ra * n + x];
      v[i].y = (rb < nrows) ? src[(int64_t)rb * n + x] : (S)0;
    }
  }
  put_twiddles(T, w, n, false);
#pragma unroll
  for (int i = 0; i < EPT; i++) {
    const int e = threadIdx.x + i * FFT_TPB;
    if (e < nbb * n) A[e] = v[i];
  }
  __syncthreads();
  C *R = lds_fft<false, NT>(A, B, T, p, nbb);
  for (int e = threadIdx.x; e < nbb * nl; e += FFT_TPB) {
    const int t = e / nl, l = e - t * nl;
    const int ra = r0 + 2 * t, rb = ra + 1;
    const C z = R[t * n + l];
    const C w = R[t * n + (l == 0 ? 0 : n - l)];  // Z[n-l]
    dst[(int64_t)ra * nl + l] = mkc<C, S>((z.x + w.x) / 2, (z.y - w.y) / 2);
    if (rb < nrows) dst[(int64_t)rb * nl + l] = mkc<C, S>((z.y + w.y) / 2, (w.x - z.x) / 2);
  }
}

// a block's four values (one 16-byte FP32 vector, or two FP64 pairs)
template <typename S>
struct alignas(4 * sizeof(S) > 16 ? 16 : 4 * sizeof(S)) Quad {
  S v[4];  // a = 0: (Re, Im) of the x transform, a = 1: (Re, Im)
};

// a block's derivative along x or y (kw: its wavenumber), element for element as the standalone
// diffx / diffy compute it (fft_ops.F90:266-269, :366-369)
template <typename S>
__device__ __forceinline__ Quad<S> derivative(const Quad<S> &u, int op, S kw) {
  if (op == SPEC_DX)  // pair swap along x
    return Quad<S>{((S)-1. * u.v[1]) * kw, u.v[0] * kw, ((S)-1. * u.v[3]) * kw, u.v[2] * kw};
  if (op == SPEC_DY)  // pair swap along y
    return Quad<S>{((S)-1. * u.v[2]) * kw, ((S)-1. * u.v[3]) * kw, u.v[0] * kw, u.v[1] * kw};
  return u;
}

// forward pass 2: complex FFT along y of nb adjacent columns l of one z level, then the
// (Re,Im)-pair split into the semi-spectral layout
template <typename S, int NT>
__global__ void __launch_bounds__(FFT_TPB) k_cols_fwd(Plan p, const cx_t<S> *__restrict__ tw,
                                                      FieldPtrs fp, const cx_t<S> *__restrict__ c1,
                                                      int64_t c1_field, int nl, int nb, int nzn) {
  using C = cx_t<S>;
  constexpr int EPT = lds_cols<S>(NT, false) / FFT_TPB;
  __shared__ C A[lds_cols<S>(NT, false)], B[lds_cols<S>(NT, false)], T[512];
  const int f = blockIdx.z;
  const C *src = c1 + (int64_t)f * c1_field;
  S *dst = static_cast<S *>(fp.out[f]);
  const int ny = NT ? NT : p.n;
  const int nbd = NT ? col_batch<S>(NT, false) : nb;  // the batch every workgroup but the last takes
  const int k = blockIdx.y;
  const int l0 = blockIdx.x * nb;
  const int nbb = min(nb, nl - l0);
  const C *lev = src + (int64_t)k * ny * nl;
  C w[TPT];
  S vx[EPT], vy[EPT];
  int at[EPT];
  load_twiddles(w, tw, ny);
#pragma unroll
  for (int i = 0; i < EPT; i++) {
    const int e = threadIdx.x + i * FFT_TPB;
    const int y = e / nbd, t = e - y * nbd;
    at[i] = (y < ny && t < nbb) ? t * ny + y : -1;
    vx[i] = 0;
    vy[i] = 0;
    if (at[i] >= 0) {
      const C u = lev[(int64_t)y * nl + l0 + t];
      vx[i] = u.x;
      vy[i] = u.y;
    }
  }
  put_twiddles(T, w, ny, false);
#pragma unroll
  for (int i = 0; i < EPT; i++)
    if (at[i] >= 0) A[at[i]] = mkc<C, S>(vx[i], vy[i]);
  __syncthreads();
  C *R = lds_fft<false, NT>(A, B, T, p, nbb);
  const int nm = ny / 2 + 1;
  for (int e = threadIdx.x; e < nbd * nm; e += FFT_TPB) {
    const int m = e / nbd, t = e - m * nbd;
    if (t >= nbb) continue;
    const int l = l0 + t;
    C g = R[t * ny + m];
    C h = R[t * ny + ((ny - m) % ny)];
    C s = mkc<C, S>(g.x + h.x, g.y + h.y);
    C d = mkc<C, S>(g.x - h.x, g.y - h.y);
    *reinterpret_cast<Quad<S> *>(dst + spec_at(nzn, nl, k, m, l)) =
        Quad<S>{s.x / 2, s.y / 2, d.y / 2, -d.x / 2};
  }
}

// inverse pass 1: per (k, m) build H = A_m + i B_m over l in [0, nx) from the two real
// x-spectra (imaginary parts of the DC and Nyquist bins dropped as c2r drops them), inverse
// FFT along x, scale 1/nx -> C2[k][m][x].  A thread loads a block (m, l) once and forms H at l and
// at nx - l.  Of a filtered field (9 of vort2vel's 14, whose 2/3 rule passes 35 % of the blocks) only
// what the filter passes is read, and rows past it are left out: 223 -> 187 us a call at 256x256x128
// FP32, 99 -> 87 at 128x128x128 FP64.
template <typename S, int NT>
__global__ void __launch_bounds__(FFT_TPB) k_rows_inv(Plan p, const cx_t<S> *__restrict__ tw,
                                                      FieldPtrs fp, cx_t<S> *__restrict__ c2,
                                                      int64_t c2_field, int nrows, int nm,
                                                      float rnm, int nb, int nzn) {
  using C = cx_t<S>;
  // blocks per thread: nl = nx / 2 + 1 of nb = lds_rows / nx rows
  constexpr int EPT = NT > 0 ? (lds_rows<S>() / NT * (NT / 2 + 1) + FFT_TPB - 1) / FFT_TPB
                             : ept_rows<S>();
  __shared__ C A[lds_rows<S>()], B[lds_rows<S>()], T[512];
  const int f = blockIdx.y;
  const S *src = static_cast<const S *>(fp.in[f]);
  const int op = fp.op[f] & 3;
  const bool filtered = fp.op[f] & SPEC_FILTERED;
  C *dst = c2 + (int64_t)f * c2_field;
  const int nx = NT ? NT : p.n, nl = nx / 2 + 1;
  const int r0 = blockIdx.x * nb;
  const int nbb = min(nb, nrows - r0);
  if (filtered) {  // all rows past the filter: nothing to write, k_cols_c2r reads none of them
    int m;
    div_small(r0, nm, rnm, m);
    if (m >= fp.mcut && m + nbb <= nm) return;
  }
  C w[TPT];
  Quad<S> q[EPT];
  load_twiddles(w, tw, nx);
#pragma unroll
  for (int i = 0; i < EPT; i++) {
    const int e = threadIdx.x + i * FFT_TPB;
    if (e < nbb * nl) {
      const int t = e / nl, l = e - t * nl;
      int m;
      const int k = div_small(r0 + t, nm, rnm, m);  // row = k * nm + m
      q[i] = Quad<S>{0, 0, 0, 0};
      if (filtered && l >= fp.lcut[m]) continue;
      q[i] = *reinterpret_cast<const Quad<S> *>(src + spec_at(nzn, nl, k, m, l));
      if (op != SPEC_PLAIN) {
        // kx depends on l and ky on m only
        const S kw = (S)(op == SPEC_DX ? fp.kx[2 * l] : fp.ky[(int64_t)(2 * m) * (2 * nl)]);
        q[i] = derivative(q[i], op, kw);
      }
    }
  }
  put_twiddles(T, w, nx, true);
#pragma unroll
  for (int i = 0; i < EPT; i++) {
    const int e = threadIdx.x + i * FFT_TPB;
    if (e < nbb * nl) {
      const int t = e / nl, l = e - t * nl;
      const S ar = q[i].v[0], ai = q[i].v[1], br = q[i].v[2], bi = q[i].v[3];
      if (l == 0 || 2 * l == nx) {
        A[t * nx + l] = mkc<C, S>(ar, br);
      } else {
        A[t * nx + l] = mkc<C, S>(ar - bi, ai + br);
        A[t * nx + nx - l] = mkc<C, S>(ar + bi, -ai + br);
      }
    }
  }
  __syncthreads();
  C *R = lds_fft<true, NT>(A, B, T, p, nbb);
  const S dn = (S)1 / (S)nx;
  for (int e = threadIdx.x; e < nbb * nx; e += FFT_TPB) {
    int t = e / nx, x = e - t * nx;
    C v = R[t * nx + x];
    dst[(int64_t)(r0 + t) * nx + x] = mkc<C, S>(v.x * dn, v.y * dn);
  }
}

// inverse pass 2: c2r along y for 2 nb adjacent x columns of one z level.  The Hermitian
// spectra of two columns a, b share one complex inverse transform of H_a + i H_b, whose real
// and imaginary parts are the two real columns.
template <typename S, int NT>
__global__ void __launch_bounds__(FFT_TPB) k_cols_c2r(Plan p, const cx_t<S> *__restrict__ tw,
                                                      FieldPtrs fp, const cx_t<S> *__restrict__ c2,
                                                      int64_t c2_field, int nx, int nb) {
  using C = cx_t<S>;
  constexpr int EPT = lds_cols<S>(NT, true) / FFT_TPB;
  __shared__ C A[lds_cols<S>(NT, true)], B[lds_cols<S>(NT, true)], T[512];
  const int f = blockIdx.z;
  const C *src = c2 + (int64_t)f * c2_field;
  double *dst = static_cast<double *>(fp.out[f]);
  const int ny = NT ? NT : p.n, nm = ny / 2 + 1;
  const int nbd = NT ? col_batch<S>(NT, true) : nb;  // the batch every workgroup but the last takes
  const int k = blockIdx.y;
  const int x0 = blockIdx.x * 2 * nb;
  const int nbb = min(nb, (nx - x0 + 1) / 2);
  const C *lev = src + (int64_t)k * nm * nx;
  const int mlim = (fp.op[f] & SPEC_FILTERED) ? fp.mcut : nm;  // rows past it are zero
  const bool even = (ny % 2) == 0;
  C w[TPT], va[EPT], vb[EPT];
  load_twiddles(w, tw, ny);
#pragma unroll
  for (int i = 0; i < EPT; i++) {
    const int e = threadIdx.x + i * FFT_TPB;
    const int y = e / nbd, t = e - y * nbd;
    if (y < ny && t < nbb) {
      const int xa = x0 + 2 * t, xb = xa + 1;
      const int m = (y < nm) ? y : ny - y;
      va[i] = m < mlim ? lev[(int64_t)m * nx + xa] : mkc<C, S>(0, 0);
      vb[i] = m < mlim && xb < nx ? lev[(int64_t)m * nx + xb] : mkc<C, S>(0, 0);
    }
  }
  put_twiddles(T, w, ny, true);
#pragma unroll
  for (int i = 0; i < EPT; i++) {
    const int e = threadIdx.x + i * FFT_TPB;
    const int y = e / nbd, t = e - y * nbd;
    if (y < ny && t < nbb) {
      const int m = (y < nm) ? y : ny - y;
      C wa = va[i], wb = vb[i];
      if (m == 0 || (even && m == ny / 2)) { wa.y = 0; wb.y = 0; }
      if (y >= nm) { wa.y = -wa.y; wb.y = -wb.y; }
      A[t * ny + y] = mkc<C, S>(wa.x - wb.y, wa.y + wb.x);
    }
  }
  __syncthreads();
  C *R = lds_fft<true, NT>(A, B, T, p, nbb);
  const S dn = (S)1 / (S)ny;
  // either output may be absent: the FP32-bulk form keeps some fields only in FP32
  double *out = dst ? dst + (int64_t)k * ny * nx : nullptr;
  float *o32 = fp.out32[f] ? fp.out32[f] + (int64_t)k * ny * nx : nullptr;
  for (int e = threadIdx.x; e < nbd * ny; e += FFT_TPB) {
    const int y = e / nbd, t = e - y * nbd;
    if (t >= nbb) continue;
    const int xa = x0 + 2 * t, xb = xa + 1;
    const C v = R[t * ny + y];
    if (out) {
      out[(int64_t)y * nx + xa] = v.x * dn;
      if (xb < nx) out[(int64_t)y * nx + xb] = v.y * dn;
    }
    if (o32) {
      o32[(int64_t)y * nx + xa] = (float)(v.x * dn);
      if (xb < nx) o32[(int64_t)y * nx + xb] = (float)(v.y * dn);
    }
  }
}

// ---- both passes of a plane in one workgroup ----
// A small plane fits the LDS whole: its x and y transforms are then one launch, without the
// intermediate in memory.  Small grids are bound by the latency of a launch and of its chain of
// loads, stages and stores, not by the rate.  The forward and inverse calls of a timestep, before
// and after: 11.0 + 17.4 -> 8.5 + 13.5 us at 48^3 FP32, 16.6 + 32 -> 12.1 + 20.3 at 90x60x41 FP32,
// 8.9 + 10.0 -> 5.7 + 5.7 at 12x10x8 FP64, each with a gap between launches less.  The transforms
// are the two-pass kernels', value for value.

// exact q = a / d for a < 2^23 and 0 < d <= 512, m = floor(2^32 / d) + 1 (0 stands for 2^32, d = 1)
__device__ __forceinline__ int div_magic(int a, uint32_t m) {
  return m ? (int)__umulhi((uint32_t)a, m) : a;
}
inline uint32_t magic_of(int d) { return d == 1 ? 0u : (uint32_t)((1ull << 32) / d) + 1u; }

// a transform of a plane: `count` of them of length n, and the stages' divisors
struct PlanePass {
  Plan p;
  int count;
  uint32_t mn, mnq[10], mns[10];
};
PlanePass plane_pass(int n, int count) {
  PlanePass pp{};
  pp.p = make_plan(n);
  pp.count = count;
  pp.mn = magic_of(n);
  int ns = 1;
  for (int s = 0; s < pp.p.nrad; s++) {
    const int r = (int)((pp.p.code >> (4 * s)) & 15u);
    pp.mnq[s] = magic_of(n / r);
    pp.mns[s] = magic_of(ns);
    ns *= r;
  }
  return pp;
}

template <int R, bool INV, int TPBP, typename C>
__device__ __forceinline__ void plane_stage(const C *x, C *y, const C *tw, int n, int Ns, int nb,
                                            uint32_t mnq, uint32_t mns) {
  const int nq = n / R;  // R divides n
  const int tstep = div_magic(nq, mns);
  const int tot = nb * nq;
  for (int bi = threadIdx.x; bi < tot; bi += TPBP) {
    const int t = div_magic(bi, mnq), i = bi - t * nq;
    const int j = div_magic(i, mns), k = i - j * Ns;
    const C *xs = x + t * n + i;
    C v[R];
#pragma unroll
    for (int q = 0; q < R; q++) {
      const C e = xs[q * nq];
      v[q] = (q == 0 || k == 0) ? e : cmul(e, tw[q * k * tstep]);
    }
    dft<R, INV>(v);
    C *ys = y + t * n + j * Ns * R + k;
#pragma unroll
    for (int o = 0; o < R; o++) ys[o * Ns] = v[o];
  }
}

template <bool INV, int TPBP, typename C>
__device__ __forceinline__ void plane_fft(C *&a, C *&b, const C *tw, const PlanePass &pp) {
  int Ns = 1;
  for (int s = 0; s < pp.p.nrad; s++) {
    const int r = (int)((pp.p.code >> (4 * s)) & 15u);
    const uint32_t mq = pp.mnq[s], ms = pp.mns[s];
    if (r == 4) plane_stage<4, INV, TPBP>(a, b, tw, pp.p.n, Ns, pp.count, mq, ms);
    else if (r == 2) plane_stage<2, INV, TPBP>(a, b, tw, pp.p.n, Ns, pp.count, mq, ms);
    else if (r == 3) plane_stage<3, INV, TPBP>(a, b, tw, pp.p.n, Ns, pp.count, mq, ms);
    else plane_stage<5, INV, TPBP>(a, b, tw, pp.p.n, Ns, pp.count, mq, ms);
    __syncthreads();
    C *sw = a;
    a = b;
    b = sw;
    Ns *= r;
  }
}

// loads of a thread in flight at once
constexpr int PLANE_BATCH = 4;

// forward: x rows in pairs, as k_rows_r2c takes them, then the columns, as k_cols_fwd does
template <typename S, int TPBP>
__global__ void __launch_bounds__(TPBP) k_plane_fwd(PlanePass px, PlanePass py,
                                                    const cx_t<S> *__restrict__ twx,
                                                    const cx_t<S> *__restrict__ twy, FieldPtrs fp,
                                                    int cap, int nzn, uint32_t mnl, uint32_t mrows) {
  using C = cx_t<S>;
  extern __shared__ double2 plane_lds[];
  C *a = reinterpret_cast<C *>(plane_lds), *b = a + cap, *tx = b + cap, *ty = tx + px.p.n;
  const int k = blockIdx.x, f = blockIdx.y, tid = threadIdx.x;
  const int nx = px.p.n, ny = py.p.n, nl = nx / 2 + 1, rows = px.count;
  const S *src = static_cast<const S *>(fp.in[f]) + (int64_t)k * ny * nx;
  for (int e = tid; e < nx; e += TPBP) tx[e] = twx[e];
  for (int e = tid; e < ny; e += TPBP) ty[e] = twy[e];
  for (int e0 = tid; e0 < rows * nx; e0 += PLANE_BATCH * TPBP) {
    C v[PLANE_BATCH];
#pragma unroll
    for (int i = 0; i < PLANE_BATCH; i++) {
      const int e = e0 + i * TPBP;
      if (e < rows * nx) {
        const int t = div_magic(e, px.mn), x = e - t * nx;
        v[i].x = src[2 * t * nx + x];
        v[i].y = 2 * t + 1 < ny ? src[(2 * t + 1) * nx + x] : (S)0;
      }
    }
#pragma unroll
    for (int i = 0; i < PLANE_BATCH; i++)
      if (e0 + i * TPBP < rows * nx) a[e0 + i * TPBP] = v[i];
  }
  __syncthreads();
  plane_fft<false, TPBP>(a, b, tx, px);
  // columns: transform l, element y at l ny + y
  for (int e = tid; e < nl * rows; e += TPBP) {
    const int l = div_magic(e, mrows), t = e - l * rows;
    const C z = a[t * nx + l], w = a[t * nx + (l == 0 ? 0 : nx - l)];
    b[l * ny + 2 * t] = mkc<C, S>((z.x + w.x) / 2, (z.y - w.y) / 2);
    if (2 * t + 1 < ny) b[l * ny + 2 * t + 1] = mkc<C, S>((z.y + w.y) / 2, (w.x - z.x) / 2);
  }
  __syncthreads();
  plane_fft<false, TPBP>(b, a, ty, py);
  S *dst = static_cast<S *>(fp.out[f]);
  for (int e = tid; e < (ny / 2 + 1) * nl; e += TPBP) {
    const int m = div_magic(e, mnl), l = e - m * nl;
    const C g = b[l * ny + m], h = b[l * ny + (m == 0 ? 0 : ny - m)];
    const C s = mkc<C, S>(g.x + h.x, g.y + h.y), d = mkc<C, S>(g.x - h.x, g.y - h.y);
    *reinterpret_cast<Quad<S> *>(dst + spec_at(nzn, nl, k, m, l)) =
        Quad<S>{s.x / 2, s.y / 2, d.y / 2, -d.x / 2};
  }
}

// inverse: the rows m as k_rows_inv takes them, then the columns in pairs, as k_cols_c2r does
template <typename S, int TPBP>
__global__ void __launch_bounds__(TPBP) k_plane_inv(PlanePass px, PlanePass py,
                                                    const cx_t<S> *__restrict__ twx,
                                                    const cx_t<S> *__restrict__ twy, FieldPtrs fp,
                                                    int cap, int nzn, uint32_t mnl, uint32_t mcols) {
  using C = cx_t<S>;
  constexpr int BATCH = PLANE_BATCH * 4 / sizeof(S);  // half as many FP64 blocks
  extern __shared__ double2 plane_lds[];
  C *a = reinterpret_cast<C *>(plane_lds), *b = a + cap, *tx = b + cap, *ty = tx + px.p.n;
  const int k = blockIdx.x, f = blockIdx.y, tid = threadIdx.x, op = fp.op[f] & 3;
  const int nx = px.p.n, ny = py.p.n, nl = nx / 2 + 1, nm = px.count, cols = py.count;
  const S *src = static_cast<const S *>(fp.in[f]);
  for (int e = tid; e < nx; e += TPBP) tx[e] = mkc<C, S>(twx[e].x, -twx[e].y);
  for (int e = tid; e < ny; e += TPBP) ty[e] = mkc<C, S>(twy[e].x, -twy[e].y);
  for (int e0 = tid; e0 < nm * nl; e0 += BATCH * TPBP) {
    Quad<S> q[BATCH];
    S kw[BATCH];
#pragma unroll
    for (int i = 0; i < BATCH; i++) {
      const int e = e0 + i * TPBP;
      if (e < nm * nl) {
        const int m = div_magic(e, mnl), l = e - m * nl;
        q[i] = *reinterpret_cast<const Quad<S> *>(src + spec_at(nzn, nl, k, m, l));
        if (op != SPEC_PLAIN)
          kw[i] = (S)(op == SPEC_DX ? fp.kx[2 * l] : fp.ky[(int64_t)(2 * m) * (2 * nl)]);
      }
    }
#pragma unroll
    for (int i = 0; i < BATCH; i++) {
      const int e = e0 + i * TPBP;
      if (e < nm * nl) {
        const int m = div_magic(e, mnl), l = e - m * nl;
        const Quad<S> u = derivative(q[i], op, kw[i]);
        const S ar = u.v[0], ai = u.v[1], br = u.v[2], bi = u.v[3];
        if (l == 0 || 2 * l == nx) {
          a[m * nx + l] = mkc<C, S>(ar, br);
        } else {
          a[m * nx + l] = mkc<C, S>(ar - bi, ai + br);
          a[m * nx + nx - l] = mkc<C, S>(ar + bi, -ai + br);
        }
      }
    }
  }
  __syncthreads();
  plane_fft<true, TPBP>(a, b, tx, px);
  const S dnx = (S)1 / (S)nx, dny = (S)1 / (S)ny;
  const bool even = (ny % 2) == 0;
  // columns 2 t, 2 t + 1 as one transform: element y at t ny + y
  for (int e = tid; e < cols * ny; e += TPBP) {
    const int y = div_magic(e, mcols), t = e - y * cols;
    const int m = y < nm ? y : ny - y;
    C wa = a[m * nx + 2 * t], wb = 2 * t + 1 < nx ? a[m * nx + 2 * t + 1] : mkc<C, S>(0, 0);
    wa.x *= dnx; wa.y *= dnx; wb.x *= dnx; wb.y *= dnx;
    if (m == 0 || (even && m == ny / 2)) { wa.y = 0; wb.y = 0; }
    if (y >= nm) { wa.y = -wa.y; wb.y = -wb.y; }
    b[t * ny + y] = mkc<C, S>(wa.x - wb.y, wa.y + wb.x);
  }
  __syncthreads();
  plane_fft<true, TPBP>(b, a, ty, py);
  double *out = static_cast<double *>(fp.out[f]);
  float *o32 = fp.out32[f];
  for (int e = tid; e < cols * ny; e += TPBP) {
    const int y = div_magic(e, mcols), t = e - y * cols;
    const C v = b[t * ny + y];
    const int64_t at = ((int64_t)k * ny + y) * nx + 2 * t;
    if (out) {
      out[at] = v.x * dny;
      if (2 * t + 1 < nx) out[at + 1] = v.y * dny;
    }
    if (o32) {
      o32[at] = (float)(v.x * dny);
      if (2 * t + 1 < nx) o32[at + 1] = (float)(v.y * dny);
    }
  }
}

// W_n^e for e in [0, n), in FP64 and rounded to FP32
int upload_twiddles(int n, double2 **dptr, float2 **dptr32) {
  std::vector<double2> h(n);
  std::vector<float2> h32(n);
  for (int e = 0; e < n; e++) {
    // quarter turns are exact so that purely real or imaginary inputs stay so
    if ((4L * e) % n == 0) {
      const int q = (int)((4L * e) / n);
      const double re[4] = {1.0, 0.0, -1.0, 0.0}, im[4] = {0.0, -1.0, 0.0, 1.0};
      h[e] = make_double2(re[q], im[q]);
    } else {
      long double ang = -2.0L * 3.14159265358979323846264338327950288L * (long double)e / (long double)n;
      h[e] = make_double2((double)cosl(ang), (double)sinl(ang));
    }
    h32[e] = make_float2((float)h[e].x, (float)h[e].y);
  }
  PMPIC_CHECK(hipMalloc(dptr, sizeof(double2) * n));
  PMPIC_CHECK(hipMemcpy(*dptr, h.data(), sizeof(double2) * n, hipMemcpyHostToDevice));
  PMPIC_CHECK(hipMalloc(dptr32, sizeof(float2) * n));
  PMPIC_CHECK(hipMemcpy(*dptr32, h32.data(), sizeof(float2) * n, hipMemcpyHostToDevice));
  return PMPIC_OK;
}

template <typename S> const cx_t<S> *twiddles_x(const Ctx *c);
template <> const double2 *twiddles_x<double>(const Ctx *c) { return c->tw_x; }
template <> const float2 *twiddles_x<float>(const Ctx *c) { return c->tw_x32; }
template <typename S> const cx_t<S> *twiddles_y(const Ctx *c);
template <> const double2 *twiddles_y<double>(const Ctx *c) { return c->tw_y; }
template <> const float2 *twiddles_y<float>(const Ctx *c) { return c->tw_y32; }

}  // namespace

int fft_setup(Ctx *c) {
  if (c->g.nx > 512 || c->g.ny > 512) return PMPIC_ERR_FFT_SIZE;
  if (make_plan(c->g.nx).nrad < 0 || make_plan(c->g.ny).nrad < 0) return PMPIC_ERR_FFT_SIZE;
  PMPIC_TRY(upload_twiddles(c->g.nx, &c->tw_x, &c->tw_x32));
  PMPIC_TRY(upload_twiddles(c->g.ny, &c->tw_y, &c->tw_y32));
  return PMPIC_OK;
}

static int64_t c1_field_size(const Geometry &g) { return (int64_t)g.nzn * g.ny * (g.nx / 2 + 1); }
static int64_t c2_field_size(const Geometry &g) { return (int64_t)g.nzn * (g.ny / 2 + 1) * g.nx; }

// f(std::integral_constant<int, N>) with N = n for a length in FIXED_N, else N = 0
template <class F>
int with_length(int n, F &&f) {
  switch (n) {
    case 16: return f(std::integral_constant<int, 16>{});
    case 32: return f(std::integral_constant<int, 32>{});
    case 48: return f(std::integral_constant<int, 48>{});
    case 64: return f(std::integral_constant<int, 64>{});
    case 96: return f(std::integral_constant<int, 96>{});
    case 128: return f(std::integral_constant<int, 128>{});
    case 256: return f(std::integral_constant<int, 256>{});
    case 512: return f(std::integral_constant<int, 512>{});
    default: return f(std::integral_constant<int, 0>{});
  }
}
static_assert(sizeof(FIXED_N) / sizeof(int) == 8, "with_length lists every fixed length");

// LDS of a plane kernel (two buffers of `cap` elements and the twiddles), or 0 where the two-pass
// kernels run: planes past 64 KB, and grids of more than 2^18 nodes whose lengths both have kernels
// compiled for them (the two passes then run at the memory's rate).  FP32 steps, plane / two-pass:
// 48^3 524 / 548 us, 72x72x30 614 / 682, 80x80x48 851 / 928, but 64^3 834 / 822, 96x64x64 1045 /
// 1028; FP64 64x48x64 1203 / 1245 us.
constexpr size_t PLANE_LDS = 64 * 1024;
constexpr int64_t PLANE_NODES = (int64_t)1 << 18;
inline bool fixed_length(int n) {
  for (int f : FIXED_N)
    if (f == n) return true;
  return false;
}
template <typename S>
static size_t plane_lds(const Geometry &g, int &cap) {
  const int nl = g.nx / 2 + 1, nm = g.ny / 2 + 1;
  cap = std::max(std::max((g.ny + 1) / 2 * g.nx, nl * g.ny),
                 std::max(nm * g.nx, (g.nx + 1) / 2 * g.ny));
  const size_t bytes = sizeof(cx_t<S>) * (2 * (size_t)cap + g.nx + g.ny);
  if (fixed_length(g.nx) && fixed_length(g.ny) && (int64_t)g.nzn * g.ny * g.nx > PLANE_NODES) return 0;
  return bytes <= PLANE_LDS ? bytes : 0;
}
// two wavefronts for planes of up to 512 points, eight above
constexpr int PLANE_SMALL = 512;

template <typename S>
int fft_forward_t(Ctx *c, int nf, const S *const *src, S *const *dst) {
  const Geometry &g = c->g;
  if (nf < 1 || nf > MAXF) return PMPIC_ERR_ARG;
  FieldPtrs fp{};
  for (int f = 0; f < nf; f++) { fp.in[f] = src[f]; fp.out[f] = dst[f]; }
  int cap;
  if (const size_t lds = plane_lds<S>(g, cap)) {
    const int rows = (g.ny + 1) / 2, nl = g.nx / 2 + 1;
    const bool small = g.nx * g.ny <= PLANE_SMALL;
    auto kernel = small ? k_plane_fwd<S, 128> : k_plane_fwd<S, 512>;
    hipLaunchKernelGGL(kernel, dim3(g.nzn, nf), dim3(small ? 128 : 512), lds, c->stream,
                       plane_pass(g.nx, rows), plane_pass(g.ny, nl), twiddles_x<S>(c),
                       twiddles_y<S>(c), fp, cap, g.nzn, magic_of(nl), magic_of(rows));
    PMPIC_CHECK(hipGetLastError());
    return PMPIC_OK;
  }
  const Plan px = make_plan(g.nx), py = make_plan(g.ny);
  const int64_t c1f = c1_field_size(g);
  const int nrows = g.nzn * g.ny;
  cx_t<S> *cb = reinterpret_cast<cx_t<S> *>(c->cbuf);
  const int nbx = lds_rows<S>() / g.nx;  // transforms per workgroup, two rows each
  with_length(g.nx, [&](auto N) {
    hipLaunchKernelGGL((k_rows_r2c<S, decltype(N)::value>), dim3(cdiv(nrows, 2 * nbx), nf),
                       dim3(FFT_TPB), 0, c->stream, px, twiddles_x<S>(c), fp, cb, c1f, nrows, nbx);
    return 0;
  });
  const int nl = g.nx / 2 + 1;
  const int nby = col_batch<S>(g.ny, false);
  with_length(g.ny, [&](auto N) {
    hipLaunchKernelGGL((k_cols_fwd<S, decltype(N)::value>), dim3(cdiv(nl, nby), g.nzn, nf),
                       dim3(FFT_TPB), 0, c->stream, py, twiddles_y<S>(c), fp, cb, c1f, nl, nby,
                       g.nzn);
    return 0;
  });
  PMPIC_CHECK(hipGetLastError());
  return PMPIC_OK;
}

template <typename S>
int fft_backward_t(Ctx *c, int nf, const S *const *src, double *const *dst, float *const *dst32,
                   const int *deriv) {
  const Geometry &g = c->g;
  if (nf < 1 || nf > MAXF) return PMPIC_ERR_ARG;
  FieldPtrs fp{};
  fp.kx = c->kx;
  fp.ky = c->ky;
  fp.lcut = c->lcut;
  fp.mcut = c->mcut;
  for (int f = 0; f < nf; f++) {
    fp.in[f] = src[f];
    fp.out[f] = dst[f];
    fp.out32[f] = dst32 ? dst32[f] : nullptr;
    fp.op[f] = deriv ? deriv[f] : SPEC_PLAIN;
    if ((fp.op[f] & 3) > SPEC_DY) return PMPIC_ERR_ARG;
  }
  int cap;
  if (const size_t lds = plane_lds<S>(g, cap)) {
    const int nl = g.nx / 2 + 1, cols = (g.nx + 1) / 2;
    const bool small = g.nx * g.ny <= PLANE_SMALL;
    auto kernel = small ? k_plane_inv<S, 128> : k_plane_inv<S, 512>;
    hipLaunchKernelGGL(kernel, dim3(g.nzn, nf), dim3(small ? 128 : 512), lds, c->stream,
                       plane_pass(g.nx, g.ny / 2 + 1), plane_pass(g.ny, cols), twiddles_x<S>(c),
                       twiddles_y<S>(c), fp, cap, g.nzn, magic_of(nl), magic_of(cols));
    PMPIC_CHECK(hipGetLastError());
    return PMPIC_OK;
  }
  const Plan px = make_plan(g.nx), py = make_plan(g.ny);
  const int64_t c2f = c2_field_size(g);
  const int nm = g.ny / 2 + 1;
  const int nrows = g.nzn * nm;
  if (nrows >= (1 << 22)) return PMPIC_ERR_ARG;  // the row split's reciprocal division
  const float rnm = (float)(1.0 / nm);
  cx_t<S> *cb = reinterpret_cast<cx_t<S> *>(c->cbuf);
  const int nbx = lds_rows<S>() / g.nx;
  with_length(g.nx, [&](auto N) {
    hipLaunchKernelGGL((k_rows_inv<S, decltype(N)::value>), dim3(cdiv(nrows, nbx), nf),
                       dim3(FFT_TPB), 0, c->stream, px, twiddles_x<S>(c), fp, cb, c2f, nrows, nm,
                       rnm, nbx, g.nzn);
    return 0;
  });
  const int nby = col_batch<S>(g.ny, true);  // transforms per workgroup, two x columns each
  with_length(g.ny, [&](auto N) {
    hipLaunchKernelGGL((k_cols_c2r<S, decltype(N)::value>), dim3(cdiv(g.nx, 2 * nby), g.nzn, nf),
                       dim3(FFT_TPB), 0, c->stream, py, twiddles_y<S>(c), fp, cb, c2f, g.nx, nby);
    return 0;
  });
  PMPIC_CHECK(hipGetLastError());
  return PMPIC_OK;
}

template int fft_forward_t<double>(Ctx *, int, const double *const *, double *const *);
template int fft_forward_t<float>(Ctx *, int, const float *const *, float *const *);
template int fft_backward_t<double>(Ctx *, int, const double *const *, double *const *,
                                    float *const *, const int *);
template int fft_backward_t<float>(Ctx *, int, const float *const *, double *const *,
                                   float *const *, const int *);

int fft_forward(Ctx *c, int nf, const double *const *src, double *const *dst) {
  return fft_forward_t<double>(c, nf, src, dst);
}

int fft_backward(Ctx *c, int nf, const double *const *src, double *const *dst,
                 float *const *dst32, const int *deriv) {
  return fft_backward_t<double>(c, nf, src, dst, dst32, deriv);
}

}  // namespace pmpic
