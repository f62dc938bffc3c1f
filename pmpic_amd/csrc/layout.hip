// Conversions between the library's device layouts (common.h) and the reference's host layouts
// (z fastest; include/pmpic_hip.h), on the device, so that a transfer is one copy in the host's
// own order.
//
// Every conversion is a transposition of (x or lane, z) for each y or tile: both sides have long
// contiguous runs, along x (or a tile's 64 lanes) on one side and along z on the other, so a
// 32 x 32 block goes through LDS and is read and written in 256-byte runs.  Bound by memory; the
// host loops it replaces took 64 ms for a 256x256x129 grid, the copy to the host takes 4-7.
#include "common.h"

namespace pmpic {

namespace {

constexpr int TD = 32;   // block edge
constexpr int TY = 8;    // thread rows of a 32 x 8 workgroup

// grid rows in[(k ny + j) nx + i] (every `stride`-th value) <-> ref[(ih nyh + jh) nz + k], with
// h halo cells in x and y holding periodic copies (to the reference) or left alone (from it)
template <typename T>
__global__ void k_rows_to_ref(const T *__restrict__ in, int stride, int nx, int ny, int nz, int h,
                              double *__restrict__ ref) {
  __shared__ double t[TD][TD + 1];
  const int jh = blockIdx.z, nyh = ny + 2 * h;
  int j = jh - h;
  j = j < 0 ? j + ny : j >= ny ? j - ny : j;
  const int ih0 = blockIdx.x * TD, k0 = blockIdx.y * TD;
  int i = ih0 + (int)threadIdx.x - h;
  i = i < 0 ? i + nx : i >= nx ? i - nx : i;
  const bool in_x = ih0 + (int)threadIdx.x < nx + 2 * h;
  for (int r = threadIdx.y; r < TD; r += TY) {
    const int k = k0 + r;
    if (in_x && k < nz) t[r][threadIdx.x] = (double)in[(((int64_t)k * ny + j) * nx + i) * stride];
  }
  __syncthreads();
  const int k = k0 + (int)threadIdx.x;
  for (int r = threadIdx.y; r < TD; r += TY) {
    const int ih = ih0 + r;
    if (ih < nx + 2 * h && k < nz) ref[((int64_t)ih * nyh + jh) * nz + k] = t[threadIdx.x][r];
  }
}

__global__ void k_ref_to_rows(const double *__restrict__ ref, int nx, int ny, int nz, int h,
                              double *__restrict__ out) {
  __shared__ double t[TD][TD + 1];
  const int j = blockIdx.z, nyh = ny + 2 * h;
  const int i0 = blockIdx.x * TD, k0 = blockIdx.y * TD;
  const int k = k0 + (int)threadIdx.x;
  for (int r = threadIdx.y; r < TD; r += TY) {
    const int i = i0 + r;
    if (i < nx && k < nz) t[threadIdx.x][r] = ref[((int64_t)(i + h) * nyh + (j + h)) * nz + k];
  }
  __syncthreads();
  const int i = i0 + (int)threadIdx.x;
  for (int r = threadIdx.y; r < TD; r += TY)
    if (i < nx && k0 + r < nz) out[((int64_t)(k0 + r) * ny + j) * nx + i] = t[r][threadIdx.x];
}

// spectral tiles <-> ref[(ii sy + jj) nz + k]; half a tile (32 lanes, 8 blocks) and 32 levels a
// workgroup
template <bool TO_REF, typename T>
__global__ void k_tiles_ref(T *__restrict__ tiles, int nl, int sy, int nz,
                            double *__restrict__ ref) {
  __shared__ double t[TD][TD + 1];
  const int lane0 = (blockIdx.x & 1) * TD, tile = blockIdx.x >> 1, k0 = blockIdx.y * TD;
  T *base = tiles + ((int64_t)tile * nz) * 64 + lane0;
  auto ref_at = [&](int lane, int k) {  // < 0 past the last block
    const int blk = tile * 16 + (lane >> 2), m = blk / nl, l = blk - m * nl;
    if (m >= sy / 2) return (int64_t)-1;
    return ((int64_t)(2 * l + (lane & 1)) * sy + 2 * m + ((lane >> 1) & 1)) * nz + k;
  };
  if (TO_REF) {
    for (int r = threadIdx.y; r < TD; r += TY)
      if (k0 + r < nz) t[r][threadIdx.x] = (double)base[(int64_t)(k0 + r) * 64 + threadIdx.x];
    __syncthreads();
    const int k = k0 + (int)threadIdx.x;
    for (int r = threadIdx.y; r < TD; r += TY) {
      const int64_t o = ref_at(lane0 + r, k);
      if (k < nz && o >= 0) ref[o] = t[threadIdx.x][r];
    }
  } else {
    const int k = k0 + (int)threadIdx.x;
    for (int r = threadIdx.y; r < TD; r += TY) {
      const int64_t o = ref_at(lane0 + r, k);
      t[threadIdx.x][r] = k < nz && o >= 0 ? ref[o] : 0.;
    }
    __syncthreads();
    for (int r = threadIdx.y; r < TD; r += TY)
      if (k0 + r < nz) base[(int64_t)(k0 + r) * 64 + threadIdx.x] = (T)t[r][threadIdx.x];
  }
}

dim3 row_blocks(int nx, int nz, int ny) {
  return dim3((unsigned)cdiv(nx, TD), (unsigned)cdiv(nz, TD), (unsigned)ny);
}

}  // namespace

template <typename T>
int grid_to_ref(Ctx *c, const T *src, int stride, double *ref) {
  const Geometry &g = c->g;
  hipLaunchKernelGGL(k_rows_to_ref<T>, row_blocks(g.nx + 4, g.nzn, g.ny + 4), dim3(TD, TY), 0,
                     c->stream, src, stride, g.nx, g.ny, g.nzn, 2, ref);
  PMPIC_CHECK(hipGetLastError());
  return PMPIC_OK;
}
template int grid_to_ref<double>(Ctx *, const double *, int, double *);
template int grid_to_ref<float>(Ctx *, const float *, int, double *);

int ref_to_grid(Ctx *c, const double *ref, double *grid) {
  const Geometry &g = c->g;
  hipLaunchKernelGGL(k_ref_to_rows, row_blocks(g.nx, g.nzn, g.ny), dim3(TD, TY), 0, c->stream, ref,
                     g.nx, g.ny, g.nzn, 2, grid);
  PMPIC_CHECK(hipGetLastError());
  return PMPIC_OK;
}

int planes_to_ref(Ctx *c, const double *planes, double *ref) {
  const Geometry &g = c->g;
  hipLaunchKernelGGL(k_rows_to_ref<double>, row_blocks(g.sx, g.nzn, g.sy), dim3(TD, TY), 0,
                     c->stream, planes, 1, g.sx, g.sy, g.nzn, 0, ref);
  PMPIC_CHECK(hipGetLastError());
  return PMPIC_OK;
}

int ref_to_planes(Ctx *c, const double *ref, double *planes) {
  const Geometry &g = c->g;
  hipLaunchKernelGGL(k_ref_to_rows, row_blocks(g.sx, g.nzn, g.sy), dim3(TD, TY), 0, c->stream, ref,
                     g.sx, g.sy, g.nzn, 0, planes);
  PMPIC_CHECK(hipGetLastError());
  return PMPIC_OK;
}

template <typename S>
int tiles_to_ref(Ctx *c, const S *tiles, double *ref) {
  const Geometry &g = c->g;
  hipLaunchKernelGGL((k_tiles_ref<true, S>), dim3(2 * spec_tiles(g), cdiv(g.nzn, TD)),
                     dim3(TD, TY), 0, c->stream, const_cast<S *>(tiles), g.sx / 2, g.sy, g.nzn,
                     ref);
  PMPIC_CHECK(hipGetLastError());
  return PMPIC_OK;
}
template int tiles_to_ref<double>(Ctx *, const double *, double *);
template int tiles_to_ref<float>(Ctx *, const float *, double *);

int ref_to_tiles(Ctx *c, const double *ref, double *tiles) {
  const Geometry &g = c->g;
  hipLaunchKernelGGL((k_tiles_ref<false, double>), dim3(2 * spec_tiles(g), cdiv(g.nzn, TD)),
                     dim3(TD, TY), 0, c->stream, tiles, g.sx / 2, g.sy, g.nzn,
                     const_cast<double *>(ref));
  PMPIC_CHECK(hipGetLastError());
  return PMPIC_OK;
}

}  // namespace pmpic
