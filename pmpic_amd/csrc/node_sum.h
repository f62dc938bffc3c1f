// Node sums of par2grid's and mixing's x-combined corner sums (both forms).
#pragma once
#include "common.h"

namespace pmpic {

// One accumulation's entries and the node grids they make.  tileres (may be null): the tiles
// whose entries were written; the others' contribute zero.
template <typename T, typename TO>
struct NodeSums {
  const T *partial;
  TO *p[7];  // null: a plane not written
  const uint8_t *tileres;
  T zmul;  // raw sums: the factor on the z boundaries
};

// Node (i, j, k) adds, for each corner pair bb = (by, bz) in a fixed order, the entry of cell row
// (j - by, k - bz) at its position, and at a tile boundary (tiles of eight cells of an x row) the
// left tile's last entry before it.  NF values: the weight, then NF - 1 weighted sums.  NORM:
// divided by the summed weights (par2grid, parcel_interpolation.F90:463-469) into NF - 1 grids;
// otherwise NF raw sums, times zmul on the z boundaries (2 for mixing's kept grids,
// parcel_mixing.F90:141-152).  gridDim.y = 2: both sets by one launch.
template <typename T, typename TO, int NF, bool NORM>
__global__ void k_node_sum(Geometry g, NodeSums<T, TO> first, NodeSums<T, TO> second) {
  const int64_t nnode = (int64_t)g.nzn * g.ny * g.nx;
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= nnode) return;
  const NodeSums<T, TO> &s_ = blockIdx.y ? second : first;
  const uint8_t *tileres = s_.tileres;
  const int i = (int)(t % g.nx);
  const int j = (int)((t / g.nx) % g.ny);
  const int k = (int)(t / ((int64_t)g.nx * g.ny));
  const int ntx = (g.nx + 7) / 8, tx = i >> 3, pos = i & 7, txl = tx == 0 ? ntx - 1 : tx - 1;
  const int64_t nrows = (int64_t)g.ny * g.ncz, W = g.nx + ntx, fstride = 4 * nrows * W;
  const int own = 9 * tx + pos, left = tx == 0 ? (int)W - 1 : 9 * tx - 1;
  T v[4][NF], vl[4][NF];
  bool ok[4], okl[4];
#pragma unroll
  for (int bb = 0; bb < 4; bb++) {
    const int by = bb & 1, bz = bb >> 1;
    int cj = j - by;
    if (cj < 0) cj += g.ny;
    const int ck = k - bz;
    const bool in = ck >= 0 && ck < g.ncz;
    const int64_t crow = in ? (int64_t)ck * g.ny + cj : 0;
    ok[bb] = in && (!tileres || tileres[crow * ntx + tx]);
    okl[bb] = in && pos == 0 && (!tileres || tileres[crow * ntx + txl]);
    const T *e = s_.partial + ((int64_t)bb * nrows + crow) * W;
#pragma unroll
    for (int f = 0; f < NF; f++) {
      v[bb][f] = ok[bb] ? e[f * fstride + own] : (T)0;
      vl[bb][f] = okl[bb] ? e[f * fstride + left] : (T)0;
    }
  }
  T s[NF];
#pragma unroll
  for (int f = 0; f < NF; f++) s[f] = 0;
#pragma unroll
  for (int bb = 0; bb < 4; bb++)
#pragma unroll
    for (int f = 0; f < NF; f++)
      if (ok[bb] || okl[bb]) s[f] = s[f] + (pos == 0 ? vl[bb][f] + v[bb][f] : v[bb][f]);
  if constexpr (NORM) {
    T w = s[0];
    if (w == (T)0) w = 1;
#pragma unroll
    for (int f = 1; f < NF; f++)
      if (s_.p[f - 1]) s_.p[f - 1][t] = (TO)(s[f] / w);
  } else {
    const T mul = k == 0 || k == g.nzn - 1 ? s_.zmul : (T)1;
#pragma unroll
    for (int f = 0; f < NF; f++)
      if (s_.p[f]) s_.p[f][t] = (TO)(s[f] * mul);
  }
}

template <typename T, typename TO, int NF, bool NORM>
void launch_node_sum(Ctx *c, const NodeSums<T, TO> &first,
                     const NodeSums<T, TO> *second = nullptr) {
  const int64_t nnode = (int64_t)c->g.nzn * c->g.ny * c->g.nx;
  hipLaunchKernelGGL((k_node_sum<T, TO, NF, NORM>), dim3(cdiv(nnode, 256), second ? 2 : 1),
                     dim3(256), 0, c->stream, c->g, first, second ? *second : first);
}

}  // namespace pmpic
