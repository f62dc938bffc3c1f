// pmpic_par2grid_noalloc: par2grid of a device array that allocates nothing.
//
// The same binning and per-cell sums as pmpic_par2grid (k_bin_count, k_bin_alloc, k_bin_scatter,
// k_cell_accum, k_node_sum), so the grid it returns is bit-identical to that entry point's.  Its
// working memory (cell and rank of each parcel, the per-cell counts and offsets, the cell-sorted
// parcel list, the corner partial sums and the interior grid) is carved out of `scratch`, one
// static device array per GPU that lives until the process ends, instead of the context's buffers
// or hipMalloc.  Inputs and the output are the caller's device arrays.
//
// Every call on a GPU shares that GPU's array, so calls that overlap (two host threads) take turns:
// a call holds the GPU's lock until the device has finished, as it waits for its status anyway.  The
// per-cell counts are zero at load and each call leaves them zero again; after one that failed the
// next clears them first.  Every other region is written in full before it is read, so nothing from
// an earlier call leaks into a later one.
#include "common.h"

#include <mutex>

#include "../../include/pmpic_hip.h"

namespace pmpic {
namespace {

constexpr int64_t NA_MAX_PARCELS = PMPIC_NOALLOC_MAX_PARCELS;
constexpr int64_t NA_MAX_CELLS = PMPIC_NOALLOC_MAX_CELLS;
constexpr size_t NA_ALIGN = 256;
constexpr size_t na_round(size_t b) { return (b + NA_ALIGN - 1) / NA_ALIGN * NA_ALIGN; }

// byte offsets of the regions inside `scratch`
constexpr size_t NA_CELL = 0;
constexpr size_t NA_RANK = NA_CELL + na_round(4 * NA_MAX_PARCELS);
constexpr size_t NA_SORTED = NA_RANK + na_round(4 * NA_MAX_PARCELS);
constexpr size_t NA_COUNT = NA_SORTED + na_round(4 * NA_MAX_PARCELS);
constexpr size_t NA_START = NA_COUNT + na_round(4 * (NA_MAX_CELLS + 1));
// at most 12 doubles a cell of x-combined (weight, weight * value) sums
constexpr size_t NA_PARTIAL = NA_START + na_round(4 * (NA_MAX_CELLS + 1));
// interior grid [nzn][ny][nx]: nzn * ny * nx = ncell + nx * ny <= 2 ncell since nz >= 2
constexpr size_t NA_GRID = NA_PARTIAL + na_round(8 * 16 * NA_MAX_CELLS);
constexpr size_t NA_CURSOR = NA_GRID + na_round(8 * 2 * NA_MAX_CELLS);
// (the size stays what pmpic_hip.h publishes)
constexpr size_t NA_TOTAL = NA_CURSOR + 256 * 1024;
static_assert(NA_TOTAL == PMPIC_NOALLOC_SCRATCH_BYTES, "scratch size in pmpic_hip.h");

// Host code must not pass `scratch` itself to a kernel: on the host the name is a stand-in, not
// the device address.  scratch_addr() gives each device's address of it.
static __device__ __align__(256) unsigned char scratch[NA_TOTAL];

constexpr int NA_MAX_DEVICES = 64;

// A device's array: its address, once looked up, and whether the last call left the counts at zero
struct Shared {
  std::mutex turn;
  unsigned char *addr;
  bool unclean;
};
Shared na_shared[NA_MAX_DEVICES];

// the address of `scratch` on `device`, looked up with that device current
int scratch_addr(int device, unsigned char **out) {
  if (!*out) {
    int prev = 0;
    PMPIC_CHECK(hipGetDevice(&prev));
    if (prev != device) PMPIC_CHECK(hipSetDevice(device));
    void *p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (prev != device) PMPIC_CHECK(hipSetDevice(prev));
    if (e != hipSuccess || p == nullptr) return PMPIC_ERR_HIP;
    *out = static_cast<unsigned char *>(p);
  }
  return PMPIC_OK;
}

int par2grid_in(Ctx *c, Shared &s, const double *var, double *grid) {
  PMPIC_TRY(scratch_addr(c->device, &s.addr));
  unsigned char *const base = s.addr;
  BinWork w;
  w.cell = reinterpret_cast<int32_t *>(base + NA_CELL);
  w.rank = reinterpret_cast<int32_t *>(base + NA_RANK);
  w.sorted = reinterpret_cast<int32_t *>(base + NA_SORTED);
  w.count = reinterpret_cast<int32_t *>(base + NA_COUNT);
  w.start = reinterpret_cast<int32_t *>(base + NA_START);
  w.partial = reinterpret_cast<double *>(base + NA_PARTIAL);
  w.cursor = reinterpret_cast<int32_t *>(base + NA_CURSOR);
  double *interior = reinterpret_cast<double *>(base + NA_GRID);
  if (s.unclean) {
    PMPIC_TRY(zero_i32(c, w.count, NA_MAX_CELLS));
    PMPIC_TRY(zero_i32(c, w.cursor, 1));
  }
  s.unclean = true;
  PMPIC_TRY(par2grid_single_ws(c, c->n, var, interior, w));
  PMPIC_TRY(grid_to_ref(c, interior, 1, grid));
  PMPIC_TRY(take_status(c));
  s.unclean = false;
  return PMPIC_OK;
}

}  // namespace
}  // namespace pmpic

using namespace pmpic;

extern "C" int pmpic_par2grid_noalloc(pmpic_ctx *ctx, const double *var, double *grid) {
  if (!ctx || !var || !grid || ctx->c.precision != 0) return PMPIC_ERR_ARG;
  Ctx *c = &ctx->c;
  if (c->n > NA_MAX_PARCELS || c->ncell > NA_MAX_CELLS) return PMPIC_ERR_ARG;
  if (c->device < 0 || c->device >= NA_MAX_DEVICES) return PMPIC_ERR_ARG;
  Shared &s = na_shared[c->device];
  std::lock_guard<std::mutex> turn(s.turn);
  const int st = par2grid_in(c, s, var, grid);
  if (st != PMPIC_OK) (void)hipStreamSynchronize(c->stream);  // the array is the next call's
  return st;
}
