// Entry points of the library's host-side code for the tests that run without a GPU.
#include "common.h"

using namespace pmpic;

extern "C" {

// cell and head lane through their packed form
void host_run_round_trip(int32_t cell, int32_t head, int32_t out[2]) {
  const uint32_t run = pack_run(cell, head);
  out[0] = run_cell(run);
  out[1] = run_head(run);
}

}  // extern "C"
