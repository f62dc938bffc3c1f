// Entry points of the library's host-side code for the tests that run without a GPU.
#include "common.h"

#include <string.h>

#include <atomic>

// The HIP calls of transfer.hip, on host memory: "device" memory is host memory, every command ends
// at once, and pinned memory runs out after pinned_left blocks.
namespace fake {
thread_local hipError_t pending = hipSuccess;  // what hipGetLastError reports
std::atomic<int> pinned_left{0}, pinned_taken{0}, copies{0}, waits{0};
std::atomic<size_t> largest{0};  // copy command
// each thread's current device; an event belongs to the one it was created on, the stream to device 1
thread_local int device = 0;
constexpr int STREAM_DEVICE = 1;

hipError_t fail(hipError_t e) { return pending = e; }
hipError_t host_malloc(void **p, size_t n) {
  if (pinned_left.fetch_sub(1) <= 0) return fail(hipErrorOutOfMemory);
  pinned_taken++;
  *p = malloc(n);
  return hipSuccess;
}
hipError_t host_free(void *p) {
  free(p);
  return hipSuccess;
}
hipError_t memcpy_async(void *to, const void *from, size_t n, hipMemcpyKind, hipStream_t) {
  copies++;
  if (n > largest) largest = n;
  memcpy(to, from, n);
  return hipSuccess;
}
hipError_t event_create(hipEvent_t *e, unsigned) {
  *e = reinterpret_cast<hipEvent_t>((intptr_t)device + 1);
  return hipSuccess;
}
hipError_t event(hipEvent_t) { return hipSuccess; }
hipError_t event_record(hipEvent_t e, hipStream_t) {
  return e == reinterpret_cast<hipEvent_t>((intptr_t)STREAM_DEVICE + 1) ? hipSuccess
                                                                        : fail(hipErrorInvalidHandle);
}
hipError_t stream(hipStream_t) {
  waits++;
  return hipSuccess;
}
hipError_t set_device(int d) {
  device = d;
  return hipSuccess;
}
hipError_t get_device(int *d) {
  *d = device;
  return hipSuccess;
}
hipError_t last_error() {
  const hipError_t e = pending;
  pending = hipSuccess;
  return e;
}
}  // namespace fake
#define hipHostMalloc fake::host_malloc
#define hipHostFree fake::host_free
#define hipMemcpyAsync fake::memcpy_async
#define hipEventCreateWithFlags fake::event_create
#define hipEventSynchronize fake::event
#define hipEventDestroy fake::event
#define hipEventRecord fake::event_record
#define hipStreamSynchronize fake::stream
#define hipSetDevice fake::set_device
#define hipGetDevice fake::get_device
#define hipGetLastError fake::last_error
#include "transfer.hip"

using namespace pmpic;

extern "C" {

// cell and head lane through their packed form
void host_run_round_trip(int32_t cell, int32_t head, int32_t out[2]) {
  const uint32_t run = pack_run(cell, head);
  out[0] = run_cell(run);
  out[1] = run_head(run);
}

// `parts` copies of n bytes each, one after another in `host` and `dev`, with pinned memory for
// `pinned` threads' slots, by a thread whose current device is `device`.  out: the status, the error
// left pending, the blocks of pinned memory taken, the copy commands issued, the thread's device
// afterwards, the waits for the stream and the largest copy's bytes
void host_copy(char *host, char *dev, int64_t n, int parts, int to_host, int pinned, int device,
               int out[7]) {
  Ctx *c = new Ctx();
  c->device = fake::STREAM_DEVICE;
  fake::device = device;
  HostPart part[32];
  for (int i = 0; i < parts; i++) part[i] = {host + i * n, dev + i * n, (size_t)n};
  fake::pinned_left = pinned;
  fake::pinned_taken = fake::copies = fake::waits = 0;
  fake::largest = 0;
  out[0] = to_host ? copy_to_host(c, part, parts, false) : copy_to_device(c, part, parts);
  out[1] = (int)fake::last_error();
  out[2] = fake::pinned_taken;
  out[3] = fake::copies;
  out[4] = fake::device;
  out[5] = fake::waits;
  out[6] = (int)fake::largest;
  free_host_slots(c);
  delete c;
}

}  // extern "C"
