// Copies between the caller's arrays and the device.
//
// The caller's memory is pageable.  The runtime's copy to the host passes through one thread, 17 GB/s
// (11 where the pages are new) of a link that carries 57 to pinned memory; and from about a megabyte
// on it pins the caller's pages for the copy, which can stall the program for milliseconds when it
// next maps or releases memory.  Here such a copy is cut into chunks that threads (a large one's four,
// else the caller's alone) carry through pinned slots of their own, two each, the link moving one while
// the thread copies the other.
//
// From the host it goes through the runtime's own staging, in pieces below the megabyte: 34 GB/s, where
// the runtime's copy of a whole array, whose pages it pins, does 29 and leaves the stall behind.  17
// arrays of 1.9, 6.9, 15, 38 MB: 1.03, 4.7, 10.0, 24.6 ms whole, 0.96, 3.5, 7.7, 19.4 in pieces of 1000
// KB (1.13, 3.8, 8.0, 19.6 of 768 KB, 1.9, 6.6, 14.5, 35.6 of 256), 1.21, 4.0, 8.9, 21.7 through slots by
// four threads; FP32-bulk arrays, one after another, of 1.9, 6.9, 15 MB 1.2, 4.7, 10.0 whole, 1.15, 3.7,
// 7.8 in pieces, 1.8, 5.5, 11.9 through one thread's slots.
#include "common.h"

#include <string.h>

#include <atomic>
#include <system_error>
#include <thread>

namespace pmpic {

namespace {

constexpr size_t CHUNK = (size_t)1 << 20;
constexpr int THREADS = HOST_THREADS;  // the caller's and three more, for the length of the call
// To the host, below this the runtime's own copy, which doesn't pin.  Above it, a 60x180x28 run's
// exports of 2.7 MB left the program's next allocation waiting 4 ms in the median (pass 18.4 ms, now
// 11.9), and eight members' 59 ms a pass is 57.
constexpr size_t LEAST_PINNED = CHUNK;
// Nor does the runtime pin arrays below a megabyte, and slots cost some 40 us at a call's start and a
// chunk for each array: of arrays below LEAST_PART, or LEAST_SUM in all and LEAST_PART_OF_MANY, they
// take longer (4 arrays of 64, 256, 512, 768 KB: 43, 75, 118, 159 us through the runtime, 88, 107,
// 132, 157 through slots; 8 of 256, 512 KB 180, 266 and 183, 230; 17 of 128, 256, 512 KB 265, 355, 537
// and 311, 354, 448).
constexpr size_t LEAST_PART = 3 * CHUNK / 4;
constexpr size_t LEAST_SUM = 4 * CHUNK, LEAST_PART_OF_MANY = CHUNK / 4;
// A caller of several copies may wait for the stream once for all of them, but above this the wait comes
// with each: the runtime's next copy waits longer by itself.  FP32-bulk get_parcels, whose fields are
// converted and copied one after another, of 2,048 parcels 0.41 ms with a wait for each field and 0.30
// with one, of 2,049 0.37 and 0.41, of 20,000 0.47 and 0.50.
constexpr size_t LEAST_WAITED = (size_t)16 << 10;
// Below this one thread: the others' start and, where the caller's pages are new, their contention
// for the address space cost more than they save (a dump of ten grids of 5.4 MB: 4.7 ms through the
// runtime, 4.3 with one thread, 4.2 at best and 10 in the median with four).
constexpr size_t LEAST_THREADS = (size_t)16 << 20;

// an upload's pieces, and the size that the runtime pins from (pieces of exactly that took as long as
// whole arrays: 17 of 15 MB 10.1 ms, of 1000 KB 7.6)
constexpr size_t UPLOAD_PIECE = (size_t)1000 << 10, PINNED_FROM = (size_t)1 << 20;

// the threads that carry a copy to the host through pinned slots, 0 for the runtime's own
int slot_threads(size_t total, int nparts) {
  const size_t least = total < LEAST_SUM ? LEAST_PART : LEAST_PART_OF_MANY;
  if (total < LEAST_PINNED || total < nparts * least) return 0;
  return total < LEAST_THREADS ? 1 : THREADS;
}

struct Copy {
  Ctx *c;
  const HostPart *part;
  int nparts;
  int64_t nchunks;
  std::atomic<int64_t> next{0};
  std::atomic<int> failed{0};

  // chunk i: its host and device addresses and length
  void chunk(int64_t i, char *&host, char *&dev, size_t &len) const {
    for (int k = 0; k < nparts; k++) {
      const int64_t m = (int64_t)((part[k].bytes + CHUNK - 1) / CHUNK);
      if (i < m) {
        const size_t at = (size_t)i * CHUNK;
        host = static_cast<char *>(part[k].host) + at;
        dev = static_cast<char *>(part[k].dev) + at;
        len = part[k].bytes - at < CHUNK ? part[k].bytes - at : CHUNK;
        return;
      }
      i -= m;
    }
    len = 0;
  }
  bool ok(hipError_t e) {
    if (e == hipSuccess) return true;
    failed.store(1);
    return false;
  }
  // one thread's share, through slots 2 w and 2 w + 1
  void run(int w) {
    char *const slot[2] = {c->hc_pin[w], c->hc_pin[w] + CHUNK};
    hipEvent_t *const ev = c->hc_ev + 2 * w;
    char *host[2], *dev[2];
    size_t len[2] = {0, 0};
    auto issue = [&](int s) {
      len[s] = 0;
      const int64_t i = next.fetch_add(1);
      if (i >= nchunks || failed.load()) return;
      chunk(i, host[s], dev[s], len[s]);
      if (!ok(hipMemcpyAsync(slot[s], dev[s], len[s], hipMemcpyDeviceToHost, c->stream)) ||
          !ok(hipEventRecord(ev[s], c->stream)))
        len[s] = 0;
    };
    issue(0);
    for (int s = 0; len[s]; s ^= 1) {
      issue(s ^ 1);
      if (!ok(hipEventSynchronize(ev[s]))) return;
      memcpy(host[s], slot[s], len[s]);
    }
  }
};

// two slots and their events for each of up to n threads: how many threads have them.  One that
// gets none is done without, so the error is taken off the runtime's record, where the caller's next
// check of a launch would find it.
int ensure_slots(Ctx *c, int n) {
  for (int w = 0; w < n; w++) {
    for (int i = 2 * w; i < 2 * w + 2; i++)
      if (!c->hc_ev[i] &&
          hipEventCreateWithFlags(&c->hc_ev[i], hipEventDisableTiming) != hipSuccess) {
        c->hc_ev[i] = nullptr;
        (void)hipGetLastError();
        return w;
      }
    if (c->hc_pin[w]) continue;
    void *p = nullptr;
    if (hipHostMalloc(&p, 2 * CHUNK) != hipSuccess) {
      (void)hipGetLastError();
      return w;
    }
    c->hc_pin[w] = static_cast<char *>(p);
  }
  return n;
}

// Makes the context's device the calling thread's current one for the length of the copy.
struct OnDevice {
  int was = -1;
  bool ok = false;
  explicit OnDevice(int device) {
    if (hipGetDevice(&was) != hipSuccess) return;
    ok = was == device || hipSetDevice(device) == hipSuccess;
    if (was == device) was = -1;
  }
  ~OnDevice() {
    if (was >= 0) (void)hipSetDevice(was);
  }
};

}  // namespace

int copy_to_device(Ctx *c, const HostPart *part, int nparts) {
  for (int k = 0; k < nparts; k++)
    for (size_t at = 0, n; at < part[k].bytes; at += n) {
      n = part[k].bytes - at;
      if (n >= PINNED_FROM) n = UPLOAD_PIECE;
      PMPIC_CHECK(hipMemcpyAsync(static_cast<char *>(part[k].dev) + at,
                                 static_cast<const char *>(part[k].host) + at, n,
                                 hipMemcpyHostToDevice, c->stream));
    }
  return PMPIC_OK;
}

int copy_to_host(Ctx *c, const HostPart *part, int nparts, bool wait) {
  size_t total = 0;
  Copy job{c, part, nparts, 0};
  for (int k = 0; k < nparts; k++) {
    total += part[k].bytes;
    job.nchunks += (int64_t)((part[k].bytes + CHUNK - 1) / CHUNK);
  }
  OnDevice on(c->device);  // the events are its own
  if (!on.ok) return PMPIC_ERR_HIP;
  const int threads = ensure_slots(c, slot_threads(total, nparts));
  if (threads == 0) {
    for (int k = 0; k < nparts; k++)
      if (part[k].bytes)
        PMPIC_CHECK(hipMemcpyAsync(part[k].host, part[k].dev, part[k].bytes, hipMemcpyDeviceToHost,
                                   c->stream));
    if (wait || total > LEAST_WAITED) PMPIC_CHECK(hipStreamSynchronize(c->stream));
    return PMPIC_OK;
  }
  std::thread th[THREADS - 1];
  for (int w = 1; w < threads; w++) {
    try {
      th[w - 1] = std::thread([&job, w]() {
        if (job.ok(hipSetDevice(job.c->device))) job.run(w);
      });
    } catch (const std::system_error &) {
      break;  // fewer threads
    }
  }
  job.run(0);
  for (std::thread &t : th)
    if (t.joinable()) t.join();
  if (!job.failed.load()) return PMPIC_OK;
  (void)hipStreamSynchronize(c->stream);  // what is still on its way into a slot
  return PMPIC_ERR_HIP;
}

void free_host_slots(Ctx *c) {
  for (char *p : c->hc_pin)
    if (p) hipHostFree(p);
  for (hipEvent_t e : c->hc_ev)
    if (e) hipEventDestroy(e);
}

}  // namespace pmpic
