// ox_hostcopy.hip -- a result's way from the device into the caller's memory.
//
// The caller's memory is ordinary as a rule: an array that it may keep, resize or
// hand to a forked child.  (Page-locked memory is a shared mapping of the driver's
// that a child does not get.)  The runtime's copy into ordinary memory takes 68 ms
// for the 720 MB of a 256^3 state, 41 ms if the pages have been touched before: one
// thread brings in the pages and moves the data.  Here the copy engine
// fills page-locked slots and several threads empty them into the caller's pages
// behind it: 15.5 ms for these 720 MB, 4.2 for the 183 MB of 160^3, 1.3 for 41 MB,
// 0.5 for 14.  Bound by the copy engine (56 GB/s, 12.9 ms).  Memory that is
// page-locked already is the copy's own target.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <new>
#include <thread>

#include "ox_solver.hpp"

namespace {

// Bytes of a slot: 256^3 took 46 ms with 1 MB (the threads' hand-over shows), 26 with
// 2, 17 with 4, 15.5 with 8, 14.6 with 16, whose slots take longer to allocate.
constexpr size_t CHUNK = 8u << 20;
constexpr int SLOTS = 4;
constexpr int MAX_WORKERS = 8;

// The page-locked slots of one copy in flight.
struct Stage {
  int device = 0;
  char* buf = nullptr;
  hipEvent_t ev[SLOTS] = {};
};

void free_stage(Stage* s) {
  if (!s) return;
  for (hipEvent_t e : s->ev)
    if (e) hipEventDestroy(e);
  if (s->buf) hipHostFree(s->buf);
  delete s;
}

// Stages between copies: every copy in flight holds one of its own, and up to four
// (128 MB) are kept for the next, until the process ends.
constexpr int KEEP = 4;
std::mutex g_mu;
Stage* g_kept[KEEP] = {};

Stage* take_stage(int device) {
  {
    std::lock_guard<std::mutex> lk(g_mu);
    for (Stage*& k : g_kept)
      if (k && k->device == device) {
        Stage* s = k;
        k = nullptr;
        return s;
      }
  }
  Stage* s = new (std::nothrow) Stage();
  if (!s) return nullptr;
  s->device = device;
  bool ok = hipHostMalloc((void**)&s->buf, SLOTS * CHUNK, hipHostMallocDefault) == hipSuccess;
  for (hipEvent_t& e : s->ev) ok = ok && hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess;
  if (ok) return s;
  (void)hipGetLastError();  // the caller copies without a stage
  free_stage(s);
  return nullptr;
}

void give_stage(Stage* s) {
  {
    std::lock_guard<std::mutex> lk(g_mu);
    for (Stage*& k : g_kept)
      if (!k) {
        k = s;
        return;
      }
  }
  free_stage(s);
}

// One copy: chunk c lies in slot c % SLOTS.
struct Job {
  char* dst;
  const char* stage;
  size_t bytes, chunks;
  int workers = 0;
  std::mutex mu;
  std::condition_variable cv;
  size_t ready = 0;       // chunks that have arrived in their slots
  int left[SLOTS] = {};   // workers that have yet to empty a slot
  bool stop = false;

  size_t length(size_t c) const { return std::min(CHUNK, bytes - c * CHUNK); }
  // part w of the parts that chunk c is cut into
  void move(size_t c, int w, int parts) const {
    const size_t len = length(c), part = ((len + parts - 1) / parts + 4095) & ~(size_t)4095;
    const size_t at = std::min(len, (size_t)w * part);
    std::memcpy(dst + c * CHUNK + at, stage + (c % SLOTS) * CHUNK + at, std::min(part, len - at));
  }
};

void work(Job* j, int w) {
  for (size_t c = 0; c < j->chunks; ++c) {
    {
      std::unique_lock<std::mutex> lk(j->mu);
      j->cv.wait(lk, [&] { return j->stop || j->ready > c; });
      if (j->stop) return;
    }
    j->move(c, w, j->workers);
    std::lock_guard<std::mutex> lk(j->mu);
    if (--j->left[c % SLOTS] == 0) j->cv.notify_all();
  }
}

hipError_t staged_copy(Job& j, Stage* s, const char* src, hipStream_t st) {
  size_t issued = 0;
  auto issue = [&]() {
    const int slot = issued % SLOTS;
    {
      std::unique_lock<std::mutex> lk(j.mu);
      j.cv.wait(lk, [&] { return j.left[slot] == 0; });
      j.left[slot] = j.workers;
    }
    hipError_t e = hipMemcpyAsync(s->buf + slot * CHUNK, src + issued * CHUNK, j.length(issued), hipMemcpyDeviceToHost, st);
    if (e == hipSuccess) e = hipEventRecord(s->ev[slot], st);
    ++issued;
    return e;
  };
  for (size_t c = 0; c < j.chunks; ++c) {
    // ahead of chunk c, up to the slot that was handed to the workers two chunks ago
    while (issued < std::min(j.chunks, c + SLOTS - 1)) {
      const hipError_t e = issue();
      if (e != hipSuccess) return e;
    }
    const hipError_t e = hipEventSynchronize(s->ev[c % SLOTS]);
    if (e != hipSuccess) return e;
    if (j.workers == 0) {
      j.move(c, 0, 1);
      continue;
    }
    std::lock_guard<std::mutex> lk(j.mu);
    j.ready = c + 1;
    j.cv.notify_all();
  }
  return hipSuccess;
}

}  // namespace

int copy_to_host(int device, void* dst, const void* src, size_t bytes, hipStream_t st) {
  hipPointerAttribute_t at{};
  const hipError_t known = hipPointerGetAttributes(&at, dst);
  if (known != hipSuccess) (void)hipGetLastError();  // ordinary memory, to runtimes that call it an error
  const bool ordinary = known != hipSuccess || at.type == hipMemoryTypeUnregistered;
  Stage* s = ordinary ? take_stage(device) : nullptr;
  if (!s) {
    OX_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, st));
    OX_HIP(hipStreamSynchronize(st));
    return OX_OK;
  }
  Job j;
  j.dst = (char*)dst;
  j.stage = s->buf;
  j.bytes = bytes;
  j.chunks = (bytes + CHUNK - 1) / CHUNK;
  // a worker for every 2 MB; one thread alone is this one
  const int want = (int)std::min<size_t>({bytes >> 21, (size_t)MAX_WORKERS, (size_t)std::thread::hardware_concurrency()});
  std::thread th[MAX_WORKERS];
  if (want > 1) {
    try {
      for (; j.workers < want; ++j.workers) th[j.workers] = std::thread(work, &j, j.workers);
    } catch (...) {  // no more threads: those that have started do the work
    }
  }
  const hipError_t e = staged_copy(j, s, (const char*)src, st);
  if (e != hipSuccess) {
    std::lock_guard<std::mutex> lk(j.mu);
    j.stop = true;
    j.cv.notify_all();
  }
  for (int w = 0; w < j.workers; ++w) th[w].join();
  const hipError_t idle = e == hipSuccess ? hipSuccess : hipStreamSynchronize(st);
  // a slot that may still be written to is not for another copy
  if (idle == hipSuccess) give_stage(s);
  if (e != hipSuccess) return ox_fail(OX_EDEVICE, std::string("copy of a result: ") + hipGetErrorString(e));
  return OX_OK;
}
