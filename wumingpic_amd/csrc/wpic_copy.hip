// wpic_copy.hip -- large copies from device memory into the caller's host
// arrays.
//
// hipMemcpyAsync into pageable memory goes through the runtime's own staging
// on one thread, which also takes the page faults of a fresh array: 0.84 GB
// (the fields of 256^3) took 85 ms, 10 GB/s.  Here the chunks go into a ring of
// pinned slots and a few threads move them on, so that the link, the faults
// and the copies overlap: 22 ms; 0.15 GB 15.5 -> 5.1, 0.05 GB 5.1 -> 1.9.  A
// context's first such copy also makes the ring, which costs about what it
// saves at 0.05 GB: smaller copies than MIN_THREADED stay with the runtime.  So
// do copies into memory that HIP made or registered: the link writes there by
// itself (0.84 GB into a pinned array 15.5 ms, through the slots 21).
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <thread>

#include "wpic_internal.h"

namespace wpic {

namespace {
constexpr size_t CHUNK = size_t(2) << 20;
constexpr int NSLOT = HostRing::NSLOT;
constexpr int NTHREAD = 6;
// below this there is less to gain than making the ring and starting threads costs
constexpr size_t MIN_THREADED = size_t(32) << 20;

bool ring_ready(HostRing& r) {
  if (r.buf) return true;
  if (hipHostMalloc((void**)&r.buf, CHUNK * NSLOT, hipHostMallocDefault) != hipSuccess) {
    (void)hipGetLastError();
    r.buf = nullptr;
    return false;
  }
  for (int k = 0; k < NSLOT; k++)
    if (hipEventCreateWithFlags(&r.ev[k], hipEventDisableTiming) != hipSuccess) {
      (void)hipGetLastError();
      r.ev[k] = nullptr;
      ring_free(r);
      return false;
    }
  return true;
}
// memory that HIP made or registered (pinned, managed): no page of the host's own
bool known_to_hip(const void* p) {
  hipPointerAttribute_t at;
  if (hipPointerGetAttributes(&at, p) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return at.type != hipMemoryTypeUnregistered;
}
}  // namespace

void ring_free(HostRing& r) {
  for (int k = 0; k < NSLOT; k++) {
    if (r.ev[k]) (void)hipEventDestroy(r.ev[k]);
    r.ev[k] = nullptr;
  }
  if (r.buf) (void)hipHostFree(r.buf);
  r.buf = nullptr;
}

hipError_t copy_to_host(HostRing& ring, int device, hipStream_t st, void* dst, const void* src, size_t bytes) {
  const size_t nchunk = (bytes + CHUNK - 1) / CHUNK;
  auto plain = [&]() {
    const hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, st);
    return e != hipSuccess ? e : hipStreamSynchronize(st);
  };
  if (bytes < MIN_THREADED || known_to_hip(dst) || !ring_ready(ring)) return plain();

  std::mutex mu;
  std::condition_variable cv;
  size_t queued = 0;            // chunks whose device copy is on the stream
  bool stop = false;            // no more will come
  bool busy[NSLOT] = {};        // a slot's chunk is not moved on yet
  std::atomic<size_t> next{0};  // the next chunk a thread takes
  hipError_t err = hipSuccess;
  auto len = [&](size_t c) { return c + 1 < nchunk ? CHUNK : bytes - c * CHUNK; };

  auto work = [&]() {
    hipError_t e = hipSetDevice(device);
    for (;;) {
      const size_t c = next.fetch_add(1);
      if (c >= nchunk) return;
      const int slot = (int)(c % NSLOT);
      {
        std::unique_lock<std::mutex> lk(mu);
        cv.wait(lk, [&]() { return c < queued || stop; });
        if (c >= queued) return;
      }
      if (e == hipSuccess) e = hipEventSynchronize(ring.ev[slot]);
      if (e == hipSuccess) std::memcpy((char*)dst + c * CHUNK, ring.buf + slot * CHUNK, len(c));
      std::lock_guard<std::mutex> lk(mu);
      if (e != hipSuccess && err == hipSuccess) err = e;
      busy[slot] = false;
      cv.notify_all();
    }
  };

  std::thread th[NTHREAD];
  int nth = 0;
  try {
    for (; nth < NTHREAD; nth++) th[nth] = std::thread(work);
  } catch (...) {  // no more threads to be had: those that started do the work
  }
  if (nth == 0) return plain();
  for (size_t c = 0; c < nchunk; c++) {
    const int slot = (int)(c % NSLOT);
    {
      std::unique_lock<std::mutex> lk(mu);
      cv.wait(lk, [&]() { return !busy[slot]; });
      if (err != hipSuccess) break;
      busy[slot] = true;
    }
    hipError_t e = hipMemcpyAsync(ring.buf + slot * CHUNK, (const char*)src + c * CHUNK, len(c),
                                  hipMemcpyDeviceToHost, st);
    if (e == hipSuccess) e = hipEventRecord(ring.ev[slot], st);
    std::lock_guard<std::mutex> lk(mu);
    if (e != hipSuccess) {
      err = e;
      break;
    }
    queued = c + 1;
    cv.notify_all();
  }
  {
    std::lock_guard<std::mutex> lk(mu);
    stop = true;
    cv.notify_all();
  }
  for (int k = 0; k < nth; k++) th[k].join();
  const hipError_t e = hipStreamSynchronize(st);
  return err != hipSuccess ? err : e;
}

}  // namespace wpic
