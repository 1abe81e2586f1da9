// Copies from the device to the caller's pageable arrays, for the host-pointer
// entry points: through a small ring of page-locked chunks, so that the CPU
// empties one chunk while the DMA engine fills the others.  hipMemcpy moves
// such a result at 17 GB/s, the ring at 25 GB/s; towards the device hipMemcpy
// reaches 34 GB/s by itself, the ring 28, so inputs don't use it.
#include <string.h>

#include <map>
#include <mutex>

#include "sfx_api_internal.h"

namespace sfx {

namespace {

// Ring of a device: N_CHUNK x CHUNK bytes, the bound on what is kept.  Each
// copy costs some 15 us beside its bytes: 8 MB take 611 us in chunks of
// 256 KB, 399 of 512 KB, 342 of 1 MB and 355 of 2 MB (hipMemcpy 490).
constexpr int N_CHUNK = 4;
constexpr size_t CHUNK = (size_t)1 << 20;
// Shorter copies have too few chunks to overlap and go to hipMemcpy: 1 MB takes
// 62 us there and 70 in the ring, 2 MB 126 and 110, 4 MB 247 and 189.
constexpr size_t RING_MIN = 2 * CHUNK;
// Longer ones go there too.  Up to this length the ring was never slower, whole
// calls in ms, ring / hipMemcpy: one result of 4 MB 0.46 / 0.52, of 31 MB 3.43 /
// 3.97; two of 2.1 MB 0.69 / 0.76, of 31 MB 10.5 / 11.6; three of 2.1 MB 0.85 /
// 0.93, of 31 MB 9.8 / 11.3; into new arrays as into old ones.  Beyond it times
// went both ways: three of 58 MB 18.8 / 21.6, of 77 MB 24.9 / 28.3, but in an
// earlier run one of 58 MB 14.4 against 7.4 where several results were written
// in turn, which was not seen again and is not explained.
constexpr size_t RING_MAX = 32 * CHUNK;

struct Ring {
  char* base = nullptr;
  hipEvent_t ev[N_CHUNK] = {nullptr};
};

std::mutex g_ring_mu;
std::map<int, Ring> g_ring;

void ring_free(Ring& r) {
  for (int i = 0; i < N_CHUNK; ++i)
    if (r.ev[i]) (void)hipEventDestroy(r.ev[i]);
  if (r.base) (void)hipHostFree(r.base);
  r = Ring();
}

// The current device's ring, made at its first use; null: none can be had
// (the caller copies without it).
Ring* ring_get() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return nullptr;
  Ring& r = g_ring[dev];
  if (r.base) return &r;
  bool ok = hipHostMalloc((void**)&r.base, N_CHUNK * CHUNK, hipHostMallocDefault) == hipSuccess;
  if (!ok) r.base = nullptr;
  for (int i = 0; ok && i < N_CHUNK; ++i) {
    ok = hipEventCreateWithFlags(&r.ev[i], hipEventDisableTiming) == hipSuccess;
    if (!ok) r.ev[i] = nullptr;
  }
  if (ok) return &r;
  ring_free(r);
  (void)hipGetLastError();
  return nullptr;
}

// Memory that HIP does not know is the caller's pageable memory, which the
// CPU may read and write; page-locked, managed or device memory goes to
// hipMemcpy, as does a null pointer.
bool pageable(const void* h) {
  if (!h) return false;
  hipPointerAttribute_t at;
  const hipError_t e = hipPointerGetAttributes(&at, h);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    return e == hipErrorInvalidValue;
  }
  return at.type == hipMemoryTypeUnregistered;
}

}  // namespace

// Device to host, behind the work queued on the null stream: on return the
// destination holds the copy.  One thread has the ring; another that comes
// meanwhile takes hipMemcpy.
hipError_t copy_out(void* h, const void* d, size_t n) {
  std::unique_lock<std::mutex> lk(g_ring_mu, std::defer_lock);
  Ring* r = nullptr;
  if (n >= RING_MIN && n <= RING_MAX && pageable(h) && lk.try_lock()) r = ring_get();
  if (!r) return hipMemcpy(h, d, n, hipMemcpyDeviceToHost);
  hipError_t e = hipSuccess;
  size_t asked = 0, done = 0;   // bytes queued, bytes delivered
  for (int tail = 0, head = 0; done < n; head = (head + 1) % N_CHUNK) {
    for (; asked < n && asked - done < N_CHUNK * CHUNK; tail = (tail + 1) % N_CHUNK) {
      const size_t len = n - asked < CHUNK ? n - asked : CHUNK;
      e = hipMemcpyAsync(r->base + (size_t)tail * CHUNK, (const char*)d + asked, len, hipMemcpyDeviceToHost, nullptr);
      if (e == hipSuccess) e = hipEventRecord(r->ev[tail], nullptr);
      if (e != hipSuccess) break;
      asked += len;
    }
    if (e == hipSuccess) e = hipEventSynchronize(r->ev[head]);
    if (e != hipSuccess) {
      (void)hipStreamSynchronize(nullptr);   // no copy into the ring outlives the call
      return e;
    }
    const size_t len = n - done < CHUNK ? n - done : CHUNK;
    memcpy((char*)h + done, r->base + (size_t)head * CHUNK, len);
    done += len;
  }
  return hipSuccess;
}

// Give the current device's ring back.
hipError_t release_hostcopy() {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  std::lock_guard<std::mutex> lk(g_ring_mu);
  auto it = g_ring.find(dev);
  if (it == g_ring.end()) return hipSuccess;
  ring_free(it->second);
  g_ring.erase(it);
  return hipSuccess;
}

}  // namespace sfx
