// A HIP runtime in host memory for tests of libsfx's host code: "device"
// memory is malloc'd, asynchronous copies wait in one queue until an event or
// a stream is waited for, and a capture makes the calls fail that a stream
// capture does not allow.  Kernel launches are recorded, not run.
#include <hip/hip_runtime.h>
#include <stdlib.h>
#include <string.h>

#include <deque>
#include <map>
#include <set>
#include <string>
#include <thread>

#include "sfx_api_internal.h"
#include "sfx_exact_body.h"
#include "sfx_kernels.h"

namespace {

struct Copy { void* d; const void* s; size_t n; };
std::deque<Copy> g_queue;
long g_run = 0, g_asked = 0;                 // copies run and queued so far
std::map<hipEvent_t, long> g_events;         // event -> copies queued before it
std::map<std::string, long> g_count;
std::map<void*, size_t> g_dev;
std::set<const void*> g_pinned;
size_t g_used = 0, g_limit = ~(size_t)0;
hipStream_t g_capturing = nullptr;           // stream under capture
bool g_capture = false, g_broken = false;    // in a capture; a call not allowed in it came
thread_local hipStreamCaptureMode g_mode = hipStreamCaptureModeGlobal;
hipError_t g_last = hipSuccess;
int g_fail_copy = -1, g_fail_record = -1;    // calls left before one that fails
void (*g_hook)() = nullptr;                  // runs once, at the next event wait

hipError_t err(hipError_t e) { if (e != hipSuccess) g_last = e; return e; }
bool unsafe() {
  if (!g_capture || g_mode == hipStreamCaptureModeRelaxed) return false;
  g_broken = true;
  return true;
}
bool waits(hipStream_t s) {                  // a wait for the captured stream, or for all work
  if (!g_capture || (s && s != g_capturing)) return false;
  g_broken = true;
  return true;
}
void run_until(long k) {
  for (; g_run < k && !g_queue.empty(); ++g_run) {
    memcpy(g_queue.front().d, g_queue.front().s, g_queue.front().n);
    g_queue.pop_front();
  }
}

}  // namespace

extern "C" {

hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
const char* hipGetErrorString(hipError_t e) { return e == hipSuccess ? "success" : "fake HIP error"; }
hipError_t hipGetLastError(void) { hipError_t e = g_last; g_last = hipSuccess; return e; }
hipError_t hipMalloc(void** p, size_t n) {
  ++g_count["malloc"];
  if (unsafe()) return err(hipErrorStreamCaptureUnsupported);
  if (n > g_limit - g_used) return err(hipErrorOutOfMemory);
  *p = malloc(n);
  g_dev[*p] = n;
  g_used += n;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  ++g_count["free"];
  if (unsafe()) return err(hipErrorStreamCaptureUnsupported);
  if (!p) return hipSuccess;
  if (!g_dev.count(p)) abort();
  g_used -= g_dev[p];
  g_dev.erase(p);
  free(p);
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
  ++g_count["memcpy"];
  if (waits(nullptr)) return err(hipErrorStreamCaptureImplicit);
  run_until(g_asked);
  memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  ++g_count["copy"];
  if (g_fail_copy >= 0 && g_fail_copy-- == 0) return err(hipErrorUnknown);
  g_queue.push_back({d, s, n});
  ++g_asked;
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
  ++g_count["sync"];
  if (waits(s)) return err(hipErrorStreamCaptureUnsupported);
  run_until(g_asked);
  return hipSuccess;
}
hipError_t hipDeviceSynchronize(void) { return hipStreamSynchronize(nullptr); }
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* st) {
  *st = g_capture && s == g_capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode* m) {
  std::swap(*m, g_mode);
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  ++g_count["event"];
  *e = (hipEvent_t)malloc(1);
  g_events[*e] = 0;
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) { g_events.erase(e); free((void*)e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
  if (g_fail_record >= 0 && g_fail_record-- == 0) return err(hipErrorUnknown);
  g_events.at(e) = g_asked;
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
  run_until(g_events.at(e));
  if (g_hook) { auto h = g_hook; g_hook = nullptr; h(); }
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  ++g_count["hostmalloc"];
  if (n > g_limit) return err(hipErrorOutOfMemory);
  *p = malloc(n);
  memset(*p, 0xff, n);
  g_pinned.insert(*p);
  return hipSuccess;
}
hipError_t hipHostFree(void* p) { ++g_count["hostfree"]; g_pinned.erase(p); free(p); return hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
  memset(a, 0, sizeof(*a));
  a->type = g_pinned.count(p) ? hipMemoryTypeHost : hipMemoryTypeUnregistered;
  return hipSuccess;
}

// ---- what the tests ask and set
long fake_count(const char* what) { return g_count[what]; }
void fake_reset_counts(void) { g_count.clear(); }
void fake_limit(size_t n) { g_limit = n ? n : ~(size_t)0; }
size_t fake_used(void) { return g_used; }
void fake_capture(void* stream, int on) { g_capture = on; g_capturing = (hipStream_t)stream; g_broken = false; }
int fake_capture_broken(void) { return g_broken; }
void fake_pin(const void* p, int on) { if (on) g_pinned.insert(p); else g_pinned.erase(p); }
void fake_fail(int copies, int records) { g_fail_copy = copies; g_fail_record = records; }
long fake_pending(void) { return g_asked - g_run; }
int fake_last_error(void) { return (int)hipGetLastError(); }

int host_copy_out(void* h, const void* d, size_t n) { return (int)sfx::copy_out(h, d, n); }

// A second thread's copy while the first one is in its own.
static void* s_h;
static const void* s_d;
static size_t s_n;
static int s_rc;
void host_copy_out_meanwhile(void* h, const void* d, size_t n) {
  s_h = h; s_d = d; s_n = n; s_rc = -1;
  g_hook = [] { std::thread([] { s_rc = (int)sfx::copy_out(s_h, s_d, s_n); }).join(); };
}
int host_copy_out_meanwhile_rc(void) { return s_rc; }

}  // extern "C"

// ---- kernel launches
namespace sfx {

hipError_t launch_fftprod(int, const FftProdArgs&, hipStream_t) { return hipSuccess; }
hipError_t launch_exact(int op, const ExactArgs& a, double*, hipStream_t) {
  ++g_count[a.mmtab ? "matrix" : "twopass"];


  return hipSuccess;
}
hipError_t launch_exact_emom(const ExactArgs&, double*, hipStream_t) { return hipSuccess; }
hipError_t launch_exact_velstat(const ExactArgs&, double*, double*, hipStream_t) { return hipSuccess; }
hipError_t launch_exact_checkif(const double*, int32_t*, hipStream_t) { return hipSuccess; }
int64_t exact_velstat_blocks(int, int64_t np, int) { return np; }
int64_t exact_grid_blocks(int, int, int64_t np, int) { return np; }
int64_t exact_emom_blocks(int64_t np, int, int) { return np; }

}  // namespace sfx
