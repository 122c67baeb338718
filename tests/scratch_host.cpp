// Host model of the HIP calls nebo_scratch.hip makes, and checks of the cache over it:
// streams that run only when told to, events, allocations with a budget, and the
// capture mode each thread is in.  `scratch_host NAME` runs one check.
#include "../spatialops-threadfix_amd/csrc/nebo_internal.h"

#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <thread>
#include <vector>

#define CHECK(c)                                                         \
  do {                                                                   \
    if (!(c)) {                                                          \
      std::fprintf(stderr, "%s:%d: %s\n", __FILE__, __LINE__, #c);       \
      std::exit(1);                                                      \
    }                                                                    \
  } while (0)

namespace fake {
struct Event { void* stream = nullptr; long at = 0; bool recorded = false; };
struct Stream { long queued = 0, done = 0; };
std::map<void*, Stream> streams;
size_t total = size_t(64) << 30, used = 0, host_bytes = 0;
std::map<void*, size_t> live;
int captures = 0;                 // streams captured in global mode
int waits = 0;                    // times the host waited for a stream
bool fail_copy = false;
void* captured = nullptr;         // a stream under capture
thread_local hipStreamCaptureMode mode = hipStreamCaptureModeGlobal;

bool allowed()   // allocations are refused while another thread captures, unless relaxed
{
  return captures == 0 || mode == hipStreamCaptureModeRelaxed;
}
hipError_t take(void** p, size_t n)
{
  if (!allowed()) return hipErrorStreamCaptureUnsupported;
  if (used + n > total) return hipErrorOutOfMemory;
  static char* next = (char*)0x10000000;
  *p = next;
  next += n + 4096;
  live[*p] = n;
  used += n;
  return hipSuccess;
}
hipError_t drop(void* p)
{
  if (!p) return hipSuccess;
  CHECK(live.count(p));
  used -= live[p];
  live.erase(p);
  return hipSuccess;
}
void finish(void* s)   // the host waits until stream s is empty
{
  Stream& q = streams[s];
  if (q.done < q.queued) ++waits;
  q.done = q.queued;
}
}  // namespace fake
using namespace fake;

extern "C" {
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* c)
{
  *c = (captured && captured == (void*)s) ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode* m) { std::swap(*m, mode); return hipSuccess; }
hipError_t hipMemGetInfo(size_t* f, size_t* t) { *f = total - used; *t = total; return hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) { return take(p, n); }
hipError_t hipFree(void* p)
{
  for (auto& s : streams) finish(s.first);   // the runtime's hipFree waits for the device
  return drop(p);
}
hipError_t hipMallocAsync(void** p, size_t n, hipStream_t) { return take(p, n); }
hipError_t hipFreeAsync(void* p, hipStream_t s) { ++streams[s].queued; return drop(p); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned)
{
  if (!allowed()) return hipErrorStreamCaptureUnsupported;
  *p = std::malloc(n);
  host_bytes += n;
  return hipSuccess;
}
hipError_t hipHostFree(void* p) { std::free(p); host_bytes = 0; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = (hipEvent_t) new Event; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { delete (Event*)e; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
  *(Event*)e = Event{(void*)s, ++streams[s].queued, true};
  return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t e)
{
  const Event* v = (Event*)e;
  return streams[v->stream].done >= v->at ? hipSuccess : hipErrorNotReady;
}
hipError_t hipEventSynchronize(hipEvent_t e) { finish(((Event*)e)->stream); return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t, unsigned) { ++streams[s].queued; return hipSuccess; }
hipError_t hipMemcpyAsync(void*, const void*, size_t, hipMemcpyKind, hipStream_t s)
{
  if (fail_copy) return hipErrorInvalidValue;
  ++streams[s].queued;
  return hipSuccess;
}
hipError_t hipDeviceGetDefaultMemPool(hipMemPool_t* p, int) { *p = nullptr; return hipSuccess; }
hipError_t hipMemPoolTrimTo(hipMemPool_t, size_t) { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error"; }
}

namespace nebo {
int check_hip(int st, const char*) { return st == hipSuccess ? NEBO_OK : NEBO_ERR_HIP; }
}

using namespace nebo;
static void* const A = (void*)0x1;
static void* const B = (void*)0x2;

// While another thread captures in global mode, a call's scratch and its slot come
// without an allocation that would be refused, and the thread's mode is as it was.
static void other_threads_capture()
{
  captures = 1;
  void *slot = nullptr, *scratch = nullptr;
  CHECK(host_slot_take(&slot, "t") == NEBO_OK && slot);
  CHECK(scratch_alloc(&scratch, 1 << 20, A, "t") == NEBO_OK && scratch);
  CHECK(mode == hipStreamCaptureModeGlobal);
  host_slot_give(slot);
  scratch_free(scratch, A);
  CHECK(mode == hipStreamCaptureModeGlobal);
}

// Slots are used again, one per call in progress, and given back by a trim.
static void slots_are_reused()
{
  void *a = nullptr, *b = nullptr, *c = nullptr;
  CHECK(host_slot_take(&a, "t") == NEBO_OK && host_slot_take(&b, "t") == NEBO_OK && a != b);
  host_slot_give(a);
  CHECK(host_slot_take(&c, "t") == NEBO_OK && c == a);
  host_slot_give(b);
  host_slot_give(c);
  CHECK(host_bytes == 2 * kHostSlotBytes);
  scratch_trim(0);
  CHECK(host_bytes == 0);
}

// A copy that fails holds no block: a trim leaves nothing allocated.
static void failed_upload()
{
  const int host[4] = {1, 2, 3, 4};
  void* p = nullptr;
  CHECK(scratch_upload(&p, host, sizeof host, A, "t") == NEBO_OK && p);
  scratch_free(p, A);
  fail_copy = true;
  CHECK(scratch_upload(&p, host, sizeof host, A, "t") == NEBO_ERR_HIP && !p);
  scratch_trim(0);
  CHECK(used == 0);
}

int main(int argc, char** argv)
{
  const struct { const char* name; void (*fn)(); } checks[] = {
      {"other_threads_capture", other_threads_capture}, {"slots_are_reused", slots_are_reused},
      {"failed_upload", failed_upload}};
  for (const auto& c : checks)
    if (argc == 2 && !std::strcmp(argv[1], c.name)) {
      c.fn();
      return 0;
    }
  return 2;
}
