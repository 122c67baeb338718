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
hipError_t hipDeviceGetMemPool(hipMemPool_t* p, int) { *p = nullptr; return hipSuccess; }
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

static constexpr size_t MB = size_t(1) << 20;

static void* get(size_t bytes, void* stream)
{
  void* p = nullptr;
  CHECK(scratch_alloc(&p, bytes, stream, "t") == NEBO_OK && p);
  return p;
}

// Blocks given back, of whatever sizes and streams, never pass 1/32 of the memory, and
// neither taking nor giving waits on the host, with all of the streams' work undone.
static void kept_within_the_limit()
{
  for (int i = 0; i < 40; ++i) {
    void* s = i % 2 ? A : B;
    void* p = get((100 + 90 * i) * MB, s);   // the largest pass the limit of 2048 MB
    scratch_free(p, s);
    CHECK(used <= total / 32);
  }
  CHECK(waits == 0);
}

// Blocks lent at one time may pass the limit; those past it are not kept.
static void lent_together()
{
  std::vector<void*> p;
  for (int i = 0; i < 8; ++i) p.push_back(get(500 * MB, A));
  CHECK(used >= 4000 * MB);
  for (void* q : p) scratch_free(q, A);
  CHECK(used <= total / 32 && used >= 1500 * MB);
  CHECK(waits == 0);
}

// The limit follows what others leave free.
static void little_memory_left()
{
  used = total - 4096 * MB;      // another program's
  const size_t others = used;
  void* p = get(400 * MB, A);
  scratch_free(p, A);
  CHECK(used - others == 416 * MB && get(400 * MB, A) == p);   // in steps of 32 MB
  scratch_free(p, A);
  p = get(600 * MB, A);          // more than an eighth of 4096 MB
  scratch_free(p, A);
  CHECK(used - others <= 512 * MB);
  CHECK(waits == 0);
}

// Another stream's block whose work is not over is taken only where a new one would pass
// the limit, and then after a wait queued on the taking stream.
static void blocks_between_streams()
{
  void* p = get(1500 * MB, A);
  scratch_free(p, A);
  CHECK(get(1500 * MB, A) == p);           // its own stream: at once
  scratch_free(p, A);
  void* small = get(400 * MB, B);
  CHECK(small != p);                        // fits the block, but a new one fits the limit
  scratch_free(small, B);
  const long before = streams[B].queued;
  CHECK(get(1400 * MB, B) == p && streams[B].queued > before);
  scratch_free(p, B);
  CHECK(waits == 0);
  streams[B].done = streams[B].queued;
  CHECK(get(1500 * MB, A) == p);           // its last use is over
}

// When memory runs out, what is kept idle goes, and the call succeeds.
static void memory_runs_out()
{
  void* p = get(1024 * MB, A);
  scratch_free(p, A);
  used = total - 300 * MB;                  // others took the rest
  void* q = get(1200 * MB, B);
  CHECK(live.count(p) == 0 && used == total - 300 * MB - 1024 * MB + 1200 * MB);
  scratch_free(q, B);
  CHECK(used == total - 300 * MB - 1024 * MB);
  void* r = nullptr;
  used = total;
  CHECK(scratch_alloc(&r, 600 * MB, A, "t") == NEBO_ERR_HIP && !r);
}

// The same for memory a program allocates to keep.
static void program_memory_runs_out()
{
  void* p = get(1024 * MB, A);
  scratch_free(p, A);
  used = total - 300 * MB;
  void* q = nullptr;
  CHECK(device_alloc(&q, 1200 * MB, "t") == NEBO_OK && q && live.count(p) == 0);
  CHECK(device_alloc(&q, 1200 * MB, "t") == NEBO_ERR_HIP);
}

// A captured stream takes the graph's own allocation nodes.
static void captured_stream()
{
  void* p = get(10 * MB, A);
  scratch_free(p, A);
  captured = B;
  void* q = get(10 * MB, B);
  CHECK(q != p);
  scratch_free(q, B);
  CHECK(live.count(q) == 0 && live.count(p) == 1);
}

int main(int argc, char** argv)
{
  const struct { const char* name; void (*fn)(); } checks[] = {
      {"other_threads_capture", other_threads_capture}, {"slots_are_reused", slots_are_reused},
      {"failed_upload", failed_upload}, {"kept_within_the_limit", kept_within_the_limit},
      {"lent_together", lent_together}, {"little_memory_left", little_memory_left},
      {"blocks_between_streams", blocks_between_streams}, {"memory_runs_out", memory_runs_out},
      {"program_memory_runs_out", program_memory_runs_out}, {"captured_stream", captured_stream}};
  for (const auto& c : checks)
    if (argc == 2 && !std::strcmp(argv[1], c.name)) {
      c.fn();
      return 0;
    }
  return 2;
}
