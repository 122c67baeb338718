// nebo_scratch.hip -- memory that a call borrows: device scratch and page-locked slots.
// Host code only.

#include "nebo_internal.h"

#include <hip/hip_runtime_api.h>

#include <map>
#include <mutex>
#include <unordered_map>
#include <vector>

namespace nebo {

// ---- scratch memory of a call ---------------------------------------------------
// The runtime's stream-ordered pool returns its memory to the driver at every
// synchronisation and mapped it anew for a call that followed closely on another:
// 13.8 ms of a 14.7 ms scatter of 2M particles (250 MB of scratch).  Freed blocks
// are kept here instead, up to 1/32 of the device's memory per GPU, and given back
// beyond that and by nebo_pool_trim.  A block carries an event recorded after its
// last use; whoever takes it waits for that event on its own stream first, so
// blocks move between streams and threads safely.
namespace {
struct ScratchBlock {
  void* p;
  size_t bytes;
  hipEvent_t done;     // recorded on `stream` when the block was given back
  void* stream;
};
struct ScratchCache {
  std::vector<ScratchBlock> idle;   // oldest first
  size_t kept = 0;                  // bytes of idle and lent blocks
  size_t limit = 0;
};
std::mutex g_scratch_mu;
std::map<int, ScratchCache> g_scratch_cache;
struct LentBlock {
  int device;
  ScratchBlock block;
};
std::unordered_map<void*, LentBlock> g_scratch_lent;
std::mutex g_slot_mu;
std::vector<void*> g_slots_free;

// Another thread's capture in global mode forbids this thread's allocations and
// event queries on streams that have nothing to do with it; they are safe.
struct RelaxedCapture {
  hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
  RelaxedCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
  ~RelaxedCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
};

// Sizes are rounded up to an eighth of their power of two, so that calls whose
// scratch differs a little (another particle set) take each other's blocks.
size_t scratch_size(size_t bytes)
{
  size_t step = size_t(1) << 16;
  while (step * 16 <= bytes) step *= 2;
  return (bytes + step - 1) / step * step;
}

// Frees idle blocks, oldest first, until at most `most` bytes are kept.
void scratch_evict(ScratchCache& c, size_t most)
{
  while (!c.idle.empty() && c.kept > most) {
    const ScratchBlock b = c.idle.front();
    c.idle.erase(c.idle.begin());
    c.kept -= b.bytes;
    (void)hipEventSynchronize(b.done);
    (void)hipFree(b.p);
    (void)hipEventDestroy(b.done);
  }
}
}  // namespace

int scratch_alloc(void** out, size_t bytes, void* stream, const char* ctx)
{
  *out = nullptr;
  hipStream_t s = (hipStream_t)stream;
  int device = 0;
  int rc = check_hip(hipGetDevice(&device), ctx);
  if (rc) return rc;
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(s, &capture) != hipSuccess) (void)hipGetLastError();
  // a captured graph holds its own allocation nodes
  if (capture != hipStreamCaptureStatusNone) return check_hip(hipMallocAsync(out, bytes ? bytes : 1, s), ctx);
  const RelaxedCapture relaxed;
  const size_t want = scratch_size(bytes ? bytes : 1);
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  ScratchCache& c = g_scratch_cache[device];
  if (!c.limit) {
    size_t free_b = 0, total_b = 0;
    if (hipMemGetInfo(&free_b, &total_b) != hipSuccess) (void)hipGetLastError();
    c.limit = total_b / 32 + 1;
  }
  if (want > c.limit) return check_hip(hipMallocAsync(out, bytes, s), ctx);
  // the smallest block that fits within four times the size: this stream's own, or
  // one whose last use is over; another stream's unfinished one only when a new
  // block would pass the limit
  int pick = -1;
  bool ready = false;
  for (int i = 0; i < (int)c.idle.size(); ++i) {
    const ScratchBlock& b = c.idle[i];
    if (b.bytes < want || b.bytes > 4 * want) continue;
    const bool r = b.stream == stream || hipEventQuery(b.done) == hipSuccess;
    if (!r) (void)hipGetLastError();   // hipErrorNotReady
    if (pick < 0 || (r && !ready) || (r == ready && b.bytes < c.idle[pick].bytes)) {
      pick = i;
      ready = r;
    }
  }
  if (pick >= 0 && (ready || c.kept + want > c.limit)) {
    const ScratchBlock b = c.idle[pick];
    if ((rc = check_hip(hipStreamWaitEvent(s, b.done, 0), ctx))) return rc;
    c.idle.erase(c.idle.begin() + pick);
    g_scratch_lent[b.p] = LentBlock{device, b};
    *out = b.p;
    return NEBO_OK;
  }
  scratch_evict(c, c.limit - want);
  ScratchBlock b{nullptr, want, nullptr, stream};
  if ((rc = check_hip(hipEventCreateWithFlags(&b.done, hipEventDisableTiming), ctx))) return rc;
  hipError_t st = hipMalloc(&b.p, want);
  if (st != hipSuccess) {   // out of memory: what is kept idle goes first
    (void)hipGetLastError();
    scratch_evict(c, 0);
    st = hipMalloc(&b.p, want);
  }
  if ((rc = check_hip(st, ctx))) {
    (void)hipEventDestroy(b.done);
    return rc;
  }
  c.kept += want;
  g_scratch_lent[b.p] = LentBlock{device, b};
  *out = b.p;
  return NEBO_OK;
}

void scratch_free(void* p, void* stream)
{
  if (!p) return;
  const RelaxedCapture relaxed;
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  const auto it = g_scratch_lent.find(p);
  if (it == g_scratch_lent.end()) {
    (void)hipFreeAsync(p, (hipStream_t)stream);
    return;
  }
  LentBlock l = it->second;
  g_scratch_lent.erase(it);
  ScratchCache& c = g_scratch_cache[l.device];
  l.block.stream = stream;
  if (hipEventRecord(l.block.done, (hipStream_t)stream) != hipSuccess) {
    // no way to tell when its last use ends: hipFree waits for the device
    (void)hipGetLastError();
    (void)hipFree(p);
    (void)hipEventDestroy(l.block.done);
    c.kept -= l.block.bytes;
    return;
  }
  c.idle.push_back(l.block);
  scratch_evict(c, c.limit);   // blocks lent together may have passed the limit
}

int scratch_upload(void** out, const void* host, size_t bytes, void* stream, const char* ctx)
{
  int rc = scratch_alloc(out, bytes, stream, ctx);
  if (rc) return rc;
  rc = check_hip(hipMemcpyAsync(*out, host, bytes, hipMemcpyHostToDevice, (hipStream_t)stream), ctx);
  if (rc) {
    scratch_free(*out, stream);
    *out = nullptr;
  }
  return rc;
}

void scratch_trim(int device)
{
  const RelaxedCapture relaxed;
  {
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    scratch_evict(g_scratch_cache[device], 0);
  }
  std::lock_guard<std::mutex> lk(g_slot_mu);
  for (void* p : g_slots_free) (void)hipHostFree(p);
  g_slots_free.clear();
}

// ---- page-locked slots ----------------------------------------------------------
int host_slot_take(void** out, const char* ctx)
{
  *out = nullptr;
  const RelaxedCapture relaxed;
  std::lock_guard<std::mutex> lk(g_slot_mu);
  if (!g_slots_free.empty()) {
    *out = g_slots_free.back();
    g_slots_free.pop_back();
    return NEBO_OK;
  }
  return check_hip(hipHostMalloc(out, kHostSlotBytes, hipHostMallocPortable | hipHostMallocMapped), ctx);
}

void host_slot_give(void* p)
{
  if (!p) return;
  std::lock_guard<std::mutex> lk(g_slot_mu);
  g_slots_free.push_back(p);
}

}  // namespace nebo
