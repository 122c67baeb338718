// nebo_scratch.hip -- memory that a call borrows: device scratch and page-locked slots.
// Host code only.

#include "nebo_internal.h"

#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <map>
#include <mutex>
#include <unordered_map>
#include <vector>

namespace nebo {

// ---- scratch memory of a call ---------------------------------------------------
// The runtime's stream-ordered pool returns its memory to the driver at every
// synchronisation and mapped it anew for a call that followed closely on another:
// 13.8 ms of a 14.7 ms scatter of 2M particles (250 MB of scratch).  Blocks of that pool
// are therefore kept here between calls, on each GPU up to 1/32 of its memory and to
// an eighth of what others leave free of it; nebo_pool_trim gives them back, and so does
// an allocation that finds no memory.  A block carries an event recorded after its
// last use; whoever takes it waits for that event on its own stream first, so
// blocks move between streams and threads safely.  What does not fit the limit comes
// from the pool and goes back to it, and blocks that make room for others go back in the
// order of the stream that takes their place: the host waits for no stream here.
namespace {
struct ScratchBlock {
  void* p;
  size_t bytes;
  hipEvent_t done;     // recorded on `stream` when the block was given back
  void* stream;
};
struct ScratchCache {
  std::vector<ScratchBlock> idle;   // oldest first
  size_t kept = 0;                  // bytes of idle and lent blocks, and of those being allocated
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

// Bytes the current device's cache may keep, of which it keeps `kept` now.
size_t scratch_limit(size_t kept)
{
  size_t free_b = 0, total_b = 0;
  if (hipMemGetInfo(&free_b, &total_b) != hipSuccess) {
    (void)hipGetLastError();
    return 0;
  }
  return std::min(total_b / 32, (free_b + kept) / 8);
}

// Gives every idle block of a device back to the driver; false when there was none.
// The host waits for their last uses.
bool scratch_drop(int device)
{
  const RelaxedCapture relaxed;
  std::vector<ScratchBlock> blocks;
  {
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    ScratchCache& c = g_scratch_cache[device];
    blocks.swap(c.idle);
    for (const ScratchBlock& b : blocks) c.kept -= b.bytes;
  }
  for (const ScratchBlock& b : blocks) {
    (void)hipEventSynchronize(b.done);
    (void)hipFree(b.p);
    (void)hipEventDestroy(b.done);
  }
  hipMemPool_t pool;
  if (hipDeviceGetMemPool(&pool, device) != hipSuccess || hipMemPoolTrimTo(pool, 0) != hipSuccess)
    (void)hipGetLastError();
  return !blocks.empty();
}

// From the runtime's stream-ordered pool; what is kept idle goes when there is no memory.
int pool_alloc(void** out, size_t bytes, int device, hipStream_t s, const char* ctx)
{
  hipError_t st = hipMallocAsync(out, bytes, s);
  if (st == hipErrorOutOfMemory) {
    (void)hipGetLastError();
    if (scratch_drop(device)) st = hipMallocAsync(out, bytes, s);
  }
  return check_hip(st, ctx);
}
}  // namespace

int scratch_alloc(void** out, size_t bytes, void* stream, const char* ctx)
{
  *out = nullptr;
  hipStream_t s = (hipStream_t)stream;
  int device = 0;
  int rc = check_hip(hipGetDevice(&device), ctx);
  if (rc) return rc;
  if (bytes == 0) bytes = 1;
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(s, &capture) != hipSuccess) (void)hipGetLastError();
  // a captured graph holds its own allocation nodes
  if (capture != hipStreamCaptureStatusNone) return check_hip(hipMallocAsync(out, bytes, s), ctx);
  const RelaxedCapture relaxed;
  const size_t want = scratch_size(bytes);
  bool keep = false;
  std::vector<ScratchBlock> leaving;
  {
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    ScratchCache& c = g_scratch_cache[device];
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
    const size_t limit = ready ? 0 : scratch_limit(c.kept);
    if (pick >= 0 && (ready || c.kept + want > limit)) {
      const ScratchBlock b = c.idle[pick];
      if ((rc = check_hip(hipStreamWaitEvent(s, b.done, 0), ctx))) return rc;
      c.idle.erase(c.idle.begin() + pick);
      g_scratch_lent[b.p] = LentBlock{device, b};
      *out = b.p;
      return NEBO_OK;
    }
    // room for a new block: the oldest idle ones go, where that makes enough
    size_t lent = c.kept;
    for (const ScratchBlock& b : c.idle) lent -= b.bytes;
    if (lent + want <= limit) {
      keep = true;
      while (c.kept + want > limit) {
        leaving.push_back(c.idle.front());
        c.idle.erase(c.idle.begin());
        c.kept -= leaving.back().bytes;
      }
      c.kept += want;
    }
  }
  for (const ScratchBlock& b : leaving) {
    if (hipStreamWaitEvent(s, b.done, 0) == hipSuccess) {
      (void)hipFreeAsync(b.p, s);
    } else {   // hipFree waits for the device
      (void)hipGetLastError();
      (void)hipFree(b.p);
    }
    (void)hipEventDestroy(b.done);
  }
  if (!keep) return pool_alloc(out, bytes, device, s, ctx);
  ScratchBlock b{nullptr, want, nullptr, stream};
  rc = check_hip(hipEventCreateWithFlags(&b.done, hipEventDisableTiming), ctx);
  if (!rc && (rc = pool_alloc(&b.p, want, device, s, ctx))) (void)hipEventDestroy(b.done);
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (rc) {
    g_scratch_cache[device].kept -= want;
    return rc;
  }
  g_scratch_lent[b.p] = LentBlock{device, b};
  *out = b.p;
  return NEBO_OK;
}

void scratch_free(void* p, void* stream)
{
  if (!p) return;
  const RelaxedCapture relaxed;
  std::unique_lock<std::mutex> lk(g_scratch_mu);
  const auto it = g_scratch_lent.find(p);
  if (it == g_scratch_lent.end()) {
    lk.unlock();
    (void)hipFreeAsync(p, (hipStream_t)stream);
    return;
  }
  LentBlock l = it->second;
  g_scratch_lent.erase(it);
  ScratchCache& c = g_scratch_cache[l.device];
  l.block.stream = stream;
  if (hipEventRecord(l.block.done, (hipStream_t)stream) == hipSuccess) {
    c.idle.push_back(l.block);
    return;
  }
  // no way to tell when its last use ends: hipFree waits for the device
  c.kept -= l.block.bytes;
  lk.unlock();
  (void)hipGetLastError();
  (void)hipFree(p);
  (void)hipEventDestroy(l.block.done);
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

int device_alloc(void** out, size_t bytes, const char* ctx)
{
  int device = 0;
  int rc = check_hip(hipGetDevice(&device), ctx);
  if (rc) return rc;
  hipError_t st = hipMalloc(out, bytes);
  if (st == hipErrorOutOfMemory) {
    (void)hipGetLastError();
    if (scratch_drop(device)) st = hipMalloc(out, bytes);
  }
  return check_hip(st, ctx);
}

void scratch_trim(int device)
{
  (void)scratch_drop(device);
  const RelaxedCapture relaxed;
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
