// Per-call workspaces of the prompt GEMM (host code only).
#include "qm_workspace.h"

#include <stdint.h>

#include <mutex>

namespace qm {

// One memory pool per device for the per-call workspace (stream-ordered: concurrent calls on different streams get
// different buffers; the pool keeps freed memory for the next call).
static hipError_t call_pool(hipMemPool_t* out) {
  static std::mutex mu;
  static hipMemPool_t pools[64] = {};
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= 64) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(mu);
  if (!pools[dev]) {
    hipMemPoolProps props{};
    props.allocType = hipMemAllocationTypePinned;
    props.location.type = hipMemLocationTypeDevice;
    props.location.id = dev;
    hipMemPool_t p;
    e = hipMemPoolCreate(&p, &props);
    if (e != hipSuccess) return e;
    uint64_t thr = ~0ull;
    e = hipMemPoolSetAttribute(p, hipMemPoolAttrReleaseThreshold, &thr);
    if (e != hipSuccess) return e;
    pools[dev] = p;
  }
  *out = pools[dev];
  return hipSuccess;
}

hipError_t pool_alloc(void** out, size_t bytes, hipStream_t s) {
  hipMemPool_t pool = nullptr;
  const hipError_t e = call_pool(&pool);
  return e == hipSuccess ? hipMallocFromPoolAsync(out, bytes, pool, s) : e;
}

// Kept workspaces. Taking a workspace from the pool and freeing it costs the host 10 to 30 us a call, and 50 to 70 us more
// when other memory of the process was freed in between, which short prompts wait for. Up to 8 buffers a device
// (32 MiB steps, 128 MiB at most each) stay allocated instead; each has an event recorded behind its last use. A call takes the one
// that its stream used last (behind the event: a stream's handle only says which to prefer, handles are reused), or one whose work
// has ended, or a new one in place of an empty slot or of a smaller buffer of these two kinds, or else memory of the pool, so
// that no stream waits for another's work. A buffer is out of the list while a call enqueues its work. They are returned when the last weight is released.
constexpr int kKeptMax = 8;
constexpr size_t kKeptStep = (size_t)32 << 20, kKeptBytes = (size_t)128 << 20;
struct KeptWs {
  void* p = nullptr;
  size_t bytes = 0;
  hipEvent_t ev = nullptr;
  hipStream_t last = nullptr;
  bool busy = false;
};
// whether the work of a buffer's last call has ended
static bool ended(const KeptWs& k) {
  if (hipEventQuery(k.ev) == hipSuccess) return true;
  (void)hipGetLastError();
  return false;
}

// A capture that the thread has open on another stream is none of a call's business: event queries, allocations and frees made here
// are no part of it and must not end it.
struct Relaxed {
  hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
  Relaxed() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
  ~Relaxed() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
};

static std::mutex g_kept_mu;
static KeptWs g_kept[64][kKeptMax];

static hipError_t take(CallWs* ws, size_t bytes, bool capturing, hipStream_t s) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  *ws = CallWs{};
  if (!capturing && dev >= 0 && dev < 64 && bytes <= kKeptBytes) {
    Relaxed relaxed;
    std::lock_guard<std::mutex> lock(g_kept_mu);
    int pick = -1, place = -1;  // a buffer to take; the slot of a new one: the stream's own, an empty one, the smallest that has ended
    for (int i = 0; i < kKeptMax; ++i) {
      const KeptWs& k = g_kept[dev][i];
      if (k.busy) continue;
      const bool own = k.p && k.last == s;
      if (k.bytes >= bytes && (own || (pick < 0 && ended(k)))) {
        pick = i;
        if (own) break;
      } else if (k.bytes < bytes) {
        const KeptWs* q = place < 0 ? nullptr : &g_kept[dev][place];
        if (!q || own || (!(q->p && q->last == s) && k.bytes < q->bytes))
          if (own || !k.p || ended(k)) place = i;
      }
    }
    if (pick < 0 && place >= 0) {
      KeptWs& k = g_kept[dev][place];
      if (k.p) {  // (freed behind the work of its last call)
        if (hipStreamWaitEvent(s, k.ev, 0) != hipSuccess || hipFreeAsync(k.p, s) != hipSuccess) {
          (void)hipGetLastError();
          return pool_alloc(&ws->p, bytes, s);
        }
        k.p = nullptr;
        k.bytes = 0;
      }
      const size_t size = (bytes + kKeptStep - 1) / kKeptStep * kKeptStep;
      e = k.ev ? hipSuccess : hipEventCreateWithFlags(&k.ev, hipEventDisableTiming);
      if (e == hipSuccess) e = pool_alloc(&k.p, size, s);
      if (e == hipSuccess) {
        k.bytes = size;
        k.last = s;
        k.busy = true;
        *ws = CallWs{k.p, place};
        return hipSuccess;
      }
      k.p = nullptr;
      (void)hipGetLastError();
    }
    if (pick >= 0) {
      KeptWs& k = g_kept[dev][pick];
      e = hipStreamWaitEvent(s, k.ev, 0);
      if (e == hipSuccess) {
        k.last = s;
        k.busy = true;
        *ws = CallWs{k.p, pick};
        return hipSuccess;
      }
      (void)hipGetLastError();
    }
  }
  return pool_alloc(&ws->p, bytes, s);
}

hipError_t workspace_take(CallWs* ws, size_t need, size_t extra, bool capturing, hipStream_t s) {
  hipError_t e = take(ws, need + extra, capturing, s);
  if (e != hipSuccess && need && extra) {
    (void)hipGetLastError();
    e = take(ws, need, capturing, s);
    ws->all = false;
  }
  if (e != hipSuccess) ws->p = nullptr;
  return e;
}

hipError_t workspace_done(const CallWs& ws, hipStream_t s) {
  if (ws.kept < 0) return hipFreeAsync(ws.p, s);
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;  // (the buffer stays out of the list)
  e = hipEventRecord(g_kept[dev][ws.kept].ev, s);
  if (e != hipSuccess) return e;
  std::lock_guard<std::mutex> lock(g_kept_mu);
  g_kept[dev][ws.kept].busy = false;
  return hipSuccess;
}

bool workspaces_give_back() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return false;
  bool any = false;
  Relaxed relaxed;
  std::lock_guard<std::mutex> lock(g_kept_mu);
  for (int d = 0; d < 64; ++d) {
    bool here = false;
    for (int i = 0; i < kKeptMax; ++i) {
      KeptWs& k = g_kept[d][i];
      if (!k.p || k.busy) continue;
      if (hipSetDevice(d) != hipSuccess || hipEventSynchronize(k.ev) != hipSuccess || hipFreeAsync(k.p, nullptr) != hipSuccess) {
        (void)hipGetLastError();
        continue;
      }
      k.p = nullptr;
      k.bytes = 0;
      here = true;
    }
    // (a freed buffer stays the pool's, out of reach of any other allocation, until the pool is trimmed)
    hipMemPool_t pool = nullptr;
    if (here && (hipStreamSynchronize(nullptr) != hipSuccess || call_pool(&pool) != hipSuccess || hipMemPoolTrimTo(pool, 0) != hipSuccess))
      (void)hipGetLastError();
    any = any || here;
  }
  (void)hipSetDevice(dev);
  return any;
}

struct Shared {
  std::mutex mu;
  hipEvent_t ev = nullptr;
};
static Shared g_shared[64];

hipError_t shared_enter(hipStream_t s) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= 64) return hipErrorInvalidDevice;
  Shared& g = g_shared[dev];
  Relaxed relaxed;
  g.mu.lock();
  e = g.ev ? hipStreamWaitEvent(s, g.ev, 0) : hipEventCreateWithFlags(&g.ev, hipEventDisableTiming);
  if (e != hipSuccess) g.mu.unlock();
  return e;
}

hipError_t shared_leave(hipStream_t s) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  e = hipEventRecord(g_shared[dev].ev, s);
  g_shared[dev].mu.unlock();
  return e;
}

}  // namespace qm
