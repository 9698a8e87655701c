// The memory, stream and event calls that qm_workspace.hip makes, on a device of `capacity` bytes that exists on paper, and the
// scenarios of tests/test_workspace.py: each prints what it saw.
#include <stdio.h>
#include <string.h>

#include <map>
#include <set>
#include <vector>

#include "qm_workspace.h"

static size_t capacity = ~(size_t)0, live = 0, reserved = 0;  // allocated; held by the pool (allocated or not given back)
static std::map<void*, size_t> blocks;
static std::vector<size_t> asked;
static uintptr_t next_ptr = 4096;
static std::map<hipEvent_t, bool> done;  // an event's last record: has its work ended?
static int waits = 0, syncs = 0;
static hipError_t last = hipSuccess;

static hipError_t ret(hipError_t e) {
  if (e != hipSuccess) last = e;
  return e;
}
extern "C" {
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError() {
  const hipError_t e = last;
  last = hipSuccess;
  return e;
}
hipError_t hipMemPoolCreate(hipMemPool_t* p, const hipMemPoolProps*) { return *p = (hipMemPool_t)1, hipSuccess; }
hipError_t hipMemPoolSetAttribute(hipMemPool_t, hipMemPoolAttr, void*) { return hipSuccess; }
hipError_t hipMemPoolTrimTo(hipMemPool_t, size_t) { return reserved = live, hipSuccess; }
hipError_t hipMallocFromPoolAsync(void** p, size_t n, hipMemPool_t, hipStream_t) {
  asked.push_back(n);
  if (live + n > capacity) return ret(hipErrorOutOfMemory);
  *p = (void*)(next_ptr += 4096);
  blocks[*p] = n;
  live += n;
  if (live > reserved) reserved = live;
  return hipSuccess;
}
hipError_t hipFreeAsync(void* p, hipStream_t) {
  if (!blocks.count(p)) return ret(hipErrorInvalidValue);
  live -= blocks[p];
  blocks.erase(p);
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  *e = (hipEvent_t)(next_ptr += 4096);
  done[*e] = true;
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) { return done[e] = false, hipSuccess; }
hipError_t hipEventQuery(hipEvent_t e) { return done[e] ? hipSuccess : ret(hipErrorNotReady); }
hipError_t hipEventSynchronize(hipEvent_t e) { return done[e] = true, ++syncs, hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t e, unsigned) { return waits += !done[e], hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return ++syncs, hipSuccess; }
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode*) { return hipSuccess; }
}

constexpr size_t MiB = (size_t)1 << 20;
static hipStream_t stream(int i) { return (hipStream_t)(uintptr_t)(i + 1); }
static bool call(size_t need, size_t extra, int s, bool* all = nullptr, bool capturing = false) {
  qm::CallWs ws;
  const bool ok = qm::workspace_take(&ws, need, extra, capturing, stream(s)) == hipSuccess;
  if (all) *all = ok && ws.all;
  if (ok) (void)qm::workspace_done(ws, stream(s));
  return ok;
}
static void gpu_idle() {
  for (auto& e : done) e.second = true;
}

int main(int argc, char** argv) {
  const char* what = argc > 1 ? argv[1] : "";
  if (!strcmp(what, "need_alone")) {
    capacity = 24 * MiB;
    bool all = true;
    const bool ok = call(20 * MiB, 30 * MiB, 0, &all);
    printf("%d %d %d\n", ok, all, (int)last);
  } else if (!strcmp(what, "streams")) {  // twelve streams with work in flight, twice; then one more stream, all work done
    bool ok = true;
    for (int turn = 0; turn < 2; ++turn)
      for (int s = 0; s < 12; ++s) ok = ok && call(20 * MiB, 0, s);
    const size_t kept = blocks.size(), calls = asked.size();
    gpu_idle();
    ok = ok && call(20 * MiB, 0, 99);
    printf("%d %d %d %d %d\n", ok, waits - 8, (int)kept, (int)(asked.size() - calls), (int)last);  // (8: their own last calls)
  } else if (!strcmp(what, "grow")) {  // eight streams' small buffers, then one stream's larger call, three times; and a stream's own
    bool ok = true;
    for (int s = 0; s < 8; ++s) ok = ok && call(20 * MiB, 0, s);
    gpu_idle();
    size_t calls = asked.size();
    for (int i = 0; i < 3; ++i) ok = ok && call(100 * MiB, 0, 99);
    const int first = (int)(asked.size() - calls), kept = (int)blocks.size();
    for (int s = 0; s < 8; ++s) ok = ok && call(20 * MiB, 0, s);  // (work in flight on every stream again)
    calls = asked.size();
    for (int i = 0; i < 3; ++i) ok = ok && call(50 * MiB, 0, 3);
    printf("%d %d %d %d %d\n", ok, first, kept, (int)(asked.size() - calls), (int)blocks.size());
  } else if (!strcmp(what, "give_back")) {  // three streams' buffers, one of them in a call that is still enqueueing
    bool ok = true;
    for (int s = 0; s < 2; ++s) ok = ok && call(20 * MiB, 0, s);
    qm::CallWs ws;
    ok = ok && qm::workspace_take(&ws, 20 * MiB, 0, false, stream(2)) == hipSuccess;
    qm::workspaces_give_back();
    const int left = (int)blocks.size(), held = (int)(reserved / MiB);
    ok = ok && qm::workspace_done(ws, stream(2)) == hipSuccess;
    qm::workspaces_give_back();
    ok = ok && call(20 * MiB, 0, 0);  // (and on as before)
    printf("%d %d %d %d %d %d\n", ok, left, held, (int)blocks.size(), (int)(reserved / MiB), (int)last);
  } else if (!strcmp(what, "shared")) {  // two streams' use of the one array, in turn
    bool ok = true;
    for (int i = 0; i < 4; ++i) {
      ok = ok && qm::shared_enter(stream(i & 1)) == hipSuccess;
      ok = ok && qm::shared_leave(stream(i & 1)) == hipSuccess;
    }
    printf("%d %d\n", ok, waits);
  }
  return 0;
}
