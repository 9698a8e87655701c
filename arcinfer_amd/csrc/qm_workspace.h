// Per-call workspaces of the prompt GEMM (qm_workspace.hip; host code, no kernels).
#pragma once
#include <hip/hip_runtime_api.h>
#include <stddef.h>

namespace qm {

// A per-device stream-ordered memory pool for per-call workspaces
hipError_t pool_alloc(void** out, size_t bytes, hipStream_t s);
// A per-call workspace of the current device, for work enqueued on s between the two calls: a buffer kept from an earlier call
// (not on a capturing stream), ordered after that call's work, or memory of the pool. `need` bytes, and `extra` behind them as far as
// memory goes (all: they are there). workspaces_give_back waits for the kept buffers that no call is using, on every device, and
// returns their memory to the device; false: there were none.
struct CallWs {
  void* p = nullptr;
  int kept = -1;  // index of the kept buffer, -1: the pool's
  bool all = true;
};
hipError_t workspace_take(CallWs* ws, size_t need, size_t extra, bool capturing, hipStream_t s);
hipError_t workspace_done(const CallWs& ws, hipStream_t s);
bool workspaces_give_back();

// Use of the current device's static partial-tile array by work enqueued on s between enter and leave: behind the work of the call
// that used it before, on whatever stream, and other threads' calls wait outside. Not on a capturing stream.
hipError_t shared_enter(hipStream_t s);
hipError_t shared_leave(hipStream_t s);

}  // namespace qm
