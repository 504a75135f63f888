// runtime.hh -- per-stream workspaces and error reporting of the backend.
#pragma once

#include <hip/hip_runtime.h>

#include <condition_variable>
#include <cstdint>
#include <mutex>
#include <string>

#include "backend.hh"

namespace honei {
namespace hipx {

// Persistent scratch owned by the library, one per (device, stream): the
// cross-block reduction slots plus a small array of device scalars.  Created
// on first use with hipMalloc, kept until honei_hip_shutdown(); no per-call
// allocation on any path.
struct Workspace {
    // Held by a call while it enqueues launches that use the slots or scalars
    // (another thread's on the same stream then follow all of them), and by a
    // solve, which also reads back between them, until it returns.
    std::mutex use;
    ReduceSlots slots;
    double *scalars = nullptr;   // kScalars doubles
    static constexpr int kScalars = 256;
    static constexpr int kSlotCapacity = 1 << 17;   // blocks
    static constexpr int kSlotLanes = 4;
    // Results of reductions that return to the host (ReturnSlot): pinned,
    // written by the reduction's last kernel itself.
    static constexpr int kReturns = 64;
    double *returns = nullptr;
    uint64_t returns_free = ~uint64_t(0);   // bit k: returns[k] has no owner
    std::mutex returns_mutex;
    std::condition_variable returned;
    void *scratch = nullptr;     // grows on demand, never shrinks
    size_t scratch_bytes = 0;
    // Returns a buffer of at least `bytes` (reallocating only when larger
    // than any earlier request), or nullptr on allocation failure.
    void *ensure_scratch(size_t bytes);
};

// One of a workspace's results, owned by a call from before its launches until
// it has read the value; a call that finds none free waits for another's (an
// owner waits for its launches only).
class ReturnSlot {
  public:
    explicit ReturnSlot(Workspace &w);
    ~ReturnSlot();
    ReturnSlot(const ReturnSlot &) = delete;
    ReturnSlot &operator=(const ReturnSlot &) = delete;
    double *get() const { return w_.returns + k_; }

  private:
    Workspace &w_;
    int k_;
};

// Returns nullptr (and records the error) when allocation fails.
Workspace *workspace_for(hipStream_t s);
void release_workspaces();

void set_error(const std::string &msg);
const char *last_error();

}  // namespace hipx
}  // namespace honei
