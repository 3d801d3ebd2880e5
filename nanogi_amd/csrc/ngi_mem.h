// Device workspaces kept between calls, and results read back through pinned
// memory.
//
// Both serve the whole process (every scene lives on device 0), are bounded,
// and are given back when the last resident scene goes (pinned memory the first
// time only: see GiveBack).
#pragma once

#include <stddef.h>

#include <functional>

#include <hip/hip_runtime.h>

namespace ngi {

// hipMalloc that gives the kept workspaces back and tries again when the
// device is out of memory.
hipError_t device_malloc(void** p, size_t bytes);
template <typename T>
hipError_t device_malloc(T** p, size_t bytes) { return device_malloc(reinterpret_cast<void**>(p), bytes); }

// Workspaces of sessions and adjoints (films, counters, shadow rings, queues,
// records): workspace_free keeps the newest of them, up to 512 MB, for the next
// workspace_alloc.  The caller has waited for every kernel that uses a block
// before it frees it, so a block may move between scenes and streams.
// Contents are undefined.
hipError_t workspace_alloc(void** p, size_t bytes);
template <typename T>
hipError_t workspace_alloc(T** p, size_t bytes) { return workspace_alloc(reinterpret_cast<void**>(p), bytes); }
void workspace_free(void* p);

// Scenes with a device copy: +1 / -1.
void resident_scenes(int delta);

// Copies `bytes` results of stream `st` into pageable host memory.  `emit`
// enqueues the production of bytes [at, at + n) into the pinned buffer `dst`
// (a copy, or a kernel: the buffer is mapped) and returns an NGI status; at is
// a multiple of 1 MiB.  The caller has waited for the work before.  Returns an
// NGI status, or NGI_NOT_PINNED, with nothing done, where no memory can be
// pinned (or NGI_PINNED=0 is in the environment) or another thread reads back:
// the caller then copies through the runtime, so no thread waits for
// another's results.
#define NGI_NOT_PINNED (-1)
bool pinned_free();   // whether read_pinned would start now
int read_pinned(hipStream_t st, void* out, size_t bytes, const std::function<int(size_t at, size_t n, void* dst)>& emit);

// A block of mapped pinned memory for a small exchange, one of 16: its
// address, or null when all are in use, for more bytes than a block's, or where
// no memory can be pinned.  The holder may wait for its stream.
#define NGI_PIN_BLOCK_BYTES ((size_t)65536)
class PinnedBlock {
public:
    explicit PinnedBlock(size_t bytes);
    ~PinnedBlock();
    PinnedBlock(const PinnedBlock&) = delete;
    PinnedBlock& operator=(const PinnedBlock&) = delete;
    void* get() const { return p; }

private:
    void* p = nullptr;
};

}  // namespace ngi
