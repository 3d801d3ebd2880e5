// Kept device workspaces and the pinned read-back (ngi_mem.h).
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <memory>
#include <mutex>
#include <thread>
#include <unordered_map>
#include <vector>

#include "ngi_copy.h"
#include "ngi_dev.h"
#include "ngi_mem.h"

namespace ngi {

#define NGI_KEPT_BYTES ((size_t)512 << 20)
// The pinned buffer is a ring of NGI_PIN_SLOTS slots.
#define NGI_PIN_SLOT ((size_t)1 << 20)
#define NGI_PIN_SLOTS 16
#define NGI_PIN_THREADS 8
#define NGI_PIN_HELP ((size_t)8 << 20)
// Blocks of PinnedBlock.
#define NGI_PIN_BLOCKS 16

namespace {

bool may_pin() {
    const char* e = getenv("NGI_PINNED");
    return !(e && !strcmp(e, "0"));
}

struct Workspaces {
    std::mutex mu;
    std::unordered_map<void*, size_t> size;   // of every block handed out or kept
    std::vector<void*> kept;                  // oldest first
    size_t kept_bytes = 0;
    int scenes = 0;

    // Takes the oldest kept blocks out until at most `bytes` are kept; the
    // caller frees them once it has let go of mu, since hipFree may wait for
    // the device.
    std::vector<void*> trim(size_t bytes) {
        std::vector<void*> out;
        size_t n = 0;
        for (; kept_bytes > bytes; ++n) {
            kept_bytes -= size[kept[n]];
            size.erase(kept[n]);
            out.push_back(kept[n]);
        }
        kept.erase(kept.begin(), kept.begin() + (long)n);
        return out;
    }
};

void free_all(const std::vector<void*>& blocks) {
    for (void* p : blocks) (void)hipFree(p);
}

// Pinned memory is given back with the last resident scene, but only once: a
// program that has to pin it again holds one scene after another, and fresh
// pages cost it more than the copies they serve (host queries of 1M rays on a
// new scene each: 4.6 ms with pages pinned anew, 2.8 with kept ones, 3.2
// through the runtime).
struct GiveBack {
    bool given = false, kept = false;
    void pinned() { kept = given; }   // memory has been pinned
    bool due() {                      // the last scene is gone
        given = true;
        return !kept;
    }
};

// hipHostMalloc, and the events of `done`, on the device of every scene: the
// calling thread's may be another one.
char* pin(size_t bytes, hipEvent_t* done = nullptr, int events = 0) {
    int dev = 0;
    if (hipGetDevice(&dev) == hipSuccess && dev != 0) (void)hipSetDevice(0);
    void* q = nullptr;
    bool ok = hipHostMalloc(&q, bytes, hipHostMallocDefault) == hipSuccess;
    for (int i = 0; i < events && ok; ++i)
        if (!done[i] && hipEventCreateWithFlags(&done[i], hipEventDisableTiming) != hipSuccess) {
            done[i] = nullptr;
            (void)hipHostFree(q);
            ok = false;
        }
    if (!ok) (void)hipGetLastError();
    if (dev != 0) (void)hipSetDevice(dev);
    return ok ? static_cast<char*>(q) : nullptr;
}

struct Pinned {
    std::mutex mu;   // held while the buffer is in use
    char* p = nullptr;
    GiveBack back;
    hipEvent_t done[NGI_PIN_SLOTS] = {};
    std::unique_ptr<CopyHelpers> helpers;

    bool ensure() {   // mu held
        if (!may_pin()) return false;
        if (p) return true;
        p = pin(NGI_PIN_SLOT * NGI_PIN_SLOTS, done, NGI_PIN_SLOTS);
        if (p) back.pinned();
        return p != nullptr;
    }
    void release() {   // mu held
        helpers.reset();
        if (p) (void)hipHostFree(p);
        p = nullptr;
        for (hipEvent_t& e : done) {
            if (e) (void)hipEventDestroy(e);
            e = nullptr;
        }
    }
};

struct Blocks {
    std::mutex mu;   // never held while the device is waited for
    char* p = nullptr;
    uint32_t used = 0;
    GiveBack back;
};

// Never destroyed: calls may come from other static destructors.
Workspaces& workspaces() {
    static Workspaces* w = new Workspaces();
    return *w;
}
Pinned& pinned() {
    static Pinned* p = new Pinned();
    return *p;
}
Blocks& blocks() {
    static Blocks* b = new Blocks();
    return *b;
}

}  // namespace

hipError_t device_malloc(void** p, size_t bytes) {
    hipError_t e = hipMalloc(p, bytes);
    if (e != hipErrorOutOfMemory) return e;
    (void)hipGetLastError();
    Workspaces& w = workspaces();
    std::vector<void*> all;
    {
        std::lock_guard<std::mutex> lock(w.mu);
        all = w.trim(0);
    }
    free_all(all);
    return hipMalloc(p, bytes);
}

hipError_t workspace_alloc(void** p, size_t bytes) {
    Workspaces& w = workspaces();
    {
        std::lock_guard<std::mutex> lock(w.mu);
        size_t best = w.kept.size();
        for (size_t i = 0; i < w.kept.size(); ++i) {
            const size_t n = w.size[w.kept[i]];
            // Not a block much larger than needed: it may be wanted as it is.
            if (n >= bytes && n <= 2 * bytes + 65536 && (best == w.kept.size() || n < w.size[w.kept[best]])) best = i;
        }
        if (best < w.kept.size()) {
            *p = w.kept[best];
            w.kept_bytes -= w.size[*p];
            w.kept.erase(w.kept.begin() + (long)best);
            return hipSuccess;
        }
    }
    const hipError_t e = device_malloc(p, bytes);
    if (e != hipSuccess) return e;
    std::lock_guard<std::mutex> lock(w.mu);
    w.size[*p] = bytes;
    return hipSuccess;
}

void workspace_free(void* p) {
    if (!p) return;
    Workspaces& w = workspaces();
    std::vector<void*> old;
    {
        std::lock_guard<std::mutex> lock(w.mu);
        const auto it = w.size.find(p);
        if (it == w.size.end()) return;
        // The newest block is the likeliest to be wanted again: older ones make
        // room for it, unless it is more than may be kept by itself.
        if (w.scenes > 0 && it->second <= NGI_KEPT_BYTES) {
            w.kept.push_back(p);
            w.kept_bytes += it->second;
            old = w.trim(NGI_KEPT_BYTES);
        } else {
            w.size.erase(it);
            old.push_back(p);
        }
    }
    free_all(old);
}

void resident_scenes(int delta) {
    Workspaces& w = workspaces();
    std::vector<void*> all;
    {
        std::lock_guard<std::mutex> lock(w.mu);
        w.scenes += delta;
        if (w.scenes > 0) return;
        all = w.trim(0);
    }
    free_all(all);
    Pinned& b = pinned();
    {
        std::lock_guard<std::mutex> ring(b.mu);
        if (b.p && b.back.due()) b.release();
    }
    Blocks& k = blocks();
    std::lock_guard<std::mutex> small(k.mu);
    if (k.p && !k.used && k.back.due()) {
        (void)hipHostFree(k.p);
        k.p = nullptr;
    }
}

PinnedBlock::PinnedBlock(size_t bytes) {
    if (bytes > NGI_PIN_BLOCK_BYTES || !may_pin()) return;
    Blocks& k = blocks();
    std::lock_guard<std::mutex> lock(k.mu);
    if (!k.p) {
        k.p = pin(NGI_PIN_BLOCK_BYTES * NGI_PIN_BLOCKS);
        if (!k.p) return;
        k.back.pinned();
    }
    static_assert(NGI_PIN_BLOCKS < 32, "bits of used");
    const int i = __builtin_ctz(~k.used);
    if (i >= NGI_PIN_BLOCKS) return;
    k.used |= 1u << i;
    p = k.p + NGI_PIN_BLOCK_BYTES * i;
}
PinnedBlock::~PinnedBlock() {
    if (!p) return;
    Blocks& k = blocks();
    std::lock_guard<std::mutex> lock(k.mu);
    k.used &= ~(1u << ((static_cast<char*>(p) - k.p) / NGI_PIN_BLOCK_BYTES));
}

bool pinned_free() {
    Pinned& b = pinned();
    std::unique_lock<std::mutex> lock(b.mu, std::try_to_lock);
    return lock && b.ensure();
}

// The runtime's copy into pageable memory reads back 7 GB/s, on one thread
// that mostly touches the caller's pages for the first time.  Here the device
// fills the ring's slots (kernels write finished results straight into mapped
// memory) while the calling thread, and helpers from NGI_PIN_HELP bytes on,
// copy filled slots out.
// Measured, whole calls, ms (with the kept workspaces): a 1280x720 film after
// 1.2 ms of rendering 3.39 -> 2.17, a 1024x1024 film and its variance after
// 32 ms 52.1 -> 34.1.  Up to 8 MiB the calling thread alone is as fast in a
// quiet process (700x500 pixels 0.77 ms, with helpers 0.84) and steadier beside
// busy threads: median and 90% of a gradient step by autograd on 500x380 pixels
// at 1 spp, ms: the runtime's copy 3.0 / 3.1, helpers from 1 MiB on that were
// joined 3.9 / 4.7, now 1.7 / 2.0; on 1024x768 pixels at 4 spp 9.2 / 9.5, 7.3 /
// 7.6, 6.3 / 6.9.
int read_pinned(hipStream_t st, void* out, size_t bytes, const std::function<int(size_t, size_t, void*)>& emit) {
    if (bytes == 0) return NGI_OK;
    Pinned& b = pinned();
    std::unique_lock<std::mutex> lock(b.mu, std::try_to_lock);
    if (!lock || !b.ensure()) return NGI_NOT_PINNED;
    if (bytes <= NGI_PIN_SLOT) {   // one slot: nothing to overlap
        const int s = emit(0, bytes, b.p);
        if (hipStreamSynchronize(st) != hipSuccess) return fail(NGI_ERR_DEVICE, "reading results back failed");
        if (s == NGI_OK) memcpy(out, b.p, bytes);
        return s;
    }
    const size_t chunks = (bytes + NGI_PIN_SLOT - 1) / NGI_PIN_SLOT;
    const auto size = [=](size_t k) { return std::min(NGI_PIN_SLOT, bytes - k * NGI_PIN_SLOT); };
    const auto job = std::make_shared<ChunkJob>(chunks, (size_t)NGI_PIN_SLOTS, [&b, out, size](size_t k) {
        if (hipEventSynchronize(b.done[k % NGI_PIN_SLOTS]) != hipSuccess) return (int)NGI_ERR_DEVICE;
        memcpy(static_cast<char*>(out) + k * NGI_PIN_SLOT, b.p + k % NGI_PIN_SLOTS * NGI_PIN_SLOT, size(k));
        return (int)NGI_OK;
    });
    const size_t want = std::min<size_t>(NGI_PIN_THREADS - 1, std::max(1u, std::thread::hardware_concurrency()) - 1);
    const bool help = bytes >= NGI_PIN_HELP && want;
    if (help) {
        if (!b.helpers) b.helpers.reset(new CopyHelpers());
        b.helpers->post(job, (unsigned)want);
    }
    const int s = job->run([&](size_t k) {
        const int e = emit(k * NGI_PIN_SLOT, size(k), b.p + k % NGI_PIN_SLOTS * NGI_PIN_SLOT);
        return e != NGI_OK ? e : hipEventRecord(b.done[k % NGI_PIN_SLOTS], st) == hipSuccess ? (int)NGI_OK : (int)NGI_ERR_DEVICE;
    });
    if (help) b.helpers->withdraw();
    if (s != NGI_OK) {
        (void)hipStreamSynchronize(st);   // nothing writes the buffer once it is let go
        return s == NGI_ERR_DEVICE ? fail(NGI_ERR_DEVICE, "reading results back failed") : s;
    }
    return NGI_OK;
}

}  // namespace ngi
