// Host side of the pinned read-back: chunks that the device fills are copied
// out by the calling thread and by helper threads (host code only).
#pragma once

#include <stddef.h>
#include <stdint.h>

#include <atomic>
#include <condition_variable>
#include <functional>
#include <memory>
#include <mutex>
#include <thread>
#include <utility>
#include <vector>

namespace ngi {

// `chunks` chunks through a ring of `slots` slots.  A thread claims a chunk
// that has been emitted before it copies it, and run() waits for claimed chunks
// only: a helper that comes late, or never, costs nothing, and touches nothing
// but this object (hold it by shared_ptr).  Joining helpers instead made a call
// wait until the scheduler had run each of them once: beside busy threads (the
// spinning workers of a torch operation) a gradient step on a 190k-pixel image
// took 4.0 ms where the runtime's copy took 3.0.
class ChunkJob {
public:
    // copy(k) copies chunk k out of its slot; 0 or an error, which ends the job.
    ChunkJob(size_t chunks, size_t slots, std::function<int(size_t)> copy)
        : chunks(chunks), slots(slots), copy(std::move(copy)), copied(new std::atomic<size_t>[slots]) {
        for (size_t i = 0; i < slots; ++i) copied[i].store(0);
    }

    // The calling thread's part: emit(k) has chunk k produced into its slot (0
    // or an error).  Returns once every chunk has been copied, or nothing is
    // being copied any more after an error, which it returns.
    int run(const std::function<int(size_t)>& emit) {
        for (size_t k = 0; k < chunks && !status.load(); ) {
            if (copied[k % slots].load(std::memory_order_acquire) < k / slots) {   // the slot's previous chunk
                if (!copy_one()) std::this_thread::yield();
                continue;
            }
            const int s = emit(k);
            if (s) status.store(s);
            else emitted.store(++k, std::memory_order_release);
        }
        while (copy_one()) {
        }
        // No chunk can be claimed any more: the rest, if any, is lost to an error.
        const size_t claimed = taken.exchange(chunks);
        while (done.load(std::memory_order_acquire) < claimed) std::this_thread::yield();
        return status.load();
    }

    // A helper's part: copies chunks until there is none left.
    void help() {
        while (!status.load() && taken.load() < chunks)
            if (!copy_one()) std::this_thread::yield();
    }

private:
    bool copy_one() {   // false: no chunk to claim now
        if (status.load()) return false;
        size_t k = taken.load();
        do {
            if (k >= emitted.load(std::memory_order_acquire)) return false;
        } while (!taken.compare_exchange_weak(k, k + 1));
        const int s = copy(k);
        if (s) status.store(s);
        copied[k % slots].fetch_add(1, std::memory_order_release);
        done.fetch_add(1, std::memory_order_release);
        return true;
    }

    const size_t chunks, slots;
    const std::function<int(size_t)> copy;
    const std::unique_ptr<std::atomic<size_t>[]> copied;   // chunks copied out of each slot
    std::atomic<size_t> emitted{0}, taken{0}, done{0};
    std::atomic<int> status{0};
};

// Threads that sleep between jobs and help with one at a time.  They are let go
// with this object, which waits for none of them.
class CopyHelpers {
public:
    CopyHelpers() : st(std::make_shared<State>()) {}
    ~CopyHelpers() {
        std::lock_guard<std::mutex> lock(st->mu);
        st->quit = true;
        st->job.reset();
        st->cv.notify_all();
    }
    CopyHelpers(const CopyHelpers&) = delete;
    CopyHelpers& operator=(const CopyHelpers&) = delete;

    // Asks `n` threads to help with the job (fewer where no more can be had).
    void post(const std::shared_ptr<ChunkJob>& job, unsigned n) {
        std::lock_guard<std::mutex> lock(st->mu);
        st->job = job;
        st->wanted = n;
        try {
            for (; threads < n; ++threads) std::thread(work, st).detach();
        } catch (...) {
        }
        st->cv.notify_all();
    }
    // The job is over: helpers that have not come yet go on sleeping.
    void withdraw() {
        std::lock_guard<std::mutex> lock(st->mu);
        st->job.reset();
        st->wanted = 0;
    }

private:
    struct State {
        std::mutex mu;
        std::condition_variable cv;
        std::shared_ptr<ChunkJob> job;
        unsigned wanted = 0;
        bool quit = false;
    };
    static void work(std::shared_ptr<State> s) {
        std::unique_lock<std::mutex> lock(s->mu);
        for (;;) {
            s->cv.wait(lock, [&] { return s->quit || (s->job && s->wanted); });
            if (s->quit) return;
            s->wanted--;
            std::shared_ptr<ChunkJob> job = s->job;
            lock.unlock();
            job->help();
            job.reset();
            lock.lock();
        }
    }
    const std::shared_ptr<State> st;
    unsigned threads = 0;
};

}  // namespace ngi
