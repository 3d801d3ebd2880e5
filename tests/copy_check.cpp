// Host check of the read-back's copying (ngi_copy.h): every chunk is copied
// once, through any number of slots, with any number of helpers; a helper that
// comes late keeps nobody waiting and touches neither buffer; an error ends the
// job.  Prints "ok" and exits 0, or says what is wrong and exits 1.
#include <chrono>
#include <cstdio>

#include "ngi_copy.h"

using namespace ngi;
using Clock = std::chrono::steady_clock;

static int g_bad = 0;
static void check(bool ok, const char* what, size_t a = 0, size_t b = 0) {
    if (!ok) printf("%s (%zu, %zu)\n", what, a, b), g_bad = 1;
}

// Chunk k is the number k + 1, written into its slot and copied to out[k].
struct Transfer {
    std::vector<size_t> ring, out;
    std::shared_ptr<ChunkJob> job;
    Transfer(size_t chunks, size_t slots, size_t fail_at = ~(size_t)0)
        : ring(slots), out(chunks), job(std::make_shared<ChunkJob>(chunks, slots, [this, slots, fail_at](size_t k) {
              if (k == fail_at) return 7;
              out[k] += ring[k % slots];
              return 0;
          })) {}
    int run(size_t refuse = ~(size_t)0) {
        return job->run([&](size_t k) {
            if (k == refuse) return 9;
            ring[k % ring.size()] = k + 1;
            return 0;
        });
    }
    bool whole() const {
        for (size_t k = 0; k < out.size(); ++k)
            if (out[k] != k + 1) return false;
        return true;
    }
};

int main() {
    for (size_t slots : {1, 2, 16})
        for (size_t chunks : {1, 2, 15, 16, 17, 333})
            for (unsigned helpers : {0u, 1u, 7u}) {
                CopyHelpers pool;
                for (int again = 0; again < 20; ++again) {
                    Transfer t(chunks, slots);
                    if (helpers) pool.post(t.job, helpers);
                    check(t.run() == 0 && t.whole(), "chunks lost", chunks, slots);
                    if (helpers) pool.withdraw();
                }
            }
    {
        // A helper that the scheduler runs only after half a second.
        auto t = std::make_unique<Transfer>(40, 16);
        std::shared_ptr<ChunkJob> job = t->job;
        std::thread late([job] {
            std::this_thread::sleep_for(std::chrono::milliseconds(500));
            job->help();
        });
        const auto t0 = Clock::now();
        check(t->run() == 0 && t->whole(), "chunks lost beside a late helper");
        check(Clock::now() - t0 < std::chrono::milliseconds(250), "waited for a late helper");
        t.reset();   // the buffers are gone before it comes
        late.join();
    }
    for (unsigned helpers : {0u, 3u}) {
        CopyHelpers pool;
        for (size_t at : {0, 1, 39}) {
            Transfer t(40, 16, at), u(40, 16);
            if (helpers) pool.post(t.job, helpers);
            check(t.run() == 7, "a copy's error is lost", at);
            if (helpers) pool.withdraw(), pool.post(u.job, helpers);
            check(u.run(at) == 9, "a producer's error is lost", at);
            if (helpers) pool.withdraw();
        }
    }
    if (!g_bad) printf("ok\n");
    return g_bad;
}
