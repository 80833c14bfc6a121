// Copies of finished frames from pinned memory to the caller's buffers. One thread
// moves ~28 GB/s, half the rate at which the GPU delivers frames over PCIe, so a
// large copy is shared by the caller and a few helper threads (with reused result
// arrays: 8 requests delivered to the host 6.5 -> 3.0 ms, two presented 1280x720
// frames 571 -> 358 us; five or seven helpers gave no more). New pinned memory is
// mapped by the same threads, each taking large pages of its own.
#include <sched.h>
#include <unistd.h>

#include <atomic>
#include <condition_variable>
#include <cstdint>
#include <cstring>
#include <mutex>
#include <thread>

#include "gorender_hip.h"
#include "gr_copy.h"
#include "gr_error.h"

namespace {

constexpr size_t kShared = 512u << 10;  // least bytes worth waking the helpers for
constexpr size_t kPiece = 128u << 10;   // bytes a thread takes at a time
constexpr size_t kPage = 2u << 20;      // bytes a fault of pinned memory maps at most
constexpr int kHelpers = 3;

// The helper threads of the process. They live until it ends: the pool is never
// destroyed, and a thread that waits holds nothing. The caller copies too and
// takes every piece no helper has taken, so a copy never depends on them (a forked
// child, which has none, copies alone). The library is linked never to be unloaded,
// since they wait in its code.
class CopyPool {
public:
    void copy(char* dst, const char* src, size_t n) {
        run(Job{dst, src, n, 0, kPiece, (n + kPiece - 1) / kPiece, 0});
    }
    // Clears a byte of every page of [p, p + n), large page by large page.
    void touch(char* p, size_t n) {
        const size_t skew = (uintptr_t)p % kPage;
        run(Job{p, nullptr, n, skew, kPage, (skew + n + kPage - 1) / kPage, 0});
    }

private:
    // Piece k is what lies in [0, n) of [k * piece - skew, (k + 1) * piece - skew).
    struct Job {
        char* dst;
        const char* src;  // null: dst is touched
        size_t n, skew, piece, pieces;
        uint64_t id;
        void one(size_t k) const {
            const size_t b = k == 0 ? 0 : k * piece - skew;
            const size_t e = (k + 1) * piece - skew < n ? (k + 1) * piece - skew : n;
            if (src)
                std::memcpy(dst + b, src + b, e - b);
            else
                for (size_t i = b; i < e; i += 4096 - (uintptr_t)(dst + i) % 4096)
                    ((volatile char*)dst)[i] = 0;
        }
    };

    void run(Job job) {
        // One shared job at a time; another thread's is not waited for. A forked
        // child has no helpers.
        std::unique_lock<std::mutex> turn(turn_, std::try_to_lock);
        if (!turn.owns_lock() || !start() || getpid() != owner_) {
            for (size_t k = 0; k < job.pieces; k++) job.one(k);
            return;
        }
        {
            std::lock_guard<std::mutex> lk(mu_);
            job.id = ++id_;
            job_ = job;
            done_.store(0, std::memory_order_relaxed);
            next_.store(job.id << 32, std::memory_order_relaxed);
        }
        wake_.notify_all();
        work(job);
        while (done_.load(std::memory_order_acquire) != job.pieces) std::this_thread::yield();
    }

    // Takes pieces of `job` until none is left. `next_` holds the job's number with
    // the next piece's, so a helper that comes late takes none of a later job's.
    void work(const Job& job) {
        for (;;) {
            uint64_t at = next_.load(std::memory_order_acquire);
            do {
                if (at >> 32 != (job.id & 0xFFFFFFFFu) || (at & 0xFFFFFFFFu) >= job.pieces) return;
            } while (!next_.compare_exchange_weak(at, at + 1, std::memory_order_acq_rel));
            job.one((size_t)(at & 0xFFFFFFFFu));
            done_.fetch_add(1, std::memory_order_acq_rel);
        }
    }

    void help() {
        uint64_t seen = 0;
        for (;;) {
            Job job;
            {
                std::unique_lock<std::mutex> lk(mu_);
                wake_.wait(lk, [&] { return id_ != seen; });
                seen = id_;
                job = job_;
            }
            work(job);
        }
    }

    // Whether there are helpers; starts them on first use. Called in turn.
    bool start() {
        if (started_) return helpers_ > 0;
        started_ = true;
        owner_ = getpid();
        cpu_set_t cpus;
        CPU_ZERO(&cpus);
        if (sched_getaffinity(0, sizeof cpus, &cpus) != 0 || CPU_COUNT(&cpus) <= kHelpers)
            return false;
        try {
            for (; helpers_ < kHelpers; helpers_++) std::thread([this] { help(); }).detach();
        } catch (...) {
            // As many as the system gave.
        }
        return helpers_ > 0;
    }

    std::mutex turn_, mu_;
    std::condition_variable wake_;
    Job job_{};
    uint64_t id_ = 0;
    std::atomic<uint64_t> next_{0};
    std::atomic<size_t> done_{0};
    bool started_ = false;
    pid_t owner_ = 0;  // the process that has the helper threads
    int helpers_ = 0;
};

CopyPool& pool() {
    static CopyPool* p = new CopyPool;
    return *p;
}

}  // namespace

namespace gr_internal {

void host_copy(void* dst, const void* src, size_t n) {
    if (n < kShared)
        std::memcpy(dst, src, n);
    else
        pool().copy((char*)dst, (const char*)src, n);
}

void host_touch(void* p, size_t n) {
    if (n) pool().touch((char*)p, n);
}

}  // namespace gr_internal

extern "C" gr_status gr_host_copy(void* dst, const void* src, size_t bytes) {
    try {
        if (bytes && (!dst || !src))
            return gr_internal::fail(GR_ERR_INVALID_ARGUMENT, "null argument");
        if (bytes) gr_internal::host_copy(dst, src, bytes);
        return GR_OK;
    } catch (...) {
        return gr_internal::fail(GR_ERR_OUT_OF_MEMORY, "host allocation failed");
    }
}
