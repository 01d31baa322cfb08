// Host side of sending results (output.hpp): the ring the device writes its
// pieces to, the helper threads that copy them out, and the loop that runs a
// send.  No HIP in here, so the loop is tested on its own with a device that
// the test plays.
#pragma once

#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstdint>
#include <cstring>
#include <exception>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>

#include "../../include/ascetic.h"

namespace asc {

constexpr uint32_t kOutPiece = 1u << 15;   // 32-bit words per piece (128 KiB: 2.3 us of the link, ~16 us of a thread)
// Pieces per launch and workgroups per piece: a launch takes ~10 us beside its
// bytes' time on the link, and more workgroups only add system fences (16 MB
// result: 8 pieces of 16 workgroups 520 us, of 4 450; 16 of 16 480, of 8 430,
// of 4 400, of 2 410; 32 of 4 400).
constexpr int kOutGroup = 16;
// pieces in flight: two groups, one on the link while the other is copied
// (page-locking its 4 MiB takes ~290 us once, where 2 MiB take ~35)
constexpr int kOutRing = 2 * kOutGroup;
constexpr uint64_t kOutAlone = 2;          // up to this many pieces the calling thread copies alone
constexpr int kOutHelpers = 7;             // threads that help it with more
constexpr double kOutLateMs = 50.0;        // without a piece for so long the device is asked

// Written by the device, a cache line each.
struct OutPub {
    unsigned long long seq;
    unsigned long long pad[15];
};

// One result being copied out.  Pieces are taken in order by whoever is free;
// a helper that wakes late finds none left and drops its reference.
struct OutJob {
    const OutPub* pub = nullptr;
    const uint32_t* buf = nullptr;
    uint32_t* const* dst = nullptr;
    uint64_t words = 0, pieces = 0, per_part = 0;
    unsigned long long seq0 = 0;
    std::atomic<uint64_t> ready{0};      // pieces that have arrived (all before it too)
    std::atomic<uint64_t> next{0};       // pieces taken
    std::atomic<uint64_t> copied[2] = {};   // pieces copied of the group in either half of the ring
    std::atomic<uint64_t> done{0};
    std::atomic<bool> stop{false};
    bool lost = false;                   // a queued piece never came

    uint64_t groups() const { return (pieces + kOutGroup - 1) / kOutGroup; }
    uint64_t group_size(uint64_t g) const { return std::min<uint64_t>(kOutGroup, pieces - g * kOutGroup); }
    bool arrived(uint64_t i) const {
        return __atomic_load_n(&pub[i % kOutRing].seq, __ATOMIC_ACQUIRE) == seq0 + i + 1;
    }
    // Takes an arrived piece; false when none is waiting.
    bool take(uint64_t& i) {
        i = next.load(std::memory_order_relaxed);
        do {
            if (i >= ready.load(std::memory_order_acquire)) return false;
        } while (!next.compare_exchange_weak(i, i + 1, std::memory_order_acq_rel));
        return true;
    }
    void copy(uint64_t i) {
        const uint64_t first = (i % per_part) * kOutPiece, n = std::min<uint64_t>(kOutPiece, words - first);
        std::memcpy(dst[i / per_part] + first, buf + (i % kOutRing) * kOutPiece, 4 * n);
        copied[(i / kOutGroup) & 1].fetch_add(1, std::memory_order_acq_rel);
        done.fetch_add(1, std::memory_order_acq_rel);
    }
    bool copy_one() {
        uint64_t i;
        if (!take(i)) return false;
        copy(i);
        return true;
    }
    // A helper: until every piece is taken.
    void help() {
        while (!stop.load(std::memory_order_acquire) && next.load(std::memory_order_relaxed) < pieces)
            if (!copy_one()) __builtin_ia32_pause();
    }
};

class OutHelpers {
public:
    // As many as the system grants, up to n: a thread that cannot be had must
    // not end a query (or the process), the calling thread copies alone.
    explicit OutHelpers(int n) {
        try {
            for (int i = 0; i < n; i++) threads_.emplace_back([this] { loop(); });
        } catch (const std::exception&) {
        }
    }
    ~OutHelpers() {
        {
            std::lock_guard<std::mutex> lk(mu_);
            quit_ = true;
        }
        cv_.notify_all();
        for (auto& t : threads_) t.join();
    }
    void post(const std::shared_ptr<OutJob>& j) {
        {
            std::lock_guard<std::mutex> lk(mu_);
            job_ = j;
            gen_++;
        }
        cv_.notify_all();
    }
    void drop(const std::shared_ptr<OutJob>& j) {
        std::lock_guard<std::mutex> lk(mu_);
        if (job_ == j) job_.reset();
    }

private:
    void loop() {
        uint64_t seen = 0;
        for (;;) {
            std::shared_ptr<OutJob> j;
            {
                std::unique_lock<std::mutex> lk(mu_);
                cv_.wait(lk, [&] { return quit_ || gen_ != seen; });
                if (quit_) return;
                seen = gen_;
                j = job_;
            }
            if (j) j->help();
        }
    }
    std::vector<std::thread> threads_;
    std::mutex mu_;
    std::condition_variable cv_;
    std::shared_ptr<OutJob> job_;
    uint64_t gen_ = 0;
    bool quit_ = false;
};

// Runs a send to its end on the calling thread, which sees the pieces arrive,
// sends the next group once its half of the ring has been copied, and copies
// too while it waits.  queue(g) queues the kernel of group g; settle() waits
// for what was queued and reports a launch that failed.  The device is held to
// be late only while a queued piece is outstanding: with all of them here the
// wait is for a helper, which may be descheduled or take page faults for as
// long as the system likes (every piece of a full ring in, one helper stopped
// for 50 ms: the run was refused for a device that had delivered).
template <class Queue, class Settle>
int out_collect(OutJob& job, Queue&& queue, Settle&& settle) {
    auto now = [] {
        return std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now().time_since_epoch()).count();
    };
    const uint64_t np = job.pieces, groups = job.groups();
    uint64_t queued = 0, ready = 0;
    int r = ASC_OK;
    while (r == ASC_OK && queued < std::min<uint64_t>(2, groups)) r = queue(queued++);
    double t_wait = now();
    uint32_t spins = 0;
    while (r == ASC_OK && job.done.load(std::memory_order_acquire) < np) {
        bool moved = false;
        const uint64_t sent = std::min(np, queued * kOutGroup);
        while (ready < sent && job.arrived(ready)) {
            ready++;
            moved = true;
        }
        if (moved) job.ready.store(ready, std::memory_order_release);
        if (queued < groups) {
            const uint64_t g = queued - 2;   // the group whose half of the ring comes next
            if (job.copied[g & 1].load(std::memory_order_acquire) == job.group_size(g)) {
                job.copied[g & 1].store(0, std::memory_order_relaxed);
                r = queue(queued++);
                moved = true;
            }
        }
        if (job.copy_one()) moved = true;
        if (moved) {
            t_wait = now();
            spins = 0;
        } else if ((++spins & 1023) == 0) {
            if (ready < sent && now() - t_wait > kOutLateMs) {
                r = settle();
                if (r == ASC_OK && !job.arrived(ready)) {
                    job.lost = true;
                    r = ASC_ERR_DEVICE;
                }
                t_wait = now();
            } else if (ready == sent) {
                std::this_thread::yield();   // to the helper waited for
            }
        }
    }
    if (r != ASC_OK) {
        // helpers may be inside a copy: let those end before dst and the ring go away
        job.stop = true;
        job.ready.store(0, std::memory_order_release);
        const uint64_t taken = std::min(job.next.exchange(np), np);
        while (job.done.load(std::memory_order_acquire) < taken) std::this_thread::yield();
    }
    return r;
}

}  // namespace asc
