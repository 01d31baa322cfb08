// Sending results to the caller's pageable array (output.hpp).
#include <algorithm>
#include <memory>

#include "output.hpp"
#include "traverse.hpp"

namespace asc {

namespace {

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

    // Copies one arrived piece; false when none is waiting.
    bool copy_one() {
        uint64_t i = next.load(std::memory_order_relaxed);
        do {
            if (i >= ready.load(std::memory_order_acquire)) return false;
        } while (!next.compare_exchange_weak(i, i + 1, std::memory_order_acq_rel));
        const uint64_t first = (i % per_part) * kOutPiece, n = std::min<uint64_t>(kOutPiece, words - first);
        std::memcpy(dst[i / per_part] + first, buf + (i % kOutRing) * kOutPiece, 4 * n);
        copied[(i / kOutGroup) & 1].fetch_add(1, std::memory_order_acq_rel);
        done.fetch_add(1, std::memory_order_acq_rel);
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
    OutHelpers() {
        const int n = std::min(kOutHelpers, hardware_threads() - 1);
        for (int i = 0; i < n; i++) threads_.emplace_back([this] { loop(); });
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

OutHelpers& out_helpers() {
    static OutHelpers h;
    return h;
}

}  // namespace

OutStage::~OutStage() {
    if (arrived) (void)hipFree(arrived);
}

int OutStage::ensure(uint64_t result_words) {
    const uint64_t want = std::min<uint64_t>(result_words, (uint64_t)kOutPiece * kOutRing);
    if (!arrived) {
        ASC_TRY(pub.alloc(kOutRing, true));
        for (int i = 0; i < kOutRing; i++) pub[i].seq = 0;
        ASC_HIP(hipHostGetDevicePointer((void**)&d_pub, pub.p, 0));
        ASC_HIP(hipMalloc(&arrived, 4 * kOutRing * 32));
        ASC_HIP(hipMemset(arrived, 0, 4 * kOutRing * 32));
    }
    if (words < want) {
        words = 0;
        ASC_TRY(buf.alloc(want, true));
        ASC_HIP(hipHostGetDevicePointer((void**)&d_buf, buf.p, 0));
        words = want;
    }
    return ASC_OK;
}

int out_send(OutStage& o, uint32_t* const* dst, uint32_t parts, uint64_t words, hipStream_t s,
             const std::function<int(const OutGroup&, int)>& launch) {
    if (parts == 0 || words == 0) return ASC_OK;
    // a helper may still look at the job after this returns, so it is shared
    auto job = std::make_shared<OutJob>();
    job->per_part = (words + kOutPiece - 1) / kOutPiece;
    job->pieces = job->per_part * parts;
    if (job->pieces >= 0xFFFFFFFFull) return ASC_ERR_RANGE;
    ASC_TRY(o.ensure(job->pieces == 1 ? words : job->pieces * kOutPiece));
    job->pub = o.pub.p;
    job->buf = o.buf.p;
    job->dst = dst;
    job->words = words;
    job->seq0 = o.seq;
    const uint64_t np = job->pieces, groups = (np + kOutGroup - 1) / kOutGroup;
    auto group_size = [&](uint64_t g) { return std::min<uint64_t>(kOutGroup, np - g * kOutGroup); };
    auto queue = [&](uint64_t g) -> int {
        OutGroup og;
        og.buf = o.d_buf;
        og.pub = o.d_pub;
        og.arrived = o.arrived;
        og.seq = job->seq0 + g * kOutGroup + 1;
        og.words = words;
        og.piece = (uint32_t)(g * kOutGroup);
        og.ring = (uint32_t)(g * kOutGroup % kOutRing);
        og.per_part = (uint32_t)job->per_part;
        og.blocks = (uint32_t)std::max<uint64_t>(
            1, std::min<uint64_t>(kOutBlocks, (std::min<uint64_t>(words, kOutPiece) + 4 * kBlock - 1) / (4 * kBlock)));
        o.seq = og.seq + group_size(g) - 1;
        return launch(og, (int)(og.blocks * group_size(g)));
    };
    const bool helped = np > kOutAlone;
    if (helped) out_helpers().post(job);   // they wake while the first group is on its way
    uint64_t queued = 0, ready = 0;
    int r = ASC_OK;
    while (r == ASC_OK && queued < std::min<uint64_t>(2, groups)) r = queue(queued++);
    // this thread sees the pieces arrive, sends the next group once its half
    // of the ring has been copied, and copies too while it waits
    double t_wait = now_ms();
    uint32_t spins = 0;
    while (r == ASC_OK && job->done.load(std::memory_order_acquire) < np) {
        bool moved = false;
        while (ready < np && ready < queued * kOutGroup &&
               ((const volatile OutPub*)o.pub.p)[ready % kOutRing].seq == job->seq0 + ready + 1) {
            std::atomic_thread_fence(std::memory_order_acquire);
            ready++;
            moved = true;
        }
        if (moved) job->ready.store(ready, std::memory_order_release);
        if (queued < groups) {
            const uint64_t g = queued - 2;   // the group whose half of the ring comes next
            if (job->copied[g & 1].load(std::memory_order_acquire) == group_size(g)) {
                job->copied[g & 1].store(0, std::memory_order_relaxed);
                r = queue(queued++);
                moved = true;
            }
        }
        if (job->copy_one()) moved = true;
        if (moved) {
            t_wait = now_ms();
            spins = 0;
        } else if ((++spins & 1023) == 0 && now_ms() - t_wait > 50.0 && ready < np) {
            // nothing for long: let the runtime report a failed launch
            if (hipStreamSynchronize(s) != hipSuccess ||
                ((const volatile OutPub*)o.pub.p)[ready % kOutRing].seq != job->seq0 + ready + 1) {
                set_last_error("the device did not deliver its results");
                r = ASC_ERR_DEVICE;
            }
            t_wait = now_ms();
        }
    }
    if (r != ASC_OK) {
        // helpers may be inside a copy: let those end before dst and the ring go away
        job->stop = true;
        job->ready.store(0, std::memory_order_release);
        const uint64_t taken = std::min(job->next.exchange(np), np);
        while (job->done.load(std::memory_order_acquire) < taken) {
        }
    }
    if (helped) out_helpers().drop(job);
    return r;
}

__global__ __launch_bounds__(kBlock) void k_out_copy(const uint32_t* src, OutGroup g) {
    const OutSlot s = out_slot(g);
    const uint32_t n4 = s.n / 4, i0 = s.block * kBlock + threadIdx.x, step = s.blocks * kBlock;
    const uint4* in = (const uint4*)(src + s.first);   // pieces start at multiples of 128 KiB
    for (uint32_t i = i0; i < n4; i += step) ((uint4*)s.dst)[i] = in[i];
    for (uint32_t i = 4 * n4 + i0; i < s.n; i += step) s.dst[i] = src[s.first + i];
    out_done(s);
}

int out_copy(OutStage& o, const uint32_t* src, uint64_t words, uint32_t* dst, hipStream_t s) {
    return out_send(o, &dst, 1, words, s, [&](const OutGroup& g, int grid) -> int {
        hipLaunchKernelGGL(k_out_copy, dim3(grid), dim3(kBlock), 0, s, src, g);
        ASC_HIP(hipGetLastError());
        return ASC_OK;
    });
}

}  // namespace asc
