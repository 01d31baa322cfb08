// Plays the device to the ring loop (out_ring.hpp) on the CPU.
#include <sys/resource.h>

#include <cstdio>
#include <cstring>

#include "out_ring.hpp"

using namespace asc;

namespace {

struct Ring {
    std::vector<uint32_t> buf = std::vector<uint32_t>((size_t)kOutRing * kOutPiece);
    std::vector<OutPub> pub = std::vector<OutPub>(kOutRing);
    std::vector<uint32_t> out;
    uint32_t* parts[1];
    std::shared_ptr<OutJob> job = std::make_shared<OutJob>();
    int settled = 0;

    explicit Ring(uint64_t words) : out(words) {
        parts[0] = out.data();
        job->pub = pub.data();
        job->buf = buf.data();
        job->dst = parts;
        job->words = words;
        job->per_part = job->pieces = (words + kOutPiece - 1) / kOutPiece;
    }
    // word w of the result is 3 w + 1
    void deliver(uint64_t piece) {
        uint32_t* p = buf.data() + (piece % kOutRing) * kOutPiece;
        for (uint64_t i = 0; i < kOutPiece; i++) p[i] = (uint32_t)(3 * (piece * kOutPiece + i) + 1);
        __atomic_store_n(&pub[piece % kOutRing].seq, job->seq0 + piece + 1, __ATOMIC_RELEASE);
    }
    int deliver_group(uint64_t g) {
        for (uint64_t k = 0; k < job->group_size(g); k++) deliver(g * kOutGroup + k);
        return ASC_OK;
    }
    bool right() const {
        for (uint64_t i = 0; i < out.size(); i++)
            if (out[i] != (uint32_t)(3 * i + 1)) return false;
        return true;
    }
};

void nap(int ms) { std::this_thread::sleep_for(std::chrono::milliseconds(ms)); }

#define CHECK(x)                                                \
    do {                                                        \
        if (!(x)) {                                             \
            printf("line %d: %s does not hold\n", __LINE__, #x); \
            return 1;                                           \
        }                                                       \
    } while (0)

// A helper stops inside a copy while every queued piece is in: the send waits.
int slow_helper() {
    bool stopped = false;
    for (int tries = 0; tries < 50 && !stopped; tries++) {
        Ring r((uint64_t)(kOutRing + kOutGroup + 2) * kOutPiece + 77);
        std::thread helper([&] {
            uint64_t i;
            while (!r.job->take(i))
                if (r.job->next >= r.job->pieces) return;
            // a piece of the first two groups: the third is not queued before it is copied
            stopped = i < (uint64_t)kOutRing;
            nap(stopped ? 200 : 0);
            r.job->copy(i);
        });
        const int rc = out_collect(*r.job, [&](uint64_t g) { return r.deliver_group(g); },
                                   [&] { r.settled++; return (int)ASC_OK; });
        helper.join();
        CHECK(rc == ASC_OK && !r.job->lost && r.settled == 0 && r.right());
    }
    CHECK(stopped);
    return 0;
}

// A late device is waited for; one that ends without a piece is an error.
int late_device() {
    Ring r(3 * kOutPiece);
    std::thread device([&] {
        nap(150);
        r.deliver_group(0);
    });
    int rc = out_collect(*r.job, [](uint64_t) { return (int)ASC_OK; }, [&] {
        device.join();
        r.settled++;
        return (int)ASC_OK;
    });
    CHECK(rc == ASC_OK && r.settled == 1 && r.right());
    Ring l(3 * kOutPiece);
    l.deliver(0);
    l.deliver(1);
    rc = out_collect(*l.job, [](uint64_t) { return (int)ASC_OK; }, [] { return (int)ASC_OK; });
    CHECK(rc == ASC_ERR_DEVICE && l.job->lost);
    return 0;
}

// A launch that fails between two groups ends the send with its error.
int failed_launch(OutHelpers& helpers) {
    Ring r((uint64_t)5 * kOutGroup * kOutPiece);
    helpers.post(r.job);
    const int rc = out_collect(*r.job, [&](uint64_t g) { return g == 3 ? (int)ASC_ERR_NOMEM : r.deliver_group(g); },
                               [] { return (int)ASC_OK; });
    helpers.drop(r.job);
    CHECK(rc == ASC_ERR_NOMEM && !r.job->lost);
    return 0;
}

int with_helpers(OutHelpers& helpers) {
    for (uint64_t pieces : {1, 2, 3, kOutGroup, kOutRing, kOutRing + 1, 5 * kOutGroup + 3}) {
        Ring r((pieces - 1) * kOutPiece + 5);
        helpers.post(r.job);
        const int rc = out_collect(*r.job, [&](uint64_t g) { return r.deliver_group(g); }, [] { return (int)ASC_OK; });
        helpers.drop(r.job);
        CHECK(rc == ASC_OK && r.right());
    }
    return 0;
}

// No room for another thread's stack (8 MiB by default).
int no_threads() {
    Ring r(3 * kOutPiece);
    std::thread([] {}).join();   // the runtime's own first allocations
    unsigned long pages = 0;
    FILE* f = fopen("/proc/self/statm", "r");
    CHECK(f && fscanf(f, "%lu", &pages) == 1);
    fclose(f);
    // glibc keeps the stack of a thread that ended, so one more may start
    const rlimit lim{pages * 4096 + (2u << 20), RLIM_INFINITY};
    CHECK(setrlimit(RLIMIT_AS, &lim) == 0);
    OutHelpers helpers(4);
    helpers.post(r.job);
    const int rc = out_collect(*r.job, [&](uint64_t g) { return r.deliver_group(g); }, [] { return (int)ASC_OK; });
    helpers.drop(r.job);
    CHECK(rc == ASC_OK && r.right());
    return 0;
}

}  // namespace

int main(int argc, char** argv) {
    if (argc > 1 && !strcmp(argv[1], "no-threads")) {
        const int bad = no_threads();
        if (!bad) printf("ok\n");
        return bad;
    }
    OutHelpers helpers(3);
    const int bad = slow_helper() + late_device() + with_helpers(helpers) + failed_launch(helpers);
    if (!bad) printf("ok\n");
    return bad;
}
