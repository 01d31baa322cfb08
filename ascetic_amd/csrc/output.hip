// Sending results to the caller's pageable array (output.hpp).
#include <algorithm>
#include <memory>

#include "output.hpp"
#include "traverse.hpp"

namespace asc {

namespace {

OutHelpers& out_helpers() {
    static OutHelpers h(std::min(kOutHelpers, hardware_threads() - 1));
    return h;
}

}  // namespace

OutStage::~OutStage() {
    if (arrived) (void)hipFree(arrived);
}

int OutStage::ensure(uint64_t result_words, hipStream_t s) {
    const uint64_t want = std::min<uint64_t>(result_words, (uint64_t)kOutPiece * kOutRing);
    if (!arrived) {
        ASC_TRY(pub.alloc(kOutRing, true));
        for (int i = 0; i < kOutRing; i++) pub[i].seq = 0;
        ASC_HIP(hipHostGetDevicePointer((void**)&d_pub, pub.p, 0));
        // cleared on the stream of the kernels that count in it: it does not
        // wait for the null stream, and hipMemset need not wait for the device
        DevTmp<uint32_t> count;
        ASC_HIP(hipMalloc(&count.p, 4 * kOutRing * 32));
        ASC_HIP(hipMemsetAsync(count.p, 0, 4 * kOutRing * 32, s));
        std::swap(arrived, count.p);
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
    ASC_TRY(o.ensure(job->pieces == 1 ? words : job->pieces * kOutPiece, s));
    job->pub = o.pub.p;
    job->buf = o.buf.p;
    job->dst = dst;
    job->words = words;
    job->seq0 = o.seq;
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
        o.seq = og.seq + job->group_size(g) - 1;
        return launch(og, (int)(og.blocks * job->group_size(g)));
    };
    auto settle = [&]() -> int {
        ASC_HIP(hipStreamSynchronize(s));
        return ASC_OK;
    };
    const bool helped = job->pieces > kOutAlone;
    if (helped) out_helpers().post(job);   // they wake while the first group is on its way
    const int r = out_collect(*job, queue, settle);
    if (job->lost) set_last_error("the device did not deliver its results");
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
