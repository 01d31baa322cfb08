// Results on their way to the caller's pageable array: the device writes them
// in pieces to mapped page-locked memory and the host copies each piece out as
// it arrives.
//
// hipMemcpy into pageable memory moved 16 MB in ~1.2 ms (one thread, staging
// inside the runtime), and a pass of the host over the values for the reached
// count and the value convention took about as long again; the link carries
// them in 0.28 ms.  The kernels that write a piece apply the convention and
// count on the way, and a few host threads copy, which also take the page
// faults of a fresh array in parallel.
#pragma once

#include "device_common.hpp"
#include "internal.hpp"
#include "out_ring.hpp"

namespace asc {

constexpr int kOutBlocks = 4;              // workgroups per piece, at most (kOutGroup)

struct OutStage {
    HostBuf<uint32_t> buf;          // kOutRing pieces (fewer for a small result)
    uint32_t* d_buf = nullptr;      // the same, as the device sees it
    HostBuf<OutPub> pub;            // one per ring slot
    OutPub* d_pub = nullptr;
    uint32_t* arrived = nullptr;    // device: workgroups done with a slot's piece (kept at zero between pieces)
    uint64_t words = 0;             // capacity
    unsigned long long seq = 0;     // pieces sent so far
    ~OutStage();
    int ensure(uint64_t result_words, hipStream_t s);   // s: the stream of every send
};

// A group of consecutive pieces, for the kernel that writes them: `blocks`
// workgroups a piece.  The result is `parts` arrays of `words` words each, cut
// into `per_part` pieces each.
struct OutGroup {
    uint32_t* buf;                  // mapped ring
    OutPub* pub;
    uint32_t* arrived;
    unsigned long long seq;         // of the group's first piece
    uint64_t words;
    uint32_t piece, ring, per_part, blocks;
};

// A workgroup's piece: words [first, first + n) of part `part`, to dst[0..n);
// it is workgroup `block` of the piece's `blocks`.
struct OutSlot {
    uint32_t* dst;
    OutPub* pub;
    uint32_t* arrived;
    unsigned long long seq;
    uint64_t first;
    uint32_t n, part, block, blocks;
};

__device__ __forceinline__ OutSlot out_slot(const OutGroup& g) {
    const uint32_t k = blockIdx.x / g.blocks, p = g.piece + k, r = (g.ring + k) % kOutRing;
    OutSlot s;
    s.dst = g.buf + (size_t)r * kOutPiece;
    s.pub = g.pub + r;
    s.arrived = g.arrived + 32 * r;
    s.seq = g.seq + k;
    s.part = p / g.per_part;
    s.first = (uint64_t)(p % g.per_part) * kOutPiece;
    const uint64_t left = g.words - s.first;
    s.n = (uint32_t)(left < kOutPiece ? left : kOutPiece);
    s.block = blockIdx.x % g.blocks;
    s.blocks = g.blocks;
    return s;
}

// Ends a piece: once every workgroup of it has called this (all lanes, after
// their stores to s.dst), the piece is published.  The stores are plain ones
// (storing every word through to the host carries 0.1 GB/s); what orders them
// is the chain lane -> its workgroup's lane 0 by the barrier -> the lane 0 that
// counts last by the acquiring and releasing count -> the host by that lane's
// releasing store of the sequence number and the host's acquiring load.  Each
// lane's fence sends its stores on their way to the host before the count, from
// whichever XCD's L2 they are in (1.1 M pieces of 128 and 512 KiB checked: none
// seen early).
__device__ __forceinline__ void out_done(const OutSlot& s) {
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x != 0) return;
    if (__hip_atomic_fetch_add(s.arrived, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) != s.blocks - 1) return;
    *s.arrived = 0;
    host_publish(&s.pub->seq, s.seq);
}

// Sends `parts` results of `words` words, part p to dst[p]: launch(group, grid)
// queues, on stream s, a kernel of `grid` workgroups of kBlock lanes that
// writes the group's pieces (out_slot, out_done).  Returns once all have been
// copied out.
int out_send(OutStage& o, uint32_t* const* dst, uint32_t parts, uint64_t words, hipStream_t s,
             const std::function<int(const OutGroup&, int)>& launch);

// The words of a device array as they are.
int out_copy(OutStage& o, const uint32_t* src, uint64_t words, uint32_t* dst, hipStream_t s);

}  // namespace asc
