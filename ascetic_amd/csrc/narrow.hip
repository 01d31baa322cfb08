// Runs of narrow steps in one launch.
//
// A step of the host-stepped loops costs a launch or two, a publish and a
// host round trip (~40 us) whatever its size, and graphs with long paths
// (meshes, road networks, the first and last levels of any traversal) take
// thousands of steps of a few hundred edges.  k_narrow runs such steps back to
// back in a single workgroup, where a step costs its dependent memory round
// trips: the edges of the frontier, the probes of their ends, then the value
// atomics and, beside them, the offsets of the vertices they lower.  The
// frontier (vertex, value, first edge and the running edge count, so edges are
// dealt to lanes evenly) sits in LDS; what outgrows it goes to the engine's
// global queue, and the wide kernels take the frontier from there.  SSSP's far
// pile stays in global memory and is split in the same launch.
// SSSP over a 1201 x 1033 mesh (1.24 M vertices, 4.5 M edges): 283 ms in 8369
// wide steps, 31 ms in ~3000 narrow ones.  What bounds it now is one CU's rate
// of scattered accesses (~4 ns an edge); loading the offsets and trying the
// atomics of every edge beside the probes, a round trip less, took 40 ms.
#include <algorithm>
#include <type_traits>

#include "device_common.hpp"
#include "internal.hpp"
#include "frontier.hpp"
#include "traverse.hpp"

namespace asc {

constexpr int kNwBlock = 1024;
constexpr int kNwUnroll = 4;                   // edges per lane and pass
constexpr uint32_t kNwMaxSteps = 16384;        // steps and splits per launch (~30 ms)
constexpr uint32_t kNwLdsBits = 1u << 18;      // BFS: visited bitmap in LDS up to this V
constexpr int kNwFarPer = kNarrowFar / kNwBlock;
constexpr int kNwCntShift = 40;                // frontier counter: (vertices << 40) | edges
constexpr unsigned long long kNwCntMask = (1ull << kNwCntShift) - 1;

struct NarrowArgs {
    uint32_t* q[2];               // q[level & 1]: the frontier of `level`
    uint32_t* far[2];
    Piles* piles;
    NarrowPub* pub;
    unsigned long long seq;
    uint32_t level, n_in;
    uint32_t n_far, fcur;
    uint32_t theta, delta, most;    // band; the next band's width, doubled at every split up to `most`
    uint32_t edge_limit, V;
};

__device__ __forceinline__ uint32_t nw_load(const uint32_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // past the CU's L1
}
__device__ __forceinline__ void nw_store(uint32_t* p, uint32_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <int ALGO, class OffT, class EdgeT, bool LDSBITS>
__global__ __launch_bounds__(kNwBlock) void k_narrow(TravArgs<OffT, EdgeT> a, NarrowArgs na) {
    constexpr bool BFS = ALGO == ALG_BFS;
    __shared__ unsigned long long s_beg[2][kNarrowCap];
    __shared__ uint32_t s_v[2][kNarrowCap];
    __shared__ uint32_t s_sv[BFS ? 1 : 2][BFS ? 1 : kNarrowCap];
    __shared__ uint32_t s_base[2][kNarrowCap];
    __shared__ uint32_t s_bits[LDSBITS ? kNwLdsBits / 32 : 1];
    // counters of levels L, L + 1 (being filled) and L + 2 (cleared during L)
    __shared__ unsigned long long s_cnt[3];
    __shared__ uint32_t s_nfar[2], s_min;
    const uint32_t tid = threadIdx.x;
    const unsigned long long t_begin = wall_clock64();
    uint32_t level = na.level, fcur = na.fcur, theta = na.theta, width = na.delta;
    unsigned long long nodes = 0, edges = 0;
    uint32_t steps = 0, splits = 0;

    // Appends v (value sv, edges [beg, beg + deg)) to the frontier of `lv`.
    auto push = [&](uint32_t lv, uint32_t v, uint32_t sv, OffT beg, uint64_t deg) {
        const unsigned long long old = atomicAdd(&s_cnt[lv % 3], (1ull << kNwCntShift) | deg);
        const uint32_t i = (uint32_t)(old >> kNwCntShift);
        if (i < kNarrowCap) {
            s_v[lv & 1][i] = v;
            if (!BFS) s_sv[BFS ? 0 : lv & 1][BFS ? 0 : i] = sv;
            s_beg[lv & 1][i] = (unsigned long long)beg;
            s_base[lv & 1][i] = (uint32_t)old;
        } else {
            na.q[lv & 1][i] = v;   // the step ends the run, and the wide kernels go on
        }
    };

    if (tid < 3) s_cnt[tid] = 0;
    if (tid < 2) s_nfar[tid] = tid == fcur ? na.n_far : 0;
    if (tid == 0) s_min = 0xFFFFFFFFu;
    if (LDSBITS)
        for (uint32_t i = tid; i < (na.V + 31) / 32; i += kNwBlock) s_bits[i] = a.visited[i];
    // the whole input frontier is read before any of it is written back
    uint32_t u_in[kNarrowCap / kNwBlock];
#pragma unroll
    for (int j = 0; j < kNarrowCap / kNwBlock; j++) {
        const uint32_t i = j * kNwBlock + tid;
        u_in[j] = i < na.n_in ? na.q[level & 1][i] : 0xFFFFFFFFu;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kNarrowCap / kNwBlock; j++) {
        const uint32_t u = u_in[j];
        if ((uint32_t)(j * kNwBlock) + tid >= na.n_in) continue;
        const OffT b = a.off[u], e = a.off[u + 1];
        uint32_t sv = 0;
        bool pend = true;
        if (!BFS) {
            sv = nw_load(a.val + u);
            pend = a.done[u] != sv;
        }
        if (BFS || (pend && e > b)) push(level, u, sv, b, (uint64_t)(e - b));
    }

    for (;;) {
        __syncthreads();
        const unsigned long long c = s_cnt[level % 3];
        const uint32_t n = (uint32_t)(c >> kNwCntShift);
        const unsigned long long total = c & kNwCntMask;
        if (n > kNarrowCap || total > na.edge_limit || steps == kNwMaxSteps) break;
        if (n == 0) {
            if (ALGO != ALG_SSSP) break;
            // advance the band past the smallest pending far value and split
            // the far pile: entries below the band to the frontier, the rest
            // to the other far array
            const uint32_t nfar = s_nfar[fcur];
            if (nfar == 0 || nfar > kNarrowFar) break;
            __builtin_amdgcn_s_waitcnt(0);   // this wave's far entries have reached the L2
            __syncthreads();
            uint32_t fv[kNwFarPer], fd[kNwFarPer];
            uint32_t lmin = 0xFFFFFFFFu;
#pragma unroll
            for (int j = 0; j < kNwFarPer; j++) {
                const uint32_t i = j * kNwBlock + tid;
                fv[j] = i < nfar ? nw_load(na.far[fcur] + i) : 0xFFFFFFFFu;
            }
#pragma unroll
            for (int j = 0; j < kNwFarPer; j++) {
                const uint32_t i = j * kNwBlock + tid;
                fd[j] = 0;
                if (i >= nfar) continue;
                fd[j] = nw_load(a.val + fv[j]);
                if (fd[j] < theta && nw_load(a.done + fv[j]) == fd[j]) fv[j] = 0xFFFFFFFFu;   // expanded already
                else lmin = min(lmin, fd[j]);
            }
#pragma unroll
            for (int d = kWave / 2; d > 0; d >>= 1) lmin = min(lmin, (uint32_t)__shfl_xor(lmin, d, kWave));
            if (lane_id() == 0 && lmin != 0xFFFFFFFFu) atomicMin(&s_min, lmin);
            __syncthreads();
            const uint32_t m = s_min;
            theta = (uint32_t)min((unsigned long long)max(theta, m == 0xFFFFFFFFu ? 0u : m) + width, 0xFFFFFFFFull);
            width = (uint32_t)min(2ull * width, (unsigned long long)na.most);
#pragma unroll
            for (int j = 0; j < kNwFarPer; j++) {
                const uint32_t i = j * kNwBlock + tid;
                if (i >= nfar || fv[j] == 0xFFFFFFFFu) continue;
                if (fd[j] >= theta) {
                    nw_store(na.far[fcur ^ 1] + atomicAdd(&s_nfar[fcur ^ 1], 1u), fv[j]);
                } else {
                    const OffT b = a.off[fv[j]], e = a.off[fv[j] + 1];
                    if (e > b) push(level, fv[j], fd[j], b, (uint64_t)(e - b));
                }
            }
            __syncthreads();
            if (tid == 0) {
                s_nfar[fcur] = 0;
                s_min = 0xFFFFFFFFu;
            }
            fcur ^= 1;
            steps++;
            splits++;
            continue;
        }
        if (tid == 0) s_cnt[(level + 2) % 3] = 0;
        const uint32_t p = level & 1, T = (uint32_t)total;
        uint32_t top = 1;   // largest power of two <= n
        while (top * 2 <= n) top *= 2;
        // U edges per lane from e0 on; lanes past the end repeat the last edge
        // (no branch around the loads, so they are in flight together)
        auto expand = [&](auto unroll, uint32_t e0) {
            constexpr int U = decltype(unroll)::value;
            uint32_t kk[U], uu[U], vv[U], cc[U], now[U], pr[U];
            unsigned long long at[U];
            EdgeT ed[U];
            bool ok[U];
#pragma unroll
            for (int j = 0; j < U; j++) kk[j] = 0;
            for (uint32_t step = top; step > 0; step >>= 1)
#pragma unroll
                for (int j = 0; j < U; j++) {
                    const uint32_t e = min(e0 + j * kNwBlock + tid, T - 1), t = min(kk[j] + step, n - 1);
                    if (s_base[p][t] <= e) kk[j] = t;
                }
#pragma unroll
            for (int j = 0; j < U; j++) {
                const uint32_t e = min(e0 + j * kNwBlock + tid, T - 1);
                uu[j] = s_v[p][kk[j]];
                at[j] = s_beg[p][kk[j]] + (e - s_base[p][kk[j]]);
            }
#pragma unroll
            for (int j = 0; j < U; j++) {
                ed[j] = a.edges[at[j]];
                // a frontier vertex lowered again since it was appended is in
                // the frontier with its lower value too
                if (!BFS) now[j] = nw_load(a.val + uu[j]);
            }
#pragma unroll
            for (int j = 0; j < U; j++) {
                vv[j] = edge_dst(ed[j]);
                if (BFS) pr[j] = LDSBITS ? s_bits[vv[j] >> 5] : a.visited[vv[j] >> 5];
                else pr[j] = a.val[vv[j]];
            }
#pragma unroll
            for (int j = 0; j < U; j++) {
                const uint32_t e = e0 + j * kNwBlock + tid;
                ok[j] = e < T;
                if (BFS) {
                    cc[j] = level + 2;
                    ok[j] = ok[j] && !(pr[j] & (1u << (vv[j] & 31)));
                } else {
                    const uint32_t sv = s_sv[BFS ? 0 : p][BFS ? 0 : kk[j]];
                    cc[j] = candidate<ALGO>(sv, edge_w(ed[j]));
                    if (ok[j] && e == s_base[p][kk[j]]) a.done[uu[j]] = sv;
                    ok[j] = ok[j] && now[j] >= sv && cc[j] < pr[j];
                }
            }
            // the atomics of the edges that lower something, and beside them
            // the offsets of the vertices they lower
            OffT b[U], e1[U];
            uint32_t old[U];
#pragma unroll
            for (int j = 0; j < U; j++) {
                const uint32_t v = vv[j];
                old[j] = BFS ? ~0u : 0u;
                b[j] = e1[j] = 0;
                if (!ok[j]) continue;
                if (BFS) {
                    old[j] = LDSBITS ? atomicOr(&s_bits[v >> 5], 1u << (v & 31))
                                     : atomicOr(a.visited + (v >> 5), 1u << (v & 31));
                } else {
                    old[j] = atomicMin(a.val + v, cc[j]);
                }
                b[j] = a.off[v];
                e1[j] = a.off[v + 1];
            }
#pragma unroll
            for (int j = 0; j < U; j++) {
                const uint32_t v = vv[j];
                if (BFS) {
                    if (old[j] & (1u << (v & 31))) continue;
                    a.val[v] = cc[j];
                    push(level + 1, v, 0, b[j], (uint64_t)(e1[j] - b[j]));
                    continue;
                }
                if (old[j] <= cc[j]) continue;
                // (the 16-bit value filter is left as it is: an older entry is larger)
                if (ALGO == ALG_SSSP && cc[j] >= theta) {
                    // a vertex reached before is in the pile
                    if (old[j] == a.unreached) nw_store(na.far[fcur] + atomicAdd(&s_nfar[fcur], 1u), v);
                    continue;
                }
                if (e1[j] > b[j]) push(level + 1, v, cc[j], b[j], (uint64_t)(e1[j] - b[j]));
            }
        };
        uint32_t e0 = 0;
        for (; T - e0 > 2 * kNwBlock; e0 += min(T - e0, (uint32_t)(kNwBlock * kNwUnroll)))
            expand(std::integral_constant<int, kNwUnroll>{}, e0);
        for (; e0 < T; e0 += min(T - e0, (uint32_t)kNwBlock)) expand(std::integral_constant<int, 1>{}, e0);
        nodes += n;
        edges += T;
        steps++;
        level++;
    }
    // every lane has left the loop at the same point; the counters are final
    const unsigned long long c = s_cnt[level % 3];
    for (uint32_t i = tid; i < min((uint32_t)(c >> kNwCntShift), kNarrowCap); i += kNwBlock)
        na.q[level & 1][i] = s_v[level & 1][i];
    if (LDSBITS)
        for (uint32_t i = tid; i < (na.V + 31) / 32; i += kNwBlock) a.visited[i] = s_bits[i];
    if (tid < 4) {
        Slot* z = a.slots + tid;
        z->n_res = tid == (level & 3) ? (uint32_t)(c >> kNwCntShift) : 0;
        z->heavy = 0;
    }
    if (tid == 0) {
        na.piles->n_far[fcur] = s_nfar[fcur];
        na.piles->n_far[fcur ^ 1] = 0;
        a.stats->edges_local += edges;
        a.stats->verts_local += nodes;
        a.stats->ticks += wall_clock64() - t_begin;
        NarrowPub* o = na.pub;
        host_store(&o->level, level);
        host_store(&o->n, (uint32_t)(c >> kNwCntShift));
        host_store(&o->edges, c & kNwCntMask);
        host_store(&o->n_far, s_nfar[fcur]);
        host_store(&o->fcur, fcur);
        host_store(&o->theta, theta);
        host_store(&o->splits, splits);
        host_store(&o->nodes, nodes);
        host_store(&o->expanded, edges);
        host_publish(&o->seq, na.seq);
    }
}

template <int ALGO, class OffT, class EdgeT>
int narrow_run(asc_graph* g, const TravArgs<OffT, EdgeT>& a, uint32_t n_in, uint32_t n_far, uint32_t delta,
               uint32_t most, NarrowState& io) {
    TravState* t = g->trav;
    hipStream_t s = g->ctx->s_main;
    const bool prof = g->ctx->cfg.profile != 0;
    NarrowArgs na{};
    for (int i = 0; i < 2; i++) {
        na.q[i] = t->q[i];
        na.far[i] = t->far[i];
    }
    na.piles = t->piles;
    na.pub = &t->d_h->narrow;
    na.seq = ++t->narrow_seq;
    na.level = io.level;
    na.n_in = n_in;
    na.n_far = n_far;
    na.fcur = io.fcur;
    na.theta = a.theta;
    na.delta = delta;
    na.most = most;
    na.edge_limit = kNarrowEdges;
    na.V = (uint32_t)g->h.V;
    ASC_TRY(timed_launch(t, prof, KERN_LOCAL, s, [&] {
        if (ALGO == ALG_BFS && g->h.V <= kNwLdsBits)
            hipLaunchKernelGGL((k_narrow<ALGO, OffT, EdgeT, ALGO == ALG_BFS>), dim3(1), dim3(kNwBlock), 0, s, a, na);
        else
            hipLaunchKernelGGL((k_narrow<ALGO, OffT, EdgeT, false>), dim3(1), dim3(kNwBlock), 0, s, a, na);
    }));
    ASC_TRY(wait_host_seq(&t->h[0].narrow.seq, na.seq, s));
    const volatile NarrowPub* o = &t->h[0].narrow;
    io.level = o->level;
    io.n = o->n;
    io.edges = o->edges;
    io.n_far = o->n_far;
    io.fcur = o->fcur;
    io.theta = o->theta;
    io.splits = o->splits;
    io.nodes = o->nodes;
    io.expanded = o->expanded;
    return ASC_OK;
}

#define ASC_NARROW(ALGO, OffT, EdgeT)                                                                          \
    template int narrow_run<ALGO, OffT, EdgeT>(asc_graph*, const TravArgs<OffT, EdgeT>&, uint32_t, uint32_t, \
                                               uint32_t, uint32_t, NarrowState&);
#define ASC_NARROW_ALL(ALGO)           \
    ASC_NARROW(ALGO, uint32_t, uint32_t) \
    ASC_NARROW(ALGO, uint64_t, uint32_t) \
    ASC_NARROW(ALGO, uint32_t, WEdge)    \
    ASC_NARROW(ALGO, uint64_t, WEdge)
ASC_NARROW_ALL(ALG_BFS)
ASC_NARROW_ALL(ALG_CC)
ASC_NARROW_ALL(ALG_SSSP)

}  // namespace asc
