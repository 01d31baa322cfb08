// PageRank over the in-CSR (BCSC input, GraphMeta.cuh:159-162).
//
// Normalised mode: r0 = 1/V; r' = (1-d)/V + d*(sum_{u->v} r[u]/outdeg[u] +
// dangling/V) for a fixed number of iterations.  Ranks and the gathered
// contributions c[u] = r[u]/outdeg[u] are FP32 (4 bytes per random gather);
// each vertex's in-edge sum (64-bit fixed point in the blocked schedule, FP32
// in the tiled one), the residual sum |r'-r| and the dangling mass are
// accumulated in FP64.  Large resident graphs take the propagation-blocked
// schedule, smaller ones row blocks, streamed rows the same sums without a
// plan; a set pr_group keeps the pull in which G lanes share a vertex.  The
// residual and dangling sums are produced inside the same kernels, so
// iterations run back-to-back without a host synchronisation.
//
// Reference mode (gpu_kernels.cuh:533-594, CalculateOpt.cu:547-721): FP64,
// 0.15 + 0.85*sum over active vertices, threshold 0.001, loop while any
// vertex is active.  Each active vertex's sum runs sequentially in CSR order
// and no multiply-add is fused, so results equal a sequential FP64
// evaluation of the same formula.
#include <algorithm>

#include "device_common.hpp"
#include "internal.hpp"
#include "traverse.hpp"

namespace asc {

// An iteration's count of vertices that moved, as the device publishes it to
// mapped host memory; seq is written last.
struct PrRefPub {
    unsigned long long moved;
    unsigned long long seq;
};

struct PrState {
    uint64_t V = 0;
    float* rank[2] = {nullptr, nullptr};
    float* contrib[2] = {nullptr, nullptr};
    double* acc = nullptr;        // ring of kAccSlots slots of kAccSlot sums (PrArgs::acc_in / acc_out)
    double* resid = nullptr;      // residual of each iteration
    int resid_iters = 0;
    HostBuf<double> h_resid;      // the same on the host, and a sequence number behind them (mapped)
    double* d_hresid = nullptr;
    unsigned long long resid_seq = 0;
    hipEvent_t ev[2] = {nullptr, nullptr};   // first and last kernel of a run
    OutStage out;
    // reference mode
    double* val64 = nullptr;
    double* contrib64[2] = {nullptr, nullptr};   // read by / written for the next iteration
    uint8_t* active = nullptr;
    uint32_t* count = nullptr;    // kPrLines counters, one per 128-byte line
    HostBuf<PrRefPub> h_refpub;   // ring written by the device through d_refpub (mapped)
    PrRefPub* d_refpub = nullptr;
    unsigned long long ref_seq = 0;
    // row blocks and heavy rows of the resident vertices (RowPlan)
    void* rows_blocks = nullptr;
    uint32_t* rows_heavy = nullptr;
    uint32_t rows_n = 0, rows_cap = 0, rows_front = 0, rows_back = 0;
    bool heavy_built = false, rows_built = false;
    // on-demand in-edges: vertex-range chunks [v0, v1) whose in-edges
    // [off[v0], off[v1]) fit one part buffer, copied from the pinned tail
    struct Chunk {
        uint64_t v0, v1, e0, e1;
    };
    std::vector<Chunk> chunks;
    uint32_t* part[2] = {nullptr, nullptr};
    uint64_t part_edges = 0;
    hipEvent_t ev_copy[2] = {nullptr, nullptr}, ev_kern[2] = {nullptr, nullptr};
    uint64_t streamed_edges = 0;  // per pull sweep
    // propagation-blocked normalised mode (every edge resident): the light
    // in-edges regrouped by (source slice, destination bin) into runs, each
    // padded to whole quads of edges
    int pb_state = 0;             // 0 not built, 1 built, -1 not possible
    bool outdeg_sums = false;     // the out-degrees were found to sum to E
    uint32_t pb_sbits = 0, pb_dbits = 0, pb_nbins = 0, pb_nitems = 0;
    void* pb_src = nullptr;       // u16 slice-local sources, in slice order
    void* pb_dst = nullptr;       // u16 bin-local destinations, in bin order
    uint32_t* pb_pos = nullptr;   // in bin order: an oct's place in slice order
    float* pb_vals = nullptr;     // contributions on their way, in slice order
    void *pb_bins = nullptr, *pb_items = nullptr;
    // source-segmented normalised mode (every edge resident): the light
    // in-edges regrouped into tiles (destination block d, source segment s),
    // tile (d, s) at tl_edges[tl_off[d * tl_ns + s] ...], one u32 word per
    // edge (block-local destination << kTlSrcBits | segment-local source)
    int tl_state = 0;             // 0 not built, 1 built, -1 not possible
    uint32_t tl_sb = 0, tl_db = 0, tl_nd = 0, tl_ns = 0;
    uint64_t tl_edges_n = 0;
    uint32_t* tl_edges = nullptr;
    unsigned long long* tl_off = nullptr;
    uint32_t* tl_heavy = nullptr; // bitmap of destinations left to k_pr_pull_heavy
};

void pr_free(PrState* p) {
    if (!p) return;
    auto f = [](void* x) {
        if (x) (void)hipFree(x);
    };
    f(p->rank[0]); f(p->rank[1]); f(p->contrib[0]); f(p->contrib[1]);
    f(p->acc); f(p->resid); f(p->val64); f(p->contrib64[0]); f(p->contrib64[1]); f(p->active);
    f(p->count); f(p->rows_heavy); f(p->rows_blocks);
    f(p->part[0]); f(p->part[1]);
    f(p->pb_src); f(p->pb_dst); f(p->pb_vals); f(p->pb_pos); f(p->pb_bins); f(p->pb_items);
    f(p->tl_edges); f(p->tl_off); f(p->tl_heavy);
    for (int i = 0; i < 2; i++) {
        if (p->ev[i]) (void)hipEventDestroy(p->ev[i]);
        if (p->ev_copy[i]) (void)hipEventDestroy(p->ev_copy[i]);
        if (p->ev_kern[i]) (void)hipEventDestroy(p->ev_kern[i]);
    }
    delete p;
}

// Plans the on-demand chunks of a partially resident PageRank graph (once).
static int pr_plan_chunks(asc_graph* g, PrState* p) {
    const uint64_t V = g->h.V, vs = g->static_vertices;
    if (vs >= V || !p->chunks.empty()) return ASC_OK;
    const uint64_t* off = g->h.off.p;
    uint64_t maxdeg = 0;
    for (uint64_t v = vs; v < V; v++) maxdeg = std::max<uint64_t>(maxdeg, off[v + 1] - off[v]);
    // a part holds at least the largest on-demand in-list
    p->part_edges = std::max<uint64_t>(g->part_edges, maxdeg);
    uint64_t v = vs;
    while (v < V) {
        uint64_t v1 = v;
        while (v1 < V && off[v1 + 1] - off[v] <= p->part_edges) v1++;
        if (v1 == v) v1 = v + 1;
        p->chunks.push_back({v, v1, off[v], off[v1]});
        v = v1;
    }
    p->streamed_edges = off[V] - off[vs];
    for (int i = 0; i < 2; i++) {
        ASC_HIP(hipMalloc(&p->part[i], 4 * std::max<uint64_t>(p->part_edges, 1)));
        ASC_HIP(hipEventCreateWithFlags(&p->ev_copy[i], hipEventDisableTiming));
        ASC_HIP(hipEventCreateWithFlags(&p->ev_kern[i], hipEventDisableTiming));
        // recorded once so that every copy can wait for the buffer's last reader
        ASC_HIP(hipEventRecord(p->ev_kern[i], g->ctx->s_main));
    }
    return ASC_OK;
}

// Enqueues, for every on-demand chunk, its copy from the pinned tail on the
// copy stream (double-buffered) and `pull(src, e_base, v0, v1)` on the compute
// stream.  No host synchronisation: every copy waits for the previous kernel
// that read its buffer, also across iterations.
template <class F>
static int pr_stream_chunks(asc_graph* g, PrState* p, F&& pull) {
    asc_ctx* ctx = g->ctx;
    const uint64_t S = g->static_edges;
    for (size_t c = 0; c < p->chunks.size(); c++) {
        const auto& ch = p->chunks[c];
        const int b = (int)(c & 1);
        ASC_HIP(hipStreamWaitEvent(ctx->s_copy, p->ev_kern[b], 0));
        ASC_HIP(hipMemcpyAsync(p->part[b], g->zc_tail.p + (ch.e0 - S), 4 * (ch.e1 - ch.e0), hipMemcpyHostToDevice,
                               ctx->s_copy));
        ASC_HIP(hipEventRecord(p->ev_copy[b], ctx->s_copy));
        ASC_HIP(hipStreamWaitEvent(ctx->s_main, p->ev_copy[b], 0));
        ASC_TRY(pull(p->part[b], ch.e0, ch.v0, ch.v1));
        ASC_HIP(hipEventRecord(p->ev_kern[b], ctx->s_main));
    }
    return ASC_OK;
}

// ---- row sums ---------------------------------------------------------------
// Resident rows (in-lists) are summed in row blocks: at most 256 consecutive
// vertices whose lists start within one window of kRowsWindow edges and hold
// fewer than kRowsHeavy edges each (a longer row ends a block), so a block is
// one contiguous stretch of at most kRowsTile edges whatever the degrees (cut
// once per graph, below).  A workgroup reads the stretch's ids, gathers their
// contributions into LDS, and each vertex's lane adds its own part in CSR
// order.  Longer rows are left to a wave or a workgroup each.
constexpr int kRowsPer = 8;
constexpr int kRowsTile = kBlock * kRowsPer;
constexpr uint32_t kRowsWindow = 1536;
constexpr uint32_t kRowsHeavy = 512;
static_assert(kRowsWindow + kRowsHeavy <= kRowsTile, "a row block is one tile");
constexpr uint32_t kRowsLong = 4096;    // rows summed by a whole workgroup, started before all others
constexpr int kPrLines = 16;            // counters spread over this many 128-byte lines
constexpr int kPrLineWords = 32;

// s + x[0] + x[1] + ... in that order, B values read ahead of their adds.
template <uint32_t B, class T>
__device__ __forceinline__ double add_in_order(double s, const T* x, uint32_t n) {
    uint32_t k = 0;
    for (; k + B <= n; k += B) {
        T y[B];
#pragma unroll
        for (uint32_t j = 0; j < B; j++) y[j] = x[k + j];
#pragma unroll
        for (uint32_t j = 0; j < B; j++) s += (double)y[j];
    }
    for (; k < n; k++) s += (double)x[k];
    return s;
}

// Sums the rows of at most 256 vertices [base, end) of any length (streamed
// chunks, whose rows have no plan): their concatenated edges a tile at a time,
// the owner of an edge found by a binary search of the degree prefix in LDS.
// take(v): whether v is summed; fin(v, sum) is called for those.
template <class OffT, class T, class Take, class Fin>
__device__ __forceinline__ void pull_rows(const OffT* off, const uint32_t* src, const T* contrib, uint64_t base,
                                          uint64_t end, T* s_val, Take take, Fin fin) {
    using PT = unsigned long long;
    __shared__ PT s_pref[kBlock];
    __shared__ OffT s_beg[kBlock];
    __shared__ PT s_tmp[kWavesPerBlock];
    const uint32_t tid = threadIdx.x;
    const uint64_t v = base + tid;
    const bool mine = v < end && take(v);
    OffT b = 0;
    PT deg = 0;
    if (mine) {
        b = off[v];
        deg = (PT)(off[v + 1] - b);
    }
    PT total;
    const PT pre = block_scan_excl(deg, s_tmp, total);
    s_pref[tid] = pre;
    s_beg[tid] = b;
    __syncthreads();
    double s = 0;
    for (PT t0 = 0; t0 < total; t0 += kRowsTile) {
        uint32_t u[kRowsPer];
        T c[kRowsPer];
#pragma unroll
        for (int j = 0; j < kRowsPer; j++) {
            const PT e = min((PT)(t0 + j * kBlock + tid), (PT)(total - 1));
            uint32_t k = 0;
#pragma unroll
            for (uint32_t step = kBlock / 2; step > 0; step >>= 1)
                if (s_pref[k + step] <= e) k += step;
            u[j] = src[s_beg[k] + (OffT)(e - s_pref[k])];
        }
#pragma unroll
        for (int j = 0; j < kRowsPer; j++) c[j] = contrib[u[j]];
        if (t0) __syncthreads();   // the previous tile's adds are done
#pragma unroll
        for (int j = 0; j < kRowsPer; j++) s_val[j * kBlock + tid] = c[j];
        __syncthreads();
        const PT t1 = total - t0 > kRowsTile ? (PT)(t0 + kRowsTile) : total;
        const PT lo = max(pre, t0), hi = min((PT)(pre + deg), t1);
        if (lo < hi) s = add_in_order<8>(s, s_val + (uint32_t)(lo - t0), (uint32_t)(hi - lo));
    }
    if (mine) fin(v, s);
    __syncthreads();
}

// Row blocks of the vertices [0, n), written in any order.
struct RowBlock {
    unsigned long long e;           // first edge
    uint32_t v, n, edges;           // vertices [v, v + n), their edges
    uint32_t pad;
};

template <class OffT>
__global__ __launch_bounds__(kBlock) void k_row_blocks(const OffT* off, uint64_t n, RowBlock* blocks, uint32_t* cnt) {
    __shared__ uint64_t s_break[kWavesPerBlock];
    __shared__ uint32_t s_count[kWavesPerBlock], s_at;
    const uint32_t lane = lane_id(), w = wave_id();
    for (uint64_t base = (uint64_t)blockIdx.x * kBlock; base < n; base += (uint64_t)gridDim.x * kBlock) {
        const uint64_t v = base + threadIdx.x;
        uint64_t b = 0, d = 0;
        bool heavy = false, starts = false;
        if (v < n) {
            b = (uint64_t)off[v];
            d = (uint64_t)off[v + 1] - b;
            heavy = d >= kRowsHeavy;
            // a new block at every multiple of 256, in every window and after a heavy row
            starts = !heavy && (threadIdx.x == 0 || (uint64_t)off[v - 1] / kRowsWindow != b / kRowsWindow ||
                                b - (uint64_t)off[v - 1] >= kRowsHeavy);
        }
        const uint64_t brk = wave_ballot(starts || heavy || v >= n);
        if (lane == 0) s_break[w] = brk;
        const uint64_t m = wave_ballot(starts);
        // one global atomic per 256 vertices
        if (lane == 0) s_count[w] = (uint32_t)__popcll(m);
        __syncthreads();
        if (threadIdx.x == 0) {
            uint32_t all = 0;
            for (int i = 0; i < kWavesPerBlock; i++) all += s_count[i];
            s_at = all ? atomicAdd(cnt, all) : 0;
        }
        __syncthreads();
        uint32_t at = s_at;
        for (uint32_t i = 0; i < w; i++) at += s_count[i];
        if (starts) {
            // the next break after this lane ends the block
            uint32_t end = kBlock;
            uint64_t rest = lane == kWave - 1 ? 0 : brk & (~0ull << (lane + 1));
            for (uint32_t i = w; i < (uint32_t)kWavesPerBlock; i++) {
                if (i > w) rest = s_break[i];
                if (rest) {
                    end = i * kWave + (uint32_t)__builtin_ctzll(rest);
                    break;
                }
            }
            const uint32_t cntv = end - threadIdx.x;
            blocks[at + lanes_below(m)] =
                RowBlock{b, (uint32_t)v, cntv, (uint32_t)((uint64_t)off[v + cntv] - b), 0u};
        }
        __syncthreads();
    }
}

// Sums the rows of a row block.  s_val: kRowsTile values of LDS.  pre(v) reads
// what fin(v, sum, pre(v)) needs of a vertex, ahead of the gathers.
template <class OffT, class T, class Pre, class Fin>
__device__ __forceinline__ void pull_block(const OffT* off, const uint32_t* src, const T* contrib, const RowBlock& rb,
                                           T* s_val, Pre pre, Fin fin) {
    const uint32_t tid = threadIdx.x;
    const uint32_t* ids = src + rb.e;
    uint32_t u[kRowsPer];
#pragma unroll
    for (int j = 0; j < kRowsPer; j++) u[j] = rb.edges ? ids[min(j * (uint32_t)kBlock + tid, rb.edges - 1)] : 0u;
    const bool mine = tid < rb.n;
    const uint32_t v = rb.v + (mine ? tid : 0);
    const uint32_t lo = (uint32_t)((uint64_t)off[v] - rb.e), hi = (uint32_t)((uint64_t)off[v + 1] - rb.e);
    const auto own = pre(v);
    T c[kRowsPer];
#pragma unroll
    for (int j = 0; j < kRowsPer; j++) c[j] = contrib[u[j]];
#pragma unroll
    for (int j = 0; j < kRowsPer; j++) s_val[j * kBlock + tid] = c[j];
    __syncthreads();
    if (mine) fin(v, add_in_order<8>(0.0, s_val + lo, hi - lo), own);
    __syncthreads();   // s_val is free again
}

// Rows of kRowsHeavy edges and more among the vertices [0, n): those of
// kRowsLong edges from the front of `list`, the others from its back.
template <class OffT>
__global__ __launch_bounds__(kBlock) void k_rows_heavy_list(const OffT* off, uint64_t n, uint32_t* list, uint32_t cap,
                                                            uint32_t* cnt) {
    for (uint64_t base = (uint64_t)blockIdx.x * kBlock; base < n; base += (uint64_t)gridDim.x * kBlock) {
        const uint64_t v = base + threadIdx.x;
        const uint64_t d = v < n ? (uint64_t)(off[v + 1] - off[v]) : 0;
        const bool front = d >= kRowsLong, back = d >= kRowsHeavy && !front;
        const uint64_t mf = wave_ballot(front), mb = wave_ballot(back);
        uint32_t at = 0;
        if (lane_id() == 0 && mf) at = atomicAdd(cnt, (uint32_t)__popcll(mf));
        at = __shfl(at, 0, kWave);
        if (front) list[at + lanes_below(mf)] = (uint32_t)v;
        if (lane_id() == 0 && mb) at = atomicAdd(cnt + 1, (uint32_t)__popcll(mb));
        at = __shfl(at, 0, kWave);
        if (back) list[cap - 1 - (at + lanes_below(mb))] = (uint32_t)v;
    }
}

// The row plan of a graph's resident vertices.
struct RowPlan {
    const RowBlock* blocks;
    const uint32_t* heavy;        // rows >= kRowsLong from the front, >= kRowsHeavy from the back
    uint32_t n_blocks, cap, n_front, n_back;
    __device__ __forceinline__ uint32_t front(uint32_t i) const { return heavy[i]; }
    __device__ __forceinline__ uint32_t back(uint32_t i) const { return heavy[cap - 1 - i]; }
};

// ---- normalised mode --------------------------------------------------------

// The residual and dangling sums of an iteration: every workgroup adds its
// share to one of kPrLines cache lines of a slot (same-address atomics of a
// whole grid take ~9 ns each, 18 us for 2048 workgroups), and the readers add
// the lines up.  Slot it & 3 holds the dangling mass of the ranks iteration
// `it` reads and the residual of iteration it - 1; iteration `it` clears slot
// (it + 2) & 3.  Beside them, the largest contribution that iteration `it`
// gathers (float bits; the blocked schedule's scale).
constexpr int kAccLine = 16;                            // doubles per 128-byte line
constexpr int kAccDang = kPrLines * kAccLine;           // the dangling lines follow the residual lines
constexpr int kAccMax = 2 * kAccDang;                   // and the maximum's follow those
constexpr int kAccSlot = 3 * kAccDang;
constexpr int kAccSlots = 4;

// Sum of a slot's lines (the residual's at `p`, the dangling mass's at
// p + kAccDang), in every lane of the calling wave.
__device__ __forceinline__ double acc_lines(const double* p) {
    const uint32_t l = lane_id();
    return wave_sum(l < (uint32_t)kPrLines ? p[l * kAccLine] : 0.0);
}

// What a lane adds up over the vertices it finishes.
struct PrSums {
    double res = 0, dang = 0;
    uint32_t most = 0;           // float bits of the largest contribution written (they order as the values do)
    __device__ __forceinline__ void wrote(float c) { most = max(most, __float_as_uint(c)); }
};

// Workgroup sums, added to this workgroup's lines of `acc`.
template <int THREADS>
__device__ __forceinline__ void acc_add(const PrSums& a, double* acc) {
    __shared__ double s_r[THREADS / kWave], s_d[THREADS / kWave];
    __shared__ uint32_t s_m[THREADS / kWave];
    const double res = wave_sum(a.res), dang = wave_sum(a.dang);
    uint32_t most = a.most;
#pragma unroll
    for (int d = kWave / 2; d > 0; d >>= 1) most = max(most, (uint32_t)__shfl_xor(most, d, kWave));
    if (lane_id() == 0) {
        s_r[wave_id()] = res;
        s_d[wave_id()] = dang;
        s_m[wave_id()] = most;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double r = 0, d = 0;
        uint32_t m = 0;
        for (int i = 0; i < THREADS / kWave; i++) {
            r += s_r[i];
            d += s_d[i];
            m = max(m, s_m[i]);
        }
        double* line = acc + (blockIdx.x % kPrLines) * kAccLine;
        if (r != 0) atomicAdd(line, r);
        if (d != 0) atomicAdd(line + kAccDang, d);
        if (m) atomicMax((uint32_t*)(line + kAccMax), m);
    }
}

__global__ void k_pr_fill(uint32_t* p, uint64_t n, uint32_t v) {
    for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
        p[i] = v;
}

__global__ __launch_bounds__(kBlock) void k_pr_init(float* rank, float* contrib, const uint32_t* outdeg, uint64_t V,
                                                    double* acc) {
    const float r0 = (float)(1.0 / (double)V);
    PrSums sums;
    for (uint64_t v = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; v < V; v += (uint64_t)gridDim.x * blockDim.x) {
        const uint32_t d = outdeg[v];
        const float c = d ? r0 / (float)d : 0.0f;
        rank[v] = r0;
        contrib[v] = c;
        sums.wrote(c);
        if (!d) sums.dang += (double)r0;
    }
    acc_add<kBlock>(sums, acc);
}

// The last iteration's residual, then all of them to mapped host memory and
// the sequence number the host polls for behind them (one wave).
__global__ void k_pr_residuals(const double* slot, double* resid, int iters, double* host, unsigned long long seq) {
    const double r = acc_lines(slot);
    for (int i = threadIdx.x; i < iters; i += kWave) host_store(host + i, i == iters - 1 ? r : resid[i]);
    __threadfence_system();   // every lane's, before the one lane publishes
    __builtin_amdgcn_wave_barrier();
    if (threadIdx.x == 0) host_publish((unsigned long long*)(host + iters), seq);
}

struct PrArgs {
    const void* off;              // OffT[V+1]
    const uint32_t* src;          // in-edges: edge k at src[k - e_base]
    unsigned long long e_base;
    unsigned long long v_begin, v_end;  // vertices pulled by this launch
    int skip_heavy;               // leave in-degree >= heavy_thr to k_pr_pull_heavy
    const uint32_t* outdeg;
    const float* rank_in;
    const float* contrib_in;
    float* rank_out;
    float* contrib_out;
    const double* acc_in;         // slot with the dangling mass of rank_in
    double* acc_out;              // slot of this iteration's residual and rank_out's dangling mass
    double* acc_clear;            // slot to clear (the iteration's first launch; else null)
    double* resid_prev;           // where that launch stores the previous iteration's residual (or null)
    uint64_t V;
    float damping;
    double damping64;
    uint32_t heavy_thr;
};

// What a vertex's new rank is finished with.
struct PrOwn {
    uint32_t outdeg;
    float rank;
};

__device__ __forceinline__ PrOwn pr_own(const PrArgs& a, uint64_t v) { return PrOwn{a.outdeg[v], a.rank_in[v]}; }

__device__ __forceinline__ void pr_finish_vertex(const PrArgs& a, uint64_t v, double s, const PrOwn& own, double base,
                                                 PrSums& sums) {
    const float nr = (float)(base + a.damping64 * s);
    const float c = own.outdeg ? nr / (float)own.outdeg : 0.0f;
    sums.res += fabs((double)nr - (double)own.rank);
    sums.wrote(c);
    a.rank_out[v] = nr;
    a.contrib_out[v] = c;
    if (!own.outdeg) sums.dang += (double)nr;
}

__device__ __forceinline__ void pr_finish_vertex(const PrArgs& a, uint64_t v, double s, double base, PrSums& sums) {
    pr_finish_vertex(a, v, s, pr_own(a, v), base, sums);
}

// Rank of a vertex whose in-sum is zero, in every lane; called by the whole
// workgroup.  Workgroup 0 of an iteration's first launch also stores the
// previous residual and clears the slot of the iteration after the next.
__device__ __forceinline__ double pr_base(const PrArgs& a) {
    __shared__ double s_base;
    if (threadIdx.x < kWave) {
        const double dang = acc_lines(a.acc_in + kAccDang);
        if (threadIdx.x == 0) s_base = (1.0 - a.damping64) / (double)a.V + a.damping64 * dang / (double)a.V;
        if (blockIdx.x == 0 && a.resid_prev) {
            const double r = acc_lines(a.acc_in);
            if (threadIdx.x == 0) *a.resid_prev = r;
        }
        if (blockIdx.x == 0 && a.acc_clear)
            for (int i = threadIdx.x; i < kAccSlot; i += kWave) a.acc_clear[i] = 0;
    }
    __syncthreads();
    return s_base;
}

// Sum of one long row by the whole workgroup (the result in thread 0): 8
// gathers in flight per lane.  s_sum: one double per wave.
template <class OffT>
__device__ __forceinline__ double pull_long_row(const uint32_t* src, const float* contrib, OffT b, OffT e,
                                                double* s_sum) {
    constexpr int U = 8;
    double s = 0;
    for (OffT k = b + threadIdx.x; k < e; k += (OffT)U * kBlock) {
        uint32_t u[U];
        float c[U];
#pragma unroll
        for (int j = 0; j < U; j++) u[j] = src[min((OffT)(k + j * kBlock), (OffT)(e - 1))];
#pragma unroll
        for (int j = 0; j < U; j++) c[j] = contrib[u[j]];
#pragma unroll
        for (int j = 0; j < U; j++)
            if (k + (OffT)(j * kBlock) < e) s += (double)c[j];
    }
    s = wave_sum(s);
    if (lane_id() == 0) s_sum[wave_id()] = s;
    __syncthreads();
    double t = 0;
    if (threadIdx.x == 0)
        for (int j = 0; j < kWavesPerBlock; j++) t += s_sum[j];
    __syncthreads();
    return t;
}

// The same by one wave (the result in every lane).
template <class OffT>
__device__ __forceinline__ double pull_wave_row(const uint32_t* src, const float* contrib, OffT b, OffT e) {
    constexpr int U = 8;
    double s = 0;
    for (OffT k = b + lane_id(); k < e; k += (OffT)U * kWave) {
        uint32_t u[U];
        float c[U];
#pragma unroll
        for (int j = 0; j < U; j++) u[j] = src[min((OffT)(k + j * kWave), (OffT)(e - 1))];
#pragma unroll
        for (int j = 0; j < U; j++) c[j] = contrib[u[j]];
#pragma unroll
        for (int j = 0; j < U; j++)
            if (k + (OffT)(j * kWave) < e) s += (double)c[j];
    }
    return wave_sum(s);
}

// The pull of an iteration: over the resident rows (HEAVY: the first `hb`
// workgroups take the rows above kRowsHeavy, longest first, the others the
// row blocks), or over the vertices [v_begin, v_end) of a streamed chunk.
template <class OffT, bool HEAVY>
__global__ __launch_bounds__(kBlock) void k_pr_rows(PrArgs a, RowPlan rows, uint32_t hb) {
    __shared__ float s_val[kRowsTile];
    __shared__ double s_sum[kWavesPerBlock];
    const OffT* off = (const OffT*)a.off;
    const uint32_t* src = a.src - a.e_base;
    const double base = pr_base(a);
    PrSums sums;
    if (HEAVY && blockIdx.x < hb) {
        for (uint32_t i = blockIdx.x; i < rows.n_front; i += hb) {
            const uint32_t v = rows.front(i);
            const double s = pull_long_row<OffT>(src, a.contrib_in, off[v], off[v + 1], s_sum);
            if (threadIdx.x == 0) pr_finish_vertex(a, v, s, base, sums);
        }
        for (uint32_t i = blockIdx.x * kWavesPerBlock + wave_id(); i < rows.n_back; i += hb * kWavesPerBlock) {
            const uint32_t v = rows.back(i);
            const double s = pull_wave_row<OffT>(src, a.contrib_in, off[v], off[v + 1]);
            if (lane_id() == 0) pr_finish_vertex(a, v, s, base, sums);
        }
    } else {
        const uint32_t bid = blockIdx.x - (HEAVY ? hb : 0), nblk = gridDim.x - (HEAVY ? hb : 0);
        if (HEAVY) {
            auto pre = [&](uint64_t v) { return pr_own(a, v); };
            auto fin = [&](uint64_t v, double s, const PrOwn& own) { pr_finish_vertex(a, v, s, own, base, sums); };
            for (uint32_t i = bid; i < rows.n_blocks; i += nblk)
                pull_block(off, src, a.contrib_in, rows.blocks[i], s_val, pre, fin);
        } else {
            auto take = [](uint64_t) { return true; };
            auto fin = [&](uint64_t v, double s) { pr_finish_vertex(a, v, s, base, sums); };
            for (uint64_t v = a.v_begin + (uint64_t)bid * kBlock; v < a.v_end; v += (uint64_t)nblk * kBlock)
                pull_rows(off, src, a.contrib_in, v, a.v_end, s_val, take, fin);
        }
    }
    acc_add<kBlock>(sums, a.acc_out);
}

// G lanes per vertex (asc_config.pr_group or a tuned graph); vertices with
// in-degree >= heavy_thr are skipped here.
template <int G, class OffT>
__global__ __launch_bounds__(kBlock) void k_pr_pull(PrArgs a) {
    const OffT* off = (const OffT*)a.off;
    const double base = pr_base(a);
    const uint32_t sub = threadIdx.x % G;
    const uint64_t groups_per_grid = (uint64_t)gridDim.x * (blockDim.x / G);
    const uint32_t* src = a.src - a.e_base;
    PrSums sums;
    for (uint64_t v = a.v_begin + blockIdx.x * (uint64_t)(blockDim.x / G) + threadIdx.x / G; v < a.v_end;
         v += groups_per_grid) {
        const OffT b = off[v], e = off[v + 1];
        const bool heavy = a.skip_heavy && (uint64_t)(e - b) >= a.heavy_thr;
        double s = 0;
        if (!heavy) {
            // four edges per lane per pass: their source ids, then their
            // contributions, are loaded back to back (a lane past the end
            // re-reads the list's first edge and drops it)
            for (OffT k = b + sub; k < e; k += 4 * G) {
                uint32_t u[4];
#pragma unroll
                for (int j = 0; j < 4; j++) u[j] = src[k + (OffT)(j * G) < e ? k + (OffT)(j * G) : b];
                float c[4];
#pragma unroll
                for (int j = 0; j < 4; j++) c[j] = a.contrib_in[u[j]];
#pragma unroll
                for (int j = 0; j < 4; j++)
                    if (k + (OffT)(j * G) < e) s += (double)c[j];
            }
        }
#pragma unroll
        for (int d = G / 2; d > 0; d >>= 1) s += __shfl_xor(s, d, G);
        if (sub == 0 && !heavy) pr_finish_vertex(a, v, s, base, sums);
    }
    acc_add<kBlock>(sums, a.acc_out);
}

template <class OffT>
__global__ __launch_bounds__(kBlock) void k_pr_pull_heavy(PrArgs a, const uint32_t* heavy, uint32_t n_heavy) {
    __shared__ double s_sum[kWavesPerBlock];
    const OffT* off = (const OffT*)a.off;
    const double base = pr_base(a);
    PrSums sums;
    for (uint32_t i = blockIdx.x; i < n_heavy; i += gridDim.x) {
        const uint32_t v = heavy[i];
        const double s = pull_long_row<OffT>(a.src, a.contrib_in, off[v], off[v + 1], s_sum);
        if (threadIdx.x == 0) pr_finish_vertex(a, v, s, base, sums);
    }
    acc_add<kBlock>(sums, a.acc_out);
}

// ---- propagation-blocked normalised mode -----------------------------------
// A pull's random 4-byte gathers each bring a 128-byte line from L2 into L1,
// and a CU takes 64 bytes a clock: 3.3 ps an edge over the chip at best (the
// row blocks measure 5.2 to 6.8 while the contributions fit the L2s, 16 at V =
// 2^23 Erdos-Renyi), and the tiled pull below measures 5.8 to 400.  Here every
// random access is to LDS and memory is only streamed, 12.5 bytes an edge:
//   scatter  a workgroup loads the contributions of one slice of sources into
//            LDS and writes, for each of a stretch of the slice's edges, the
//            contribution of its source (2-byte local id) to the edge's place;
//   gather   a workgroup per bin of destinations adds the values of the bin's
//            edges into LDS sums (2-byte local ids) and finishes its vertices.
// A slice's edges of one bin are a run, padded to octs.  Sources and values
// lie in slice order, so the scatter reads and writes straight through;
// destinations lie in bin order, with each oct's place in slice order, so the
// gather's lanes are busy whatever the runs' lengths and its value reads are
// runs of a few KB.  Bins are cut by vertices and by edges, so skewed graphs
// get bins of equal work; a row of kRowsLong edges and more is a bin of its
// own, summed in registers.  The layout depends on the graph alone and is
// built once (2^28 edges: 14 ms).
// 20 iterations in ms, this / tiled / row blocks:
//   Erdos-Renyi V = 2^23, 2^28 edges  14.8 / 31.3 / 86.2 (scatter 328 us and
//                                     gather 408 us an iteration, both at the
//                                     ~5 TB/s that memory gives)
//   R-MAT scale 23, 2.6e8 edges       17.1 / 152 / 41.0
//   R-MAT scale 20, 3.1e7 edges       2.27 / 109 / 3.28
//   Erdos-Renyi V = 2^18, 2^23 edges  0.66 / 13.5 / 1.07
//   R-MAT scale 18, 7.6e6 edges       0.91 / 46.0 / 0.80
//   Erdos-Renyi V = 2^22, 8.4e6 edges 0.75 / 2.19 / 2.94
constexpr int kPbBlock = 1024;
constexpr uint32_t kPbOct = 8;                  // edges a lane moves at a time; runs are padded to it
constexpr uint32_t kPbItemOcts = 1u << 14;      // octs per scatter workgroup, at most
constexpr uint32_t kPbMaxSlices = 8192;         // build histograms in LDS

struct PbBin {
    uint32_t v, n;               // vertices [v, v + n)
    uint32_t o, octs;            // octs [o, o + octs) in bin order
    uint32_t kind;               // kPbPlain / kPbAround / kPbHeavy
};
constexpr uint32_t kPbPlain = 0;
constexpr uint32_t kPbAround = 1;   // holds rows of kRowsLong edges and more, which are not its own
constexpr uint32_t kPbHeavy = 2;    // is one such row: summed in registers
struct PbRun {
    uint32_t q, n, o;            // octs [q, q + n) in slice order, [o, o + n) in bin order
};
struct PbItem {
    uint32_t slice, q0, q1;
};
typedef unsigned short PbIds __attribute__((ext_vector_type(8)));   // the ids of an oct

// cnt[b * ns + s]: edges of bin b from slice s.  A workgroup per bin.
template <class OffT>
__global__ __launch_bounds__(kPbBlock) void k_pb_count(const OffT* off, const uint32_t* src, const PbBin* bins,
                                                       uint32_t ns, uint32_t bits, uint32_t* cnt) {
    __shared__ uint32_t h[kPbMaxSlices];
    const PbBin b = bins[blockIdx.x];
    for (uint32_t i = threadIdx.x; i < ns; i += kPbBlock) h[i] = 0;
    __syncthreads();
    if (b.kind == kPbAround) {
        constexpr uint32_t L = 8;
        for (uint32_t r = threadIdx.x / L; r < b.n; r += kPbBlock / L) {
            const OffT e0 = off[b.v + r], e1 = off[b.v + r + 1];
            if (e1 - e0 >= kRowsLong) continue;
            for (OffT e = e0 + threadIdx.x % L; e < e1; e += L) atomicAdd(&h[src[e] >> bits], 1u);
        }
    } else {
        const OffT e1 = off[b.v + b.n];
        for (OffT e = off[b.v] + threadIdx.x; e < e1; e += kPbBlock) atomicAdd(&h[src[e] >> bits], 1u);
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < ns; i += kPbBlock) cnt[(size_t)blockIdx.x * ns + i] = h[i];
}

// Octs of every slice (SLICES: a workgroup per slice, else per bin).
template <bool SLICES>
__global__ __launch_bounds__(kBlock) void k_pb_totals(const uint32_t* cnt, uint32_t nb, uint32_t ns, uint32_t* out) {
    __shared__ uint32_t s_sum[kWavesPerBlock];
    uint32_t sum = 0;
    for (uint32_t i = threadIdx.x; i < (SLICES ? nb : ns); i += kBlock)
        sum += (cnt[SLICES ? (size_t)i * ns + blockIdx.x : (size_t)blockIdx.x * ns + i] + kPbOct - 1) / kPbOct;
    sum = wave_sum(sum);
    if (lane_id() == 0) s_sum[wave_id()] = sum;
    __syncthreads();
    if (threadIdx.x == 0) out[blockIdx.x] = s_sum[0] + s_sum[1] + s_sum[2] + s_sum[3];
}

// The runs' places: in slice order (SLICES: a workgroup per slice goes through
// the bins), else in bin order (a workgroup per bin goes through the slices).
template <bool SLICES>
__global__ __launch_bounds__(kBlock) void k_pb_place(const uint32_t* cnt, uint32_t nb, uint32_t ns,
                                                     const uint32_t* first, PbRun* runs) {
    __shared__ uint32_t s_sum[kWavesPerBlock];
    uint32_t at = first[blockIdx.x];
    for (uint32_t i0 = 0; i0 < (SLICES ? nb : ns); i0 += kBlock) {
        const uint32_t i = i0 + threadIdx.x;
        const bool in = i < (SLICES ? nb : ns);
        const size_t k = SLICES ? (size_t)i * ns + blockIdx.x : (size_t)blockIdx.x * ns + i;
        const uint32_t n = in ? (cnt[k] + kPbOct - 1) / kPbOct : 0;
        uint32_t x = n;   // inclusive sum over the wave
#pragma unroll
        for (int d = 1; d < kWave; d <<= 1) {
            const uint32_t y = __shfl_up(x, d, kWave);
            if (lane_id() >= (uint32_t)d) x += y;
        }
        if (lane_id() == kWave - 1) s_sum[wave_id()] = x;
        __syncthreads();
        uint32_t before = 0, all = 0;
        for (uint32_t w = 0; w < (uint32_t)kWavesPerBlock; w++) {
            if (w < wave_id()) before += s_sum[w];
            all += s_sum[w];
        }
        const uint32_t place = at + before + x - n;
        if (in && SLICES) {
            runs[k].q = place;
            runs[k].n = n;
        } else if (in) {
            runs[k].o = place;
        }
        at += all;
        __syncthreads();
    }
}

// The local ids of every edge of a bin (source in the low half of a word,
// destination in the high), in arrival order within its runs.  Eight lanes
// share a row.  The LDS array is larger than the cursors need: one workgroup a
// CU keeps the runs' open lines (128 bytes a run) within the XCD's L2.
template <class OffT>
__global__ __launch_bounds__(kPbBlock) void k_pb_fill(const OffT* off, const uint32_t* src, const PbBin* bins,
                                                      const PbRun* runs, uint32_t ns, uint32_t bits, uint32_t* out) {
    constexpr uint32_t L = 8;
    __shared__ unsigned long long cur[kPbMaxSlices + kPbMaxSlices / 4 + 128];
    const PbBin b = bins[blockIdx.x];
    for (uint32_t i = threadIdx.x; i < ns; i += kPbBlock) cur[i] = (uint64_t)kPbOct * runs[(size_t)blockIdx.x * ns + i].q;
    __syncthreads();
    const uint32_t mask = (1u << bits) - 1;
    if (b.kind == kPbHeavy) {
        const OffT e1 = off[b.v + 1];
        for (OffT e = off[b.v] + threadIdx.x; e < e1; e += kPbBlock) {
            const uint32_t u = src[e];
            out[atomicAdd(&cur[u >> bits], 1ull)] = u & mask;
        }
        return;
    }
    for (uint32_t r = threadIdx.x / L; r < b.n; r += kPbBlock / L) {
        const OffT e0 = off[b.v + r], e1 = off[b.v + r + 1];
        if (b.kind == kPbAround && e1 - e0 >= kRowsLong) continue;
        for (OffT e = e0 + threadIdx.x % L; e < e1; e += L) {
            const uint32_t u = src[e];
            out[atomicAdd(&cur[u >> bits], 1ull)] = (u & mask) | (r << 16);
        }
    }
}

// Splits the pairs: sources stay in slice order, destinations go to bin order,
// where `pos` has each oct's place in slice order.  Eight lanes take a run.
__global__ __launch_bounds__(kPbBlock) void k_pb_unzip(const PbRun* runs, uint32_t ns, const uint4* in, PbIds* src,
                                                       PbIds* dst, uint32_t* pos) {
    constexpr uint32_t L = 8;
    for (uint32_t i = threadIdx.x / L; i < ns; i += kPbBlock / L) {
        const PbRun r = runs[(size_t)blockIdx.x * ns + i];
        for (uint32_t k = threadIdx.x % L; k < r.n; k += L) {
            const uint32_t q = r.q + k;
            const uint4 x = in[2 * (size_t)q], y = in[2 * (size_t)q + 1];
            src[q] = PbIds{(unsigned short)x.x, (unsigned short)x.y, (unsigned short)x.z, (unsigned short)x.w,
                           (unsigned short)y.x, (unsigned short)y.y, (unsigned short)y.z, (unsigned short)y.w};
            dst[r.o + k] = PbIds{(unsigned short)(x.x >> 16), (unsigned short)(x.y >> 16), (unsigned short)(x.z >> 16),
                                 (unsigned short)(x.w >> 16), (unsigned short)(y.x >> 16), (unsigned short)(y.y >> 16),
                                 (unsigned short)(y.z >> 16), (unsigned short)(y.w >> 16)};
            pos[r.o + k] = q;
        }
    }
}

// Consecutive items (of one slice, mostly) go to one XCD, so a slice comes
// into one L2.
template <int BITS>
__global__ __launch_bounds__(kPbBlock) void k_pb_scatter(const float* __restrict__ contrib, uint64_t V,
                                                         const PbItem* __restrict__ items, uint32_t n_items,
                                                         const ushort4* __restrict__ src, float4* __restrict__ vals) {
    __shared__ float s_c[1u << BITS];
    const uint32_t per = (n_items + 7) / 8, id = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if ((blockIdx.x >> 3) >= per || id >= n_items) return;
    const PbItem it = items[id];
    const uint64_t base = (uint64_t)it.slice << BITS;
    const uint32_t have = (uint32_t)min<uint64_t>(1u << BITS, V - base);
    for (uint32_t i = threadIdx.x; i < have / 4; i += kPbBlock)
        ((float4*)s_c)[i] = ((const float4*)(contrib + base))[i];
    for (uint32_t i = (have & ~3u) + threadIdx.x; i < have; i += kPbBlock) s_c[i] = contrib[base + i];
    __syncthreads();
    // half an oct a lane: whole lines per store
    constexpr int U = 4;
    const uint32_t q1 = 2 * it.q1;
    for (uint32_t q = 2 * it.q0 + threadIdx.x; q < q1; q += U * kPbBlock) {
        ushort4 u[U];
#pragma unroll
        for (int j = 0; j < U; j++) u[j] = src[min(q + j * kPbBlock, q1 - 1)];
#pragma unroll
        for (int j = 0; j < U; j++)
            if (q + j * kPbBlock < q1)
                vals[q + j * kPbBlock] = make_float4(s_c[u[j].x], s_c[u[j].y], s_c[u[j].z], s_c[u[j].w]);
    }
}

// Sums in LDS are 64-bit fixed point: a 64-lane FP32 LDS add takes 136 clocks
// on gfx950 (the lanes one after the other; FP32 sums ran 1363 us an iteration
// at V = 2^23, 2^28 edges, all of it those adds), an integer one a few.  With
// the largest contribution c below 2^e and fewer than 2^12 edges a row, units
// of 2^(e - 51) cannot overflow, a contribution of 2^-27 of the largest still
// keeps its 24 bits, and sums are exact in these units whatever their order.
// A smaller one is off by half a unit at most, 2^-51 c, and the 4095 of a row
// may all be off the same way (a clique's are equal).  Every rank is at least
// its base, so with c at most kPbSpread bases a row stays within 2^-26 of the
// rank, a quarter of what rounding it to FP32 may change (2^20 instead of 2^13
// bases: ranks of a 4095-clique beside a hub of 2^18 leaves two units off
// those of FP64 sums).  R-MAT and Erdos-Renyi graphs reach 2^3 to 2^5 bases.
// Beyond kPbSpread (a vertex with a large share of all rank and few out-edges,
// or out-degrees too small for the edges, whose ranks grow to infinity) sums
// are FP64.
constexpr double kPbSpread = 1 << 13;
__device__ __forceinline__ uint32_t pb_most(const double* slot) {
    const uint32_t l = lane_id();
    uint32_t m = l < (uint32_t)kPrLines ? *(const uint32_t*)(slot + kAccMax + l * kAccLine) : 0u;
#pragma unroll
    for (int d = kWave / 2; d > 0; d >>= 1) m = max(m, (uint32_t)__shfl_xor(m, d, kWave));
    return m;
}
__device__ __forceinline__ unsigned long long pb_fixed(float x, int shift) {
    const uint32_t bits = __float_as_uint(x);
    const int s = max((int)(bits >> 23), 1) + shift;
    const unsigned long long m = (bits & 0x7FFFFFu) | (bits >> 23 ? 0x800000u : 0u);
    return s >= 0 ? m << s : s > -25 ? (m + (1ull << (-s - 1))) >> -s : 0ull;
}

// A lane takes an oct at a time, wherever its run begins or ends (a wave per
// run left most lanes idle on R-MAT graphs, whose runs are mostly short: 1040
// us at V = 2^23).  The padding of a run adds to one sum past the bin's.
template <class OffT, int BITS>
__global__ __launch_bounds__(kPbBlock) void k_pb_gather(PrArgs a, const PbBin* __restrict__ bins,
                                                        const uint32_t* __restrict__ pos,
                                                        const ushort4* __restrict__ dst,
                                                        const float4* __restrict__ vals) {
    __shared__ unsigned long long acc[(1u << BITS) + 1];
    const PbBin b = bins[blockIdx.x];
    const OffT* off = (const OffT*)a.off;
    for (uint32_t i = threadIdx.x; i < b.n; i += kPbBlock) acc[i] = 0;
    const uint32_t big = pb_most(a.acc_in);
    // shift of a 24-bit mantissa, less its exponent field: the largest
    // contribution is below 2^(field - 126)
    const int shift = 27 - (int)max(big >> 23, 1u);
    const double base = pr_base(a);   // (ends with a barrier)
    const bool fixed = (double)__uint_as_float(big) <= kPbSpread * base, heavy = b.kind == kPbHeavy;
    double sum = 0;                   // a heavy row's (id 0; the padding has another)
    auto add = [&](uint32_t at, float x) {
        if (heavy) sum += at == 0 ? (double)x : 0.0;
        else if (fixed) atomicAdd(&acc[at], pb_fixed(x, shift));
        else atomicAdd((double*)&acc[at], (double)x);
    };
    constexpr int U = 4;
    const uint32_t end = 2 * (b.o + b.octs);
    for (uint32_t o = 2 * b.o + threadIdx.x; o < end; o += U * kPbBlock) {
        uint32_t q[U];
        ushort4 d[U];
        float4 x[U];
#pragma unroll
        for (int j = 0; j < U; j++) {
            const uint32_t at = min(o + j * kPbBlock, end - 1);
            q[j] = 2 * pos[at >> 1] + (at & 1);
            d[j] = dst[at];
        }
#pragma unroll
        for (int j = 0; j < U; j++) x[j] = vals[q[j]];
#pragma unroll
        for (int j = 0; j < U; j++) {
            if (o + j * kPbBlock >= end) continue;
            add(d[j].x, x[j].x);
            add(d[j].y, x[j].y);
            add(d[j].z, x[j].z);
            add(d[j].w, x[j].w);
        }
    }
    __syncthreads();
    // a unit is 2^(field - 126 - 51)
    const double unit = ldexp(1.0, 27 - shift - 177);
    PrSums sums;
    if (heavy) {
        __shared__ double s_sum[kPbBlock / kWave];
        sum = wave_sum(sum);
        if (lane_id() == 0) s_sum[wave_id()] = sum;
        __syncthreads();
        if (threadIdx.x == 0) {
            for (int i = 1; i < kPbBlock / kWave; i++) sum += s_sum[i];
            pr_finish_vertex(a, b.v, sum, base, sums);
        }
    }
    for (uint32_t i = threadIdx.x; !heavy && i < b.n; i += kPbBlock) {
        if (b.kind == kPbAround && off[b.v + i + 1] - off[b.v + i] >= kRowsLong) continue;
        pr_finish_vertex(a, b.v + i, fixed ? (double)acc[i] * unit : __longlong_as_double((long long)acc[i]), base, sums);
    }
    acc_add<kPbBlock>(sums, a.acc_out);
}

// ---- source-segmented normalised mode --------------------------------------
// The pull gathers one random 4-byte contribution per in-edge from an array
// of 4V bytes (256 MB at V = 2^26, beyond the 4 MB L2 of an XCD and as large
// as the MALL), so almost every gather moves a whole line from HBM.  Here the
// light in-edges are regrouped once into tiles by (destination block of 2^db
// vertices, source segment of 2^sb vertices).  One workgroup owns a
// destination block at a time: it keeps the block's sums in LDS (FP32) and
// walks the segments in order, so the gathers of a tile read one 4 * 2^sb
// byte slice of the contributions, and the workgroups resident on an XCD,
// walking the segments in the same order, share that slice in the XCD's L2.
// A tile edge is one u32 word (block-local destination << sb | segment-local
// source).  The grid is persistent: workgroup b takes blocks b, b + G, ...,
// so the resident workgroups start together and stay near each other's
// segment.  The last pass over a block finishes its vertices (rank,
// contribution, residual, dangling mass) as the pull does.  Destinations with
// in-degree >= the heavy threshold keep the FP64 pull (k_pr_pull_heavy).
constexpr int kTlMaxDstBits = 15;                          // LDS sums: up to 32768 FP32 (128 KB)
constexpr uint32_t kTlMaxSeg = 8192;                       // build histograms in LDS
constexpr int kTlBlock = 1024;                             // workgroup of the tiled pull

struct TileShape {
    uint32_t sb, db;            // source segment / destination block bits
    uint32_t ns, nd;            // segments, blocks
};

// cnt[d * ns + s] = light in-edges of destination block d from segment s.
template <class OffT>
__global__ __launch_bounds__(kBlock) void k_tl_count(const OffT* off, const uint32_t* src, uint64_t V,
                                                     uint32_t heavy_thr, TileShape ts, uint32_t* cnt) {
    __shared__ uint32_t h[kTlMaxSeg];
    const uint64_t d = blockIdx.x;
    for (uint32_t i = threadIdx.x; i < ts.ns; i += kBlock) h[i] = 0;
    __syncthreads();
    const uint64_t v0 = d << ts.db, v1 = min<uint64_t>(V, v0 + (1ull << ts.db));
    for (uint64_t v = v0 + threadIdx.x; v < v1; v += kBlock) {
        const OffT b = off[v], e = off[v + 1];
        if ((uint64_t)(e - b) >= heavy_thr) continue;
        for (OffT k = b; k < e; k++) atomicAdd(&h[src[k] >> ts.sb], 1u);
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < ts.ns; i += kBlock) cnt[d * ts.ns + i] = h[i];
}

// Writes the tile words of destination block d (positions within a tile in
// arrival order) and marks its heavy destinations in `heavy_bits`.
template <class OffT>
__global__ __launch_bounds__(kBlock) void k_tl_fill(const OffT* off, const uint32_t* src, uint64_t V,
                                                    uint32_t heavy_thr, TileShape ts,
                                                    const unsigned long long* toff, uint32_t* tiles,
                                                    uint32_t* heavy_bits) {
    __shared__ uint32_t cur[kTlMaxSeg];
    const uint64_t d = blockIdx.x;
    for (uint32_t i = threadIdx.x; i < ts.ns; i += kBlock) cur[i] = 0;
    __syncthreads();
    const uint64_t v0 = d << ts.db, v1 = min<uint64_t>(V, v0 + (1ull << ts.db));
    const unsigned long long* t = toff + d * ts.ns;
    const uint32_t smask = (1u << ts.sb) - 1;
    for (uint64_t v = v0 + threadIdx.x; v < v1; v += kBlock) {
        const OffT b = off[v], e = off[v + 1];
        if ((uint64_t)(e - b) >= heavy_thr) {
            atomicOr(&heavy_bits[v >> 5], 1u << (v & 31));
            continue;
        }
        const uint32_t dl = (uint32_t)(v - v0) << ts.sb;
        for (OffT k = b; k < e; k++) {
            const uint32_t u = src[k];
            const uint32_t s = u >> ts.sb;
            tiles[t[s] + atomicAdd(&cur[s], 1u)] = dl | (u & smask);
        }
    }
}

// Persistent: workgroup b takes destination blocks b, b + G, b + 2G, ...
// (G = gridDim.x).
// DB: the largest destination block (bits) its LDS sums hold; 2^14 blocks
// (64 KB) leave room for two workgroups per CU, 2^15 (128 KB) for one.
// Tiles are walked one by one (a flat walk across tile boundaries, each
// word's segment found by a binary search in LDS, measured 30% slower: the
// gathers of one pass then spread over several segments).  A tile is
// usually one pass (ER 2^26: ~512 words for 1024 lanes), so a pass is two
// dependent memory round trips (its words, then their gathers): the words of
// the next tile's first pass are loaded before the current tile's gathers,
// which leaves one round trip per tile.
template <int DB>
__global__ __launch_bounds__(kTlBlock) void k_pr_tiled(PrArgs a, const uint32_t* __restrict__ tiles,
                                                       const unsigned long long* __restrict__ toff, TileShape ts,
                                                       const uint32_t* heavy_bits) {
    __shared__ float acc[1u << DB];
    const uint32_t G = gridDim.x;
    const uint32_t nb = blockIdx.x < ts.nd ? (ts.nd - blockIdx.x + G - 1) / G : 0;   // blocks of this workgroup
    const uint32_t dsz = 1u << ts.db, smask = (1u << ts.sb) - 1;
    const double base = pr_base(a);
    PrSums sums;
    for (uint32_t r = 0; r < nb; r++) {
        const uint64_t d = blockIdx.x + (uint64_t)r * G;
        for (uint32_t i = threadIdx.x; i < dsz; i += kTlBlock) acc[i] = 0.0f;
        __syncthreads();
        const unsigned long long* t = toff + d * ts.ns;
        unsigned long long k0 = t[0], k1 = t[1];
        // first pass of a tile: four words per lane, lanes past its end load nothing
        uint32_t w[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const unsigned long long k = k0 + threadIdx.x + j * kTlBlock;
            w[j] = k < k1 ? tiles[k] : 0u;
        }
        for (uint32_t s = 0; s < ts.ns; s++) {
            const bool more = s + 1 < ts.ns;
            const unsigned long long k2 = more ? t[s + 2] : k1;
            uint32_t wn[4];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const unsigned long long k = k1 + threadIdx.x + j * kTlBlock;
                wn[j] = k < k2 ? tiles[k] : 0u;
            }
            const float* cseg = a.contrib_in + ((uint64_t)s << ts.sb);
            float c[4];
#pragma unroll
            for (int j = 0; j < 4; j++) c[j] = k0 + threadIdx.x + j * kTlBlock < k1 ? cseg[w[j] & smask] : 0.0f;
#pragma unroll
            for (int j = 0; j < 4; j++)
                if (k0 + threadIdx.x + j * kTlBlock < k1) atomicAdd(&acc[w[j] >> ts.sb], c[j]);
            // further passes of a tile longer than one: the words, then their
            // gathers, then the LDS adds (lanes past the end re-read its first word)
            for (unsigned long long k = k0 + threadIdx.x + 4 * kTlBlock; k < k1; k += 4 * kTlBlock) {
                uint32_t x[4];
#pragma unroll
                for (int j = 0; j < 4; j++) x[j] = tiles[k + j * kTlBlock < k1 ? k + j * kTlBlock : k0];
                float cx[4];
#pragma unroll
                for (int j = 0; j < 4; j++) cx[j] = cseg[x[j] & smask];
#pragma unroll
                for (int j = 0; j < 4; j++)
                    if (k + j * kTlBlock < k1) atomicAdd(&acc[x[j] >> ts.sb], cx[j]);
            }
#pragma unroll
            for (int j = 0; j < 4; j++) w[j] = wn[j];
            k0 = k1;
            k1 = k2;
        }
        __syncthreads();
        const uint64_t v0 = d << ts.db;
        for (uint32_t i = threadIdx.x; i < dsz; i += kTlBlock) {
            const uint64_t v = v0 + i;
            if (v >= a.V) break;
            if (heavy_bits && (heavy_bits[v >> 5] >> (v & 31) & 1u)) continue;
            pr_finish_vertex(a, v, (double)acc[i], base, sums);
        }
        __syncthreads();
    }
    acc_add<kTlBlock>(sums, a.acc_out);
}

// ---- reference mode --------------------------------------------------------

__global__ void k_prref_init(double* val, double* contrib, uint8_t* active, const uint32_t* outdeg, uint64_t V) {
    for (uint64_t v = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; v < V; v += (uint64_t)gridDim.x * blockDim.x) {
        const double r0 = 1.0 / (double)V;  // GraphMeta.cuh:418
        val[v] = r0;
        contrib[v] = outdeg[v] ? r0 / (double)outdeg[v] : 0.0;
        active[v] = 1;
    }
}

struct PrRefArgs {
    const void* off;              // OffT[V+1]
    const uint32_t* src;          // in-edges: edge k at src[k - e_base]
    unsigned long long e_base;
    unsigned long long v_begin, v_end;
    const double* contrib_in;
    double* contrib_out;
    double* val;
    uint8_t* active;
    const uint32_t* outdeg;
    uint32_t* count;              // vertices moved (kPrLines counters)
    double base, damping, threshold;
    RowPlan rows;                 // resident rows
};

// prKernel_Opt (gpu_kernels.cuh:533-552) for active vertex v with in-sum s; a
// vertex that stops keeps its value.  Its contribution is written for the
// next iteration either way, so both buffers hold it from then on.
__device__ __forceinline__ uint32_t prref_finish(const PrRefArgs& a, uint64_t v, double s) {
#pragma clang fp contract(off)
    const double t = a.base + a.damping * s;
    const double old = a.val[v];
    const double diff = t > old ? (t - old) : (old - t);
    const uint32_t d = a.outdeg[v];
    if (diff > a.threshold) {
        a.val[v] = t;
        a.contrib_out[v] = d ? t / (double)d : 0.0;
        return 1;
    }
    a.active[v] = 0;
    a.contrib_out[v] = a.contrib_in[v];
    return 0;
}

// What a stretch of a sequential FP64 sum adds to the running sum s while s
// stays in its binade, whose numbers are multiples of u: `a` if s is an even
// multiple, a + d * u if it is an odd one.  A term rounds to a whole number of
// units whatever s is, unless it lies halfway between two: then to the one that
// leaves s even.  All sums of units here are exact, and a sum that leaves the
// binade stays outside whatever is added (nothing added is negative).
struct Ordered {
    double a;
    int d;
    __device__ __forceinline__ double added(double s, double u) const {
        return __double_as_longlong(s) & 1 ? a + d * u : a;
    }
    // this stretch, then the next; base: the binade's first number, even
    __device__ __forceinline__ Ordered then(const Ordered& b, double base, double u) const {
        const double even = base + a, odd = base + u + (a + d * u);
        const double x = a + b.added(even, u), y = (a + d * u) + b.added(odd, u);
        return Ordered{x, y > x ? 1 : y < x ? -1 : 0};
    }
};

// A term c >= 0.
__device__ __forceinline__ Ordered ordered_term(double c, double base, double u) {
    const double r = (base + c) - base, e = c - r;
    return Ordered{r, fabs(e) == 0.5 * u ? (e > 0 ? 1 : -1) : 0};
}

constexpr int kOrdPer = 8;                       // terms a lane holds
constexpr uint32_t kOrdWave = kWave * kOrdPer;   // terms a wave holds
constexpr int kOrdBlock = kBlock;
static_assert(kBlock * kOrdPer <= kRowsTile, "the rows' LDS has room");

// The state of an ordered sum's binade.
struct Binade {
    double base, u, top;
    int e;
    __device__ __forceinline__ explicit Binade(double s) {
        e = (int)((unsigned long long)__double_as_longlong(s) >> 52);
        base = __longlong_as_double((long long)e << 52);
        u = __longlong_as_double((long long)max(e - 52, 0) << 52);
        top = base + base;
    }
    __device__ __forceinline__ bool tiny() const { return e < 64; }     // zero, or too small for units
    __device__ __forceinline__ bool huge() const { return e >= 2046; }  // next to infinity, or negative
};

// Inclusive sum over the wave by lane moves within the vector unit (__shfl_up
// goes through LDS, six times one after the other).
__device__ __forceinline__ double wave_scan_dpp(double x) {
#define ASC_STEP(ctrl, rows)                                                                                    \
    {                                                                                                           \
        const long long b = __double_as_longlong(x);                                                            \
        const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)b, ctrl, rows, 0xf, false);           \
        const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(b >> 32), ctrl, rows, 0xf, false);   \
        x += __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));                            \
    }
    ASC_STEP(0x111, 0xf)   // row_shr:1
    ASC_STEP(0x112, 0xf)
    ASC_STEP(0x114, 0xf)
    ASC_STEP(0x118, 0xf)
    ASC_STEP(0x142, 0xa)   // row_bcast:15
    ASC_STEP(0x143, 0xc)   // row_bcast:31
#undef ASC_STEP
    return x;
}

// The terms of the lanes from `skip` on, summed from the wave's first lane.
__device__ __forceinline__ Ordered ordered_scan(const double (&c)[kOrdPer], bool mine, const Binade& n) {
    Ordered x{0, 0};
    bool tie = false;
#pragma unroll
    for (int j = 0; j < kOrdPer; j++) {
        const Ordered t = ordered_term(c[j], n.base, n.u);
        x.a += t.a;
        tie |= t.d != 0;
    }
    if (!mine) {
        x.a = 0;
        tie = false;
    }
    if (!wave_ballot(tie)) {
        x.a = wave_scan_dpp(x.a);
        return x;
    }
    if (tie) {
        x = ordered_term(c[0], n.base, n.u);
#pragma unroll
        for (int j = 1; j < kOrdPer; j++) x = x.then(ordered_term(c[j], n.base, n.u), n.base, n.u);
    }
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
        const Ordered y{__shfl_up(x.a, d, kWave), __shfl_up(x.d, d, kWave)};
        if (lane_id() >= (uint32_t)d) x = y.then(x, n.base, n.u);
    }
    return x;
}

__device__ __forceinline__ double add_own(double s, const double (&c)[kOrdPer]) {
#pragma unroll
    for (int j = 0; j < kOrdPer; j++) s += c[j];
    return s;
}

__device__ __forceinline__ bool ordered_terms(const double (&c)[kOrdPer]) {
    bool ok = true;
#pragma unroll
    for (int j = 0; j < kOrdPer; j++) ok &= ((unsigned long long)__double_as_longlong(c[j]) >> 52) < 2047;
    return ok;   // neither negative, infinite nor NaN
}

// s + c[0] + c[1] + ... in this order, each sum rounded to FP64: lane t of the
// wave holds terms 8t to 8t + 7.  All lanes round their terms to units of s at
// once and a scan adds them; where the sum leaves its binade that lane adds
// its terms one by one, and the lanes behind it go on in the new units.
__device__ __forceinline__ double add_ordered_wave(double s, const double (&c)[kOrdPer]) {
    const uint32_t lane = lane_id();
    uint32_t skip = 0, small = 0;
    if (!wave_ballot(!ordered_terms(c))) {
        while (skip < (uint32_t)kWave) {
            const Binade n(s);
            if (n.huge()) break;
            if (n.tiny()) {
                // the first terms of a row, in which the sum doubles often, or zeros
                if (++small > 4) break;
                for (const uint32_t to = min(skip + 8, (uint32_t)kWave); skip < to; skip++)
                    s = __shfl(add_own(s, c), skip, kWave);
                continue;
            }
            const Ordered x = ordered_scan(c, lane >= skip, n);
            const double F = s + x.added(s, n.u);
            const uint64_t out = wave_ballot(F >= n.top);
            if (!out) return __shfl(F, kWave - 1, kWave);
            const uint32_t first = (uint32_t)__builtin_ctzll(out);
            const double before = __shfl_up(F, 1, kWave);
            s = __shfl(add_own(lane ? before : s, c), first, kWave);
            skip = first + 1;
        }
    }
    for (; skip < (uint32_t)kWave; skip++) s = __shfl(add_own(s, c), skip, kWave);
    return s;
}

struct OrderedLds {
    double a[2][kOrdBlock / kWave];
    int d[2][kOrdBlock / kWave];
    double s;
    uint32_t skip;
};

// The same over a workgroup of kOrdBlock lanes.
__device__ __forceinline__ double add_ordered_block(double s, const double (&c)[kOrdPer], OrderedLds& l,
                                                    uint32_t& round) {
    constexpr uint32_t W = kOrdBlock / kWave;
    const uint32_t tid = threadIdx.x, lane = lane_id(), w = wave_id();
    bool units = !__syncthreads_or(!ordered_terms(c));
    uint32_t skip = 0, small = 0;
    while (skip < (uint32_t)kOrdBlock) {
        const Binade n(s);
        units = units && !n.huge() && !(n.tiny() && ++small > 4);
        if (!units || n.tiny()) {   // eight lanes, one after the other
            const uint32_t to = min(skip + 8, (skip / kWave + 1) * kWave);
            __syncthreads();
            if (w == skip / kWave) {
                for (uint32_t i = skip; i < to; i++) s = __shfl(add_own(s, c), i % kWave, kWave);
                if (lane == 0) l.s = s;
            }
            __syncthreads();
            s = l.s;
            skip = to;
            continue;
        }
        const Ordered x = ordered_scan(c, tid >= skip, n);
        const uint32_t buf = round++ & 1;
        if (lane == kWave - 1) {
            l.a[buf][w] = x.a;
            l.d[buf][w] = x.d;
        }
        __syncthreads();
        double S = s, in = s;     // after the waves so far; before this wave
        uint32_t out = W;         // the wave in which the sum leaves its binade
#pragma unroll
        for (uint32_t i = 0; i < W; i++) {
            if (i == w) in = S;
            const double F = S + Ordered{l.a[buf][i], l.d[buf][i]}.added(S, n.u);
            if (F >= n.top) out = min(out, i);
            S = F;
        }
        if (out == W) return S;
        if (w == out) {
            const double F = in + x.added(in, n.u);
            const double before = __shfl_up(F, 1, kWave);
            const uint32_t first = (uint32_t)__builtin_ctzll(wave_ballot(F >= n.top));
            if (lane == first) {
                l.s = add_own(lane ? before : in, c);
                l.skip = tid + 1;
            }
        }
        __syncthreads();
        s = l.s;
        skip = l.skip;
    }
    return s;
}

// The in-sum of the row [b, e) by `waves` waves, this one the w-th.  While a
// tile is added (add(s, c)) the contributions of the next are gathered and the
// ids of the one after loaded.  Neighbouring lanes gather neighbouring edges
// (sources ascend along a row, so they share lines: with eight edges a lane
// R-MAT scale 20 took 461 us an iteration), and s_val, kOrdWave values of the
// wave's own, turns them into eight terms a lane.
template <class Add>
__device__ __forceinline__ double pull_ordered(const uint32_t* src, const double* contrib, uint64_t b, uint64_t e,
                                               uint32_t w, uint32_t waves, double* s_val, Add add) {
    const uint32_t lane = lane_id();
    const uint64_t tile = (uint64_t)waves * kOrdWave;
    uint32_t u[kOrdPer];
    double c0[kOrdPer], c1[kOrdPer];
    b += w * kOrdWave;   // (of this wave from here on)
    auto load_ids = [&](uint64_t t0) {
#pragma unroll
        for (int j = 0; j < kOrdPer; j++) u[j] = src[min(t0 + j * kWave + lane, e - 1)];
    };
    auto gather = [&](double (&c)[kOrdPer], uint64_t t0) {
#pragma unroll
        for (int j = 0; j < kOrdPer; j++) c[j] = t0 + j * kWave + lane < e ? contrib[u[j]] : 0.0;
    };
    auto turn = [&](double (&c)[kOrdPer]) {
#pragma unroll
        for (int j = 0; j < kOrdPer; j++) s_val[j * kWave + lane] = c[j];
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int j = 0; j < kOrdPer; j++) c[j] = s_val[lane * kOrdPer + j];
        __builtin_amdgcn_wave_barrier();
    };
    double s = 0;
    load_ids(b);
    gather(c0, b);
    load_ids(b + tile);
    for (uint64_t t0 = b;; t0 += 2 * tile) {
        gather(c1, t0 + tile);
        load_ids(t0 + 2 * tile);
        turn(c0);
        s = add(s, c0);
        if (t0 - w * kOrdWave + tile >= e) break;
        gather(c0, t0 + 2 * tile);
        load_ids(t0 + 3 * tile);
        turn(c1);
        s = add(s, c1);
        if (t0 - w * kOrdWave + 2 * tile >= e) break;
    }
    return s;
}

// One iteration over [v_begin, v_end): prSumKernel_static / _dynamic
// (gpu_kernels.cuh:554-594) and prKernel_Opt.  The result must equal a
// sequential FP64 sum in CSR order.  The first `hb` workgroups take the heavy
// rows with ordered sums, the longest first and a workgroup each, the others a
// wave each; the other workgroups run pull_block, where a lane adds a row.
// R-MAT scale 20 (31 M in-edges, longest row 64.6 k): 24.4 ms an iteration
// with one thread per row loading and adding edge by edge, 0.43 ms with one
// lane adding a heavy row out of LDS (6.6 ns an add), 0.29 ms this way, most
// of it the gathers of 8-byte contributions (8.4 MB, twice an XCD's L2).
// Launch bounds for more waves spill: 0.50 ms.
template <class OffT, bool HEAVY>
__global__ __launch_bounds__(kBlock) void k_prref_rows(PrRefArgs a, uint32_t hb) {
    __shared__ double s_val[kRowsTile];
    __shared__ uint32_t s_cnt[kWavesPerBlock];
    const OffT* off = (const OffT*)a.off;
    const uint32_t* src = a.src - a.e_base;
    const uint32_t tid = threadIdx.x;
    uint32_t moved = 0;
    if (HEAVY && blockIdx.x < hb) {
        // the longest rows, a workgroup each
        __shared__ OrderedLds s_ord;
        uint32_t round = 0;
        const uint32_t lb = min(a.rows.n_front, hb / 2);
        if (blockIdx.x < lb) {
            for (uint32_t i = blockIdx.x; i < a.rows.n_front; i += lb) {
                const uint32_t v = a.rows.front(i);
                if (!a.active[v]) continue;   // the same for the whole workgroup: only its own lane 0 clears it, below
                const double s = pull_ordered(src, a.contrib_in, off[v], off[v + 1], wave_id(), kWavesPerBlock,
                                              s_val + wave_id() * kOrdWave, [&](double s, const double (&c)[kOrdPer]) {
                                                  return add_ordered_block(s, c, s_ord, round);
                                              });
                if (tid == 0) moved += prref_finish(a, v, s);
            }
        }
        else for (uint32_t i = (blockIdx.x - lb) * kWavesPerBlock + wave_id(); i < a.rows.n_back; i += (hb - lb) * kWavesPerBlock) {
            const uint32_t v = a.rows.back(i);
            if (!a.active[v]) continue;   // the same for the whole wave: only its own lane 0 clears it, below
            const double s = pull_ordered(src, a.contrib_in, off[v], off[v + 1], 0, 1,
                                          s_val + wave_id() * kOrdWave,
                                          [](double s, const double (&c)[kOrdPer]) { return add_ordered_wave(s, c); });
            if (lane_id() == 0) moved += prref_finish(a, v, s);
        }
    } else {
        const uint32_t bid = blockIdx.x - (HEAVY ? hb : 0), nblk = gridDim.x - (HEAVY ? hb : 0);
        if (HEAVY) {
            auto pre = [&](uint64_t v) { return a.active[v] != 0; };
            auto fin = [&](uint64_t v, double s, bool act) {
                if (act) moved += prref_finish(a, v, s);
            };
            for (uint32_t i = bid; i < a.rows.n_blocks; i += nblk) {
                const RowBlock rb = a.rows.blocks[i];
                if (__syncthreads_or(tid < rb.n && a.active[rb.v + tid]))   // else every row has stopped
                    pull_block(off, src, a.contrib_in, rb, s_val, pre, fin);
            }
        } else {
            auto take = [&](uint64_t v) { return a.active[v] != 0; };
            auto fin = [&](uint64_t v, double s) { moved += prref_finish(a, v, s); };
            for (uint64_t v = a.v_begin + (uint64_t)bid * kBlock; v < a.v_end; v += (uint64_t)nblk * kBlock)
                pull_rows(off, src, a.contrib_in, v, a.v_end, s_val, take, fin);
        }
    }
    moved = wave_sum(moved);
    if (lane_id() == 0) s_cnt[wave_id()] = moved;
    __syncthreads();
    if (tid == 0) {
        uint32_t t = 0;
        for (int i = 0; i < kWavesPerBlock; i++) t += s_cnt[i];
        if (t) atomicAdd(a.count + (blockIdx.x % kPrLines) * kPrLineWords, t);
    }
}

// Sums and clears an iteration's counters and publishes the sum (one wave).
__global__ void k_prref_publish(uint32_t* count, PrRefPub* host, unsigned long long seq) {
    uint32_t n = 0;
    if (threadIdx.x < kPrLines) {
        n = count[threadIdx.x * kPrLineWords];
        count[threadIdx.x * kPrLineWords] = 0;
    }
    n = wave_sum(n);
    if (threadIdx.x == 0) {
        host_store(&host->moved, (unsigned long long)n);
        host_publish(&host->seq, seq);
    }
}

// ---- host -------------------------------------------------------------------

constexpr int kRefRing = 4;   // published iterations of the reference mode

// Lists the heavy rows of the resident vertices, once per graph.
template <class OffT>
static int pr_heavy_build(asc_graph* g, PrState* p) {
    if (p->heavy_built) return ASC_OK;
    const uint64_t n = g->static_vertices;
    const uint64_t cap = std::min<uint64_t>(n, g->static_edges / kRowsHeavy) + 1;
    hipStream_t s = g->ctx->s_main;
    DevTmp<uint32_t> d_cnt;
    uint32_t cnt[2] = {0, 0};
    if (!p->rows_heavy) ASC_HIP(hipMalloc(&p->rows_heavy, 4 * cap));
    ASC_HIP(hipMalloc(&d_cnt.p, sizeof(cnt)));
    ASC_HIP(hipMemsetAsync(d_cnt.p, 0, sizeof(cnt), s));
    if (n) {
        const int grid = (int)std::min<uint64_t>((n + kBlock - 1) / kBlock, (uint64_t)g->ctx->num_cus * 8);
        hipLaunchKernelGGL((k_rows_heavy_list<OffT>), dim3(grid), dim3(kBlock), 0, s, (const OffT*)g->d_off, n,
                           p->rows_heavy, (uint32_t)cap, d_cnt.p);
        ASC_HIP(hipGetLastError());
    }
    ASC_HIP(hipMemcpyAsync(cnt, d_cnt.p, sizeof(cnt), hipMemcpyDeviceToHost, s));
    ASC_HIP(hipStreamSynchronize(s));
    p->rows_cap = (uint32_t)cap;
    p->rows_front = cnt[0];
    p->rows_back = cnt[1];
    p->heavy_built = true;
    return ASC_OK;
}

// Cuts the resident vertices into row blocks too, once per graph.
template <class OffT>
static int pr_rows_build(asc_graph* g, PrState* p) {
    ASC_TRY(pr_heavy_build<OffT>(g, p));
    if (p->rows_built) return ASC_OK;
    const uint64_t n = g->static_vertices;
    const uint64_t bcap = std::min<uint64_t>(n, (n + kBlock - 1) / kBlock + g->static_edges / kRowsWindow +
                                                    p->rows_cap) + 1;
    hipStream_t s = g->ctx->s_main;
    DevTmp<uint32_t> d_cnt;
    uint32_t cnt = 0;
    if (!p->rows_blocks) ASC_HIP(hipMalloc(&p->rows_blocks, sizeof(RowBlock) * bcap));
    ASC_HIP(hipMalloc(&d_cnt.p, sizeof(cnt)));
    ASC_HIP(hipMemsetAsync(d_cnt.p, 0, sizeof(cnt), s));
    if (n) {
        const int grid = (int)std::min<uint64_t>((n + kBlock - 1) / kBlock, (uint64_t)g->ctx->num_cus * 8);
        hipLaunchKernelGGL((k_row_blocks<OffT>), dim3(grid), dim3(kBlock), 0, s, (const OffT*)g->d_off, n,
                           (RowBlock*)p->rows_blocks, d_cnt.p);
        ASC_HIP(hipGetLastError());
    }
    ASC_HIP(hipMemcpyAsync(&cnt, d_cnt.p, sizeof(cnt), hipMemcpyDeviceToHost, s));
    ASC_HIP(hipStreamSynchronize(s));
    p->rows_n = cnt;
    p->rows_built = true;
    return ASC_OK;
}

static RowPlan row_plan(const PrState* p) {
    return RowPlan{(const RowBlock*)p->rows_blocks, p->rows_heavy, p->rows_n, p->rows_cap, p->rows_front,
                   p->rows_back};
}

static int pr_ensure(asc_graph* g, int iters, bool ref) {
    PrState* p = g->pr;
    const uint64_t V = g->h.V;
    if (!p || p->V != V) {
        if (p) pr_free(p);
        p = new PrState();
        g->pr = p;
        p->V = V;
    }
    ASC_HIP(hipSetDevice(g->ctx->device));
    if (!ref && !p->rank[0]) {
        for (int i = 0; i < 2; i++) {
            ASC_HIP(hipMalloc(&p->rank[i], 4 * V));
            ASC_HIP(hipMalloc(&p->contrib[i], 4 * V));
        }
    }
    for (int i = 0; i < 2; i++)
        if (!p->ev[i]) ASC_HIP(hipEventCreate(&p->ev[i]));
    if (!ref && !p->acc) ASC_HIP(hipMalloc(&p->acc, sizeof(double) * kAccSlots * kAccSlot));
    if (!ref && p->resid_iters < iters) {
        if (p->resid) (void)hipFree(p->resid);
        p->resid = nullptr;
        p->resid_iters = 0;
        ASC_HIP(hipMalloc(&p->resid, sizeof(double) * (size_t)iters));
        ASC_TRY(p->h_resid.alloc((size_t)iters + 1, true));
        std::memset((void*)p->h_resid.p, 0, sizeof(double) * ((size_t)iters + 1));
        ASC_HIP(hipHostGetDevicePointer((void**)&p->d_hresid, p->h_resid.p, 0));
        p->resid_iters = iters;
    }
    if (ref && !p->val64) {
        ASC_HIP(hipMalloc(&p->contrib64[0], 8 * V));
        ASC_HIP(hipMalloc(&p->contrib64[1], 8 * V));
        ASC_HIP(hipMalloc(&p->active, V));
        ASC_HIP(hipMalloc(&p->count, 4 * kPrLines * kPrLineWords));
        ASC_TRY(p->h_refpub.alloc(kRefRing, true));
        ASC_HIP(hipHostGetDevicePointer((void**)&p->d_refpub, p->h_refpub.p, 0));
        for (int i = 0; i < kRefRing; i++) p->h_refpub[i].seq = 0;
        ASC_HIP(hipMalloc(&p->val64, 8 * V));   // last: set once all of the above are
    }
    return pr_plan_chunks(g, p);
}

// One pull over [a.v_begin, a.v_end): the row kernel (with its heavy rows when
// a.skip_heavy), or k_pr_pull with the G lanes per vertex asked for.
// Measured on R-MAT scale 18 (7.6 M in-edges): the row kernel 40 us an
// iteration; 16 lanes a vertex, heavy rows from 4096 edges on, 283 us (a group
// walks up to 4095 edges, and the heavy kernel held one gather in flight).
// What is left is mostly the 128-byte L2 line that every 4-byte gather brings
// into L1: 64 bytes a clock per CU make 7.6 M of them 25 us.
template <class OffT>
static int launch_pull(int G, int num_cus, hipStream_t s, const PrArgs& a, const PrState* p) {
    const uint64_t n = a.v_end - a.v_begin;
    const uint32_t cap = (uint32_t)num_cus * 8;
    if (G == 0) {
        if (a.skip_heavy) {
            const uint32_t hb = std::min<uint32_t>(p->rows_front + (p->rows_back + kWavesPerBlock - 1) / kWavesPerBlock,
                                                   cap / 2);
            hipLaunchKernelGGL((k_pr_rows<OffT, true>), dim3(hb + std::min(p->rows_n, cap)), dim3(kBlock), 0, s, a,
                               row_plan(p), hb);
        } else {
            const uint32_t rb = (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>((n + kBlock - 1) / kBlock, cap));
            hipLaunchKernelGGL((k_pr_rows<OffT, false>), dim3(rb), dim3(kBlock), 0, s, a, RowPlan{}, 0u);
        }
        ASC_HIP(hipGetLastError());
        return ASC_OK;
    }
    const uint32_t grid = (uint32_t)std::min<uint64_t>(cap, (n * G + kBlock - 1) / kBlock + 1);
    switch (G) {
        case 4: hipLaunchKernelGGL((k_pr_pull<4, OffT>), dim3(grid), dim3(kBlock), 0, s, a); break;
        case 8: hipLaunchKernelGGL((k_pr_pull<8, OffT>), dim3(grid), dim3(kBlock), 0, s, a); break;
        case 16: hipLaunchKernelGGL((k_pr_pull<16, OffT>), dim3(grid), dim3(kBlock), 0, s, a); break;
        case 32: hipLaunchKernelGGL((k_pr_pull<32, OffT>), dim3(grid), dim3(kBlock), 0, s, a); break;
        default: hipLaunchKernelGGL((k_pr_pull<64, OffT>), dim3(grid), dim3(kBlock), 0, s, a); break;
    }
    ASC_HIP(hipGetLastError());
    return ASC_OK;
}

// ASC_PR_BLOCKED asked for by name refuses out-degrees that do not sum to E.
static int pr_check_outdeg(const asc_graph* g, PrState* p) {
    if (p->outdeg_sums) return ASC_OK;
    std::atomic<uint64_t> sum{0};
    host_pool().parallel_for(g->h.V, [&](uint64_t b, uint64_t e) {
        uint64_t x = 0;
        for (uint64_t u = b; u < e; u++) x += g->h.outdeg[u];
        sum += x;
    });
    if (sum != g->h.E) {
        set_last_error("out-degrees sum to %llu, not E = %llu", (unsigned long long)sum.load(),
                       (unsigned long long)g->h.E);
        return ASC_ERR_FORMAT;
    }
    p->outdeg_sums = true;
    return ASC_OK;
}

// Smallest graph of the blocked schedule under ASC_PR_AUTO.
// Below, the row blocks' gathers come out of the L2s and two launches an
// iteration on few workgroups cost more (ms of 20 iterations, blocked / row
// blocks: R-MAT scale 18, 7.6e6 edges 0.91 / 0.80, Erdos-Renyi V = 2^18, 8.4e6
// edges 0.66 / 1.07, V = 2^17, 1.7e7 edges 0.85 / 1.82).  Between the first two
// points lies the line on edges, but they differ in skew more than in edges:
// on a skewed graph just above it the row blocks may still be the faster, on
// an even one just below it the blocked schedule, by what the points show.
// From V = 2^20 on the blocked schedule is taken however few the edges (V =
// 2^20, 4.2e6 edges: Erdos-Renyi 0.53 / 0.96, R-MAT 0.86 / 0.79).
constexpr uint64_t kPbMinV = uint64_t(1) << 17, kPbMinE = uint64_t(1) << 23;

// Shape of the propagation-blocked layout: 2^14 sources a slice and 2^13
// destinations a bin: 64 KB of LDS each, two workgroups a CU (V = 2^23, 2^28
// edges: 14.7 ms for 20 iterations, also with 2^15 sources, 15.0 with 2^14
// destinations; R-MAT scale 20: 2.20, 2.26, 2.57).  Larger ones where runs
// would be shorter than 64 edges; AUTO leaves graphs with less than 16 a run
// to the tiled pull, also where the layout was built by name.
struct PbShape {
    uint32_t bits = 14, dbits = 13;
    uint64_t most;                // edges of a bin
    bool long_runs;               // 16 edges a run and more
    PbShape(uint64_t V, uint64_t E, uint32_t cus) {
        most = std::max<uint64_t>(1u << 16, E / (8 * (uint64_t)cus));
        auto runs = [&] { return ((V >> bits) + 1) * (std::max(V >> dbits, E / most) + 1); };
        if (E / 64 < runs()) bits = 15;
        if (E / 64 < runs()) dbits = 14;
        long_runs = E / 16 >= runs();
    }
};

// Builds the propagation-blocked layout once (every edge resident, at most
// kPbMaxSlices slices, fewer than 2^31 octs, its arrays within free device
// memory); pb_state = -1 when it cannot be built.
template <class OffT>
static int pr_blocked_build(asc_graph* g, PrState* p, const PbShape& shape) {
    if (p->pb_state != 0) return ASC_OK;
    const uint64_t V = g->h.V, E = g->h.E;
    const uint32_t cus = (uint32_t)g->ctx->num_cus;
    const uint64_t most = shape.most;
    const uint32_t bits = shape.bits, dbits = shape.dbits;
    p->pb_state = -1;
    const uint64_t ns = (V + (1ull << bits) - 1) >> bits;
    if (g->static_vertices != V || E == 0 || E >= 0xFFFFFFFFull || V > (uint64_t(1) << 28) || ns > kPbMaxSlices)
        return ASC_OK;
    hipStream_t s = g->ctx->s_main;
    const OffT* off = (const OffT*)g->d_off;
    const uint32_t* src = (const uint32_t*)g->d_edges;
    // rows left to the pull, in order
    std::vector<uint32_t> heavy(p->rows_front);
    if (p->rows_front) {
        ASC_HIP(hipMemcpyAsync(heavy.data(), p->rows_heavy, 4 * heavy.size(), hipMemcpyDeviceToHost, s));
        ASC_HIP(hipStreamSynchronize(s));
    }
    std::sort(heavy.begin(), heavy.end());
    const uint64_t* ho = g->h.off.p;
    std::vector<PbBin> bins;
    for (uint32_t v : heavy) bins.push_back({v, 1, 0, 0, kPbHeavy});
    size_t nh = 0;
    for (uint64_t v = 0; v < V;) {
        const uint64_t lim = std::min<uint64_t>(V, v + (1ull << dbits));
        uint64_t left = most, at = v;   // (a row that is not heavy always fits an empty bin)
        uint32_t kind = kPbPlain;
        while (at < lim) {
            if (nh < heavy.size() && heavy[nh] == at) {
                kind = kPbAround;
                nh++;
                at++;
                continue;
            }
            const uint64_t seg = nh < heavy.size() ? std::min<uint64_t>(lim, heavy[nh]) : lim;
            const uint64_t* e = std::upper_bound(ho + at + 1, ho + seg + 1, ho[at] + left);
            const uint64_t v1 = (uint64_t)(e - ho) - 1;
            left -= ho[v1] - ho[at];
            at = v1;
            if (at < seg) break;
        }
        bins.push_back({(uint32_t)v, (uint32_t)(at - v), 0, 0, kind});
        v = at;
    }
    const uint64_t nb = bins.size();
    size_t free_b = 0, total_b = 0;
    ASC_HIP(hipMemGetInfo(&free_b, &total_b));
    const uint64_t padded = E + (kPbOct - 1) * nb * ns;
    if (nb == 0 || padded / kPbOct >= (uint64_t(1) << 31) || 9 * padded + 16 * nb * ns + (uint64_t(1) << 30) > free_b) return ASC_OK;
    DevTmp<uint32_t> d_cnt;
    ASC_HIP(hipMalloc(&d_cnt.p, 4 * nb * ns));
    ASC_HIP(hipMalloc(&p->pb_bins, sizeof(PbBin) * nb));
    ASC_HIP(hipMemcpyAsync(p->pb_bins, bins.data(), sizeof(PbBin) * nb, hipMemcpyHostToDevice, s));
    hipLaunchKernelGGL((k_pb_count<OffT>), dim3((uint32_t)nb), dim3(kPbBlock), 0, s, off, src,
                       (const PbBin*)p->pb_bins, (uint32_t)ns, bits, d_cnt.p);
    ASC_HIP(hipGetLastError());
    DevTmp<uint32_t> d_first;   // octs of the slices, then of the bins; then where they begin
    ASC_HIP(hipMalloc(&d_first.p, 4 * (ns + nb)));
    hipLaunchKernelGGL(k_pb_totals<true>, dim3((uint32_t)ns), dim3(kBlock), 0, s, d_cnt.p, (uint32_t)nb, (uint32_t)ns,
                       d_first.p);
    hipLaunchKernelGGL(k_pb_totals<false>, dim3((uint32_t)nb), dim3(kBlock), 0, s, d_cnt.p, (uint32_t)nb, (uint32_t)ns,
                       d_first.p + ns);
    ASC_HIP(hipGetLastError());
    std::vector<uint32_t> first(ns + nb);
    ASC_HIP(hipMemcpyAsync(first.data(), d_first.p, 4 * first.size(), hipMemcpyDeviceToHost, s));
    ASC_HIP(hipStreamSynchronize(s));
    // slice order: a slice's runs one after the other, bin by bin
    uint64_t octs = 0;
    for (uint64_t i = 0; i < ns; i++) octs += first[i];
    const uint64_t per = std::min<uint64_t>(kPbItemOcts, std::max<uint64_t>(octs / (2 * (uint64_t)cus), 1u << 11));
    std::vector<PbItem> items;
    uint32_t at = 0;
    for (uint64_t i = 0; i < ns; i++) {
        const uint32_t end = at + first[i];
        first[i] = at;
        for (uint64_t q = at; q < end; q += per)
            items.push_back({(uint32_t)i, (uint32_t)q, (uint32_t)std::min<uint64_t>(end, q + per)});
        at = end;
    }
    at = 0;
    for (uint64_t b = 0; b < nb; b++) {
        bins[b].o = at;
        bins[b].octs = first[ns + b];
        first[ns + b] = at;
        at += bins[b].octs;
    }
    const uint64_t q1 = std::max<uint64_t>(octs, 1);
    DevTmp<PbRun> d_runs;
    ASC_HIP(hipMalloc(&d_runs.p, sizeof(PbRun) * nb * ns));
    ASC_HIP(hipMemcpyAsync(d_first.p, first.data(), 4 * first.size(), hipMemcpyHostToDevice, s));
    ASC_HIP(hipMemcpyAsync(p->pb_bins, bins.data(), sizeof(PbBin) * nb, hipMemcpyHostToDevice, s));
    hipLaunchKernelGGL(k_pb_place<true>, dim3((uint32_t)ns), dim3(kBlock), 0, s, d_cnt.p, (uint32_t)nb, (uint32_t)ns,
                       d_first.p, d_runs.p);
    hipLaunchKernelGGL(k_pb_place<false>, dim3((uint32_t)nb), dim3(kBlock), 0, s, d_cnt.p, (uint32_t)nb, (uint32_t)ns,
                       d_first.p + ns, d_runs.p);
    ASC_HIP(hipGetLastError());
    ASC_HIP(hipMalloc(&p->pb_items, sizeof(PbItem) * std::max<size_t>(items.size(), 1)));
    if (!items.empty())
        ASC_HIP(hipMemcpyAsync(p->pb_items, items.data(), sizeof(PbItem) * items.size(), hipMemcpyHostToDevice, s));
    ASC_HIP(hipMalloc(&p->pb_src, sizeof(PbIds) * q1));
    ASC_HIP(hipMalloc(&p->pb_dst, sizeof(PbIds) * q1));
    ASC_HIP(hipMalloc(&p->pb_pos, 4 * q1));
    ASC_HIP(hipMalloc(&p->pb_vals, 4 * kPbOct * q1));
    // the padding's places: source 0 of the slice, the sum past the bin's.  The
    // ids are written in pairs first (the values' array holds them meanwhile):
    // two arrays of scattered 2-byte writes took twice as long
    hipLaunchKernelGGL(k_pr_fill, dim3(cus * 8), dim3(256), 0, s, (uint32_t*)p->pb_vals, kPbOct * q1,
                       1u << (dbits + 16));
    hipLaunchKernelGGL((k_pb_fill<OffT>), dim3((uint32_t)nb), dim3(kPbBlock), 0, s, off, src,
                       (const PbBin*)p->pb_bins, d_runs.p, (uint32_t)ns, bits, (uint32_t*)p->pb_vals);
    hipLaunchKernelGGL(k_pb_unzip, dim3((uint32_t)nb), dim3(kPbBlock), 0, s, d_runs.p, (uint32_t)ns,
                       (const uint4*)p->pb_vals, (PbIds*)p->pb_src, (PbIds*)p->pb_dst, p->pb_pos);
    ASC_HIP(hipGetLastError());
    ASC_HIP(hipStreamSynchronize(s));   // the host arrays above are read until here
    p->pb_sbits = bits;
    p->pb_dbits = dbits;
    p->pb_nbins = (uint32_t)nb;
    p->pb_nitems = (uint32_t)items.size();
    p->pb_state = 1;
    return ASC_OK;
}

template <class OffT, int SB, int DB>
static int launch_blocked(const PrArgs& a, const PrState* p, hipStream_t s) {
    if (p->pb_nitems)
        hipLaunchKernelGGL(k_pb_scatter<SB>, dim3((p->pb_nitems + 7) / 8 * 8), dim3(kPbBlock), 0, s, a.contrib_in,
                           a.V, (const PbItem*)p->pb_items, p->pb_nitems, (const ushort4*)p->pb_src,
                           (float4*)p->pb_vals);
    hipLaunchKernelGGL((k_pb_gather<OffT, DB>), dim3(p->pb_nbins), dim3(kPbBlock), 0, s, a, (const PbBin*)p->pb_bins,
                       p->pb_pos, (const ushort4*)p->pb_dst, (const float4*)p->pb_vals);
    ASC_HIP(hipGetLastError());
    return ASC_OK;
}

// Builds the tiles of the source-segmented mode for segments of 2^sb and
// blocks of 2^db vertices (every edge resident, at most kTlMaxSeg segments,
// sb + db <= 32, tile words within free device memory); rebuilt when the
// shape changes.  tl_state = -1 when they cannot be built.
template <class OffT>
static int pr_tiled_build(asc_graph* g, PrState* p, uint32_t sb, uint32_t db) {
    if (p->tl_state == 1 && p->tl_sb == sb && p->tl_db == db) return ASC_OK;
    auto f = [](void* x) {
        if (x) (void)hipFree(x);
    };
    f(p->tl_edges); f(p->tl_off); f(p->tl_heavy);
    p->tl_edges = nullptr;
    p->tl_off = nullptr;
    p->tl_heavy = nullptr;
    p->tl_state = -1;
    const uint64_t V = g->h.V, E = g->h.E;
    if (db < 6 || db > (uint32_t)kTlMaxDstBits || sb < 8 || sb + db > 32) return ASC_OK;
    const uint64_t ns = (V + (1ull << sb) - 1) >> sb, nd = (V + (1ull << db) - 1) >> db;
    if (g->static_vertices != V || E == 0 || ns > kTlMaxSeg || nd > 0xFFFFFFFFull) return ASC_OK;
    size_t free_b = 0, total_b = 0;
    ASC_HIP(hipMemGetInfo(&free_b, &total_b));
    const uint64_t need = 4 * E + 12 * nd * ns + 8 + (V + 31) / 32 * 4;
    if (need + (uint64_t(1) << 30) > free_b) return ASC_OK;
    hipStream_t s = g->ctx->s_main;
    const OffT* off = (const OffT*)g->d_off;
    const uint32_t* src = (const uint32_t*)g->d_edges;
    const uint32_t thr = kRowsLong;
    const TileShape ts{sb, db, (uint32_t)ns, (uint32_t)nd};
    DevTmp<uint32_t> d_cnt;
    ASC_HIP(hipMalloc(&d_cnt.p, 4 * nd * ns));
    hipLaunchKernelGGL((k_tl_count<OffT>), dim3((uint32_t)nd), dim3(kBlock), 0, s, off, src, V, thr, ts, d_cnt.p);
    ASC_HIP(hipGetLastError());
    std::vector<uint32_t> cnt(nd * ns);
    ASC_HIP(hipMemcpyAsync(cnt.data(), d_cnt.p, 4 * cnt.size(), hipMemcpyDeviceToHost, s));
    ASC_HIP(hipStreamSynchronize(s));
    std::vector<unsigned long long> toff(nd * ns + 1);
    unsigned long long acc = 0;
    for (size_t i = 0; i < cnt.size(); i++) {
        toff[i] = acc;
        acc += cnt[i];
    }
    toff[cnt.size()] = acc;
    ASC_HIP(hipMalloc(&p->tl_off, 8 * toff.size()));
    ASC_HIP(hipMemcpy(p->tl_off, toff.data(), 8 * toff.size(), hipMemcpyHostToDevice));
    ASC_HIP(hipMalloc(&p->tl_edges, 4 * std::max<unsigned long long>(acc, 1)));
    ASC_HIP(hipMalloc(&p->tl_heavy, 4 * ((V + 31) / 32)));
    ASC_HIP(hipMemsetAsync(p->tl_heavy, 0, 4 * ((V + 31) / 32), s));
    hipLaunchKernelGGL((k_tl_fill<OffT>), dim3((uint32_t)nd), dim3(kBlock), 0, s, off, src, V, thr, ts,
                       (const unsigned long long*)p->tl_off, p->tl_edges, p->tl_heavy);
    ASC_HIP(hipGetLastError());
    ASC_HIP(hipStreamSynchronize(s));
    p->tl_sb = sb;
    p->tl_db = db;
    p->tl_nd = (uint32_t)nd;
    p->tl_ns = (uint32_t)ns;
    p->tl_edges_n = acc;
    p->tl_state = 1;
    return ASC_OK;
}

template <class OffT>
static int pr_normalised(asc_graph* g, const asc_pr_opts* o, float* rank_out, double* residual_out, asc_stats* st) {
    asc_ctx* ctx = g->ctx;
    const int iters = o->iterations > 0 ? o->iterations : 20;
    ASC_TRY(pr_ensure(g, iters, false));
    PrState* p = g->pr;
    const uint64_t V = g->h.V;
    hipStream_t s = ctx->s_main;
    const int grid = ctx->num_cus * 8;
    ASC_TRY(pr_heavy_build<OffT>(g, p));
    auto slot = [&](int it) { return p->acc + (size_t)(it % kAccSlots) * kAccSlot; };
    ASC_HIP(hipMemsetAsync(p->acc, 0, sizeof(double) * kAccSlots * kAccSlot, s));
    hipLaunchKernelGGL(k_pr_init, dim3(std::max<uint64_t>(1, std::min<uint64_t>((V + kBlock - 1) / kBlock, (uint64_t)grid))), dim3(kBlock), 0,
                       s, p->rank[0], p->contrib[0], g->d_outdeg, V, slot(0));
    ASC_HIP(hipGetLastError());
    const int G = g->pr_group > 0 ? g->pr_group : 0;
    const bool by_name = o->method == ASC_PR_BLOCKED;
    const bool big = o->method == ASC_PR_AUTO && g->static_vertices == V && V >= (uint64_t(1) << 20);
    const PbShape shape(V, g->h.E, (uint32_t)ctx->num_cus);
    const bool blocks =
        by_name || (shape.long_runs &&
                    (big || (o->method == ASC_PR_AUTO && !G && V >= kPbMinV && g->h.E >= kPbMinE)));
    if (blocks) ASC_TRY(pr_blocked_build<OffT>(g, p, shape));
    const bool blocked = blocks && p->pb_state == 1;
    if (o->method == ASC_PR_BLOCKED && !blocked) {
        set_last_error("propagation-blocked PageRank needs every edge resident, E < 2^32 and room for its slots");
        return ASC_ERR_UNSUPPORTED;
    }
    if (o->method == ASC_PR_BLOCKED) ASC_TRY(pr_check_outdeg(g, p));
    // tile shape: 2^15-vertex segments (128 KB contribution slices) measured
    // fastest on Erdos-Renyi 2^26 / 2^31 edges (20 iterations: 496 ms with
    // 2^14-vertex blocks against 557-833 ms for 2^14 or 2^16-2^20-vertex
    // segments, and 821 ms for the pull); 2^15-vertex blocks (one workgroup
    // per CU, 128 KB of LDS sums, tiles twice as long) 468 ms, taken once
    // there are at least four blocks per CU; the graph's tuned shape or the
    // caller's wins
    const uint32_t sb = o->tile_src_bits > 0 ? (uint32_t)o->tile_src_bits
                        : g->pr_tile_src_bits > 0 ? (uint32_t)g->pr_tile_src_bits : 15;
    const uint32_t db_auto = (V >> 15) >= 4 * (uint64_t)ctx->num_cus ? 15u : 14u;
    const uint32_t db = o->tile_dst_bits > 0 ? (uint32_t)o->tile_dst_bits
                        : g->pr_tile_dst_bits > 0 ? (uint32_t)g->pr_tile_dst_bits : db_auto;
    // AUTO: the tiled pull where the blocked layout cannot be built or its
    // runs would be short, as on every large graph before there was that
    // layout.  On R-MAT graphs the row blocks are faster than the tiles (the
    // table above kPbBlock); no graph of that kind was measured this sparse.
    const bool want_tiled = o->method == ASC_PR_TILED || (big && !blocked);
    if (want_tiled) ASC_TRY(pr_tiled_build<OffT>(g, p, sb, db));
    const bool tiled = want_tiled && p->tl_state == 1;
    if (o->method == ASC_PR_TILED && !tiled) {
        set_last_error("source-segmented PageRank needs every edge resident, V <= 2^31 and room for its tiles");
        return ASC_ERR_UNSUPPORTED;
    }
    g->pr_schedule = tiled ? ASC_PR_TILED : blocked ? ASC_PR_BLOCKED : ASC_PR_PULL;
    if (!tiled && !blocked && !G) ASC_TRY(pr_rows_build<OffT>(g, p));
    const double t0 = now_ms();
    ASC_HIP(hipEventRecord(p->ev[0], s));
    for (int it = 0; it < iters; it++) {
        PrArgs a{};
        a.off = g->d_off;
        a.src = (const uint32_t*)g->d_edges;
        a.outdeg = g->d_outdeg;
        a.rank_in = p->rank[it & 1];
        a.contrib_in = p->contrib[it & 1];
        a.rank_out = p->rank[(it + 1) & 1];
        a.contrib_out = p->contrib[(it + 1) & 1];
        a.acc_in = slot(it);
        a.acc_out = slot(it + 1);
        // only the iteration's first launch: `led` takes these off for the others
        a.acc_clear = slot(it + 2);
        a.resid_prev = it ? p->resid + it - 1 : nullptr;
        auto led = [&] {
            a.acc_clear = nullptr;
            a.resid_prev = nullptr;
        };
        a.V = V;
        a.damping = (float)o->damping;
        a.damping64 = o->damping;
        a.heavy_thr = kRowsLong;
        // resident vertices from the device edges, heavy in-lists by workgroups
        a.e_base = 0;
        a.v_begin = 0;
        a.v_end = g->static_vertices;
        a.skip_heavy = 1;
        if (tiled) {
            const TileShape ts{p->tl_sb, p->tl_db, p->tl_ns, p->tl_nd};
            // 1024-lane workgroups: two per CU with blocks up to 2^14
            // destinations (64 KB of LDS each), one with 2^15 (128 KB)
            const bool big = p->tl_db > 14;
            const uint32_t tgrid = (uint32_t)std::min<uint64_t>((uint64_t)ctx->num_cus * (big ? 1 : 2), p->tl_nd);
            const uint32_t* hb = p->rows_front ? (const uint32_t*)p->tl_heavy : nullptr;
            if (big)
                hipLaunchKernelGGL(k_pr_tiled<15>, dim3(tgrid), dim3(kTlBlock), 0, s, a,
                                   (const uint32_t*)p->tl_edges, (const unsigned long long*)p->tl_off, ts, hb);
            else
                hipLaunchKernelGGL(k_pr_tiled<14>, dim3(tgrid), dim3(kTlBlock), 0, s, a,
                                   (const uint32_t*)p->tl_edges, (const unsigned long long*)p->tl_off, ts, hb);
            ASC_HIP(hipGetLastError());
            led();
        } else if (blocked) {
            if (p->pb_dbits == 14) ASC_TRY((launch_blocked<OffT, 15, 14>(a, p, s)));
            else if (p->pb_sbits == 15) ASC_TRY((launch_blocked<OffT, 15, 13>(a, p, s)));
            else ASC_TRY((launch_blocked<OffT, 14, 13>(a, p, s)));
            led();
        } else if (a.v_end > 0) {
            ASC_TRY(launch_pull<OffT>(G, ctx->num_cus, s, a, p));
            led();
        }
        // rows of kRowsLong edges and more (the row kernel takes them itself)
        if (p->rows_front && (tiled || (G && !blocked))) {
            hipLaunchKernelGGL((k_pr_pull_heavy<OffT>), dim3(std::min<uint32_t>(p->rows_front, grid)), dim3(kBlock), 0,
                               s, a, p->rows_heavy, p->rows_front);
            ASC_HIP(hipGetLastError());
        }
        // on-demand vertices from streamed chunks
        ASC_TRY(pr_stream_chunks(g, p, [&](const uint32_t* src, uint64_t e0, uint64_t v0, uint64_t v1) {
            PrArgs c = a;
            c.src = src;
            c.e_base = e0;
            c.v_begin = v0;
            c.v_end = v1;
            c.skip_heavy = 0;
            led();
            return launch_pull<OffT>(G, ctx->num_cus, s, c, p);
        }));
    }
    ASC_HIP(hipEventRecord(p->ev[1], s));
    // the host copies hold `iters` residuals and the sequence number right
    // behind them, whatever their capacity
    volatile unsigned long long* seq = (volatile unsigned long long*)(p->h_resid.p + iters);
    *seq = 0;
    const unsigned long long want = ++p->resid_seq;
    hipLaunchKernelGGL(k_pr_residuals, dim3(1), dim3(kWave), 0, s, (const double*)slot(iters), p->resid, iters,
                       p->d_hresid, want);
    ASC_HIP(hipGetLastError());
    ASC_TRY(wait_host_seq(seq, want, s));
    const double t1 = now_ms();
    const double* hres = p->h_resid.p;
    if (residual_out) std::memcpy(residual_out, hres, sizeof(double) * iters);
    if (rank_out) ASC_TRY(out_copy(p->out, (const uint32_t*)p->rank[iters & 1], V, (uint32_t*)rank_out, s));
    float kms = 0;
    if (hipEventElapsedTime(&kms, p->ev[0], p->ev[1]) != hipSuccess) {   // not yet seen by the runtime
        (void)hipGetLastError();
        ASC_HIP(hipEventSynchronize(p->ev[1]));
        (void)hipEventElapsedTime(&kms, p->ev[0], p->ev[1]);
    }
    if (st) {
        std::memset(st, 0, sizeof(*st));
        st->total_ms = t1 - t0;
        st->static_ms = kms;
        st->kernel_ms = kms;
        st->iterations = (uint32_t)iters;
        st->node_sum = V * (uint64_t)iters;
        st->edges_traversed = g->h.E * (uint64_t)iters;
        st->static_edges_traversed = st->edges_traversed;
        st->vertices_processed = V * (uint64_t)iters;
        st->reached = V;
        st->reached_degree_sum = g->h.E;
        st->pr_residual = hres[iters - 1];
        st->host_cores = hardware_threads();
        st->streamed_edges = p->streamed_edges * (uint64_t)iters;
        st->streamed_bytes = 4 * st->streamed_edges;
        st->kern[KERN_PART].record_bytes = p->chunks.empty() ? 0 : 4;
        st->parts = (uint32_t)(p->chunks.size() * (size_t)iters);
        st->kern[3].launches = (uint32_t)iters;
        st->kern[3].ms = kms;
        st->kern[3].edges = g->h.E * (uint64_t)iters;
        st->kern[3].vertices = V * (uint64_t)iters;
    }
    return ASC_OK;
}

template <class OffT>
static int pr_reference(asc_graph* g, const asc_pr_opts* o, double* rank_out, asc_stats* st) {
    asc_ctx* ctx = g->ctx;
    ASC_TRY(pr_ensure(g, 0, true));
    PrState* p = g->pr;
    const uint64_t V = g->h.V;
    hipStream_t s = ctx->s_main;
    const int grid = ctx->num_cus * 8;
    // 0.15 and 0.85 are the reference's literals (gpu_kernels.cuh:538)
    const double damping = o->damping;
    const double base = damping == 0.85 ? 0.15 : 1.0 - damping;
    const int maxit = o->max_iterations > 0 ? o->max_iterations : 10000;
    ASC_TRY(pr_rows_build<OffT>(g, p));
    ASC_HIP(hipMemsetAsync(p->count, 0, 4 * kPrLines * kPrLineWords, s));
    hipLaunchKernelGGL(k_prref_init, dim3(grid), dim3(256), 0, s, p->val64, p->contrib64[0], p->active, g->d_outdeg,
                       V);
    ASC_HIP(hipGetLastError());
    const double t0 = now_ms();
    // Queues iteration `it` (from 1) and the publish of its count.
    const unsigned long long seq0 = p->ref_seq;
    auto iterate = [&](int it) -> int {
        p->ref_seq = seq0 + (unsigned long long)it;
        PrRefArgs a{};
        a.off = g->d_off;
        a.contrib_in = p->contrib64[(it + 1) & 1];
        a.contrib_out = p->contrib64[it & 1];
        a.val = p->val64;
        a.active = p->active;
        a.outdeg = g->d_outdeg;
        a.count = p->count;
        a.base = base;
        a.damping = damping;
        a.threshold = o->threshold;
        if (g->static_vertices) {
            a.src = (const uint32_t*)g->d_edges;
            a.v_end = g->static_vertices;
            a.rows = row_plan(p);
            const uint32_t hb = std::min<uint32_t>(
                p->rows_front + (p->rows_back + kWavesPerBlock - 1) / kWavesPerBlock + 1, (uint32_t)grid / 2);
            const uint32_t rb = std::min<uint32_t>(p->rows_n, (uint32_t)grid);
            if (hb + rb)
                hipLaunchKernelGGL((k_prref_rows<OffT, true>), dim3(hb + rb), dim3(kBlock), 0, s, a, hb);
            ASC_HIP(hipGetLastError());
        }
        ASC_TRY(pr_stream_chunks(g, p, [&](const uint32_t* src, uint64_t e0, uint64_t v0, uint64_t v1) {
            PrRefArgs c = a;
            c.src = src;
            c.e_base = e0;
            c.v_begin = v0;
            c.v_end = v1;
            const int cgrid = (int)std::max<uint64_t>(1, std::min<uint64_t>(grid, (v1 - v0 + 255) / 256));
            hipLaunchKernelGGL((k_prref_rows<OffT, false>), dim3(cgrid), dim3(kBlock), 0, s, c, 0u);
            ASC_HIP(hipGetLastError());
            return ASC_OK;
        }));
        hipLaunchKernelGGL(k_prref_publish, dim3(1), dim3(kWave), 0, s, p->count, p->d_refpub + it % kRefRing,
                           p->ref_seq);
        ASC_HIP(hipGetLastError());
        return ASC_OK;
    };
    uint64_t node_sum = V;
    uint64_t active = V;
    // A resident graph's next iteration is queued before the count of the
    // current one arrives: after the last one it finds no active vertex and
    // changes nothing.  A streamed one would copy its tail for that.
    const int ahead = p->chunks.empty() ? 1 : 0;
    int it = 0, queued = 0;
    while (active && it < maxit) {
        it++;
        for (; queued < std::min(it + ahead, maxit);) ASC_TRY(iterate(++queued));
        ASC_TRY(wait_host_seq(&p->h_refpub.p[it % kRefRing].seq, seq0 + (unsigned long long)it, s));
        active = (uint64_t)((const volatile PrRefPub*)p->h_refpub.p)[it % kRefRing].moved;
        node_sum += active;
    }
    const double t1 = now_ms();
    // (a queued iteration past the last runs ahead of the copy and changes nothing)
    if (rank_out) ASC_TRY(out_copy(p->out, (const uint32_t*)p->val64, 2 * V, (uint32_t*)rank_out, s));
    else ASC_HIP(hipStreamSynchronize(s));
    if (st) {
        std::memset(st, 0, sizeof(*st));
        st->total_ms = t1 - t0;
        st->iterations = (uint32_t)it;
        st->node_sum = node_sum;
        st->reached = V;
        st->reached_degree_sum = g->h.E;
        st->host_cores = hardware_threads();
    }
    return ASC_OK;
}

int pagerank(asc_graph* g, const asc_pr_opts* o, float* rank_f32, double* rank_f64, double* residual_out,
             asc_stats* st) {
    if (g->h.kind != ASC_KIND_CSC) {
        set_last_error("PageRank needs a BCSC graph (in-CSR + out-degree)");
        return ASC_ERR_UNSUPPORTED;
    }
    asc_stats local;
    if (!st && g->ctx->cfg.verbose) st = &local;
    int r;
    if (o->mode == ASC_PR_REFERENCE)
        r = g->off_bytes == 4 ? pr_reference<uint32_t>(g, o, rank_f64, st) : pr_reference<uint64_t>(g, o, rank_f64, st);
    else
        r = g->off_bytes == 4 ? pr_normalised<uint32_t>(g, o, rank_f32, residual_out, st)
                              : pr_normalised<uint64_t>(g, o, rank_f32, residual_out, st);
    // per-phase timings in the reference's wording (CalculateOpt.cu:700-720)
    if (r == ASC_OK && g->ctx->cfg.verbose && st)
        printf("totalProcess time is %.3f ms\nstaticProcess time is %.3f ms\noverloadProcess time is %.3f ms\n"
               "iterations : %u\n",
               st->total_ms, st->static_ms, st->overload_ms, st->iterations);
    return r;
}

}  // namespace asc
