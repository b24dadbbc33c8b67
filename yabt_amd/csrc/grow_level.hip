// Level-batched growth with best-first results on gfx950.
//
// cgrow (yabt/_cgrow/grow.c:321-408) splits, best leaf first, until no leaf
// has a positive fp32 gain or the leaf budget is reached.  When the budget
// cannot bind -- max_leaves >= 2^max_depth, the depth-wise workloads -- every
// node above the depth cap with a positive gain is split whatever the order,
// and a node's best split depends only on its rows and on the features of its
// ancestors (the interaction boost).  So all nodes of one depth are grown
// together: one routing pass over the rows, one histogram pass for the smaller
// child of every split (counting sort of the rows by child, then per-child
// runs), in-place sibling subtraction, one scan launch for every node of the
// new depth.  The tree is then numbered as cgrow numbers it -- by replaying its
// leaf table (left child replaces the split slot, right child appended,
// first maximum of the fp32 gains above 0) over the computed gains, on the
// host -- so the node arrays, values and leaf ids are those of yabt_grow bit
// for bit (same fixed-point sums, same scan).
//
// The device decides everything on the way down: a node at place p of depth d
// has the id 2^d - 1 + p (its children 2 id + 1 and 2 id + 2) and its histogram
// slot follows from p (the subtracted child keeps the parent's, the built one
// takes the parent's + 2^(max_depth - 2 - d)), so no table is made on the host
// between depths.  The places that split are listed per depth, and every launch
// goes over that list: its work is that of the nodes that exist, not of the
// 2^d places.  The host enqueues depth after depth, two ahead of the last one
// whose splits it has seen (k_route tells it their number), so that it stops soon
// after growth does, and numbers the nodes from the records that k_pick leaves
// in its mapped memory.  Growth with its margin update: 1M x 28, depth 8 1.65 ->
// 0.92 ms, 4M x 500, depth 6 3.39 -> 1.83 ms; with a read, four small tables and
// a wait per depth the device stood idle a quarter of the first.
//
// Per depth: k_pick (best records, split decisions, children), k_route (rows to
// their children; rows per built child), k_scatter (rows of built children
// sorted by child), k_hist (their histograms), k_scan (sibling subtraction and
// both children's scans).

#include "common.h"
#include "hist.h"
#include "host.h"
#include "scan.h"
#include "yabt_hip.h"

#include <math.h>
#include <string.h>

#include <algorithm>
#include <queue>
#include <vector>

namespace yabt {
namespace lvl {

constexpr int LB = 256;             // threads of the row kernels
constexpr int LROWS = 4096;         // rows per routing / scatter block
constexpr int LCHUNK_MAX = 8192;    // sorted rows per histogram block, at most
constexpr int LHIST_BLOCKS = 1024;  // histogram blocks of a depth, about
constexpr int LSCAN = 4;            // features per scan block (one wave each, per child)
constexpr int LSCAN_BLOCKS = 4096;  // scan blocks of a depth, about: more splits are taken in strides
constexpr int LPICK_BLOCKS = 1024;
constexpr int AHEAD = 2;            // depths enqueued past the last one whose splits are known
constexpr int LDS_SLOTS = 4096;     // child counters kept in LDS up to this many
constexpr int MAX_DEPTH = 16;
constexpr int XCDS = 8;             // dies of the device; blocks go to them in turn

struct LNode {                      // node id 2^depth - 1 + place
    int64_t tot[3];                 // totals: sum q(g), sum q(h), rows
    int32_t slot;                   // histogram slot, -1: not scanned
};

struct HNode {                      // a node's record for the host (mapped memory)
    float gain;                     // of its best split
    int32_t f, b;                   // the split
    int32_t split;                  // 1: its children exist
    float value[2];                 // the children's values
};

struct HHead {
    int32_t splits[MAX_DEPTH + 1];  // splits at each depth + 1, 0: not known yet
    int32_t finite;                 // 0: non-finite g or h
    float value;                    // the root's value
};

struct Route {                      // a node's rows at its depth: f = -1: they stay
    int16_t f_lo, f_hi;             // f in two halves (F may pass 32767)
    uint8_t b;
    uint8_t built_left;             // 1: the left child is built, 0: the right one
    uint16_t s;                     // the split's number in its depth's list
};

__device__ __forceinline__ int route_f(const Route& r) { return (int)(uint16_t)r.f_lo | ((int)r.f_hi << 16); }

struct Ws {
    Quant* q;
    uint16_t* row_node;             // (n) node of each row (max_leaves <= 65535: ids below 2^16)
    uint32_t* sorted;               // (n) rows sorted by built child
    float2* gh;                     // (n) g and h interleaved, for the gathers
    uint32_t* count;                // (P) rows of each split's built child
    int64_t* off;                   // (P + 1)
    unsigned long long* cursor;     // (P)
    int32_t* nsplit;                // (MAX_DEPTH + 1) splits at each depth
    LNode* nodes;                   // (NP)
    Route* route;                   // (NP)
    uint16_t* built;                // (NP) 1 + the number of the split whose built child the node is, else 0
    int32_t* list;                  // (2, P) places that split: this depth's, and the last one's
    uint8_t* path;                  // (NP, F)
    int32_t* remap;                 // (NP) final node id
    ScanRec* rec;                   // (P, scan blocks)
    int64_t* hist;                  // (P, 3, F, 256)
    size_t bytes;
};

inline int pool_slots(int max_depth) { return 1 << (max_depth > 0 ? max_depth - 1 : 0); }

Ws carve(char* base, int64_t n, int F, int max_leaves, int max_depth) {
    Carve c{base, 0};
    Ws w;
    const int64_t nn = n > 0 ? n : 1;
    const size_t NP = 2 * (size_t)max_leaves + 1;
    const size_t P = (size_t)pool_slots(max_depth);
    const size_t sblk = (size_t)(F + LSCAN - 1) / LSCAN;
    w.q = c.take<Quant>(1);
    w.row_node = c.take<uint16_t>(nn);
    w.sorted = c.take<uint32_t>(nn);
    w.gh = c.take<float2>(nn);
    w.count = c.take<uint32_t>(P);
    w.off = c.take<int64_t>(P + 1);
    w.cursor = c.take<unsigned long long>(P);
    w.nsplit = c.take<int32_t>(MAX_DEPTH + 1);
    w.nodes = c.take<LNode>(NP);
    w.route = c.take<Route>(NP);
    w.built = c.take<uint16_t>(NP);
    w.list = c.take<int32_t>(2 * P);
    w.path = c.take<uint8_t>(NP * (size_t)F);
    w.remap = c.take<int32_t>(NP);
    w.rec = c.take<ScanRec>(P * sblk);
    w.hist = c.take<int64_t>(P * 3 * (size_t)F * NB);
    w.bytes = align_up(c.off, 256);
    return w;
}

// ---------------------------------------------------------------------------
// setup
// ---------------------------------------------------------------------------

__global__ void __launch_bounds__(LB) k_setup(const float* grad, const float* hess, int64_t n, Ws w, int F,
                                              int64_t slot_n) {
    quant_reduce<LB>(grad, hess, n, w.q, w.gh);
    const int64_t tid = (int64_t)blockIdx.x * LB + threadIdx.x, stride = (int64_t)gridDim.x * LB;
    for (int64_t i = tid; i < n; i += stride) w.row_node[i] = 0;
    for (int64_t i = tid; i < F; i += stride) w.path[i] = 0;
    for (int64_t i = tid; i < slot_n; i += stride) w.hist[i] = 0;
    for (int64_t i = tid; i <= MAX_DEPTH; i += stride) w.nsplit[i] = 0;
}

// ---------------------------------------------------------------------------
// one depth
// ---------------------------------------------------------------------------

// The nodes of depth d (the children of the last depth's splits), a block each:
// the node's best record, whether it splits (fp32 gain above 0, as cgrow's leaf
// table compares them), its rows' route and its children's totals, values
// (grow.c:371-379), paths and slots.
__global__ void __launch_bounds__(LB) k_pick(Ws w, int F, int nblk, int d, int max_depth, int P, int64_t n, float lr,
                                             float lam, int32_t* status, HNode* __restrict__ h_nodes, HHead* h_head) {
    __shared__ int s_split, s_f;
    const int lane = threadIdx.x & (WAVE - 1);
    const Quant* q = w.q;
    if (d == 0) {
        if (threadIdx.x == 0) {
            LNode& L = w.nodes[0];
            L.tot[0] = q->tot_g;
            L.tot[1] = q->const_h ? n * q->hq_const : q->tot_h;
            L.tot[2] = n;
            L.slot = max_depth > 0 ? 0 : -1;
            const double G = (double)L.tot[0] * q->ig, H = (double)L.tot[1] * q->ih;
            h_head->value = (float)(-lr * G / (H + lam));
            h_head->finite = q->nonfinite ? 0 : 1;
            status[0] = q->nonfinite ? -1 : 0;
        }
        __syncthreads();
        if (q->nonfinite) return;
    }
    const int32_t* parents = w.list + (size_t)((d + 1) & 1) * P;
    int32_t* list = w.list + (size_t)(d & 1) * P;
    const int nodes = d ? 2 * w.nsplit[d - 1] : 1;
    for (int j = blockIdx.x; j < nodes; j += gridDim.x) {
        const int p = d ? 2 * parents[j >> 1] + (j & 1) : 0, id = (1 << d) - 1 + p;
        const LNode& L = w.nodes[id];
        if (threadIdx.x < WAVE) {
            const bool scanned = L.slot >= 0;
            ScanRec r;
            no_split(r);
            if (scanned) r = wave_best_record(w.rec + (size_t)p * nblk, nblk, lane);
            if (lane == 0) {
                const int split = scanned && r.b >= 0 && (float)r.gain > 0.0f;
                HNode h{0.0f, 0, 0, split, {0.0f, 0.0f}};
                Route route{-1, -1, 0, 0, 0};
                if (split) {
                    const int s = atomicAdd(&w.nsplit[d], 1);
                    list[s] = p;
                    w.count[s] = 0;
                    // the smaller child is built, ties left (grow.c:355)
                    const bool bl = r.left[2] <= L.tot[2] - r.left[2], scan = d + 1 < max_depth;
                    route = Route{(int16_t)(r.f & 0xFFFF), (int16_t)(r.f >> 16), (uint8_t)r.b, (uint8_t)bl, (uint16_t)s};
                    h.gain = (float)r.gain;
                    h.f = r.f;
                    h.b = r.b;
                    for (int c = 0; c < 2; ++c) {
                        const int k = 2 * id + 1 + c;
                        LNode& C = w.nodes[k];
                        for (int i = 0; i < 3; ++i) C.tot[i] = c ? L.tot[i] - r.left[i] : r.left[i];
                        const double G = (double)C.tot[0] * q->ig, H = (double)C.tot[1] * q->ih;
                        h.value[c] = (float)(-lr * G / (H + lam));
                        const bool made = (c == 0) == bl;
                        C.slot = scan ? (made ? L.slot + (P >> (d + 1)) : L.slot) : -1;
                        w.built[k] = made ? (uint16_t)(s + 1) : 0;
                    }
                }
                w.route[id] = route;
                h_nodes[id] = h;
                s_split = split;
                s_f = r.f;
            }
        }
        __syncthreads();
        if (s_split) {
            const uint8_t* mine = w.path + (size_t)id * F;
            uint8_t* child = w.path + (size_t)(2 * id + 1) * F;
            for (int i = threadIdx.x; i < F; i += LB) {
                const uint8_t v = (uint8_t)(mine[i] | (i == s_f ? 1 : 0));
                child[i] = v;
                child[F + i] = v;
            }
        }
        __syncthreads();                    // s_split and s_f are read
    }
}

// Rows of depth-d nodes follow their split; with COUNT the rows of each split's
// built child are counted (in LDS up to LDS_SLOTS splits) and the built
// children's slots cleared.  The host is told the depth's splits.
template <bool COUNT>
__global__ void __launch_bounds__(LB) k_route(const uint8_t* __restrict__ bins_fm, int64_t ld, int64_t n, Ws w, int d, int P,
                                              int64_t slot_n, HHead* h_head) {
    __shared__ uint32_t s_cnt[COUNT ? LDS_SLOTS : 1];
    __shared__ int s_slot[LB];
    const int ns = w.nsplit[d], id0 = (1 << d) - 1;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        *(volatile int32_t*)&h_head->splits[d] = ns + 1;
        __threadfence_system();
    }
    if (ns == 0) return;
    const int32_t* list = w.list + (size_t)(d & 1) * P;
    const bool lds = ns <= LDS_SLOTS;
    if (COUNT) {
        if (lds)
            for (int i = threadIdx.x; i < ns; i += LB) s_cnt[i] = 0;
        // block b clears its share of every built child's slot; the slots are
        // looked up by all threads at once
        const int64_t per = (slot_n + gridDim.x - 1) / gridDim.x, z0 = per * blockIdx.x, z1 = min(slot_n, z0 + per);
        for (int base = 0; base < ns; base += LB) {
            const int s = base + threadIdx.x;
            if (s < ns) {
                const int k = 2 * (id0 + list[s]) + 1;
                s_slot[threadIdx.x] = w.nodes[w.built[k] ? k : k + 1].slot;
            }
            __syncthreads();
            for (int j = 0; j < min(LB, ns - base); ++j) {
                int64_t* h = w.hist + (size_t)s_slot[j] * slot_n;
                for (int64_t i = z0 + threadIdx.x; i < z1; i += LB) h[i] = 0;
            }
            __syncthreads();
        }
    }
    for (int64_t r0 = (int64_t)blockIdx.x * LROWS; r0 < n; r0 += (int64_t)gridDim.x * LROWS) {
        constexpr int U = 8;               // rows of a thread in flight
        for (int64_t i0 = r0 + threadIdx.x; i0 < min(n, r0 + LROWS); i0 += LB * U) {
            int k[U], f[U];
            Route R[U];
            uint8_t v[U];
#pragma unroll
            for (int u = 0; u < U; ++u) k[u] = i0 + u * LB < n ? w.row_node[i0 + u * LB] : 0;
#pragma unroll
            for (int u = 0; u < U; ++u) R[u] = w.route[k[u]];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                // rows of nodes above this depth have no route left to take
                f[u] = i0 + u * LB < n && k[u] >= id0 ? route_f(R[u]) : -1;
                v[u] = f[u] >= 0 ? bins_fm[(size_t)f[u] * ld + i0 + u * LB] : 0;
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (f[u] < 0) continue;
                const bool gl = v[u] <= R[u].b;
                w.row_node[i0 + u * LB] = (uint16_t)(2 * k[u] + (gl ? 1 : 2));
                if (COUNT && gl == (R[u].built_left != 0)) {
                    if (lds) atomicAdd(&s_cnt[R[u].s], 1u);
                    else atomicAdd(&w.count[R[u].s], 1u);
                }
            }
        }
    }
    if (COUNT && lds) {
        __syncthreads();
        for (int i = threadIdx.x; i < ns; i += LB)
            if (s_cnt[i]) atomicAdd(&w.count[i], s_cnt[i]);
    }
}

// Places of the built children's rows in `sorted`, one run per split of depth d.
__global__ void __launch_bounds__(1024) k_offsets(Ws w, int d) {
    __shared__ int64_t s_wave[1024 / WAVE];
    const int K = w.nsplit[d];
    int64_t carry = 0;
    for (int base = 0; base < K; base += 1024) {
        const int i = base + threadIdx.x;
        const int64_t c = i < K ? (int64_t)w.count[i] : 0;
        int64_t tot;
        const int64_t ex = block_excl_scan<1024, int64_t>(c, s_wave, &tot);
        if (i < K) {
            w.off[i] = carry + ex;
            w.cursor[i] = (unsigned long long)(carry + ex);
        }
        carry += tot;
    }
    if (threadIdx.x == 0) w.off[K] = carry;
}

// Rows of the built children (nodes of depth d + 1) sorted by child.  Up to
// LDS_SLOTS splits a block reserves one range per child.
__global__ void __launch_bounds__(LB) k_scatter(int64_t n, Ws w, int d) {
    __shared__ uint32_t s_cnt[LDS_SLOTS];
    __shared__ unsigned long long s_base[LDS_SLOTS];
    const int ns = w.nsplit[d], id1 = (2 << d) - 1;
    if (ns == 0) return;
    const bool lds = ns <= LDS_SLOTS;
    const int64_t lo = (int64_t)blockIdx.x * LROWS, hi = min(n, lo + LROWS);
    constexpr int U = LROWS / LB;
    int run[U];                            // -1: not a built child's row
    if (lds) {
        for (int i = threadIdx.x; i < ns; i += LB) s_cnt[i] = 0;
        __syncthreads();
    }
    uint16_t k[U];
#pragma unroll
    for (int u = 0; u < U; ++u) k[u] = lo + u * LB + threadIdx.x < hi ? w.row_node[lo + u * LB + threadIdx.x] : 0;
#pragma unroll
    for (int u = 0; u < U; ++u)
        run[u] = lo + u * LB + threadIdx.x < hi && (int)k[u] >= id1 ? (int)w.built[k[u]] - 1 : -1;
    if (!lds) {
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (run[u] >= 0) w.sorted[atomicAdd(&w.cursor[run[u]], 1ull)] = (uint32_t)(lo + u * LB + threadIdx.x);
        return;
    }
    uint32_t rank[U];
#pragma unroll
    for (int u = 0; u < U; ++u) rank[u] = run[u] >= 0 ? atomicAdd(&s_cnt[run[u]], 1u) : 0u;
    __syncthreads();
    for (int i = threadIdx.x; i < ns; i += LB)
        s_base[i] = s_cnt[i] ? atomicAdd(&w.cursor[i], (unsigned long long)s_cnt[i]) : 0ull;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < U; ++u)
        if (run[u] >= 0) w.sorted[s_base[run[u]] + rank[u]] = (uint32_t)(lo + u * LB + threadIdx.x);
}

// Unit (chunk of `per` sorted rows, tile of 16 features): one built child's
// run at a time by the row gathers of hist.h (16 bytes of a row per lane, the
// count packed beside q), added into the child's slot.  All tiles of a chunk
// run on one die, one after the other, so that a row's lines are read from
// HBM once, and a chunk is small enough for LHIST_BLOCKS units.  (Mean launch
// with the tiles a whole pass apart, 8192 rows a chunk, 16 one-byte loads per
// lane and the count in an atomic of its own -> now: 4M x 500, depth 6, h
// constant, up to 2M rows, 353 -> 126 us; 1M x 28, depth 8, both channels, up
// to 500 000 rows, 75 -> 30 us.)
__global__ void __launch_bounds__(HBLOCK) k_hist(const uint8_t* __restrict__ bins_rm, int64_t ldb,
                                                 const float* __restrict__ grad, const float* __restrict__ hess, int F,
                                                 Ws w, int d, int P, int64_t per) {
    __shared__ GatherLds L;
    const int K = w.nsplit[d], id0 = (1 << d) - 1;
    if (K == 0) return;
    const int32_t* list = w.list + (size_t)(d & 1) * P;
    const int tiles = (F + HFL - 1) / HFL;
    const int x = blockIdx.x % XCDS, u = blockIdx.x / XCDS, tile = u % tiles;
    const int64_t chunk = (int64_t)(u / tiles) * XCDS + x;
    const int64_t total = w.off[K], c0 = chunk * per, c1 = min(total, c0 + per);
    if (c0 >= c1) return;
    const Quant* q = w.q;
    const double scg = q->scg, sch = q->sch;
    const int wlog = q->wlog;
    const bool no_h = q->const_h != 0;
    int lo = 0, hi = K - 1;                 // the split whose run holds position c0: last s with off[s] <= c0
    while (lo < hi) {
        const int m = (lo + hi + 1) / 2;
        if (w.off[m] <= c0) lo = m;
        else hi = m - 1;
    }
    for (int s = lo; s < K && w.off[s] < c1; ++s) {
        const int64_t a = max(c0, w.off[s]), b = min(c1, w.off[s + 1]);
        if (a >= b) continue;               // uniform across the block
        const int k = 2 * (id0 + list[s]) + 1;
        int64_t* out = w.hist + (size_t)w.nodes[w.built[k] ? k : k + 1].slot * 3 * F * NB;
        if (no_h)
            hist_gather_rows<false, false>(L, bins_rm, ldb, grad, hess, F, scg, sch, nullptr, w.sorted, a, b, out, wlog,
                                           tile);
        else
            hist_gather_rows<true, false>(L, bins_rm, ldb, grad, hess, F, scg, sch, nullptr, w.sorted, a, b, out, wlog,
                                          tile, w.gh);
        __syncthreads();                    // the flush's LDS is read before the next run clears it
    }
}

// ---------------------------------------------------------------------------
// scan: grid (feature blocks, splits of depth d, in strides); waves 0 .. LSCAN - 1
// scan the built child's features, the others form the sibling (parent less built,
// in the parent's slot) and scan it.  d < 0: the root alone, by the first waves.
// ---------------------------------------------------------------------------

struct ScanArgs {
    const int32_t* nbins;
    const uint8_t* fmask;
    const float* imat;
    float ib;
    int use_imat;
    ScanParams sp;
    int F;
};

__global__ void __launch_bounds__(2 * LSCAN * WAVE) k_scan(ScanArgs S, Ws w, int d, int P) {
    const bool root = d < 0;
    const int lane = threadIdx.x & (WAVE - 1), wv = threadIdx.x / WAVE, side = wv / LSCAN, wf = wv % LSCAN;
    const int F = S.F, f = blockIdx.x * LSCAN + wf;
    __shared__ ScanRec s_rec[2 * LSCAN];
    if (root && side) return;
    const int ns = root ? 1 : w.nsplit[d];
    const Quant* q = w.q;
    const bool derive = q->const_h != 0;
    const int64_t hqc = q->hq_const;
    for (int s = blockIdx.y; s < ns; s += gridDim.y) {
        int node = 0;                           // the node this wave scans
        int64_t* slot = w.hist;                 // its slot
        const int64_t* built = nullptr;         // the sibling's, to subtract
        if (!root) {
            const int k = 2 * ((1 << d) - 1 + w.list[(size_t)(d & 1) * P + s]) + 1, kb = w.built[k] ? k : k + 1;
            node = side ? (kb == k ? k + 1 : k) : kb;
            const size_t slot_n = (size_t)3 * F * NB;
            slot = w.hist + (size_t)w.nodes[node].slot * slot_n;
            if (side) built = w.hist + (size_t)w.nodes[kb].slot * slot_n;
        }
        if (f < F) {
            int64_t g4[4], h4[4], c4[4];
            load_bins(slot, F, f, lane, g4, h4, c4, !derive);
            if (built) {
                int64_t gb[4], hb[4], cb[4];
                load_bins(built, F, f, lane, gb, hb, cb, !derive);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    g4[i] -= gb[i];
                    h4[i] -= hb[i];
                    c4[i] -= cb[i];
                }
                store_bins(slot, F, f, lane, g4, h4, c4, !derive);
            }
            int64_t hh[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) hh[i] = derive ? c4[i] * hqc : h4[i];
            const bool use = S.fmask[f] != 0;
            const int nb = max(0, min(NB, S.nbins[f]));
            const float bo = (S.use_imat && use) ? path_boost(w.path + (size_t)node * F, S.imat, S.ib, F, f, lane) : 1.0f;
            int64_t t256[3];
            ScanRec r = scan_feature(g4, hh, c4, nb, q->ig, q->ih, S.sp, (double)bo, lane, t256);
            if (!use) no_split(r);
            r.f = f;
            if (lane == 0) s_rec[wv] = r;
        } else if (lane == 0) {
            no_split(s_rec[wv]);
            s_rec[wv].f = -1;
        }
        __syncthreads();                        // at the root the second half has left
        if (lane == 0 && wf == 0) {
            int bi = wv;
            for (int i = wv + 1; i < wv + LSCAN; ++i)
                if (rec_beats(s_rec[i].sel, s_rec[i].f, s_rec[i].b, s_rec[bi].sel, s_rec[bi].f, s_rec[bi].b)) bi = i;
            // records by place of the new depth
            const int place = root ? 0 : node - ((2 << d) - 1);
            w.rec[(size_t)place * gridDim.x + blockIdx.x] = s_rec[bi];
        }
        __syncthreads();                        // the records are read
    }
}

// The tree in cgrow's numbering, from the host's mapped memory to the outputs
// (entries past the nodes as cgrow initialises them); h_prov: each node's id
// during growth.
struct Outputs {
    int64_t *feature, *thr, *left, *right, *depth;
    float* value;
    int32_t *status, *remap;
};

__global__ void __launch_bounds__(LB) k_emit(const int64_t* __restrict__ h_int, const float* __restrict__ h_val,
                                             const int32_t* __restrict__ h_prov, int NP, int n_nodes, Outputs o) {
    const int i = blockIdx.x * LB + threadIdx.x;
    if (i == 0) o.status[0] = n_nodes;
    if (i >= NP) return;
    const bool node = i < n_nodes;
    o.feature[i] = node ? h_int[i] : LEAF;
    o.thr[i] = node ? h_int[NP + i] : 0;
    o.left[i] = node ? h_int[2 * NP + i] : -1;
    o.right[i] = node ? h_int[3 * NP + i] : -1;
    o.depth[i] = node ? h_int[4 * NP + i] : 0;
    o.value[i] = node ? h_val[i] : 0.0f;
    if (node) o.remap[h_prov[i]] = i;
}

// out[row] = final id of the row's leaf.
__global__ void __launch_bounds__(LB) k_leaf_ids(const uint16_t* __restrict__ row_node, int64_t n,
                                                 const int32_t* __restrict__ remap, int64_t* __restrict__ out) {
    for (int64_t i = (int64_t)blockIdx.x * LB + threadIdx.x; i < n; i += (int64_t)gridDim.x * LB)
        out[i] = remap[row_node[i]];
}

}  // namespace lvl
}  // namespace yabt

using namespace yabt;
using namespace yabt::lvl;

extern "C" {

size_t yabt_grow_levelwise_workspace_bytes(int64_t n, int F, int max_leaves, int max_depth) {
    if (n < 0 || n > 0x7FFFFFFFll || F < 1 || max_depth < 0 || max_depth > MAX_DEPTH ||
        max_leaves < (1 << max_depth) || max_leaves > 65535)
        return 0;
    return carve(nullptr, n, F, max_leaves, max_depth).bytes;
}

int yabt_grow_levelwise(const uint8_t* bins_fm, int64_t ld_fm, const uint8_t* bins_rm, int64_t ld_rm,
                        const float* grad, const float* hess, const uint8_t* fmask, const float* imat, float ib,
                        int use_imat, const int32_t* nbins, const uint32_t* bin_counts, int64_t n, int F,
                        float lam, float gamma, float mcw,
                        int msl, float lr, int max_leaves, int max_depth, void* workspace, size_t workspace_bytes,
                        int64_t* out_feature, int64_t* out_thr_bin, int64_t* out_left, int64_t* out_right,
                        float* out_value, int64_t* out_depth, int64_t* out_leaf_of_row, int32_t* out_status,
                        hipStream_t stream) {
    if (F < 1 || n < 0 || n > 0x7FFFFFFFll || max_depth < 0 || max_depth > MAX_DEPTH || max_leaves > 65535)
        return fail(-2, "yabt_grow_levelwise: bad sizes (F >= 1, 0 <= n < 2^31, 0 <= max_depth <= 16)");
    if (max_leaves < (1 << max_depth))
        return fail(-3, "yabt_grow_levelwise: needs max_leaves >= 2^max_depth (the leaf budget must not bind)");
    if (ld_fm < n || ld_fm % 16 || ld_rm < F || ld_rm % 16)
        return fail(-2, "yabt_grow_levelwise: leading dimensions must be multiples of 16 covering n and F");
    if (!bins_fm || !bins_rm || !grad || !hess || !fmask || !nbins || (use_imat && !imat) || !workspace ||
        !out_feature || !out_thr_bin || !out_left || !out_right || !out_value || !out_depth || !out_status)
        return fail(-2, "yabt_grow_levelwise: null pointer argument");
    if (!aligned16(bins_fm) || !aligned16(bins_rm) || !aligned16(grad) || !aligned16(hess))
        return fail(-2, "yabt_grow_levelwise: bins, grad and hess must be 16-byte aligned");
    const Ws w = carve((char*)workspace, n, F, max_leaves, max_depth);
    if (workspace_bytes < w.bytes) return fail(-2, "yabt_grow_levelwise: workspace too small");
    const int NP = 2 * max_leaves + 1;
    const int P = pool_slots(max_depth);
    const size_t slot_n = (size_t)3 * F * NB;
    const int sblk = (F + LSCAN - 1) / LSCAN;
    const int tiles = (F + HFL - 1) / HFL;
    const int n_prov = (1 << (max_depth + 1)) - 1;    // ids of a complete tree; at most NP

    // pinned staging for the nodes' records and the numbered tree, from the
    // library's pinned pool; every return waits for the stream before it goes back
    struct Held {
        PinnedHold hold;
        hipStream_t s;
        ~Held() {
            if (hold.p) (void)hipStreamSynchronize(s);
        }
    } pin;
    pin.s = stream;
    const size_t head_bytes = align_up(sizeof(HHead), 64), rec_bytes = align_up((size_t)n_prov * sizeof(HNode), 64);
    const size_t int_bytes = (size_t)5 * NP * sizeof(int64_t);
    if (int prc = pin.hold.take(head_bytes + rec_bytes + int_bytes + (size_t)NP * (sizeof(float) + sizeof(int32_t)),
                                hipHostMallocMapped | hipHostMallocCoherent))
        return prc;
    HHead* h_head = (HHead*)pin.hold.p;
    HNode* h_nodes = (HNode*)((char*)pin.hold.p + head_bytes);     // by id, those at depths above the cap that exist
    int64_t* h_int = (int64_t*)((char*)pin.hold.p + head_bytes + rec_bytes);   // feature, bin, left, right, depth
    float* h_val = (float*)((char*)h_int + int_bytes);
    int32_t* h_prov = (int32_t*)(h_val + NP);
    memset(h_head, 0, sizeof *h_head);

    ScanArgs S;
    S.nbins = nbins;
    S.fmask = fmask;
    S.imat = imat;
    S.ib = ib;
    S.use_imat = use_imat ? 1 : 0;
    S.sp = ScanParams{(double)lam, (double)gamma, (double)mcw, msl};
    S.F = F;

    // root
    k_quant_clear<<<1, 1, 0, stream>>>(w.q);
    k_setup<<<launch_grid(max(n, (int64_t)slot_n), LB * 16, 1024), LB, 0, stream>>>(grad, hess, n, w, F, (int64_t)slot_n);
    launch_quant_resid(stream, grad, hess, n, w.q);
    if (n > 0) {
        launch_hist_root(stream, bins_fm, ld_fm, grad, hess, n, F, w.q, 0.0, 0.0, 0, nullptr, bin_counts, w.q, w.hist,
                         1, nullptr);
    }
    if (max_depth > 0) k_scan<<<dim3(sblk, 1), 2 * LSCAN * WAVE, 0, stream>>>(S, w, -1, P);
    k_pick<<<1, LB, 0, stream>>>(w, F, sblk, 0, max_depth, P, n, lr, lam, out_status, h_nodes, h_head);
    // the splits of depth d, once k_route has told them: waits for it
    const auto splits = [&](int d, int* count) -> int {
        const volatile int32_t* at = &h_head->splits[d];
        for (SpinWait sw; *at == 0;) {
            if (!sw.stream_check()) continue;
            const hipError_t e = hipStreamQuery(stream);
            if (e == hipSuccess && *at == 0) return fail(-4, "yabt_grow_levelwise: stream finished without a depth's splits");
            if (e != hipSuccess && e != hipErrorNotReady) return hip_fail(e, "yabt_grow_levelwise: depth");
        }
        *count = *at - 1;
        return 0;
    };
    int rc = 0;
    const int rb = (int)((n + LROWS - 1) / LROWS);
    for (int d = 0; d < max_depth && n > 0; ++d) {
        if (d >= AHEAD) {
            int count = 0;
            if ((rc = launch_status("yabt_grow_levelwise launch")) || (rc = splits(d - AHEAD, &count))) return rc;
            if (count == 0) break;
        }
        const int K = 1 << d;                      // splits of this depth, at most
        if (d + 1 == max_depth) {
            k_route<false><<<rb, LB, 0, stream>>>(bins_fm, ld_fm, n, w, d, P, (int64_t)slot_n, h_head);
        } else {
            // few rows: more blocks, which only clear
            const int zb = std::max(rb, launch_grid((int64_t)K * (int64_t)slot_n, LB * 32, 512));
            k_route<true><<<zb, LB, 0, stream>>>(bins_fm, ld_fm, n, w, d, P, (int64_t)slot_n, h_head);
            k_offsets<<<1, 1024, 0, stream>>>(w, d);
            k_scatter<<<rb, LB, 0, stream>>>(n, w, d);
            // the built children together hold at most half of the rows
            const int64_t most = std::max<int64_t>(1, n / 2);
            const int64_t even = (most * tiles + LHIST_BLOCKS - 1) / LHIST_BLOCKS;
            const int64_t per = std::min<int64_t>(LCHUNK_MAX, std::max<int64_t>(HSTEP, (even + HSTEP - 1) / HSTEP * HSTEP));
            const int64_t chunks = ((most + per - 1) / per + XCDS - 1) / XCDS * XCDS;
            k_hist<<<(unsigned)(chunks * tiles), HBLOCK, 0, stream>>>(bins_rm, ld_rm, grad, hess, F, w, d, P, per);
            const int sy = std::min(K, std::max(64, LSCAN_BLOCKS / sblk));
            k_scan<<<dim3(sblk, sy), 2 * LSCAN * WAVE, 0, stream>>>(S, w, d, P);
            k_pick<<<std::min(2 * K, LPICK_BLOCKS), LB, 0, stream>>>(w, F, sblk, d + 1, max_depth, P, n, lr, lam, out_status,
                                                                     h_nodes, h_head);
        }
    }
    if ((rc = launch_status("yabt_grow_levelwise launch"))) return rc;
    hipError_t e = hipStreamSynchronize(stream);   // the nodes' records are in
    if (e != hipSuccess) return hip_fail(e, "yabt_grow_levelwise: growth");
    if (!h_head->finite) return 0;                 // non-finite g/h: out_status[0] = -1, like yabt_grow

    // cgrow's numbering (grow.c:321-408) replayed over the computed gains: the
    // leaf table's first maximum above 0, left child in the split entry's place,
    // right child appended; a node at the depth cap carries gain -inf
    // (grow.c:316,392,402) and was never scanned
    struct Entry {
        float gain;
        int place, node;
        bool operator<(const Entry& o) const { return gain != o.gain ? gain < o.gain : place > o.place; }
    };
    std::priority_queue<Entry> table;
    int n_leaves = 1, n_nodes = 0;
    const auto add = [&](int k, int depth, float value, int place) {   // node k of growth is node n_nodes
        h_int[n_nodes] = LEAF;
        h_int[NP + n_nodes] = 0;
        h_int[2 * NP + n_nodes] = h_int[3 * NP + n_nodes] = -1;
        h_int[4 * NP + n_nodes] = depth;
        h_val[n_nodes] = value;
        h_prov[n_nodes] = k;
        if (depth < max_depth && h_nodes[k].split) table.push(Entry{h_nodes[k].gain, place, n_nodes});
        ++n_nodes;
    };
    add(0, 0, h_head->value, 0);
    while (n_leaves < max_leaves && !table.empty()) {
        const Entry t = table.top();
        table.pop();
        const int i = t.node, k = h_prov[i];
        const HNode& h = h_nodes[k];
        h_int[i] = h.f;
        h_int[NP + i] = h.b;
        h_int[2 * NP + i] = n_nodes;
        h_int[3 * NP + i] = n_nodes + 1;
        h_val[i] = 0.0f;
        const int depth = (int)h_int[4 * NP + i] + 1;
        add(2 * k + 1, depth, h.value[0], t.place);
        add(2 * k + 2, depth, h.value[1], n_leaves);
        ++n_leaves;
    }
    k_emit<<<(NP + LB - 1) / LB, LB, 0, stream>>>(h_int, h_val, h_prov, NP, n_nodes,
                                                  Outputs{out_feature, out_thr_bin, out_left, out_right, out_depth,
                                                          out_value, out_status, w.remap});
    if (out_leaf_of_row && n > 0)
        k_leaf_ids<<<launch_grid(n, LB * 8, 4096), LB, 0, stream>>>(w.row_node, n, w.remap, out_leaf_of_row);
    if ((rc = launch_status("yabt_grow_levelwise launch"))) return rc;
    e = hipStreamSynchronize(stream);              // the kernels read the pinned memory
    return e == hipSuccess ? 0 : hip_fail(e, "yabt_grow_levelwise: final synchronisation");
}

}  // extern "C"
