// The boosting step around the grower on gfx950: gradients/hessians of the
// losses and the margin update, so consecutive trees need no host copies.
//
//   yabt_grad_hess      LogLoss / MSELoss grad_hess (yabt/boosting.py:35-38, 52-54), at the
//                       margin or at margin + value[leaf] (yabt/neural_leaves.py:147)
//   yabt_margin_update  margin += value[leaf] + sum_j linear[leaf][j] * clamp(x_j, lo, hi)
//                       (yabt/boosting.py:508-511 with Tree.net_contribution,
//                       yabt/tree.py:118-128)
//   yabt_predict        out = base + sum over trees of Tree.predict (yabt/boosting.py:536-545,
//                       yabt/tree.py:82-135), all trees of a forest in one launch

#include "common.h"
#include "host.h"
#include "yabt_hip.h"

#include <algorithm>

namespace yabt {

constexpr int BB = 256;

// loss 0: squared error, g = m - y, h = 1; loss 1: logistic, p = 1 / (1 + e^-m),
// g = p - y, h = max(p (1 - p), 1e-6), in fp32 as the reference's torch code.
template <bool AT_LEAF>
__global__ void __launch_bounds__(BB) k_grad_hess(int loss, const float* __restrict__ margin,
                                                  const int64_t* __restrict__ leaf, const float* __restrict__ value,
                                                  int64_t n_nodes, const float* __restrict__ y, int64_t n,
                                                  float* __restrict__ g, float* __restrict__ h) {
    for (int64_t i = (int64_t)blockIdx.x * BB + threadIdx.x; i < n; i += (int64_t)gridDim.x * BB) {
        float m = margin[i];
        if (AT_LEAF) {
            const int64_t l = leaf[i];
            if (l >= 0 && l < n_nodes) m = m + value[l];
        }
        const float t = y[i];
        if (loss == 0) {
            g[i] = m - t;
            h[i] = 1.0f;
        } else {
            const float p = 1.0f / (1.0f + expf(-m));
            g[i] = p - t;
            h[i] = fmaxf(p * (1.0f - p), 1e-6f);
        }
    }
}

// One row per thread; the leaf's linear model over K inputs with the inputs
// clamped to the leaf's envelope (the reference adds the terms in input order).
template <int K>
__global__ void __launch_bounds__(BB) k_margin_update(float* __restrict__ margin, int64_t n,
                                                      const int64_t* __restrict__ leaf, int64_t n_nodes,
                                                      const float* __restrict__ value,
                                                      const int32_t* __restrict__ feats, const float* __restrict__ lin,
                                                      const float* __restrict__ lo, const float* __restrict__ hi,
                                                      int x_kind, const void* __restrict__ X, int64_t ldx) {
    __shared__ int32_t s_fs[K > 0 ? K : 1];
    if (K > 0 && threadIdx.x < K) s_fs[threadIdx.x] = feats[threadIdx.x];
    __syncthreads();
    for (int64_t i = (int64_t)blockIdx.x * BB + threadIdx.x; i < n; i += (int64_t)gridDim.x * BB) {
        const int64_t node = leaf[i];
        if (node < 0 || node >= n_nodes) continue;
        float c = value[node];
        if (K > 0) {
            float net = 0.0f;
#pragma unroll
            for (int j = 0; j < K; ++j) {
                float x = x_kind == 0   ? reinterpret_cast<const float*>(X)[(size_t)i * (size_t)ldx + s_fs[j]]
                          : x_kind == 2 ? reinterpret_cast<const float*>(X)[(size_t)s_fs[j] * (size_t)ldx + i]
                                        : (float)reinterpret_cast<const uint8_t*>(X)[(size_t)s_fs[j] * (size_t)ldx + i];
                x = fminf(fmaxf(x, lo[node * K + j]), hi[node * K + j]);
                net += lin[node * K + j] * x;
            }
            c += net;
        }
        margin[i] += c;
    }
}

template <int K>
void launch_margin(float* margin, int64_t n, const int64_t* leaf, int64_t n_nodes, const float* value,
                   const int32_t* feats, const float* lin, const float* lo, const float* hi, int x_kind, const void* X,
                   int64_t ldx, hipStream_t stream) {
    k_margin_update<K><<<launch_grid(n, BB * 8, 4096), BB, 0, stream>>>(margin, n, leaf, n_nodes, value, feats, lin,
                                                                       lo, hi, x_kind, X, ldx);
}

struct Forest {
    int T, F, K;                       // K: columns of lin, lo, hi (0: no linear leaves)
    const int64_t* node_off;
    int64_t n_total;
    const int64_t* feature;
    const float* threshold;
    const int64_t* left;
    const int64_t* right;
    const float* value;
    const int32_t* net_k;
    const int32_t* net_feats;
    const float* lin;
    const float* lo;
    const float* hi;
    int vec;                           // lin, lo, hi rows are two 16-byte aligned quads (K == 8)
};

// Tree t's nodes [off, off + nt) when they lie inside the forest, else nt 0
// (such a tree adds nothing).
__device__ __forceinline__ int64_t tree_nodes(const Forest& A, int t, int64_t* off) {
    const int64_t o = A.node_off[t], nt = A.node_off[t + 1] - o;
    *off = o;
    return (o < 0 || nt < 1 || o + nt > A.n_total) ? 0 : nt;
}

// One row's walk through a tree in global memory, as capply does
// (yabt/_cgrow/grow.c:223-239): it stops at a leaf, at an out-of-range
// feature or child, or after as many steps as the tree has nodes.  BOTH: the
// two children are loaded with the threshold, so that a step waits once; else
// only the one taken, for narrow rows enough to hide the waits (1M x 10, 1000
// leaves: 67 and 62 us; x 28 112 and 139).
template <bool BOTH = true, typename XF>
__device__ int64_t walk_global(const Forest& A, int64_t off, int64_t nt, const XF& x) {
    int64_t node = 0;
    for (int64_t s = 0; s < nt; ++s) {
        const int64_t f = A.feature[off + node];
        if (f < 0 || f >= A.F) break;
        const float thr = A.threshold[off + node];
        int64_t nxt;
        if (BOTH) {
            const int64_t l = A.left[off + node], r = A.right[off + node];
            nxt = (x((int)f) <= thr) ? l : r;
        } else {
            nxt = (x((int)f) <= thr) ? A.left[off + node] : A.right[off + node];
        }
        if (nxt < 0 || nxt >= nt) break;
        node = nxt;
    }
    return off + node;
}

// value[g] plus the node's clamped linear contribution, terms in input order.
template <typename XF>
__device__ float node_output(const Forest& A, int t, int64_t g, const XF& x) {
    float c = A.value[g];
    const int kt = A.net_k ? min(A.net_k[t], A.K) : 0;
    if (kt > 0) {
        float net = 0.0f;
        for (int j = 0; j < kt; ++j) {
            const int fj = A.net_feats[t * A.K + j];
            float xv = (fj >= 0 && fj < A.F) ? x(fj) : 0.0f;
            if (A.lo) xv = fminf(fmaxf(xv, A.lo[g * A.K + j]), A.hi[g * A.K + j]);
            net += A.lin[g * A.K + j] * xv;
        }
        c += net;
    }
    return c;
}

// Few rows: one block per row, a tree per thread, the trees' outputs added in
// order by one thread.  A row's trees are walked side by side instead of one
// after the other: bound by one walk's chain of loads (two per level) and the
// adds (1 row, 116 trees of 34 linear leaves: 401 -> 15 us).
constexpr int PRED_TC = 1024;                  // outputs kept per round
__global__ void __launch_bounds__(BB) k_predict_rows(Forest A, const float* __restrict__ X, int64_t ldx, float base,
                                                     int accumulate, float* __restrict__ out) {
    __shared__ float s_c[PRED_TC];
    const int64_t i = blockIdx.x;
    const float* row = X + (size_t)i * (size_t)ldx;
    const auto x = [row](int f) { return row[f]; };
    float acc = accumulate ? out[i] : base;
    for (int t0 = 0; t0 < A.T; t0 += PRED_TC) {
        const int nc = min(PRED_TC, A.T - t0);
        for (int k = threadIdx.x; k < nc; k += BB) {
            int64_t off;
            const int64_t nt = tree_nodes(A, t0 + k, &off);
            // -0.0f: adding it leaves every sum as it is
            s_c[k] = nt > 0 ? node_output(A, t0 + k, walk_global(A, off, nt, x), x) : -0.0f;
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            int k = 0;
            for (; k + 8 <= nc; k += 8) {
                float c[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) c[j] = s_c[k + j];
#pragma unroll
                for (int j = 0; j < 8; ++j) acc += c[j];
            }
            for (; k < nc; ++k) acc += s_c[k];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) out[i] = acc;
}

// Rows enough but little work in each (predict_flat): a row per thread, the trees
// in order.
template <bool BOTH>
__global__ void __launch_bounds__(BB) k_predict_flat(Forest A, const float* __restrict__ X, int64_t ldx, int64_t n, float base,
                                                     int accumulate, float* __restrict__ out) {
    for (int64_t i = (int64_t)blockIdx.x * BB + threadIdx.x; i < n; i += (int64_t)gridDim.x * BB) {
        const float* row = X + (size_t)i * (size_t)ldx;
        const auto x = [row](int f) { return row[f]; };
        float acc = accumulate ? out[i] : base;
        for (int t = 0; t < A.T; ++t) {
            int64_t off;
            const int64_t nt = tree_nodes(A, t, &off);
            if (nt > 0) acc += node_output(A, t, walk_global<BOTH>(A, off, nt, x), x);
        }
        out[i] = acc;
    }
}

// Many rows: a block takes up to PRED_TILES tiles of R rows and the forest in
// batches of trees that fit its LDS; every tile walks a batch before the next
// one is loaded.
//   s_x[f][row]   a tile's inputs: a lane reads its own row's bank whatever
//                 feature its node asks for, so the reads have no conflicts;
//   s_node        a batch's nodes, 8 bytes each: the threshold, then feature and
//                 left child (the right child is the next node, as every grower
//                 here numbers them).  A node where walks end has the threshold
//                 NaN, whose payload is its leaf's place, and the node before it
//                 as left child: no input is <= NaN, so a step from it stays;
//   s_leaf        per leaf of the batch: the linear model's weights and
//                 bounds and the value;
//   s_out[t][row] where the row's walk of tree t ended, then its output.
// The trees of a batch are shared out over G groups of R threads.  A lane
// walks its trees one after the other in one loop (a lane that ends early goes
// on with its next tree instead of waiting for the deepest of the wave), two
// such lists side by side; then the leaves' models are evaluated tree by tree,
// and the outputs are added in tree order.  Trees whose nodes do not have that
// form (children not neighbours or not after their parent, more than tcap nodes)
// are walked in global memory.
//
// 500 000 rows x 50 features, 200 trees of 63 leaves with 8 inputs: 1.41 ms
// (0.63 ms without linear leaves), 18.9 ms by a walk per row and tree in
// global memory, which waited on a gather of 32 node bytes and one of the
// row's input per level.  Counters: LDS active 49% and VALU 44% of the time,
// bank conflicts 17%; a wave waits 48% of its time, and the tile's LDS leaves
// no more than 16 waves a CU to cover that (a longer list of walks per thread in
// one loop, lanes going on by themselves: 2.2 ms; the end's select and its own
// slot per step: 1.75 ms; inputs not loaded ahead, batches not a multiple of the
// groups: 1.52 ms).
constexpr int PRED_TB = 32;                    // trees per batch at most
constexpr int PRED_TILES = 16;                 // tiles per block at most
constexpr int PRED_LEAF = 28;                  // floats per leaf: 8 weights, 8 lows, 8 highs, value, padding
constexpr uint32_t PRED_TERM = 0x80000000u;    // mark of a node where walks end
constexpr uint32_t PRED_NAN = 0x7FC00000u;

// fminf(fmaxf(x, lo), hi) for operands that are no signalling NaNs, without the
// compiler's quieting of each.
__device__ __forceinline__ float clamp_quiet(float x, float lo, float hi) {
    float t;
    asm("v_max_f32 %0, %1, %2\n\tv_min_f32 %0, %0, %3" : "=&v"(t) : "v"(x), "v"(lo), "v"(hi));
    return t;
}

template <int R, int G, bool XLDS, bool LIN>
__global__ void __launch_bounds__(R * G) k_predict_tile(Forest A, const float* __restrict__ X, int64_t ldx, int64_t n,
                                                        int tiles, int tb, int ncap, int tcap, int lcap, float base,
                                                        int accumulate, float* __restrict__ out) {
    constexpr int NT = R * G;
    static_assert(!XLDS || NT >= 4 * R, "rows of a tile are staged by four threads each");
    extern __shared__ char smem[];
    __shared__ int64_t s_off[PRED_TB], s_nt[PRED_TB];
    __shared__ int s_base[PRED_TB + 1];
    __shared__ int s_slow[PRED_TB];            // 1: walk in global memory, 2: adds nothing
    __shared__ int s_kt[PRED_TB];
    __shared__ __attribute__((aligned(16))) int s_feat[PRED_TB][8];
    __shared__ int s_count, s_leaves;
    constexpr int LS = LIN ? PRED_LEAF : 1;
    constexpr int CH = LIN ? 2 : 4;            // walks of a thread side by side
    constexpr int PF = 16;                     // features of a row that a thread holds ahead, four threads a row
    float* s_x = reinterpret_cast<float*>(smem);
    float* s_out = s_x + (XLDS ? (size_t)(A.F + 1) * R : 0);
    int* s_g = reinterpret_cast<int*>(s_out);  // while a batch is loaded: its leaves' nodes (tb * R places)
    float* s_acc = s_out + (size_t)tb * R;
    float* s_leaf = s_acc + (size_t)tiles * R;
    uint2* s_node = reinterpret_cast<uint2*>(s_leaf + (size_t)lcap * LS);
    const int tid = threadIdx.x, r = tid % R, grp = tid / R;
    const int64_t row0 = (int64_t)blockIdx.x * tiles * R;
    // place 1: an end, for lists shorter than the others; nodes from place 2 on
    if (tid == 0) s_node[1] = make_uint2(PRED_NAN, PRED_TERM);
    if (XLDS && tid < R) s_x[A.F * R + tid] = 0.0f;   // column F: the input that a model names wrongly
    for (int k = tid; k < tiles * R; k += NT) s_acc[k] = (accumulate && row0 + k < n) ? out[row0 + k] : base;
    // four features of sixteen rows a wave: 16-byte pieces of a row, four-way
    // conflicts on the writes into s_x
    const int f4 = tid % 4, r4 = tid / 4;
    float ahead[PF];
    const auto load_ahead = [&](int tile) {
        const float* row = X + (size_t)min(row0 + (int64_t)tile * R + r4, n - 1) * (size_t)ldx;
#pragma unroll
        for (int u = 0; u < PF; ++u)
            if (r4 < R && f4 + 4 * u < A.F) ahead[u] = row[f4 + 4 * u];
    };
    if (XLDS && A.T > 0) load_ahead(0);
    for (int t0 = 0; t0 < A.T;) {
        __syncthreads();                       // the last batch's readers are done
        if (tid < WAVE) {                      // the batch: as many trees as fit, at least one
            const int t = t0 + tid;
            int64_t off = 0, nt = 0;
            if (tid < tb && t < A.T) nt = tree_nodes(A, t, &off);
            const int fit = nt > 0 && nt <= tcap && A.F < 32767;
            const int mine = fit ? (int)nt : 0;
            int sum = mine;
#pragma unroll
            for (int d = 1; d < PRED_TB; d <<= 1) {
                const int up = __shfl_up(sum, d, WAVE);
                if (tid >= d) sum += up;
            }
            const uint64_t over = __ballot(tid < tb && (t >= A.T || sum > ncap));
            int cnt = over ? (int)__builtin_ctzll(over) : tb;
            if (cnt > G && t0 + cnt < A.T) cnt -= cnt % G;   // as many for each group
            if (tid < tb) {
                s_off[tid] = off;
                s_nt[tid] = nt;
                s_slow[tid] = fit ? 0 : (nt > 0 ? 1 : 2);
                if (LIN) {
                    const int kt = t < A.T ? min(A.net_k[t], A.K) : 0;
                    s_kt[tid] = kt;
#pragma unroll
                    for (int j = 0; j < 8; ++j) {
                        const int fj = j < kt ? A.net_feats[t * A.K + j] : -1;
                        s_feat[tid][j] = fj >= 0 && fj < A.F ? fj : A.F;
                    }
                }
                if (tid <= cnt) s_base[tid] = sum - mine;
                if (tid == cnt - 1) s_base[cnt] = sum;
            }
            if (tid == 0) {
                s_count = cnt;
                s_leaves = 0;
            }
        }
        __syncthreads();
        const int cnt = s_count, total = s_base[cnt];
        for (int k = tid; k < total; k += NT) {
            int b = 0;                         // the last tree whose base is at most k
#pragma unroll
            for (int d = PRED_TB / 2; d > 0; d >>= 1)
                if (b + d < cnt && s_base[b + d] <= k) b += d;
            const int node = k - s_base[b];
            const int nt = (int)s_nt[b];
            const int64_t g = s_off[b] + node;
            const int64_t f = A.feature[g], l = A.left[g], rt = A.right[g];
            const float thr = A.threshold[g];
            uint2 nd;
            if (f < 0 || f >= A.F) {
                const int slot = atomicAdd(&s_leaves, 1);
                if (slot < lcap) s_g[slot] = (b << 26) | node;
                else s_slow[b] = 1;
                nd = make_uint2(PRED_NAN | (uint32_t)min(slot, lcap - 1), PRED_TERM | (uint32_t)(k + 1));
            } else {
                const bool regular = l > node && rt == l + 1 && rt < nt;
                if (!regular) s_slow[b] = 1;
                nd = make_uint2(__float_as_uint(thr), ((uint32_t)f << 16) | (regular ? (uint32_t)(s_base[b] + (int)l + 2) : 0u));
            }
            s_node[k + 2] = nd;
        }
        __syncthreads();
        const int leaves = min(s_leaves, lcap);
        const auto leaf_node = [&](int k) { return s_off[(uint32_t)s_g[k] >> 26] + (s_g[k] & 0x3FFFFFF); };
        if (!LIN) {
            for (int k = tid; k < leaves; k += NT) s_leaf[k] = A.value[leaf_node(k)];
        } else if (A.vec && A.lo) {
            // whole quads, four loads in flight
            constexpr int U = 4;
            for (int k0 = tid; k0 < leaves * 8; k0 += NT * U) {
                float4 q[U];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int k = min(k0 + u * NT, leaves * 8 - 1), part = k % 8;
                    const int64_t g = leaf_node(k / 8);
                    const float* src = part < 2 ? A.lin : part < 4 ? A.lo : A.hi;
                    q[u] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                    if (part < 6) q[u] = *reinterpret_cast<const float4*>(src + g * 8 + (part & 1) * 4);
                    else if (part == 6) q[u].x = A.value[g];
                }
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int k = k0 + u * NT, part = k % 8;
                    if (k < leaves * 8 && part < 7) *reinterpret_cast<float4*>(s_leaf + (k / 8) * LS + part * 4) = q[u];
                }
            }
        } else {
            for (int k = tid; k < leaves * 25; k += NT) {
                const int slot = k / 25, j = k % 25, c = j % 8;
                const int64_t g = leaf_node(slot);
                const float* src = j < 8 ? A.lin : j < 16 ? A.lo : A.hi;
                s_leaf[slot * LS + j] = j == 24 ? A.value[g] : (src && c < A.K) ? src[g * A.K + c] : 0.0f;
            }
        }
        for (int tile = 0; tile < tiles && row0 + (int64_t)tile * R < n; ++tile) {
            const int64_t i = row0 + (int64_t)tile * R + r;
            const float* xrow = X + (size_t)min(i, n - 1) * (size_t)ldx;
            const auto x = [&](int f) { return XLDS ? s_x[f * R + r] : xrow[f]; };
            if (XLDS && r4 < R && (t0 == 0 || tiles > 1)) {
#pragma unroll
                for (int u = 0; u < PF; ++u)   // quieted, so that clamps need not be
                    if (f4 + 4 * u < A.F) s_x[(f4 + 4 * u) * R + r4] = __builtin_canonicalizef(ahead[u]);
                const float* row = X + (size_t)min(row0 + (int64_t)tile * R + r4, n - 1) * (size_t)ldx;
                for (int f = f4 + 4 * PF; f < A.F; f += 4) s_x[f * R + r4] = __builtin_canonicalizef(row[f]);
            }
            __syncthreads();                   // the tile and (first tile) the batch are in place
            // the next tile's loads go out now and are used after this tile's walks
            if (XLDS && tiles > 1) {
                const bool more = tile + 1 < tiles && row0 + (int64_t)(tile + 1) * R < n;
                load_ahead(more ? tile + 1 : 0);
            }
            // this thread's trees, CH of them side by side
            for (int b0 = grp; b0 < cnt; b0 += G * CH) {
                uint2 nd[CH];
#pragma unroll
                for (int c = 0; c < CH; ++c) {
                    const int b = b0 + G * c;
                    nd[c] = s_node[b < cnt && !s_slow[b] ? s_base[b] + 2 : 1];
                }
                while (true) {
                    uint32_t all = PRED_TERM;
#pragma unroll
                    for (int c = 0; c < CH; ++c) all &= nd[c].y;
                    if (all) break;
                    float xv[CH];
#pragma unroll
                    for (int c = 0; c < CH; ++c) xv[c] = x((int)((nd[c].y >> 16) & 0x7FFFu));
#pragma unroll
                    for (int c = 0; c < CH; ++c)
                        nd[c] = s_node[(nd[c].y & 0xFFFFu) + (xv[c] <= __uint_as_float(nd[c].x) ? 0u : 1u)];
                }
#pragma unroll
                for (int c = 0; c < CH; ++c) {
                    const int b = b0 + G * c;
                    if (b >= cnt) break;
                    const int slow = s_slow[b];
                float v = -0.0f;               // adds nothing, whatever the sum
                if (slow == 1) {
                    v = node_output(A, t0 + b, walk_global(A, s_off[b], s_nt[b], x), x);
                } else if (slow == 0) {
                    const float* lf = s_leaf + (nd[c].x & 0xFFFFu) * LS;
                    if (!LIN) {
                        v = lf[0];
                    } else {
                        v = lf[24];
                        const int kt = s_kt[b];
                        if (kt > 0) {
                            float w[8], lo[8], hi[8];
#pragma unroll
                            for (int q = 0; q < 2; ++q) {
                                *reinterpret_cast<float4*>(w + 4 * q) = reinterpret_cast<const float4*>(lf)[q];
                                *reinterpret_cast<float4*>(lo + 4 * q) = reinterpret_cast<const float4*>(lf)[2 + q];
                                *reinterpret_cast<float4*>(hi + 4 * q) = reinterpret_cast<const float4*>(lf)[4 + q];
                            }
                            float net = 0.0f;
                            const bool clamp = A.lo != nullptr;
                            if (XLDS && kt == 8 && clamp) {
                                int fj[8];
                                *reinterpret_cast<int4*>(fj) = reinterpret_cast<const int4*>(s_feat[b])[0];
                                *reinterpret_cast<int4*>(fj + 4) = reinterpret_cast<const int4*>(s_feat[b])[1];
                                float xj[8];
#pragma unroll
                                for (int j = 0; j < 8; ++j) xj[j] = s_x[fj[j] * R + r];
#pragma unroll
                                for (int j = 0; j < 8; ++j) net += w[j] * clamp_quiet(xj[j], lo[j], hi[j]);
                            } else {
#pragma unroll
                                for (int j = 0; j < 8; ++j) {
                                    if (j < kt) {
                                        const int fj = s_feat[b][j];
                                        float xj = fj < A.F ? x(fj) : 0.0f;
                                        if (clamp) xj = fminf(fmaxf(xj, lo[j]), hi[j]);
                                        net += w[j] * xj;
                                    }
                                }
                            }
                            v += net;
                        }
                    }
                }
                s_out[b * R + r] = v;
                }
            }
            __syncthreads();
            if (grp == 0) {
                float acc = s_acc[tile * R + r];
                for (int b = 0; b < cnt; ++b) acc += s_out[b * R + r];
                s_acc[tile * R + r] = acc;
            }
            __syncthreads();                   // before the next tile's inputs and ends
        }
        t0 += cnt;
    }
    __syncthreads();
    for (int k = tid; k < tiles * R; k += NT)
        if (row0 + k < n) out[row0 + k] = s_acc[k];
}

// LDS of a tile kernel with node and leaf places ncap, lcap.
size_t predict_lds(int R, bool xlds, bool lin, int F, int tiles, int tb, int ncap, int lcap) {
    return (size_t)R * 4 * ((xlds ? F + 1 : 0) + tb + tiles) + (size_t)lcap * ((lin ? PRED_LEAF : 1) * 4) +
           (size_t)(ncap + 2) * 8;
}

constexpr size_t PRED_LDS = 156 * 1024;        // dynamic LDS of a tile block (one a CU)

// Rows up to which a block per row takes less than tiles of rows.  By rows and by
// tiles, us: 200 trees of 63 linear leaves, 50 features, 2048 rows 110 and 140, 3000
// 150 and 140; 10 of 31, 28 features 26 and 27, 30 and 27; 1000 of 20 constant
// leaves 186 and 224, 263 and 224; 40 of 31 24 and 32, at 6000 rows 33 and 33; 30 of
// 255 linear leaves 33 and 60, at 6000 58 and 57.
constexpr int64_t PRED_ROW_BLOCKS = 2048;
// Rows from which tiles of 256 (each stages the forest once per 256 rows or more)
// beat tiles of 64 (four times as many blocks).  By 64 and by 256, us: 200 trees of
// 63 linear leaves, 50 features, 20 000 rows 191 and 227, 32 768 194 and 230, 40 000
// 242 and 233, 65 536 301 and 244; 30 of 255 101 and 122, 123 and 121, 158 and 122;
// 200 of 63 constant leaves 116 and 105, 117 and 105, 150 and 105.
constexpr int64_t PRED_WIDE_ROWS = 32768;

// Tiles of a block: one block a CU, in as many rounds of them as PRED_TILES asks,
// all of the same size (300 000 rows x 100, 200 trees of 63 leaves: 1403 us in 293
// blocks of 16 tiles, 961 in 469 of 10).
inline int predict_tiles_per_block(int64_t n, int R) {
    const int64_t slots = 256 * (int64_t)R, rounds = (n + slots * PRED_TILES - 1) / (slots * PRED_TILES);
    return (int)((n + slots * rounds - 1) / (slots * rounds));
}

template <int R, int G, bool XLDS, bool LIN>
int launch_predict(const Forest& A, const float* X, int64_t ldx, int64_t n, float base, int accumulate, float* out,
                   hipStream_t stream) {
    const int tiles = predict_tiles_per_block(n, R);
    const int tb = std::min(LIN ? 16 : PRED_TB, std::max(A.T, 1));
    // half the nodes of a tree are leaves: two node places per leaf place
    const size_t fixed = predict_lds(R, XLDS, LIN, A.F, tiles, tb, 0, 0);
    int64_t lcap = (int64_t)((PRED_LDS - fixed) / ((LIN ? PRED_LEAF : 1) * 4 + 16));
    lcap = std::min<int64_t>(std::min<int64_t>(lcap, 4096), std::max<int64_t>(A.n_total, 16));
    lcap = std::min<int64_t>(lcap, (int64_t)tb * R) & ~(int64_t)3;
    const int ncap = (int)(2 * lcap);
    // Trees of which a batch holds too few for the groups leave threads idle, and the
    // tile's inputs are read again for every batch: they are walked in global
    // memory instead.  Constant leaves: 20 trees of 1000, 20 000 rows x 50 219 us
    // one tree a batch, 59 walked; 300 000 x 300 14.4 ms, 0.94.  Linear leaves: 78
    // trees of 255, 20 000 x 50 300 and 237 us; of 200, 16 trees, 200 000 x 100 280
    // in LDS, four a batch, 340 walked.  Staged tiles of 256 rows fill their four
    // groups or read few batches: 40 linear trees of 500, 300 000 x 10, 893 us in
    // LDS, 1236 walked
    const int least = G == 16 ? (!LIN ? 16 : n < PRED_WIDE_ROWS ? 8 : 4) : XLDS ? 1 : 4;
    const int tcap = ncap / std::max(1, std::min(least, A.T));
    const size_t lds = predict_lds(R, XLDS, LIN, A.F, tiles, tb, ncap, (int)lcap);
    const int64_t per = (int64_t)tiles * R;
    k_predict_tile<R, G, XLDS, LIN><<<(unsigned)((n + per - 1) / per), R * G, lds, stream>>>(
        A, X, ldx, n, tiles, tb, ncap, tcap, (int)lcap, base, accumulate, out);
    return launch_status("yabt_predict launch");
}

template <int R, int G, bool XLDS>
int launch_predict(const Forest& A, const float* X, int64_t ldx, int64_t n, float base, int accumulate, float* out,
                   hipStream_t stream) {
    return A.net_k ? launch_predict<R, G, XLDS, true>(A, X, ldx, n, base, accumulate, out, stream)
                   : launch_predict<R, G, XLDS, false>(A, X, ldx, n, base, accumulate, out, stream);
}

// Staging a tile reads whole rows; the walks of a few trees touch only some of
// a wide row's lines.  1M rows x 100 features, 1 / 2 trees of 63 linear leaves: 328 /
// 342 us staged, 122 / 215 us not; 200 000 x 200, 8 trees of 31 146 and 167.  Constant
// leaves read less: there 146 and 119, 600 000 x 300, 16 trees 1089 and 489 us; 4000
// rows x 200 29 and 32.
constexpr int64_t PRED_STAGE_ROWS = 16384;
inline bool stage_rows(const Forest& A, int64_t n) {
    return A.F <= (A.net_k || n < PRED_STAGE_ROWS ? 28 : 16) * (A.T + 1);
}

// Few trees, whose walks cost less than a tile's fixed steps (about 4.5 us a tile and
// CU).  One tree: with constant leaves always (1M rows x 28, 31 leaves: 74 us by
// tiles, 63 by rows; x 10 73 and 41; 20 000 rows 28 and 22), with linear ones
// while the rows are few (20 000 x 28: 29 and 24 us; 1M x 28: 73 and 114) or the
// tree is larger than the LDS, but for rows that are little more than the walk
// reads (1M x 300, 1000 leaves: 502 and 427; x 10 194 and 151; x 28 198 and 221).
// Constant leaves: two trees, 1M x 10 75 and 60, 300 000 x 28 41 and 38, 1M x 28
// 80 and 98 us; three on narrow rows, 300 000 x 10 42 and 39, of 1000 leaves 72
// and 57; rows that are not staged, 200 000 x 100, 4 trees 74 and 69, 600 000 x 100
// 161 and 191, x 300 295 and 223; 1M x 300, 5 trees 510 and 435 us.
constexpr int64_t PRED_FLAT_INPUTS = 12'000'000;
constexpr int64_t PRED_FLAT_ROWS = 131072;
constexpr int PRED_NARROW = 16;                // features of a row within one 64-byte line
inline bool predict_flat(const Forest& A, int64_t n, bool staged) {
    const int64_t inputs = n * A.F;
    const bool narrow = A.F <= PRED_NARROW;
    if (A.T == 0) return true;
    if (A.T == 1)
        return !A.net_k || inputs < PRED_FLAT_INPUTS || (A.n_total > 1024 && (narrow || A.F > 4 * PRED_NARROW));
    if (A.net_k) return false;
    if (A.T == 2 && inputs < PRED_FLAT_INPUTS) return true;
    if (n < PRED_FLAT_ROWS) return false;
    if (A.T <= 3 && narrow) return true;
    return !staged && A.T <= 5 && A.n_total <= 4096 && (A.F > 8 * PRED_NARROW || inputs < 5 * PRED_FLAT_INPUTS / 2);
}

int predict_tiles(const Forest& A, const float* X, int64_t ldx, int64_t n, float base, int accumulate, float* out,
                  hipStream_t stream) {
    constexpr size_t TREES = 40 * 1024;        // of the block's LDS at least this for the trees
    const auto fits = [&](int R) {
        return stage_rows(A, n) && predict_lds(R, true, false, A.F, PRED_TILES, PRED_TB, 0, 0) + TREES <= PRED_LDS;
    };
    if (predict_flat(A, n, fits(64))) {
        auto flat = n < PRED_FLAT_ROWS || A.F > PRED_NARROW ? k_predict_flat<true> : k_predict_flat<false>;
        flat<<<launch_grid(n, BB, 8192), BB, 0, stream>>>(A, X, ldx, n, base, accumulate, out);
        return launch_status("yabt_predict launch");
    }
    if (n >= PRED_WIDE_ROWS && fits(256))
        return launch_predict<256, 4, true>(A, X, ldx, n, base, accumulate, out, stream);
    if (fits(64)) return launch_predict<64, 16, true>(A, X, ldx, n, base, accumulate, out, stream);
    return launch_predict<256, 4, false>(A, X, ldx, n, base, accumulate, out, stream);
}

}  // namespace yabt

using namespace yabt;

extern "C" {

int yabt_grad_hess(int loss, const float* margin, const int64_t* leaf_of_row, const float* value, int64_t n_nodes,
                   const float* y, int64_t n, float* out_g, float* out_h, hipStream_t stream) {
    if ((loss != 0 && loss != 1) || n < 0) return fail(-2, "yabt_grad_hess: loss must be 0 (MSE) or 1 (LogLoss)");
    if (n == 0) return 0;
    if (!margin || !y || !out_g || !out_h) return fail(-2, "yabt_grad_hess: null pointer argument");
    if ((leaf_of_row == nullptr) != (value == nullptr) || (leaf_of_row && n_nodes < 1))
        return fail(-2, "yabt_grad_hess: leaf_of_row and value (n_nodes >= 1) go together");
    const int grid = launch_grid(n, BB * 8, 4096);
    if (leaf_of_row)
        k_grad_hess<true><<<grid, BB, 0, stream>>>(loss, margin, leaf_of_row, value, n_nodes, y, n, out_g, out_h);
    else
        k_grad_hess<false><<<grid, BB, 0, stream>>>(loss, margin, nullptr, nullptr, 0, y, n, out_g, out_h);
    return launch_status("yabt_grad_hess launch");
}

int yabt_margin_update(float* margin, int64_t n, const int64_t* leaf_of_row, const float* value, int64_t n_nodes,
                       int K, const int32_t* feats, const float* linear, const float* lo, const float* hi, int x_kind,
                       const void* X, int64_t ldx, hipStream_t stream) {
    if (n < 0 || n_nodes < 1 || K < 0 || K > 8 || (K > 0 && (x_kind < 0 || x_kind > 2)))
        return fail(-2, "yabt_margin_update: bad sizes (n_nodes >= 1, 0 <= K <= 8, x_kind 0, 1 or 2)");
    if (n == 0) return 0;
    if (!margin || !leaf_of_row || !value || (K > 0 && (!feats || !linear || !lo || !hi || !X)))
        return fail(-2, "yabt_margin_update: null pointer argument");
    switch (K) {
        case 0: launch_margin<0>(margin, n, leaf_of_row, n_nodes, value, feats, linear, lo, hi, x_kind, X, ldx, stream); break;
        case 1: launch_margin<1>(margin, n, leaf_of_row, n_nodes, value, feats, linear, lo, hi, x_kind, X, ldx, stream); break;
        case 2: launch_margin<2>(margin, n, leaf_of_row, n_nodes, value, feats, linear, lo, hi, x_kind, X, ldx, stream); break;
        case 3: launch_margin<3>(margin, n, leaf_of_row, n_nodes, value, feats, linear, lo, hi, x_kind, X, ldx, stream); break;
        case 4: launch_margin<4>(margin, n, leaf_of_row, n_nodes, value, feats, linear, lo, hi, x_kind, X, ldx, stream); break;
        case 5: launch_margin<5>(margin, n, leaf_of_row, n_nodes, value, feats, linear, lo, hi, x_kind, X, ldx, stream); break;
        case 6: launch_margin<6>(margin, n, leaf_of_row, n_nodes, value, feats, linear, lo, hi, x_kind, X, ldx, stream); break;
        case 7: launch_margin<7>(margin, n, leaf_of_row, n_nodes, value, feats, linear, lo, hi, x_kind, X, ldx, stream); break;
        default: launch_margin<8>(margin, n, leaf_of_row, n_nodes, value, feats, linear, lo, hi, x_kind, X, ldx, stream); break;
    }
    return launch_status("yabt_margin_update launch");
}

int yabt_predict(const float* X, int64_t ldx, int64_t n, int F, int T, const int64_t* node_off, int64_t n_total,
                 const int64_t* feature, const float* threshold, const int64_t* left, const int64_t* right,
                 const float* value, int K, const int32_t* net_k, const int32_t* net_feats, const float* linear,
                 const float* lo, const float* hi, float base, int accumulate, float* out, hipStream_t stream) {
    if (n < 0 || F < 1 || ldx < F || T < 0 || n_total < 0 || K < 0 || K > 8)
        return fail(-2, "yabt_predict: bad sizes (ldx >= F >= 1, 0 <= K <= 8)");
    if (n == 0) return 0;
    if (!X || !out || (T > 0 && (!node_off || !feature || !threshold || !left || !right || !value)))
        return fail(-2, "yabt_predict: null pointer argument");
    if (net_k && (K < 1 || !net_feats || !linear || (lo == nullptr) != (hi == nullptr)))
        return fail(-2, "yabt_predict: linear leaves need K >= 1, net_feats and linear (lo and hi together)");
    const Forest A{T, F, net_k ? K : 0, node_off, n_total, feature, threshold, left, right, value, net_k, net_feats,
                   linear, lo, hi, net_k && K == 8 && aligned16(linear) && (!lo || (aligned16(lo) && aligned16(hi)))};
    if (n <= PRED_ROW_BLOCKS) {
        k_predict_rows<<<(unsigned)n, BB, 0, stream>>>(A, X, ldx, base, accumulate, out);
        return launch_status("yabt_predict launch");
    }
    return predict_tiles(A, X, ldx, n, base, accumulate, out, stream);
}

}  // extern "C"
