// Quantile binner on gfx950 (yabt/binning.py:29-129, the numpy path).
//
//   yabt_bin_fit        per feature: the quantile edges of a row sample
//                       (numpy's linear quantiles at linspace(0, 1, B+1)[1:-1],
//                       rounded to fp32, de-duplicated), the inter-quartile
//                       scale (numpy's fp32 std when it is zero) and the median
//                       of all rows (NaNs ignored, 0 if none)
//   yabt_bin_transform  bin = #{edges < x} after median imputation, written
//                       straight into the grower's feature-major and row-major
//                       layouts, plus the imputed fp32 matrix
//
// Fit, per feature: the sample column is gathered as order-preserving uint32
// keys (NaN last), sorted by a stable 4 x 8-bit radix sort, and the quantiles
// are read off the sorted keys with numpy's arithmetic: virtual index (c - 1) * q in double, d = fp32(b - a), value
// a + d * t (t < 1/2) or b - d * (1 - t) in double (numpy _lerp), rounded to
// fp32; the edges are those values sorted and de-duplicated (np.unique).
// Medians: of all rows, from the sorted keys when the sample is all rows, else
// from one pass over X that counts around a bracket taken from the sample and
// keeps what lies inside it; a 4-pass radix select over all rows when a
// bracket missed.  The two middle values are combined as numpy's float32 mean.

#include "common.h"
#include "host.h"
#include "yabt_hip.h"

#include <math.h>

#include <algorithm>

namespace yabt {
namespace bin {

constexpr int RT = 256;             // threads of a sort block
constexpr int RK = 16;              // keys per thread
constexpr int RC = RT * RK;         // keys per sort block
constexpr int HT = 16;              // features per histogram tile
constexpr int TB = 256;             // threads per select block
constexpr int MAXE = 255;           // edges per feature (max_bins - 1 <= 255)
constexpr uint32_t NAN_KEY = 0xFFFFFFFFu;

__device__ __forceinline__ uint32_t fkey(float v) {
    if (isnan(v)) return NAN_KEY;
    const uint32_t b = __float_as_uint(v);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}

__device__ __forceinline__ float kval(uint32_t k) {
    return __uint_as_float((k & 0x80000000u) ? (k & 0x7FFFFFFFu) : ~k);
}

// Bracket of a feature's median and what the pass over all rows finds about it.
struct Bracket {
    uint32_t lo, hi;       // keys; lo == hi: one value
    uint32_t below;        // rows with key < lo
    uint32_t eq_lo, eq_hi; // rows with key lo, and key hi (> lo)
    uint32_t inside;       // rows between: list entries wanted (may exceed the list)
    uint32_t valid;        // non-NaN rows
    uint32_t missed;       // the two middle values are not among them: select over all rows
};

struct FitWs {
    uint32_t* orig;        // (F, m) sample keys in sample order
    uint32_t* ka;          // (F, m) sorted keys
    uint32_t* kb;          // (F, m) radix ping-pong, then the std fallback's column, then the median lists
    uint32_t* dig;         // (F, 256, chunks) digit counts, then places
    uint32_t* need_std;    // (F) the IQR was 0
    Bracket* br;           // (F)
    uint32_t* cnt;         // (F) non-NaN rows over all n
    uint32_t* missed;      // (1) some bracket missed: select over all rows
    uint32_t* sel_hist;    // (F, 2, 256)
    uint32_t* sel_state;   // (F, 2, 2): prefix, rank
    int64_t chunks;
    size_t bytes;
};

FitWs carve_fit(char* base, int64_t m, int F) {
    Carve c{base, 0};
    FitWs w;
    const size_t fm = (size_t)F * (size_t)(m > 0 ? m : 1);
    w.chunks = (m + RC - 1) / RC;
    w.orig = c.take<uint32_t>(fm);
    w.ka = c.take<uint32_t>(fm);
    w.kb = c.take<uint32_t>(fm);
    w.dig = c.take<uint32_t>(w.chunks > 1 ? (size_t)F * NB * (size_t)w.chunks : 1);
    w.need_std = c.take<uint32_t>(F);
    w.br = c.take<Bracket>(F);
    w.cnt = c.take<uint32_t>(F);
    w.missed = c.take<uint32_t>(1);
    w.sel_hist = c.take<uint32_t>((size_t)F * 2 * NB);
    w.sel_state = c.take<uint32_t>((size_t)F * 4);
    w.bytes = c.off;
    return w;
}

// keys[f][i] = key of X[rows[i]][f] (rows == null: row i): 64 rows x 64
// features turned in LDS, so that rows are read and columns written in runs.
__global__ void __launch_bounds__(TB) k_gather_keys(const float* __restrict__ X, int64_t ldx, int F,
                                                    const int64_t* __restrict__ rows, int64_t m,
                                                    uint32_t* __restrict__ keys) {
    __shared__ uint32_t s_k[64][65];
    const int lane = threadIdx.x % 64, w = threadIdx.x / 64;
    const int64_t i0 = (int64_t)blockIdx.x * 64;
    const int f0 = blockIdx.y * 64;
    if (f0 + lane < F) {
#pragma unroll 8
        for (int q = 0; q < 16; ++q) {
            const int64_t i = min(i0 + w * 16 + q, m - 1);
            const int64_t r = rows ? rows[i] : i;
            s_k[lane][w * 16 + q] = fkey(X[(size_t)r * ldx + f0 + lane]);
        }
    }
    __syncthreads();
    if (i0 + lane < m)
        for (int j = w; j < 64 && f0 + j < F; j += TB / 64) keys[(size_t)(f0 + j) * m + i0 + lane] = s_k[j][lane];
}

// ---------------------------------------------------------------------------
// stable LSD radix sort of each feature's m keys, 4 passes of 8 bits.  A block
// takes RC keys: wave w's keys are RK rounds of 64 neighbours, so a key's rank
// among the block's equal digits is the wave's running count of the digit plus
// the lanes before it (eight ballots), with no barrier until the wave's keys
// are done.  One block sorts up to RC keys in LDS; above that a pass is a
// count, a scan of (digit, chunk) and a scatter through LDS that writes each
// digit's keys in a run.  200 000 x 50: 1607 us by one block per feature,
// which walked its tiles one after the other with five barriers each (50 of
// 256 CUs busy), 272 us by chunks
// (scatters 145, counts 90, scans 37).
// ---------------------------------------------------------------------------

struct RadixLds {
    uint32_t wc[RT / WAVE][NB];    // running counts, then the wave's start among the block's equal digits
    uint32_t start[NB];            // the digit's first place in the block
    uint32_t keys[RC];
    uint32_t scan[RT / WAVE];
};

// Places of the block's keys sorted by digit; keys past the end are NAN_KEY
// (the highest digit, after all others).
__device__ __forceinline__ void radix_places(RadixLds& L, const uint32_t (&key)[RK], int shift, uint32_t (&place)[RK]) {
    const int lane = threadIdx.x % WAVE, w = threadIdx.x / WAVE;
    for (int i = threadIdx.x; i < (RT / WAVE) * NB; i += RT) (&L.wc[0][0])[i] = 0;
    __syncthreads();
    volatile uint32_t* wc = L.wc[w];
#pragma unroll
    for (int q = 0; q < RK; ++q) {
        const uint32_t d = (key[q] >> shift) & 255u;
        uint64_t peers = ~0ull;
#pragma unroll
        for (int bit = 0; bit < 8; ++bit) {
            const bool on = (d >> bit) & 1u;
            const uint64_t bal = __ballot(on);
            peers &= on ? bal : ~bal;
        }
        const uint32_t before = lane_prefix(peers), run = wc[d];
        place[q] = run + before;
        __builtin_amdgcn_wave_barrier();       // every lane has read its count
        if (before == 0) wc[d] = run + (uint32_t)__popcll(peers);
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    uint32_t run = 0;
#pragma unroll
    for (int k = 0; k < RT / WAVE; ++k) {      // thread d: digit d
        const uint32_t c = L.wc[k][threadIdx.x];
        L.wc[k][threadIdx.x] = run;
        run += c;
    }
    uint32_t tot;
    L.start[threadIdx.x] = block_excl_scan<RT, uint32_t>(run, L.scan, &tot);
    __syncthreads();
#pragma unroll
    for (int q = 0; q < RK; ++q) {
        const uint32_t d = (key[q] >> shift) & 255u;
        place[q] += L.start[d] + L.wc[w][d];
    }
    (void)lane;
}

__device__ __forceinline__ int64_t radix_index(int q) {
    return (int64_t)(threadIdx.x / WAVE) * (RC / (RT / WAVE)) + q * WAVE + threadIdx.x % WAVE;
}

// m <= RC: the whole sort in one block per feature.
__global__ void __launch_bounds__(RT) k_sort_small(const uint32_t* __restrict__ src, uint32_t* __restrict__ dst,
                                                   int64_t m) {
    __shared__ RadixLds L;
    src += (size_t)blockIdx.x * m;
    dst += (size_t)blockIdx.x * m;
    uint32_t key[RK], place[RK];
#pragma unroll
    for (int q = 0; q < RK; ++q) key[q] = radix_index(q) < m ? src[radix_index(q)] : NAN_KEY;
    for (int shift = 0; shift < 32; shift += 8) {
        radix_places(L, key, shift, place);
#pragma unroll
        for (int q = 0; q < RK; ++q) L.keys[place[q]] = key[q];
        __syncthreads();
#pragma unroll
        for (int q = 0; q < RK; ++q) key[q] = L.keys[radix_index(q)];
        __syncthreads();
    }
#pragma unroll
    for (int q = 0; q < RK; ++q)
        if (radix_index(q) < m) dst[radix_index(q)] = key[q];
}

// dig[f][digit][chunk] = the chunk's keys with that digit.
__global__ void __launch_bounds__(RT) k_radix_count(const uint32_t* __restrict__ src, int64_t m, int shift,
                                                    int64_t chunks, uint32_t* __restrict__ dig) {
    __shared__ uint32_t s_c[NB];
    const int64_t chunk = blockIdx.x % chunks, f = blockIdx.x / chunks, c0 = chunk * RC;
    src += (size_t)f * m;
    s_c[threadIdx.x] = 0;
    __syncthreads();
#pragma unroll
    for (int q = 0; q < RK; ++q) {
        const int64_t i = c0 + q * RT + threadIdx.x;
        if (i < m) atomicAdd(&s_c[(src[i] >> shift) & 255u], 1u);
    }
    __syncthreads();
    dig[((size_t)f * NB + threadIdx.x) * chunks + chunk] = s_c[threadIdx.x];
}

// Exclusive prefix of a feature's (digit, chunk) counts.
__global__ void __launch_bounds__(1024) k_radix_scan(uint32_t* __restrict__ dig, int64_t chunks) {
    __shared__ uint32_t s_w[1024 / WAVE];
    uint32_t* d = dig + (size_t)blockIdx.x * NB * chunks;
    const int64_t total = NB * chunks;
    uint32_t carry = 0;
    for (int64_t base = 0; base < total; base += 1024 * 4) {
        const int64_t i = base + threadIdx.x * 4;
        uint32_t v[4], sum = 0;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            v[t] = i + t < total ? d[i + t] : 0u;
            sum += v[t];
        }
        uint32_t tot;
        uint32_t run = carry + block_excl_scan<1024, uint32_t>(sum, s_w, &tot);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            if (i + t < total) d[i + t] = run;
            run += v[t];
        }
        carry += tot;
    }
}

__global__ void __launch_bounds__(RT) k_radix_scatter(const uint32_t* __restrict__ src, uint32_t* __restrict__ dst,
                                                      int64_t m, int shift, int64_t chunks,
                                                      const uint32_t* __restrict__ dig) {
    __shared__ RadixLds L;
    __shared__ uint32_t s_to[NB];              // the digit's first place in dst, less its place in the block
    const int64_t chunk = blockIdx.x % chunks, f = blockIdx.x / chunks, c0 = chunk * RC;
    src += (size_t)f * m;
    dst += (size_t)f * m;
    const uint32_t to = dig[((size_t)f * NB + threadIdx.x) * chunks + chunk];
    uint32_t key[RK], place[RK];
#pragma unroll
    for (int q = 0; q < RK; ++q) key[q] = c0 + radix_index(q) < m ? src[c0 + radix_index(q)] : NAN_KEY;
    radix_places(L, key, shift, place);
    s_to[threadIdx.x] = to - L.start[threadIdx.x];
#pragma unroll
    for (int q = 0; q < RK; ++q) L.keys[place[q]] = key[q];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < RK; ++q) {
        const uint32_t i = q * RT + threadIdx.x, k = L.keys[i];
        const uint32_t at = s_to[(k >> shift) & 255u] + i;
        if (at < (uint32_t)m) dst[at] = k;     // past the end: the filled-up keys
    }
}

// numpy's linear quantile of the c sorted keys at q (numpy _quantile/_lerp),
// in double.
__device__ double np_quantile(const uint32_t* sk, int64_t c, double q) {
    const double virt = (double)(c - 1) * q;
    int64_t lo, hi;
    double prev;
    if (virt >= (double)(c - 1)) {
        lo = hi = c - 1;
        prev = -1.0;
    } else {
        prev = floor(virt);
        lo = (int64_t)prev;
        hi = lo + 1;
    }
    const double t = virt - prev;
    const float a = kval(sk[lo]), b = kval(sk[hi]);
    const float d = b - a;
    return t >= 0.5 ? (double)b - (double)d * (1.0 - t) : (double)a + (double)d * t;
}

// One block per feature: edges, edge count, scale (or the wish for the std
// fallback); the median when the sample is all rows, else its bracket.
__global__ void __launch_bounds__(TB) k_quantiles(const uint32_t* __restrict__ sorted, int64_t m, int max_bins, int whole,
                                                  float* __restrict__ out_edges, int64_t ld_edges,
                                                  int32_t* __restrict__ out_nedges, float* __restrict__ out_scales,
                                                  float* __restrict__ out_medians, uint32_t* __restrict__ need_std,
                                                  Bracket* __restrict__ br, uint32_t* __restrict__ missed, int64_t n) {
    __shared__ float s_q[TB];
    __shared__ int s_wave[TB / WAVE];
    __shared__ int64_t s_lo, s_hi;
    __shared__ int s_bad;
    const int f = blockIdx.x, tid = threadIdx.x;
    const uint32_t* sk = sorted + (size_t)f * m;
    if (tid == 0) {
        s_lo = 0;                           // non-NaN keys sort below NAN_KEY: their count lies in [lo, hi]
        s_hi = m;
        s_bad = 0;
    }
    __syncthreads();
    while (s_hi > s_lo) {                   // TB probes a round
        const int64_t lo = s_lo, hi = s_hi, step = (hi - lo + TB - 1) / TB, at = lo + tid * step;
        const bool num = at < hi && sk[at] != NAN_KEY;
        const int n = block_sum<TB, int>(num ? 1 : 0, s_wave);   // the first n probes are numbers
        if (tid == 0) {
            s_lo = n ? lo + (n - 1) * step + 1 : lo;
            s_hi = n ? min(hi, lo + n * step) : lo;
        }
        __syncthreads();
    }
    const int64_t c = s_lo;
    const uint32_t zero_key = 0x80000000u;  // an all-NaN (or empty) column is [0.0] (binning.py:57-59)
    const uint32_t* keys = c > 0 ? sk : &zero_key;
    const int64_t cc = c > 0 ? c : 1;
    const int ne = max_bins - 1;
    const double step = 1.0 / (double)max_bins;   // np.linspace(0, 1, max_bins + 1)
    if (tid < ne) {
        const double q = (double)(tid + 1) * step + 0.0;
        s_q[tid] = (float)np_quantile(keys, cc, q);
    }
    __syncthreads();
    // np.unique: sort (NaN last) and drop repeats (NaNs count as equal).  The
    // values come in order but for the rounding of neighbours; only then one
    // thread sorts them.
    if (tid + 1 < ne) {
        const float v = s_q[tid + 1], p = s_q[tid];
        if (isnan(v) ? false : (isnan(p) || p > v)) s_bad = 1;
    }
    __syncthreads();
    if (s_bad && tid == 0) {
        for (int i = 1; i < ne; ++i) {
            const float v = s_q[i];
            int k = i - 1;
            while (k >= 0 && (isnan(v) ? false : (isnan(s_q[k]) || s_q[k] > v))) {
                s_q[k + 1] = s_q[k];
                --k;
            }
            s_q[k + 1] = v;
        }
    }
    __syncthreads();
    const float v = tid < ne ? s_q[tid] : 0.0f;
    int keep = 0;
    if (tid < ne) keep = tid == 0 || !(v == s_q[tid - 1] || (isnan(v) && isnan(s_q[tid - 1])));
    int u;
    const int at = block_excl_scan<TB, int>(keep, s_wave, &u);
    if (keep) out_edges[(size_t)f * ld_edges + at] = v;
    if (tid == 0) {
        out_nedges[f] = u;
        // scale: q75 - q25 in double, else numpy's float32 std of the column, else 1
        const double s = np_quantile(keys, cc, 0.75) - np_quantile(keys, cc, 0.25);
        need_std[f] = s == 0.0;
        out_scales[f] = (float)s;
    }
    Bracket bk = {0u, 0u, 0u, 0u, 0u, 0u, 0u, 0u};
    if (!whole && c > 0) {
        // the rows' median lies within 3 sqrt(c) sample ranks of the sample's
        // (six standard deviations of a random sample's)
        const int64_t mid = (c - 1) / 2, w = (int64_t)(3.0 * sqrt((double)c)) + 8;
        const uint32_t lo = mid >= w ? sk[mid - w] : 0u, hi = mid + 1 + w < c ? sk[mid + 1 + w] : NAN_KEY - 1;
        // the rows between the ends go into a list of m keys, n / m of them for
        // each of the sample's, and two standard deviations more.  A list that
        // would not hold them is not begun (the ends stay equal, at no value's
        // key): keys that overflow it cost an atomic each on one counter (1M x
        // 50, a sample of 2000: 1909 us with the list, 935 without; 990 by
        // counting and selecting alone)
        int in = 0;
        for (int64_t i = max(mid - w, (int64_t)-1) + 1 + tid; i < min(mid + 1 + w, c); i += TB) in += sk[i] > lo && sk[i] < hi;
        const double between = block_sum<TB, int>(in, s_wave);
        if ((double)n * (between + 2.0 * sqrt(between)) <= (double)m * (double)m) {
            bk.lo = lo;
            bk.hi = hi;
        }
    }
    if (tid == 1) {
        if (whole) {
            // np.nanmedian of the rows, 0 where all are NaN (binning.py:32-33)
            float med = 0.0f;
            if (c > 0) {
                const float a = kval(sk[(c - 1) / 2]), b = kval(sk[c / 2]);
                med = (c % 2) ? a : (a + b) / 2.0f;
                if (isnan(med)) med = 0.0f;
            }
            out_medians[f] = med;
        } else {
            br[f] = bk;
        }
    }
    if (f == 0 && tid == 2) *missed = 0;
}

// ---------------------------------------------------------------------------
// scale of a column whose IQR is zero: numpy's float32 std, in its order --
// 8192-element buffers, each summed pairwise (halves split at multiples of 8
// down to at most 128 elements, those with eight accumulators), added in order
// to an accumulator that starts at 0.  A buffer's at most 128 runs are summed
// by 128 threads and combined along the same splits.
// ---------------------------------------------------------------------------
constexpr int PB = 8192;                    // elements per buffer
constexpr int PL = 128;                     // elements per run; also the most runs of a buffer
constexpr int PD = 7;                       // levels of splits
constexpr int ST = 1024;                    // threads: eight buffers at a time

// The run that path (PD bits, first split highest) leads to in a buffer of n
// elements: its place and length; false when it is another path's (a run that
// ends above the last split is its all-zero path's).  level: stop there.
__device__ __forceinline__ bool pairwise_run(int path, int level, int n, int* off, int* len) {
    int o = 0;
    for (int d = 0; d < level; ++d) {
        const int bit = (path >> (PD - 1 - d)) & 1;
        if (n <= PL) {
            if (bit) return false;
            continue;
        }
        int h = n / 2;
        h -= h % 8;
        o += bit ? h : 0;
        n = bit ? n - h : h;
    }
    *off = o;
    *len = n;
    return true;
}

template <typename Get>
__device__ float pairwise_leaf(const Get& get, int64_t off, int n) {
    if (n < 8) {
        float res = 0.0f;
        for (int i = 0; i < n; ++i) res += get(off + i);
        return res;
    }
    float r[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) r[j] = get(off + j);
    int i = 8;
    for (; i < n - (n % 8); i += 8)
#pragma unroll
        for (int j = 0; j < 8; ++j) r[j] += get(off + i + j);
    float res = ((r[0] + r[1]) + (r[2] + r[3])) + ((r[4] + r[5]) + (r[6] + r[7]));
    for (; i < n; ++i) res += get(off + i);
    return res;
}

// numpy's float32 sum of get(0 .. k - 1), by the block.
template <typename Get>
__device__ float block_np_sum(const Get& get, int64_t k, float (*s_v)[PL]) {
    const int buf = threadIdx.x / PL, path = threadIdx.x % PL;
    float acc = 0.0f;
    for (int64_t b0 = 0; b0 < k; b0 += (int64_t)PB * (ST / PL)) {
        const int64_t first = b0 + (int64_t)buf * PB;
        const int n = (int)max((int64_t)0, min((int64_t)PB, k - first));
        int off, len;
        if (n > 0 && pairwise_run(path, PD, n, &off, &len)) s_v[buf][path] = pairwise_leaf(get, first + off, len);
        __syncthreads();
        for (int d = PD - 1; d >= 0; --d) {    // the splits of level d
            const int half = 1 << (PD - 1 - d);
            if (n > 0 && path % (2 * half) == 0 && pairwise_run(path, d, n, &off, &len) && len > PL)
                s_v[buf][path] = s_v[buf][path] + s_v[buf][path + half];
            __syncthreads();
        }
        for (int j = 0; j < ST / PL && b0 + (int64_t)j * PB < k; ++j) acc += s_v[j][0];
        __syncthreads();
    }
    return acc;
}

__global__ void __launch_bounds__(ST) k_std_scale(const uint32_t* __restrict__ orig, float* __restrict__ scratch, int64_t m,
                                                  const uint32_t* __restrict__ need_std, float* __restrict__ out_scales) {
    __shared__ float s_v[ST / PL][PL];
    __shared__ uint32_t s_wave[ST / WAVE];
    const int f = blockIdx.x, tid = threadIdx.x;
    if (!need_std[f]) return;
    const uint32_t* ok = orig + (size_t)f * m;
    float* col = scratch + (size_t)f * m;
    int64_t k = 0;                             // the column's numbers, in sample order
    for (int64_t i0 = 0; i0 < m; i0 += ST * 4) {
        uint32_t key[4], n = 0;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int64_t i = i0 + tid * 4 + t;
            key[t] = i < m ? ok[i] : NAN_KEY;
            n += key[t] != NAN_KEY;
        }
        uint32_t tot;
        int64_t at = k + block_excl_scan<ST, uint32_t>(n, s_wave, &tot);
#pragma unroll
        for (int t = 0; t < 4; ++t)
            if (key[t] != NAN_KEY) col[at++] = kval(key[t]);
        k += tot;
    }
    if (k == 0) {                              // an all-NaN column is [0.0]: std 0
        if (tid == 0) out_scales[f] = 1.0f;
        return;
    }
    __syncthreads();
    const float mean = block_np_sum([&](int64_t i) { return col[i]; }, k, s_v) / (float)k;
    const float var = block_np_sum([&](int64_t i) { const float x = col[i] - mean; return x * x; }, k, s_v) / (float)k;
    if (tid == 0) {
        const float s = sqrtf(var);
        out_scales[f] = (double)s == 0.0 ? 1.0f : s;
    }
}

// ---------------------------------------------------------------------------
// medians over all rows by the sample's bracket
// ---------------------------------------------------------------------------

// One pass over X, every thread one feature (neighbouring threads neighbouring
// features): rows below, at and between the bracket's ends; the keys between
// go into the feature's list (cap places).  At most about 6 sqrt(c) / c of the
// rows lie between (1.35% at a sample of 200 000, fewer where values are tied:
// one that holds more of them than that is an end of the bracket); a list of a
// sample's size holds them up to 14.3M rows without ties, and k_quantiles
// gives no bracket to a feature whose rows it would not hold: these rows are
// only counted.  2M x 50: 215 us (1.9
// TB/s of X) and 23 us for the lists' selects; counting the numbers and
// four digit passes over X took 1580 us and 170 us of steps between them.
constexpr int MT = 256;                        // threads
constexpr int MPEND = 12;                      // keys a thread holds back
__global__ void __launch_bounds__(MT) k_median_pass(const float* __restrict__ X, int64_t ldx, int64_t n, int F, int fw,
                                                    Bracket* __restrict__ br, uint32_t* __restrict__ lists, int64_t cap) {
    __shared__ uint32_t s_pend[MPEND][MT];
    __shared__ uint32_t s_c[5][MT];            // below, eq_lo, eq_hi, valid, pending of a feature
    __shared__ uint32_t s_base[MT];
    const int tid = threadIdx.x, j = tid % fw, f = blockIdx.y * fw + j;
    const int per = MT / fw;                   // rows a step
    const bool live = f < F && tid < per * fw;
    for (int k = 0; k < 5; ++k) s_c[k][tid] = 0;
    __syncthreads();
    const uint32_t lo = live ? br[f].lo : 0u, hi = live ? br[f].hi : 0u;
    uint32_t below = 0, eql = 0, eqh = 0, valid = 0, pend = 0;
    if (live) {
        constexpr int U = 8;
        const int64_t step = (int64_t)gridDim.x * per;
        for (int64_t r0 = (int64_t)blockIdx.x * per + tid / fw; r0 < n; r0 += step * U) {
            float x[U];
#pragma unroll
            for (int u = 0; u < U; ++u) x[u] = r0 + u * step < n ? X[(size_t)(r0 + u * step) * ldx + f] : NAN;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const uint32_t k = fkey(x[u]);
                valid += k != NAN_KEY;
                below += k < lo;
                eql += k == lo;
                eqh += k == hi && hi != lo;
                if (k > lo && k < hi) {
                    if (pend < MPEND) {
                        s_pend[pend++][tid] = k;
                    } else {
                        const uint32_t at = atomicAdd(&br[f].inside, 1u);
                        if (at < cap) lists[(size_t)f * cap + at] = k;
                    }
                }
            }
        }
    }
    uint32_t place = 0;
    if (live) {
        if (below) atomicAdd(&s_c[0][j], below);
        if (eql) atomicAdd(&s_c[1][j], eql);
        if (eqh) atomicAdd(&s_c[2][j], eqh);
        if (valid) atomicAdd(&s_c[3][j], valid);
        place = pend ? atomicAdd(&s_c[4][j], pend) : 0u;
    }
    __syncthreads();
    if (tid < fw && blockIdx.y * fw + tid < F) {
        Bracket* b = br + blockIdx.y * fw + tid;
        if (s_c[0][tid]) atomicAdd(&b->below, s_c[0][tid]);
        if (s_c[1][tid]) atomicAdd(&b->eq_lo, s_c[1][tid]);
        if (s_c[2][tid]) atomicAdd(&b->eq_hi, s_c[2][tid]);
        if (s_c[3][tid]) atomicAdd(&b->valid, s_c[3][tid]);
        s_base[tid] = s_c[4][tid] ? atomicAdd(&b->inside, s_c[4][tid]) : 0u;
    }
    __syncthreads();
    for (uint32_t q = 0; q < pend; ++q) {
        const uint32_t at = s_base[j] + place + q;
        if (at < cap) lists[(size_t)f * cap + at] = s_pend[q][tid];
    }
}

// One block per feature: the two middle order statistics from the counts and
// the list (a radix select of the list's keys), or *missed.
__global__ void __launch_bounds__(1024) k_median_finish(Bracket* __restrict__ br, const uint32_t* __restrict__ lists,
                                                        int64_t cap, uint32_t* __restrict__ cnt,
                                                        uint32_t* __restrict__ missed, float* __restrict__ out_medians) {
    __shared__ uint32_t s_h[2][NB];
    __shared__ uint32_t s_prefix[2], s_rank[2];
    const int f = blockIdx.x, tid = threadIdx.x;
    const Bracket b = br[f];
    if (tid == 0) cnt[f] = b.valid;
    if (b.valid == 0) {
        if (tid == 0) out_medians[f] = 0.0f;
        return;
    }
    const uint32_t want[2] = {(b.valid - 1) / 2, b.valid / 2};
    uint32_t key[2] = {0u, 0u};
    bool search = false, miss = b.inside > cap;
    for (int t = 0; t < 2; ++t) {
        const uint32_t r = want[t] - b.below;  // wraps below the bracket: past every count
        if (want[t] < b.below) miss = true;
        else if (r < b.eq_lo) key[t] = b.lo;
        else if (r - b.eq_lo < b.inside) search = true;
        else if (r - b.eq_lo - b.inside < b.eq_hi) key[t] = b.hi;
        else miss = true;
    }
    if (miss) {
        if (tid == 0) {
            br[f].missed = 1;
            *missed = 1;
        }
        return;
    }
    if (search) {
        if (tid < 2) {
            s_prefix[tid] = 0;
            // a rank outside the list is clamped into it and its answer not used
            const uint32_t r = want[tid] - b.below;
            s_rank[tid] = r < b.eq_lo ? 0u : min(r - b.eq_lo, b.inside - 1);
        }
        const uint32_t* l = lists + (size_t)f * cap;
        // digits of the distance from lo: the keys' common high bits would send
        // every key of a pass to one counter
        const int bits = 32 - __clz(b.hi - b.lo), passes = (bits + 7) / 8, width = (bits + passes - 1) / passes;
        for (int shift = (passes - 1) * width; shift >= 0; shift -= width) {
            if (tid < 2 * NB) (&s_h[0][0])[tid] = 0;
            __syncthreads();
            const uint32_t p0 = s_prefix[0], p1 = s_prefix[1];
            for (uint32_t i = tid; i < b.inside; i += 1024) {
                const uint32_t k = l[i] - b.lo, top = shift + width >= 32 ? 0u : k >> (shift + width),
                               d = (k >> shift) & ((1u << width) - 1u);
                if (top == p0) atomicAdd(&s_h[0][d], 1u);
                if (top == p1) atomicAdd(&s_h[1][d], 1u);
            }
            __syncthreads();
            if (tid < 2 * WAVE) {              // wave t: target t's digit, four digits a lane
                const int t = tid / WAVE, lane = tid % WAVE;
                uint32_t c[4], sum = 0;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    c[q] = s_h[t][4 * lane + q];
                    sum += c[q];
                }
                uint32_t run = wave_excl_scan<uint32_t>(sum, lane);
                const uint32_t r = s_rank[t];
                uint32_t d = 0, left = 0;
                bool mine = false;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    if (r >= run && r < run + c[q]) {
                        mine = true;
                        d = 4 * lane + q;
                        left = r - run;
                    }
                    run += c[q];
                }
                if (mine) {
                    s_prefix[t] = (s_prefix[t] << width) | d;
                    s_rank[t] = left;
                }
            }
            __syncthreads();
        }
        for (int t = 0; t < 2; ++t) {
            const uint32_t r = want[t] - b.below;
            if (r >= b.eq_lo && r - b.eq_lo < b.inside) key[t] = b.lo + s_prefix[t];
        }
    }
    if (tid == 0) {
        const float a = kval(key[0]), c = kval(key[1]);
        float med = (b.valid % 2) ? a : (a + c) / 2.0f;
        if (isnan(med)) med = 0.0f;
        out_medians[f] = med;
    }
}

// ---------------------------------------------------------------------------
// medians over all rows: radix select of the two middle order statistics, for
// the features whose bracket missed (a sample that is no random one) or that got
// none (k_quantiles: more rows than their list holds); every kernel here ends
// at once where there is no such feature
// ---------------------------------------------------------------------------

// state[f][t] = {prefix, rank}: the ranks of the two middle order statistics.
__global__ void k_select_init(const uint32_t* __restrict__ missed, const uint32_t* __restrict__ cnt, int F,
                              uint32_t* __restrict__ state, uint32_t* __restrict__ hist) {
    const int f = blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= F || !*missed) return;
    const uint32_t c = cnt[f];
    const uint32_t k1 = c == 0 ? 0 : (c % 2 ? (c - 1) / 2 : c / 2 - 1);
    const uint32_t k2 = c == 0 ? 0 : c / 2;
    state[(size_t)f * 4 + 0] = 0;
    state[(size_t)f * 4 + 1] = k1;
    state[(size_t)f * 4 + 2] = 0;
    state[(size_t)f * 4 + 3] = k2;
    for (int i = 0; i < 2 * NB; ++i) hist[(size_t)f * 2 * NB + i] = 0;
}

// Histogram of digit `shift` among keys whose higher bits equal each target's prefix.
__global__ void __launch_bounds__(TB) k_select_hist(const uint32_t* __restrict__ missed, const Bracket* __restrict__ br,
                                                    const float* __restrict__ X, int64_t ldx, int64_t n, int F, int shift,
                                                    const uint32_t* __restrict__ state, uint32_t* __restrict__ hist) {
    __shared__ uint32_t s_h[HT][2][NB];
    if (!*missed) return;
    const int f0 = blockIdx.y * HT;
    const int j = threadIdx.x % HT;
    const int f = f0 + j;
    const bool mine = f < F && br[f].missed;
    if (!__syncthreads_or(mine)) return;
    for (int i = threadIdx.x; i < HT * 2 * NB; i += TB) (&s_h[0][0][0])[i] = 0;
    __syncthreads();
    if (mine) {
        const uint32_t p1 = state[(size_t)f * 4 + 0], p2 = state[(size_t)f * 4 + 2];
        for (int64_t r = (int64_t)blockIdx.x * (TB / HT) + threadIdx.x / HT; r < n; r += (int64_t)gridDim.x * (TB / HT)) {
            const float v = X[(size_t)r * ldx + f];
            if (isnan(v)) continue;
            const uint32_t k = fkey(v);
            const uint32_t hi = shift == 24 ? 0u : (k >> (shift + 8));
            const uint32_t d = (k >> shift) & 255u;
            if (hi == p1) atomicAdd(&s_h[j][0][d], 1u);
            if (hi == p2) atomicAdd(&s_h[j][1][d], 1u);
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < HT * 2 * NB; i += TB) {
        const int jj = i / (2 * NB), rest = i % (2 * NB);
        const uint32_t v = (&s_h[0][0][0])[i];
        if (f0 + jj < F && v) atomicAdd(&hist[(size_t)(f0 + jj) * 2 * NB + rest], v);
    }
}

// Choose each target's digit; clear the histogram for the next pass.
__global__ void k_select_step(const uint32_t* __restrict__ missed, int F, uint32_t* __restrict__ state,
                              uint32_t* __restrict__ hist) {
    const int f = blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= F || !*missed) return;
    for (int t = 0; t < 2; ++t) {
        uint32_t* h = hist + (size_t)f * 2 * NB + (size_t)t * NB;
        uint32_t k = state[(size_t)f * 4 + 2 * t + 1];
        uint32_t d = 0;
        for (; d < NB - 1; ++d) {
            if (k < h[d]) break;
            k -= h[d];
        }
        state[(size_t)f * 4 + 2 * t + 0] = (state[(size_t)f * 4 + 2 * t + 0] << 8) | d;
        state[(size_t)f * 4 + 2 * t + 1] = k;
        for (int i = 0; i < NB; ++i) h[i] = 0;
    }
}

// median = x_k (odd count) or float32 (x_k1 + x_k2) / 2 (even), 0 if no value
// (np.nanmedian then np.where(isnan, 0, .), binning.py:32-33).
__global__ void k_select_finish(const uint32_t* __restrict__ missed, const Bracket* __restrict__ br,
                                const uint32_t* __restrict__ cnt, int F, const uint32_t* __restrict__ state,
                                float* __restrict__ out_medians) {
    const int f = blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= F || !*missed || !br[f].missed) return;
    const uint32_t c = cnt[f];
    float med = 0.0f;
    if (c > 0) {
        const float a = kval(state[(size_t)f * 4 + 0]), b = kval(state[(size_t)f * 4 + 2]);
        med = (c % 2) ? a : (a + b) / 2.0f;
        if (isnan(med)) med = 0.0f;
    }
    out_medians[f] = med;
}

// ---------------------------------------------------------------------------
// transform
// ---------------------------------------------------------------------------

// A block keeps its feature group's edges in LDS and takes tiles of tr rows:
//   * a tile's values are read in memory order (lanes over neighbouring
//     features), imputed and stored the same way, and each looked up by its lane
//     in its own feature's edges.  The edges lie as a complete search tree
//     in level order (node k's children 2k and 2k + 1; +inf where a feature
//     has fewer edges), so a lookup is one read, compare and add a level; it
//     starts at the root of the leftmost subtree that holds the group's longest
//     edge list, so its levels are as many as that list needs.  Tables of
//     different features start a bank apart;
//   * the bins wait in LDS as [feature][row] bytes and leave as 16 rows of a
//     feature (feature-major) and as 4 x 4 blocks turned into 4 features of a
//     row (row-major), both in whole lines.
// 2684 -> 365 us at 2M x 50 (X in, two byte layouts and the imputed matrix out:
// 1.03 GB, 2.8 TB/s, under half of a copy's rate): a tile's loads, its lookups'
// LDS reads and its stores follow one another, over the 16 waves a CU that the
// tables leave.  A row per thread, as before, read X at the row stride and
// searched sorted edges at addresses that share four of the 64 banks.
constexpr int TT = 512;                        // threads of a transform block
constexpr int TL = 8;                          // levels of a table: MAXE edges
constexpr int TSTRIDE = NB + 1;                // words between two features' tables
constexpr int TFEAT = 60;                      // features per block: two blocks' LDS on a CU
// Values of a tile, at most: with few features a tile of more rows, so that
// every thread has several values in flight between two barriers.
constexpr int TVALUES = 16384;

// log2 of a tile's rows: TVALUES / fg of them, halved (down to 16, and to a
// value a thread) while the tiles are not two blocks a CU.
inline int transform_rows_log2(int64_t n, int F, int fg, int groups) {
    int l = 4;
    while ((fg << (l + 1)) <= TVALUES) ++l;
    while (l > 4 && (std::min(F, fg) << l) > TT && ((n + (1ll << l) - 1) >> l) * groups < 512) --l;
    return l;
}

struct TransformArgs {
    const float* X;
    int64_t ldx, n;
    int F, fg, trl;                            // fg: features per group (a multiple of 4); trl: log2 of a tile's rows
    const float* edges;
    int64_t ld_edges;
    const int32_t* nedges;
    const float* medians;
    uint8_t* fm;
    int64_t ld_fm;
    uint8_t* rm;
    int64_t ld_rm;
    float* imp;
    int64_t ld_imp;
    int fm_vec, rm_vec;                        // 16-byte aligned layouts
};

__global__ void __launch_bounds__(TT) k_transform(TransformArgs A) {
    extern __shared__ char smem[];
    __shared__ int s_any;                                              // the group's edge counts, or-ed
    const int tr = 1 << A.trl, bstride = tr + 4;                       // bytes between two features' bins
    float* s_e = reinterpret_cast<float*>(smem);                       // [fg][TSTRIDE]
    float* s_med = s_e + A.fg * TSTRIDE;                               // [fg]
    uint8_t* s_b = reinterpret_cast<uint8_t*>(s_med + A.fg);           // [fg][bstride]
    const int f0 = blockIdx.y * A.fg, nf = min(A.fg, A.F - f0);
    const int tid = threadIdx.x;
    if (tid == 0) s_any = 0;
    __syncthreads();
    if (tid < nf) {
        atomicOr(&s_any, min(max(A.nedges[f0 + tid], 0), MAXE));
        s_med[tid] = A.medians[f0 + tid];
    }
    // edges and edge counts are read together: an edge past its list is not used
#pragma unroll 4
    for (int i = tid; i < nf << TL; i += TT) {
        const int j = i >> TL, k = i & (NB - 1);
        if (k == 0) continue;
        const int lv = 31 - __clz(k);                                  // node k: number k - 2^lv of level lv
        const int at = ((2 * (k - (1 << lv)) + 1) << (TL - 1 - lv)) - 1;
        const float e = A.edges[(size_t)(f0 + j) * A.ld_edges + min((int64_t)at, A.ld_edges - 1)];
        s_e[j * TSTRIDE + k] = at < min(max(A.nedges[f0 + j], 0), MAXE) ? e : INFINITY;
    }
    __syncthreads();
    const int levels = __builtin_amdgcn_readfirstlane(s_any ? 32 - __clz(s_any) : 0), root = NB >> levels;
    // the bins of the row-major layout's columns up to the next multiple of 16 are zero
    const int last = blockIdx.y + 1 == gridDim.y;
    const int nq = last && A.rm_vec ? (((A.F + 15) & ~15) - f0) / 4 : (nf + 3) / 4;
    for (int64_t r0 = (int64_t)blockIdx.x << A.trl; r0 < A.n; r0 += (int64_t)gridDim.x << A.trl) {
        const int rows = (int)min((int64_t)tr, A.n - r0);
        const int total = rows * nf, dj = TT % nf, dr = TT / nf;
        constexpr int U = 4;
        int j = tid % nf, r = tid / nf;
        for (int i0 = tid; i0 < total; i0 += TT * U) {
            float x[U];
            int jj[U], rr[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                jj[u] = j;
                rr[u] = r;
                const bool ok = i0 + u * TT < total;
                x[u] = ok ? A.X[(size_t)(r0 + r) * A.ldx + f0 + j] : 0.0f;
                j += dj;
                r += dr;
                if (j >= nf) {
                    j -= nf;
                    ++r;
                }
            }
            int k[U];
            const float* e[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (isnan(x[u])) x[u] = s_med[jj[u]];
                if (A.imp && i0 + u * TT < total) A.imp[(size_t)(r0 + rr[u]) * A.ld_imp + f0 + jj[u]] = x[u];
                k[u] = root;
                e[u] = s_e + jj[u] * TSTRIDE;
            }
            for (int lv = 0; lv < levels; ++lv) {
#pragma unroll
                for (int u = 0; u < U; ++u) k[u] = 2 * k[u] + (e[u][k[u]] < x[u] ? 1 : 0);
            }
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (i0 + u * TT < total) s_b[jj[u] * bstride + rr[u]] = (uint8_t)(k[u] - NB);
        }
        __syncthreads();
        if (A.fm) {
            for (int i = tid; i < nf << (A.trl - 4); i += TT) {
                const int jf = i >> (A.trl - 4), r16 = (i & ((tr >> 4) - 1)) * 16;
                if (r16 >= rows) continue;
                const uint32_t* src = reinterpret_cast<const uint32_t*>(s_b + jf * bstride + r16);
                uint8_t* dst = A.fm + (size_t)(f0 + jf) * A.ld_fm + r0 + r16;
                if (A.fm_vec && r16 + 16 <= rows) {
                    *reinterpret_cast<uint4*>(dst) = make_uint4(src[0], src[1], src[2], src[3]);
                } else {
                    for (int q = 0; q < 16 && r16 + q < rows; ++q) dst[q] = s_b[jf * bstride + r16 + q];
                }
            }
        }
        if (A.rm && A.rm_vec && nf <= 4 && nq == 4) {      // a row is 16 bytes: one store
            for (int i = tid; i < rows; i += TT) {
                uint32_t w = 0;
                for (int t = 0; t < nf; ++t) w |= (uint32_t)s_b[t * bstride + i] << (8 * t);
                *reinterpret_cast<uint4*>(A.rm + (size_t)(r0 + i) * A.ld_rm + f0) = make_uint4(w, 0u, 0u, 0u);
            }
        } else if (A.rm && A.rm_vec) {
            for (int i = tid; i < nq * (tr / 4); i += TT) {
                const int q = i % nq, r4 = (i / nq) * 4;
                uint32_t c[4];
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    c[t] = 4 * q + t < nf ? *reinterpret_cast<const uint32_t*>(s_b + (4 * q + t) * bstride + r4) : 0u;
                // byte t of row t4's word: byte t4 of feature t's word
                const uint32_t a0 = __builtin_amdgcn_perm(c[1], c[0], 0x05010400u), a1 = __builtin_amdgcn_perm(c[1], c[0], 0x07030602u);
                const uint32_t b0 = __builtin_amdgcn_perm(c[3], c[2], 0x05010400u), b1 = __builtin_amdgcn_perm(c[3], c[2], 0x07030602u);
                const uint32_t o[4] = {__builtin_amdgcn_perm(b0, a0, 0x05040100u), __builtin_amdgcn_perm(b0, a0, 0x07060302u),
                                       __builtin_amdgcn_perm(b1, a1, 0x05040100u), __builtin_amdgcn_perm(b1, a1, 0x07060302u)};
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    if (r4 + t < rows)
                        *reinterpret_cast<uint32_t*>(A.rm + (size_t)(r0 + r4 + t) * A.ld_rm + f0 + 4 * q) = o[t];
            }
        } else if (A.rm) {
            int jb = tid % nf, rb = tid / nf;
            for (int i = tid; i < total; i += TT) {
                A.rm[(size_t)(r0 + rb) * A.ld_rm + f0 + jb] = s_b[jb * bstride + rb];
                jb += dj;
                rb += dr;
                if (jb >= nf) {
                    jb -= nf;
                    ++rb;
                }
            }
        }
        __syncthreads();                       // the tile's bins are out
    }
}

}  // namespace bin
}  // namespace yabt

using namespace yabt;
using namespace yabt::bin;

extern "C" {

size_t yabt_bin_fit_workspace_bytes(int64_t m, int F) {
    if (m < 0 || m > 0x7FFFFFFFll || F < 1) return 0;
    return carve_fit(nullptr, m, F).bytes;
}

int yabt_bin_fit(const float* X, int64_t ldx, int64_t n, int F, const int64_t* sample_rows, int64_t m, int max_bins,
                 void* workspace, size_t workspace_bytes, float* out_edges, int64_t ld_edges, int32_t* out_nedges,
                 float* out_scales, float* out_medians, hipStream_t stream) {
    if (n < 0 || F < 1 || ldx < F || m < 0 || m > 0x7FFFFFFFll || max_bins < 2 || max_bins > 256 ||
        ld_edges < max_bins - 1)
        return fail(-2, "yabt_bin_fit: bad sizes (ldx >= F >= 1, 2 <= max_bins <= 256, ld_edges >= max_bins - 1)");
    if (!sample_rows && m != n) return fail(-2, "yabt_bin_fit: without sample_rows the sample is all n rows (m == n)");
    if (!X || !workspace || !out_edges || !out_nedges || !out_scales || !out_medians)
        return fail(-2, "yabt_bin_fit: null pointer argument");
    const FitWs w = carve_fit((char*)workspace, m, F);
    if (workspace_bytes < w.bytes) return fail(-2, "yabt_bin_fit: workspace too small");
    // quantiles and scales of the sample (an empty sample is the column [0.0])
    if (m > 0) {
        const dim3 tiles((unsigned)((m + 63) / 64), (unsigned)((F + 63) / 64));
        k_gather_keys<<<tiles, TB, 0, stream>>>(X, ldx, F, sample_rows, m, w.orig);
        if (m <= RC) {
            k_sort_small<<<F, RT, 0, stream>>>(w.orig, w.ka, m);
        } else {
            const unsigned grid = (unsigned)(w.chunks * F);
            const uint32_t* src = w.orig;
            for (int pass = 0; pass < 4; ++pass) {
                uint32_t* dst = pass & 1 ? w.ka : w.kb;
                k_radix_count<<<grid, RT, 0, stream>>>(src, m, 8 * pass, w.chunks, w.dig);
                k_radix_scan<<<F, 1024, 0, stream>>>(w.dig, w.chunks);
                k_radix_scatter<<<grid, RT, 0, stream>>>(src, dst, m, 8 * pass, w.chunks, w.dig);
                src = dst;
            }
        }
    }
    const int whole = !sample_rows;            // the sample is all rows
    k_quantiles<<<F, TB, 0, stream>>>(w.ka, m, max_bins, whole, out_edges, ld_edges, out_nedges, out_scales, out_medians,
                                      w.need_std, w.br, w.missed, n);
    k_std_scale<<<F, ST, 0, stream>>>(w.orig, reinterpret_cast<float*>(w.kb), m, w.need_std, out_scales);
    if (whole) return launch_status("yabt_bin_fit launch");
    // medians over all n rows
    const int fw = std::min(F, MT);
    const dim3 pass((unsigned)launch_grid(n, MT / fw * 64, 2048), (unsigned)((F + fw - 1) / fw));
    k_median_pass<<<pass, MT, 0, stream>>>(X, ldx, n, F, fw, w.br, w.kb, m);
    k_median_finish<<<F, 1024, 0, stream>>>(w.br, w.kb, m, w.cnt, w.missed, out_medians);
    const dim3 grid((unsigned)launch_grid(max(n, (int64_t)1), TB / HT * 8, 1024), (unsigned)((F + HT - 1) / HT));
    k_select_init<<<(F + 63) / 64, 64, 0, stream>>>(w.missed, w.cnt, F, w.sel_state, w.sel_hist);
    for (int shift = 24; shift >= 0; shift -= 8) {
        k_select_hist<<<grid, TB, 0, stream>>>(w.missed, w.br, X, ldx, n, F, shift, w.sel_state, w.sel_hist);
        k_select_step<<<(F + 63) / 64, 64, 0, stream>>>(w.missed, F, w.sel_state, w.sel_hist);
    }
    k_select_finish<<<(F + 63) / 64, 64, 0, stream>>>(w.missed, w.br, w.cnt, F, w.sel_state, out_medians);
    return launch_status("yabt_bin_fit launch");
}

int yabt_bin_transform(const float* X, int64_t ldx, int64_t n, int F, const float* edges, int64_t ld_edges,
                       const int32_t* nedges, const float* medians, uint8_t* out_fm, int64_t ld_fm, uint8_t* out_rm,
                       int64_t ld_rm, float* out_imputed, int64_t ld_imputed, hipStream_t stream) {
    if (n < 0 || F < 1 || ldx < F || ld_edges < 1 || (out_fm && ld_fm < n) || (out_imputed && ld_imputed < F))
        return fail(-2, "yabt_bin_transform: bad sizes");
    if (out_rm && ld_rm < F) return fail(-2, "yabt_bin_transform: row-major output needs ld_rm >= F");
    if (!X || !edges || !nedges || !medians || !(out_fm || out_rm || out_imputed))
        return fail(-2, "yabt_bin_transform: null pointer argument");
    if (n == 0) return 0;
    const int even = (F + TFEAT - 1) / TFEAT, fg = ((F + even - 1) / even + 3) / 4 * 4, groups = (F + fg - 1) / fg;
    const int trl = transform_rows_log2(n, F, fg, groups);
    // 16-byte row stores when every 16-feature tile of every row is 16-byte aligned
    const TransformArgs A{X, ldx, n, F, fg, trl, edges, ld_edges, nedges, medians, out_fm, ld_fm, out_rm, ld_rm, out_imputed,
                          ld_imputed, out_fm && ld_fm % 16 == 0 && aligned16(out_fm),
                          out_rm && ld_rm % 16 == 0 && aligned16(out_rm)};
    const size_t lds = (size_t)fg * (TSTRIDE * 4 + 4 + (1 << trl) + 4);
    // as many blocks as are resident stay for all tiles: each loads its edges once
    const int resident = 256 * (int)std::min<size_t>(2048 / TT, 160 * 1024 / (lds + 64));
    const dim3 grid((unsigned)launch_grid(n, 1 << trl, std::max(1, resident / groups)), (unsigned)groups);
    k_transform<<<grid, TT, lds, stream>>>(A);
    return launch_status("yabt_bin_transform launch");
}

}  // extern "C"
