// k_accept.hip — fused verify-accept over the k+1 logits rows of one verify
// step, batched over requests.
//
// Greedy mode restates the accept loop of engine/speculative.go:191-208 with
// argmaxLogit (:263-271): draft i is accepted iff the first maximum of row i
// equals it. Stochastic mode is speculative sampling with a one-hot draft
// (no reference counterpart): accept iff u < p(d), else resample from p with
// d removed; the target p follows engine/sampling.go:60-119 (drop NaN/-Inf,
// top-k in (logit desc, id asc) order, weights exp(float64(logit - max) / T),
// top-p smallest prefix).
//
// Kernels (the passes over a row are separate launches so that the exact row
// maximum is known before any exponential is taken):
//   stats:    per (request, row, chunk): maximum and its first index.
// greedy and untruncated stochastic:
//   weights:  (stochastic) per chunk: float64 sum of the weights with the
//             draft removed, and the draft's own weight.
//   finalize: one workgroup per request walks the rows in order, decides,
//             and for a rejection or the bonus row draws by inverse CDF
//             in index order (chunk prefix, then a scan inside the chunk).
// top-k / top-p:
//   bins:     per (row, chunk) histogram of the row over equal steps of the
//             logit below the row maximum.
//   collect:  the bin that holds the cut, and its members (top-k: every
//             member down to it) as a candidate list.
//   cut:      one workgroup per row finds the exact cut among the candidates
//             (or over the whole row when they do not fit), and the weight
//             sums of the kept set.
//   resample: decides every request, and sums the kept weights of the one
//             row it draws from, per chunk.
//   pick:     the draw, as finalize makes it.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <type_traits>

#include "accept_math.h"
#include "internal.h"

namespace yk {
namespace {

struct Stat {
    float v;
    int i;
};

// a beats b: larger value, or equal value and lower index. NaN never wins.
__device__ __forceinline__ bool beats(float av, int ai, float bv, int bi) {
    return av > bv || (av == bv && ai < bi);
}

struct Geo {
    int B, R, k, V, C, L;
    uint64_t stride;
    int ds;  // int32 elements between consecutive requests' drafts
};

__device__ __forceinline__ const float *row_ptr(const float *logits, const Geo &g, int b, int row) {
    return logits + ((uint64_t)b * g.R + row) * g.stride;
}

// Bytes of truncation scratch per (request, row, chunk), and the sums of a
// chunk's logits (up to 1e6 in size) that set the truncation's bin width.
constexpr uint64_t kRowArea = 3072;
struct Moments {
    float n, s1, s2, pad;
};

__device__ __forceinline__ uint8_t *row_area(uint8_t *area, const Geo &g, int b, int row) {
    return area + ((uint64_t)b * g.R + row) * g.C * kRowArea;
}

// Per (request, row, chunk) maximum (MOM: and the moments, at the start of
// the row's area). A chunk of L (a multiple of 4) logits is read by `wpc`
// waves (1: four chunks per workgroup, for short chunks; 4: one chunk per
// workgroup), with 16-byte loads when the rows are 16-byte aligned. The
// maximum under `beats` does not depend on the order in which elements are
// visited, so the split does not change the result.
template <bool MOM>
__global__ __launch_bounds__(256) void accept_stats_kernel(const float *__restrict__ logits, Geo g,
                                                           Stat *__restrict__ stats, int vec, int wpc,
                                                           uint8_t *__restrict__ area) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int c = blockIdx.x * (4 / wpc) + wave / wpc, row = blockIdx.y, b = blockIdx.z;
    const int t = (wave % wpc) * 64 + lane, nt = wpc * 64;
    const bool live = c < g.C;
    float bv = -INFINITY;
    int bi = INT_MAX;
    float mn = 0.f, m1 = 0.f, m2 = 0.f;
    auto take = [&](float v, int j) __attribute__((always_inline)) {
        if (beats(v, j, bv, bi)) { bv = v; bi = j; }
        if (MOM && fabsf(v) <= 1e6f) {
            mn += 1.f;
            m1 += v;
            m2 = fmaf(v, v, m2);
        }
    };
    if (live) {
        const float *p = row_ptr(logits, g, b, row);
        const int begin = c * g.L;
        const int end = min(begin + g.L, g.V);
        if (vec) {
            const int end4 = begin + ((end - begin) & ~3);
            auto take4 = [&](const float4 v, int j) __attribute__((always_inline)) {
                take(v.x, j);
                take(v.y, j + 1);
                take(v.z, j + 2);
                take(v.w, j + 3);
            };
            int j = begin + t * 4;
            // four 16-byte loads in flight per thread
            for (; j + 3 * nt * 4 < end4; j += 4 * nt * 4) {
                float4 v[4];
#pragma unroll
                for (int u = 0; u < 4; u++) v[u] = *reinterpret_cast<const float4 *>(p + j + u * nt * 4);
#pragma unroll
                for (int u = 0; u < 4; u++) take4(v[u], j + u * nt * 4);
            }
            for (; j < end4; j += nt * 4) take4(*reinterpret_cast<const float4 *>(p + j), j);
            const int jt = end4 + t;
            if (jt < end) take(p[jt], jt);
        } else {
            for (int j = begin + t; j < end; j += nt) take(p[j], j);
        }
    }
    for (int off = 32; off > 0; off >>= 1) {
        const float ov = __shfl_xor(bv, off);
        const int oi = __shfl_xor(bi, off);
        if (beats(ov, oi, bv, bi)) {
            bv = ov;
            bi = oi;
        }
        if (MOM) {
            mn += __shfl_xor(mn, off);
            m1 += __shfl_xor(m1, off);
            m2 += __shfl_xor(m2, off);
        }
    }
    Moments *mom = MOM && live ? reinterpret_cast<Moments *>(row_area(area, g, b, row)) + c : nullptr;
    if (wpc == 1) {
        if (live && lane == 0) {
            stats[((uint64_t)b * g.R + row) * g.C + c] = Stat{bv, bi};
            if (MOM) *mom = Moments{mn, m1, m2, 0.f};
        }
        return;
    }
    __shared__ Stat ws[4];
    __shared__ Moments wm[4];
    if (lane == 0) {
        ws[wave] = Stat{bv, bi};
        wm[wave] = Moments{mn, m1, m2, 0.f};
    }
    __syncthreads();
    if (threadIdx.x == 0 && live) {
        Stat s = ws[0];
        Moments m = wm[0];
        for (int w = 1; w < 4; w++) {
            if (beats(ws[w].v, ws[w].i, s.v, s.i)) s = ws[w];
            m.n += wm[w].n;
            m.s1 += wm[w].s1;
            m.s2 += wm[w].s2;
        }
        stats[((uint64_t)b * g.R + row) * g.C + c] = s;
        if (MOM) *mom = m;
    }
}

// Truncation cut of one row (top-k / top-p): an element is kept iff its
// order key is above `key`, or equal to it with an id of at most `id`. The
// default {0, INT_MAX} keeps every valid logit.
struct Cut {
    uint32_t key;
    int32_t id;
};

// Monotone map of a float onto uint32 (larger logit, larger key). -0 maps
// with +0, since the sampler's sort compares values (sampling.go:84-89).
__device__ __forceinline__ uint32_t order_key(float l) {
    uint32_t u = __float_as_uint(l);
    if ((u << 1) == 0u) u = 0u;
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

__device__ __forceinline__ float key_value(uint32_t key) {
    return __uint_as_float((key & 0x80000000u) ? (key & 0x7fffffffu) : ~key);
}

// NaN and -Inf are dropped (sampling.go:75-80).
__device__ __forceinline__ bool valid_logit(float l) { return l == l && l != -INFINITY; }

__device__ __forceinline__ bool in_cut(uint32_t key, int j, const Cut &c) {
    return key > c.key || (key == c.key && j <= c.id);
}

// The exponential's table in LDS: a thread's entry is loaded at a kernel's
// start and put down just before its first barrier, behind its other loads.
__device__ __forceinline__ ExpEntry exp_entry() { return kExpTab[threadIdx.x & 15]; }
__device__ __forceinline__ void put_exp_entry(ExpEntry *tab, const ExpEntry &e) {
    if (threadIdx.x < 16) tab[threadIdx.x] = e;
}

// The weight of a logit, zero outside the cut.
__device__ __forceinline__ double weight_of(float l, int j, float mx, const Temp &t, const Cut &c, const ExpEntry *tab) {
    if (!valid_logit(l) || !in_cut(order_key(l), j, c)) return 0.0;
    return soft_weight(l, mx, t, tab);
}

// Wave 0 of a workgroup: the row's maximum and its first index over the
// chunk statistics, in every lane.
__device__ __forceinline__ Stat wave_best(const Stat *__restrict__ st, int C) {
    const int lane = threadIdx.x & 63;
    Stat s{-INFINITY, INT_MAX};
    for (int cc = lane; cc < C; cc += 64)
        if (beats(st[cc].v, st[cc].i, s.v, s.i)) s = st[cc];
    for (int off = 32; off > 0; off >>= 1) {
        const float ov = __shfl_xor(s.v, off);
        const int oi = __shfl_xor(s.i, off);
        if (beats(ov, oi, s.v, s.i)) s = Stat{ov, oi};
    }
    return s;
}

__global__ __launch_bounds__(256) void accept_weights_kernel(const float *__restrict__ logits, Geo g,
                                                             const int32_t *__restrict__ drafts,
                                                             const Stat *__restrict__ stats, Temp t,
                                                             double *__restrict__ sums,
                                                             double *__restrict__ wdraft) {
    const int c = blockIdx.x, row = blockIdx.y, b = blockIdx.z;
    const float *p = row_ptr(logits, g, b, row);
    __shared__ float mx_s;
    __shared__ ExpEntry tab[16];
    const ExpEntry entry = exp_entry();
    if (threadIdx.x < 64) {
        const Stat s = wave_best(stats + ((uint64_t)b * g.R + row) * g.C, g.C);
        if (threadIdx.x == 0) mx_s = s.v;
    }
    put_exp_entry(tab, entry);
    __syncthreads();
    const float mx = mx_s;
    const int d = row < g.k ? drafts[(uint64_t)b * g.ds + row] : -1;
    const int begin = c * g.L;
    const int end = min(begin + g.L, g.V);
    double acc = 0.0;
    auto weigh = [&](float l) __attribute__((always_inline)) {
        const double w = soft_weight(l, mx, t, tab);
        return valid_logit(l) ? w : 0.0;
    };
    // eight logit loads in flight per thread; the sum keeps index order
    constexpr int kU = 8;
    int j = begin + threadIdx.x;
    for (; j + (kU - 1) * 256 < end; j += kU * 256) {
        float l[kU];
#pragma unroll
        for (int u = 0; u < kU; u++) l[u] = p[j + u * 256];
        double wv[kU];
#pragma unroll
        for (int u = 0; u < kU; u++) wv[u] = weigh(l[u]);
#pragma unroll
        for (int u = 0; u < kU; u++) {
            const double w = wv[u];
            if (j + u * 256 == d)
                wdraft[(uint64_t)b * g.R + row] = w;
            else
                acc += w;
        }
    }
    for (; j < end; j += 256) {
        const double w = weigh(p[j]);
        if (j == d)
            wdraft[(uint64_t)b * g.R + row] = w;
        else
            acc += w;
    }
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off);
    __shared__ double ws[4];
    if ((threadIdx.x & 63) == 0) ws[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) sums[((uint64_t)b * g.R + row) * g.C + c] = ws[0] + ws[1] + ws[2] + ws[3];
}

// ---------------------------------------------------------------- truncation
// Per-row cut for top-k / top-p (sampling.go:84-113) without sorting.
//
// A histogram over equal steps of the logit below the row maximum, one
// workgroup per (row, chunk), leaves a few hundred candidates around the cut
// for any smooth distribution; one workgroup per row then orders those
// exactly. (A histogram over the top byte of the order key, as a radix
// selection has it, has about five buckets in use at once — an octave or two
// each — so the 64 lanes of an LDS atomic met on the same few addresses
// (95 us at 144 rows of 151936), and its boundary bucket still held 17
// thousand members, for three more passes of one workgroup per row (136 us).)
// Candidates without room in the row's area (thousands of rows leave each a
// few KB; a sorted row puts all of them into one wave's segment) are gathered
// once more by the row's workgroup, into its own list; before that such rows
// took the radix selection over the whole row, four more passes (2500 rows of
// 151936, T 1.5, top-p 0.9: 6.20 -> 3.13 ms, top-k 2000: 4.01 -> 2.39; 420
// sorted rows of 27205, top-k 1000: 247 -> 135 us). That is left for rows
// whose list is too short as well (a bin of many equal logits) or whose cut
// lies in the open last bin; it lists a bucket's members as soon as they fit,
// as it does the boundary bin's of a top-k set that is longer than the list.
//
// Scratch of one (request, row): C * kRowArea bytes of
//   Moments [C]              per-chunk sums behind the bin width
//   double or uint32 [HC][NB]  chunk histograms: weights, or counts with top-k
//   uint32 [segs]            candidates of each collecting wave
//   Member [segs][seg]       the candidates
constexpr int kBins = 1024;    // most bins of a histogram
constexpr int kBinWaves = 8;   // waves of a bins workgroup, a histogram each
// Rows cut without bins: up to kDirectMost logits (in LDS where they fit the
// list, see SelShared), and with top-k alone and a CU for every row up to
// kDirectTopK, from memory (us, from memory / through the bins: 8200 logits,
// top-k 40 34 / 37 at 1 row, 35 / 39 at 144 rows, top-k 1000 34 / 43 and 36 /
// 45; 16000, top-k 40 38 / 37 and 41 / 42, top-k 1000 41 / 44 and 45 / 49;
// 26307, top-k 40 48 / 38, 60 / 54).
constexpr int kDirectMost = 8192;
constexpr int kDirectTopK = 16384;
constexpr int kRankMost = 512;  // candidates ordered by counting

struct Member {
    float l;
    int j;
};

struct TruncGeo {
    int NB;    // bins
    int HC;    // histogram chunks of a row
    int KC;    // collecting chunks of a row (4 waves each)
    int seg;   // candidates of one collecting wave
    int cap;   // candidates of a row
    uint32_t bins_off, cnt_off, cand_off;  // in the row's area
};

// See wave_bin_map.
struct BinMap {
    float top, scale;
};

// What collect leaves for a row.
struct RowCut {
    Cut cut;
    double rest;   // kept weight without the draft
    double wd;     // the draft's kept weight
    double total;  // (collect -> cut) all weight, draft included
    double before;       // (collect -> cut) weight above the boundary bin, draft included
    double before_rest;  // ... without the draft
    float best_v;        // row maximum
    int best_i;
    int status;
    int bnd;      // (collect -> cut) the boundary bin
    BinMap map;   // (collect -> cut) the row's bins
};
// The candidates decide; nothing is cut; scan the row; the candidates decide
// but have no room in the row's area; top-k keeps every valid logit; the
// boundary bin decides top-k's cut (the bins above it are too long a list).
enum { kCutFound = 0, kCutAll = 1, kCutRow = 2, kCutGather = 3, kCutNoTopK = 4, kCutBin = 5 };

// A row's record lies at the end of its area.
__device__ __forceinline__ RowCut &row_cut(uint8_t *area, const Geo &g, int b, int row) {
    return *reinterpret_cast<RowCut *>(row_area(area, g, b, row) + g.C * kRowArea - sizeof(RowCut));
}

// The bins of a row: `scale` of them per unit of logit below `top`, over the
// range down to three standard deviations under the mean in NB steps. Weighed
// bins (COUNT false) start at the maximum and end at 48 T if that is less (the
// weights below it are under 1e-20 of the largest); counted ones start at most
// eight deviations above the mean, or one logit far above the others would
// leave these a few bins (13 x 9 x 127103, top-k 5000, one logit of 1e4:
// 383 -> 134 us).
// Every workgroup of a row computes the same values (fixed order, every fused
// operation written out), so the bins of its passes agree. Wave 0 of a workgroup.
template <bool COUNT>
__device__ __forceinline__ BinMap wave_bin_map(const Moments *__restrict__ m, int C, float mx, const Temp &t, int NB) {
    const int lane = threadIdx.x & 63;
    float n = 0.f, s1 = 0.f, s2 = 0.f;
    for (int c = lane; c < C; c += 64) {
        n += m[c].n;
        s1 += m[c].s1;
        s2 += m[c].s2;
    }
    for (int off = 32; off > 0; off >>= 1) {
        n += __shfl_xor(n, off);
        s1 += __shfl_xor(s1, off);
        s2 += __shfl_xor(s2, off);
    }
    const float cap = fminf(fmaxf(48.f * (float)t.t, 1e-30f), 1e30f);
    const float mean = s1 / n;
    const float sd = sqrtf(fmaxf(fmaf(-mean, mean, s2 / n), 1e-6f * mean * mean));
    const float top = COUNT ? fminf(mx, fmaf(8.f, sd, mean)) : mx;  // (mx if n is 0)
    float range = fmaf(3.f, sd, top - mean);
    if (!(range > 1e-30f && range < (COUNT ? 1e30f : cap))) range = cap;
    return BinMap{top, (float)NB / range};
}

// Monotone: a larger logit never has a larger bin (each operation rounds
// monotonically; the first bin takes what is above `top`, the last one is
// open, and takes a NaN).
__device__ __forceinline__ int bin_of(float l, const BinMap &m, int NB) {
    return (int)fmaxf(fminf((m.top - l) * m.scale, (float)(NB - 1)), 0.f);
}

// Histogram of one chunk of a row, the draft's weight left out. COUNT (with
// top-k): members; otherwise their float64 weights. Each wave has its own
// histogram (an atomic's lanes add in a fixed order, waves would not), the
// waves are added in wave order.
template <bool COUNT>
__global__ __launch_bounds__(64 * kBinWaves) void accept_bins_kernel(const float *__restrict__ logits, Geo g, TruncGeo tg,
                                                                     const int32_t *__restrict__ drafts,
                                                                     const Stat *__restrict__ stats, Temp t,
                                                                     uint8_t *__restrict__ area) {
    using T = typename std::conditional<COUNT, uint32_t, double>::type;
    extern __shared__ __attribute__((aligned(16))) uint8_t bins_dyn[];
    T *hist = reinterpret_cast<T *>(bins_dyn);  // [wave][NB]
    __shared__ float mx_s;
    __shared__ BinMap map_s;
    __shared__ ExpEntry tab[16];
    const ExpEntry entry = exp_entry();
    constexpr int kT = 64 * kBinWaves;
    const int c = blockIdx.x, row = blockIdx.y, b = blockIdx.z;
    const float *p = row_ptr(logits, g, b, row);
    uint8_t *ra = row_area(area, g, b, row);
    const int begin = (int)((int64_t)g.V * c / tg.HC), end = (int)((int64_t)g.V * (c + 1) / tg.HC);
    constexpr int kU = 8;  // loads in flight per thread
    float lv[kU];
    int j0 = begin + threadIdx.x;
#pragma unroll
    for (int u = 0; u < kU; u++) lv[u] = j0 + kT * u < end ? p[j0 + kT * u] : NAN;
    for (int i = threadIdx.x; i < kBinWaves * tg.NB; i += kT) hist[i] = (T)0;
    if (threadIdx.x < 64) {
        const Stat s = wave_best(stats + ((uint64_t)b * g.R + row) * g.C, g.C);
        const BinMap map = wave_bin_map<COUNT>(reinterpret_cast<const Moments *>(ra), g.C, s.v, t, tg.NB);
        if (threadIdx.x == 0) {
            mx_s = s.v;
            map_s = map;
        }
    }
    put_exp_entry(tab, entry);
    __syncthreads();
    const float mx = mx_s;
    const BinMap map = map_s;
    const int d = !COUNT && row < g.k ? drafts[(uint64_t)b * g.ds + row] : -1;
    T *mine = hist + (threadIdx.x >> 6) * tg.NB;
    while (j0 < end) {
        float nx[kU];
        const int jn = j0 + kU * kT;
#pragma unroll
        for (int u = 0; u < kU; u++) nx[u] = jn + kT * u < end ? p[jn + kT * u] : NAN;
        if constexpr (COUNT) {
#pragma unroll
            for (int u = 0; u < kU; u++)
                if (valid_logit(lv[u])) atomicAdd(&mine[bin_of(lv[u], map, tg.NB)], 1u);
        } else {
            // four weights at a time without branches: their chains of
            // dependent float64 operations interleave
            constexpr int kW = 4;
#pragma unroll
            for (int u0 = 0; u0 < kU; u0 += kW) {
                double w[kW];
#pragma unroll
                for (int u = 0; u < kW; u++) w[u] = soft_weight(lv[u0 + u], mx, t, tab);
#pragma unroll
                for (int u = 0; u < kW; u++) {
                    const float l = lv[u0 + u];
                    if (valid_logit(l) && w[u] != 0.0 && j0 + kT * (u0 + u) != d)
                        unsafeAtomicAdd(&mine[bin_of(l, map, tg.NB)], w[u]);
                }
            }
        }
#pragma unroll
        for (int u = 0; u < kU; u++) lv[u] = nx[u];
        j0 = jn;
    }
    __syncthreads();
    T *out = reinterpret_cast<T *>(ra + tg.bins_off) + (uint64_t)c * tg.NB;
    for (int i = threadIdx.x; i < tg.NB; i += kT) {
        T v = hist[i];
#pragma unroll
        for (int w = 1; w < kBinWaves; w++) v += hist[w * tg.NB + i];
        out[i] = v;
    }
}

// The boundary bin of a row — the first where the members reach top_k
// (COUNT) or the weight reaches the top_p share — and the chunk's members of
// it (COUNT: of it and the bins above), each wave into its own segment in
// (iteration, lane) order. Every workgroup of a row finds the boundary again
// (a few KB from L2); the first one writes it down.
template <bool COUNT>
__global__ __launch_bounds__(256) void accept_collect_kernel(const float *__restrict__ logits, Geo g, TruncGeo tg,
                                                             const int32_t *__restrict__ drafts,
                                                             const Stat *__restrict__ stats, int top_k, float top_p,
                                                             Temp t, uint8_t *__restrict__ area) {
    using T = typename std::conditional<COUNT, uint32_t, double>::type;
    __shared__ float mx_s;
    __shared__ BinMap map_s;
    __shared__ int best_i_s, bnd_s;
    __shared__ T wave_tot[4];
    __shared__ T before_s, upto_s;
    __shared__ ExpEntry tab[16];
    const ExpEntry entry = exp_entry();
    const int c = blockIdx.x, row = blockIdx.y, b = blockIdx.z;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const float *p = row_ptr(logits, g, b, row);
    uint8_t *ra = row_area(area, g, b, row);
    // thread i owns bins [per i, per i + per): the chunks' sums in chunk order
    constexpr int kPer = kBins / 256;
    const int per = max(1, tg.NB / 256), lo = (int)threadIdx.x * per;
    T h[kPer];
#pragma unroll
    for (int i = 0; i < kPer; i++) h[i] = (T)0;
    const T *hist = reinterpret_cast<const T *>(ra + tg.bins_off);
    for (int ch = 0; ch < tg.HC; ch++)
#pragma unroll
        for (int i = 0; i < kPer; i++)
            if (i < per && lo + i < tg.NB) h[i] += hist[(uint64_t)ch * tg.NB + lo + i];
    if (threadIdx.x < 64) {
        const Stat s = wave_best(stats + ((uint64_t)b * g.R + row) * g.C, g.C);
        const BinMap map = wave_bin_map<COUNT>(reinterpret_cast<const Moments *>(ra), g.C, s.v, t, tg.NB);
        if (threadIdx.x == 0) {
            mx_s = s.v;
            map_s = map;
            best_i_s = s.i;
            bnd_s = tg.NB;
            before_s = upto_s = (T)0;
        }
    }
    T sum = (T)0;
#pragma unroll
    for (int i = 0; i < kPer; i++) sum += h[i];
    T inc = sum;  // inclusive prefix over the wave
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const T v = __shfl_up(inc, off);
        if (lane >= off) inc += v;
    }
    T exc = __shfl_up(inc, 1);
    if (lane == 0) exc = (T)0;
    if (lane == 63) wave_tot[wave] = inc;
    put_exp_entry(tab, entry);
    __syncthreads();
    const float mx = mx_s;
    const BinMap map = map_s;
    T tot = (T)0;
    for (int w = 0; w < 4; w++) {
        if (w == wave) exc += tot;
        tot += wave_tot[w];
    }
    // the draft's own weight and bin
    const int d = row < g.k ? drafts[(uint64_t)b * g.ds + row] : -1;
    double wd = 0.0;
    int dbin = tg.NB;
    if (!COUNT && d >= 0 && d < g.V && valid_logit(p[d])) {
        wd = soft_weight(p[d], mx, t, tab);
        dbin = bin_of(p[d], map, tg.NB);
    }
    const double total = (double)tot + wd;
    {
        T cum = exc;
        int pick = -1;
        T before = (T)0, upto = (T)0;
#pragma unroll
        for (int i = 0; i < kPer; i++) {
            if (i >= per || lo + i >= tg.NB || pick >= 0) continue;
            const T next = cum + h[i];
            bool hit;
            if constexpr (COUNT) hit = next >= (uint32_t)top_k;
            else hit = next + (lo + i >= dbin ? wd : 0.0) >= (double)top_p * total && (h[i] > 0.0 || lo + i == dbin);
            if (hit) {
                pick = lo + i;
                before = cum;
                upto = next;
            }
            cum = next;
        }
        if (pick >= 0) atomicMin(&bnd_s, pick);
        __syncthreads();
        if (pick >= 0 && bnd_s == pick) {
            before_s = before;
            upto_s = upto;
        }
    }
    __syncthreads();
    const int bnd = bnd_s;
    int status = kCutFound;
    if (COUNT) {
        if (tot <= (T)top_k) status = kCutNoTopK;
        else if (bnd >= tg.NB - 1) status = kCutRow;
        else if (upto_s > (T)tg.cap) status = upto_s - before_s <= (T)(tg.cap / 4 * 3) ? kCutBin : kCutRow;
        else if (upto_s > (T)(tg.KC * 4 * tg.seg)) status = kCutGather;
    } else {
        if (!(total > 0.0) || isinf(total) || bnd >= tg.NB) status = kCutAll;
        else if (bnd == tg.NB - 1) status = kCutRow;
    }
    if (c == 0 && threadIdx.x == 0) {
        RowCut &o = row_cut(area, g, b, row);
        o.cut = Cut{0u, INT_MAX};
        o.rest = (double)tot;  // (kCutAll)
        o.wd = wd;
        o.total = total;
        o.before = (double)before_s + (dbin < bnd ? wd : 0.0);
        o.before_rest = (double)before_s;
        o.best_v = mx;
        o.best_i = best_i_s;
        o.status = status;
        o.bnd = bnd;
        o.map = map;
    }
    const int w = c * 4 + wave;
    uint32_t found = 0u;
    if (status == kCutFound) {
        Member *out = reinterpret_cast<Member *>(ra + tg.cand_off) + (uint64_t)w * tg.seg;
        const int begin = (int)((int64_t)g.V * c / tg.KC), end = (int)((int64_t)g.V * (c + 1) / tg.KC);
        constexpr int kU = 8;
        for (int j0 = begin + threadIdx.x; j0 - (int)threadIdx.x < end; j0 += kU * 256) {
            float l[kU];
#pragma unroll
            for (int u = 0; u < kU; u++) l[u] = j0 + 256 * u < end ? p[j0 + 256 * u] : NAN;
#pragma unroll
            for (int u = 0; u < kU; u++) {
                const int bin = bin_of(l[u], map, tg.NB);
                const bool take = valid_logit(l[u]) && (COUNT ? bin <= bnd : bin == bnd);
                const uint64_t m = __ballot(take);
                if (!m) continue;
                const uint32_t at = found + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
                if (take && at < (uint32_t)tg.seg) out[at] = Member{l[u], j0 + 256 * u};
                found += (uint32_t)__popcll(m);
            }
        }
    }
    if (lane == 0) reinterpret_cast<uint32_t *>(ra + tg.cnt_off)[w] = found;
}

// ---- exact cut among a row's elements or its candidates: radix selection
// over the 32-bit order key, histograms in LDS. Each wave fills its own
// histogram and the waves are combined in wave order, so weight sums do not
// depend on wave scheduling.
//
// A workgroup of W waves: sixteen and a long candidate list while every row
// can have a CU, else eight and a list that lets a CU hold two workgroups
// (2160 rows of 8192, top-k 40: 202 -> 132 us; 1350 of 8200, top-k 1000: 139
// -> 99; 2070 of 151936, T 1.5, top-p 0.9: 1.59 -> 1.45 ms).
constexpr int cand_most(int W) { return W == 16 ? 8192 : 6144; }

template <int W>
struct SelShared {
    uint32_t cnt[W][256];
    double wsum[W][256];
    uint32_t tc[256];
    double tw[256];
    uint32_t prefix;    // digits chosen so far
    int bucket;         // bucket chosen by the last scan (-1: none)
    uint32_t before_c;  // count of the buckets ahead of it in scan order
    double before_w;    // their weight
    double total_w;     // all weight of the first pass
    uint32_t total_c;
    int id;             // result of an id selection
    uint32_t seg_n[W];  // gather: members of each wave
    ExpEntry tab[16];
};

// The elements a selection runs over: a candidate list in LDS, or (list
// null) the whole row.
struct SelSrc {
    const float *p;
    int V;
    const Member *list;
    int n;
    bool top;  // the list is the row's top, top_k members or more
};

// f(logit, id) for every valid element, in a fixed order per thread.
template <int W, class F>
__device__ __forceinline__ void for_each(const SelSrc &src, F f) {
    constexpr int kStride = W * 64;
    if (src.list) {
        for (int i = threadIdx.x; i < src.n; i += kStride)
            if (valid_logit(src.list[i].l)) f(src.list[i].l, src.list[i].j);
        return;
    }
    // eight loads in flight per thread (the row is read from L2 / the
    // Infinity Cache once per pass: latency, not bandwidth, bounds the pass)
    constexpr int kU = 8;
    for (int j0 = threadIdx.x; j0 < src.V; j0 += kU * kStride) {
        float l[kU];
#pragma unroll
        for (int u = 0; u < kU; u++) l[u] = j0 + u * kStride < src.V ? src.p[j0 + u * kStride] : NAN;
#pragma unroll
        for (int u = 0; u < kU; u++)
            if (valid_logit(l[u])) f(l[u], j0 + u * kStride);
    }
}

// Histogram of the next digit over the elements that `sel` admits.
template <bool WEIGH, int W, class Sel>
__device__ __forceinline__ void hist_pass(const SelSrc &src, float mx, const Temp &t, SelShared<W> &s, int shift, Sel sel) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (int b = lane; b < 256; b += 64) {
        s.cnt[wave][b] = 0u;
        if (WEIGH) s.wsum[wave][b] = 0.0;
    }
    __syncthreads();
    for_each<W>(src, [&](float l, int j) __attribute__((always_inline)) {
        const uint32_t k = order_key(l);
        if (!sel(k, j)) return;
        const int b = (k >> shift) & 255u;
        const double w = WEIGH ? soft_weight(l, mx, t, s.tab) : 0.0;
        auto add = [&](uint32_t n) __attribute__((always_inline)) {
            atomicAdd(&s.cnt[wave][b], n);
            if (WEIGH) unsafeAtomicAdd(&s.wsum[wave][b], (double)n * w);
        };
        // the lanes that share the first one's key add once (64 adds to one
        // address, one after the other, are what a row of equal logits costs
        // otherwise)
        const bool same = k == (uint32_t)__builtin_amdgcn_readfirstlane((int)k);
        const uint64_t m = __ballot(same);
        if (!same) add(1u);
        else if (lane == __ffsll((unsigned long long)m) - 1) add((uint32_t)__popcll(m));
    });
    __syncthreads();
    if (threadIdx.x < 256) {
        uint32_t c = 0u;
        double w = 0.0;
        for (int q = 0; q < W; q++) {
            c += s.cnt[q][threadIdx.x];
            if (WEIGH) w += s.wsum[q][threadIdx.x];
        }
        s.tc[threadIdx.x] = c;
        s.tw[threadIdx.x] = w;
    }
    __syncthreads();
}

// Wave 0: walk the buckets in scan order (descending keys, or ascending for
// ids) to the first non-empty one where the running count reaches need_c (or
// the running weight reaches need_w); append its digit to the prefix. Lane l
// takes scan positions [4 l, 4 l + 4): its running start is the
// lanes-before-it prefix (a fixed shuffle tree, so the sums are the same on
// every run), then its own buckets in order; the first lane that reaches
// the need picks. (One thread walking 256 LDS entries took ~16 us a pass.)
template <int W>
__device__ __forceinline__ void scan_buckets(SelShared<W> &s, bool descending, bool by_weight, uint32_t need_c,
                                             double need_w, int shift) {
    const int lane = threadIdx.x & 63;
    uint32_t bc[4], lc = 0u;
    double bw[4], lw = 0.0;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int q = 4 * lane + i, b = descending ? 255 - q : q;
        bc[i] = s.tc[b];
        bw[i] = s.tw[b];
        lc += bc[i];
        lw += bw[i];
    }
    uint32_t ic = lc;  // inclusive prefix over lanes
    double iw = lw;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t tc = __shfl_up(ic, off);
        const double tw = __shfl_up(iw, off);
        if (lane >= off) {
            ic += tc;
            iw += tw;
        }
    }
    const uint32_t ec = __shfl_up(ic, 1);
    const double ew = __shfl_up(iw, 1);
    uint32_t c = s.before_c + (lane ? ec : 0u);
    double w = s.before_w + (lane ? ew : 0.0);
    int pick = -1;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        if (pick >= 0 || !bc[i]) continue;
        if (by_weight ? (w + bw[i] >= need_w) : (c + bc[i] >= need_c)) {
            pick = 4 * lane + i;
            continue;
        }
        c += bc[i];
        w += bw[i];
    }
    const uint64_t hit = __ballot(pick >= 0);
    const int first = hit ? __ffsll((unsigned long long)hit) - 1 : -1;
    if (first < 0) {
        if (lane == 0) s.bucket = -1;
        return;
    }
    if (lane == first) {
        const int b = descending ? 255 - pick : pick;
        s.bucket = b;
        s.before_c = c;
        s.before_w = w;
        s.prefix |= (uint32_t)b << shift;
    }
}

// Wave 0: the sums of the 256 bucket counts and weights (fixed tree order).
template <int W>
__device__ __forceinline__ void bucket_totals(const SelShared<W> &s, uint32_t *c_out, double *w_out) {
    const int lane = threadIdx.x & 63;
    uint32_t c = 0u;
    double w = 0.0;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        c += s.tc[4 * lane + i];
        w += s.tw[4 * lane + i];
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        c += __shfl_xor(c, off);
        w += __shfl_xor(w, off);
    }
    *c_out = c;
    *w_out = w;
}

// The need-th smallest id (1-based) among the elements with order key `key`
// that lie inside `cut`.
template <int W>
__device__ int select_id(const float *p, int V, SelShared<W> &s, uint32_t key, Cut cut, uint32_t need) {
    // One ordered sweep: 8 slices of W * 64 consecutive ids per
    // step, the matches of each wave counted by ballot, and the step where
    // the running count reaches `need` resolved by rank.
    constexpr int kT = W * 64, kU = 8;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (threadIdx.x == 0) s.id = INT_MAX;
    uint32_t before = 0u;
    for (int base = 0; base < V; base += kU * kT) {
        float l[kU];
#pragma unroll
        for (int u = 0; u < kU; u++) {
            const int j = base + u * kT + threadIdx.x;
            l[u] = p[min(j, V - 1)];
        }
        bool m[kU];
        uint64_t bal[kU];
#pragma unroll
        for (int u = 0; u < kU; u++) {
            const int j = base + u * kT + threadIdx.x;
            m[u] = j < V && valid_logit(l[u]) && order_key(l[u]) == key && in_cut(key, j, cut);
            bal[u] = __ballot(m[u]);
            if (lane == 0) s.cnt[u][wave] = (uint32_t)__popcll(bal[u]);
        }
        __syncthreads();
        uint32_t tot = 0u;
        for (int q = 0; q < kU * W; q++) tot += s.cnt[q / W][q % W];
        if (before + tot >= need) {
            uint32_t r = before;
#pragma unroll
            for (int u = 0; u < kU; u++) {
                uint32_t pw = 0u;
                for (int q = 0; q < W; q++) pw += q < wave ? s.cnt[u][q] : 0u;
                const uint32_t rank = r + pw + (uint32_t)__popcll(bal[u] & ((1ull << lane) - 1ull)) + 1u;
                if (m[u] && rank == need) s.id = base + u * kT + threadIdx.x;
                for (int q = 0; q < W; q++) r += s.cnt[u][q];
            }
            break;
        }
        before += tot;
        __syncthreads();  // the counts are read before the next step overwrites them
    }
    __syncthreads();
    const int id = s.id;
    __syncthreads();  // every thread has read the result before the state is reused
    return id;
}

// The row's elements that `take` admits side by side in the list, by one
// workgroup: each wave fills a segment in (iteration, lane) order, then the
// segments close up. Returns their number, or -1 if a segment is too short.
// Waves take every W-th 64 ids, so a run of large logits spreads over them.
template <int W, class Take>
__device__ __forceinline__ int gather(const float *__restrict__ p, int V, Member *list, uint32_t *found_s, Take take) {
    constexpr int kT = 64 * W, kSeg = cand_most(W) / W, kPer = cand_most(W) / kT, kU = 8;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    uint32_t found = 0u;
    for (int j0 = threadIdx.x; j0 - (int)threadIdx.x < V && found <= (uint32_t)kSeg; j0 += kU * kT) {
        float l[kU];
#pragma unroll
        for (int u = 0; u < kU; u++) l[u] = j0 + kT * u < V ? p[j0 + kT * u] : NAN;
#pragma unroll
        for (int u = 0; u < kU; u++) {
            const bool in = valid_logit(l[u]) && take(l[u]);
            const uint64_t m = __ballot(in);
            const uint32_t at = found + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
            if (in && at < (uint32_t)kSeg) list[wave * kSeg + at] = Member{l[u], j0 + kT * u};
            found += (uint32_t)__popcll(m);
        }
    }
    if (lane == 0) found_s[wave] = found;
    __syncthreads();
    uint32_t at[W + 1];
    at[0] = 0u;
    bool ok = true;
#pragma unroll
    for (int q = 0; q < W; q++) {
        ok = ok && found_s[q] <= (uint32_t)kSeg;
        at[q + 1] = at[q] + found_s[q];
    }
    const int n = (int)at[W];
    Member m[kPer];
#pragma unroll
    for (int u = 0; u < kPer; u++) {
        const uint32_t i = threadIdx.x + u * kT;
        if (!ok || i >= (uint32_t)n) continue;
        uint32_t from = 0u;
#pragma unroll
        for (int q = 0; q < W; q++)
            if (i >= at[q]) from = q * kSeg + i - at[q];
        m[u] = list[from];
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kPer; u++) {
        const uint32_t i = threadIdx.x + u * kT;
        if (ok && i < (uint32_t)n) list[i] = m[u];
    }
    __syncthreads();
    return ok ? n : -1;
}

// The cut of one row by radix selection over src. With `tail` (candidates of
// one bin): the weight `before` lies ahead of src's elements, of `total`.
// `room` (src is the whole row): a list of cand_most(W) for the members of
// the chosen bucket once they are few enough, so that the later passes need
// not read the row. `bin_n` of them may be there already, those of the bin
// with top-k's cut, behind `bin_before` larger ones (16 rows of 53144, top-k
// 13286: 103 -> 73 us; with a bucket's list for top-p, 37 rows of 63461, top-k
// 15865, top-p 0.95: 222 -> 180).
template <int W>
__device__ __forceinline__ Cut radix_cut(const SelSrc src, SelShared<W> &s, float mx, const Temp t, int top_k, float top_p,
                                         bool tail, double before, double total, Member *room, int bin_n,
                                         uint32_t bin_before) {
    Cut cut{0u, INT_MAX};
    // (three quarters of the list: the waves' segments fill unevenly)
    auto narrow = [&](SelSrc &cur, uint32_t mask, uint32_t pre) __attribute__((always_inline)) {
        if (!room || cur.list || s.tc[s.bucket] > (uint32_t)(cand_most(W) / 4 * 3)) return;  // uniform
        const int n = gather<W>(src.p, src.V, room, s.seg_n, [=](float l) { return (order_key(l) & mask) == pre; });
        if (n < 0) return;
        cur.list = room;
        cur.n = n;
    };
    // top-k: the top_k-th element in (logit desc, id asc) order (sampling.go:90-92).
    if (top_k > 0) {
        SelSrc cur = src;
        if (bin_n > 0) {
            cur.list = room;
            cur.n = bin_n;
            cur.top = true;
        }
        if (threadIdx.x == 0) {
            s.prefix = 0u;
            s.before_c = bin_n > 0 ? bin_before : 0u;
            s.before_w = 0.0;
        }
        __syncthreads();
        bool all = false;
        for (int pass = 0; pass < 4; pass++) {
            const int shift = 24 - 8 * pass;
            const uint32_t mask = pass ? ~0u << (shift + 8) : 0u;
            const uint32_t pre = s.prefix;
            if (pass) narrow(cur, mask, pre);
            hist_pass<false>(cur, mx, t, s, shift, [=](uint32_t k, int) { return (k & mask) == pre; });
            if (threadIdx.x < 64) {
                uint32_t tot_c = s.total_c;
                if (pass == 0) {
                    double unused;
                    bucket_totals(s, &tot_c, &unused);
                    if (threadIdx.x == 0) s.total_c = tot_c;
                }
                if (cur.top || tot_c > (uint32_t)top_k) scan_buckets(s, true, false, (uint32_t)top_k, 0.0, shift);
            }
            __syncthreads();
            if (!cur.top && s.total_c <= (uint32_t)top_k) {
                all = true;
                break;
            }
        }
        if (!all) {
            const uint32_t key = s.prefix;
            const uint32_t need = (uint32_t)top_k - s.before_c;
            const uint32_t ties = s.tc[s.bucket];
            __syncthreads();
            cut.key = key;
            cut.id = need < ties ? select_id(src.p, src.V, s, key, Cut{0u, INT_MAX}, need) : INT_MAX;
        }
    }

    // top-p: the smallest prefix whose cumulative share reaches top_p
    // (sampling.go:104-113), within the top-k set.
    if (top_p > 0.0f && top_p < 1.0f) {
        __syncthreads();
        if (threadIdx.x == 0) {
            s.prefix = 0u;
            s.before_c = 0u;
            s.before_w = tail ? before : 0.0;
        }
        __syncthreads();
        SelSrc cur = src;
        bool found = true;
        for (int pass = 0; pass < 4 && found; pass++) {
            const int shift = 24 - 8 * pass;
            const uint32_t mask = pass ? ~0u << (shift + 8) : 0u;
            const uint32_t pre = s.prefix;
            const Cut ck = cut;
            if (pass) narrow(cur, mask, pre);
            hist_pass<true>(cur, mx, t, s, shift,
                            [=](uint32_t k, int j) { return in_cut(k, j, ck) && (k & mask) == pre; });
            if (threadIdx.x < 64) {
                double tot = s.total_w;
                if (pass == 0) {
                    uint32_t unused;
                    bucket_totals(s, &unused, &tot);
                    if (tail) tot = total;
                    if (threadIdx.x == 0) s.total_w = tot;
                }
                if (tot > 0.0 && !isinf(tot))
                    scan_buckets(s, true, true, 0u, (double)top_p * tot, shift);
                else if (threadIdx.x == 0)
                    s.bucket = -1;
            }
            __syncthreads();
            found = s.bucket >= 0;
        }
        if (found) {
            if (threadIdx.x == 0) {
                const uint32_t ties = s.tc[s.bucket];
                const uint32_t m = tie_members(s.before_w, soft_weight(key_value(s.prefix), mx, t, s.tab), s.total_w,
                                               (double)top_p, ties);
                s.before_c = m;  // kept members of the tie group
                s.total_c = ties;
            }
            __syncthreads();
            const uint32_t key = s.prefix, m = s.before_c, ties = s.total_c;
            __syncthreads();
            Cut nc{key, key == cut.key ? cut.id : INT_MAX};
            if (m < ties) nc.id = select_id(src.p, src.V, s, key, cut, m);
            cut = nc;
        }
    }
    return cut;
}

// Sum over the workgroup in wave order, in every thread.
template <int W>
__device__ __forceinline__ double block_sum(double v, double *waves) {
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) waves[threadIdx.x >> 6] = v;
    __syncthreads();
    double t = 0.0;
    for (int w = 0; w < W; w++) t += waves[w];
    return t;
}

// One workgroup per row: the exact cut, and the kept weight without the
// draft and of the draft. Up to kRankMost candidates are put in order by
// counting (thread i counts what lies ahead of candidate i) and their weights
// summed in that order (some 450 candidates of one row: 63 us a call; with the
// sums taken in the counting loop 82); more take the radix selection.
// `direct`: no candidates were collected, the row itself is taken (1: into LDS).
template <int W>
__global__ __launch_bounds__(64 * W, 4) void accept_cut_kernel(const float *__restrict__ logits, Geo g, TruncGeo tg,
                                                                    const int32_t *__restrict__ drafts,
                                                                    const Stat *__restrict__ stats, int top_k, float top_p,
                                                                    Temp t, uint8_t *__restrict__ area, int direct) {
    const int row = blockIdx.x, b = blockIdx.y;
    const float *p = row_ptr(logits, g, b, row);
    uint8_t *ra = row_area(area, g, b, row);
    RowCut &rc = row_cut(area, g, b, row);
    __shared__ SelShared<W> s;
    __shared__ double waves[W];
    __shared__ uint32_t seg_at[260];
    __shared__ int n_s, end_s, last_s;
    extern __shared__ __attribute__((aligned(16))) uint8_t cut_dyn[];
    Member *list = reinterpret_cast<Member *>(cut_dyn);
    RowCut in = rc;
    const ExpEntry entry = exp_entry();
    if (direct) {
        __shared__ Stat best_s;
        if (direct == 1)
            for (int j = threadIdx.x; j < g.V; j += 64 * W) list[j] = Member{p[j], j};
        if (threadIdx.x < 64) {
            const Stat best = wave_best(stats + ((uint64_t)b * g.R + row) * g.C, g.C);
            if (threadIdx.x == 0) best_s = best;
        }
        __syncthreads();
        in.status = kCutRow;
        in.best_v = best_s.v;
        in.best_i = best_s.i;
    }
    put_exp_entry(s.tab, entry);
    const float mx = in.best_v;
    if (in.status == kCutAll) return;  // the defaults of collect hold
    const int d = row < g.k ? drafts[(uint64_t)b * g.ds + row] : -1;
    bool fits = in.status == kCutFound;
    const int segs = tg.KC * 4;
    if (fits) {  // segment starts (wave 0: up to 256 segments, 4 a lane), then the members side by side
        if (threadIdx.x < 64) {
            const uint32_t *cnt = reinterpret_cast<const uint32_t *>(ra + tg.cnt_off);
            uint32_t c[4], sum = 0u;
            bool ok = true;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int q = 4 * (int)threadIdx.x + i;
                c[i] = q < segs ? cnt[q] : 0u;
                ok = ok && c[i] <= (uint32_t)tg.seg;
                sum += c[i];
            }
            uint32_t inc = sum;
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) {
                const uint32_t v = __shfl_up(inc, off);
                if ((int)threadIdx.x >= off) inc += v;
            }
            uint32_t at = inc - sum;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                seg_at[4 * threadIdx.x + i] = at;
                at += c[i];
            }
            if (threadIdx.x == 63) seg_at[256] = at;
            const uint64_t good = __ballot(ok);
            if (threadIdx.x == 63) n_s = good == ~0ull && at <= (uint32_t)cand_most(W) ? (int)at : -1;
        }
        __syncthreads();
        fits = n_s >= 0;
    }
    if (fits) {
        const Member *src = reinterpret_cast<const Member *>(ra + tg.cand_off);
        for (int q = threadIdx.x >> 6; q < segs; q += W) {
            const uint32_t a = seg_at[q], n = seg_at[q + 1] - a;
            for (uint32_t i = threadIdx.x & 63; i < n; i += 64) list[a + i] = src[(uint64_t)q * tg.seg + i];
        }
        __syncthreads();
    }
    int n = fits ? n_s : 0;
    if (!fits && (in.status == kCutFound || in.status == kCutGather)) {
        n = gather<W>(p, g.V, list, s.seg_n, [=](float l) {
            const int bin = bin_of(l, in.map, tg.NB);
            return top_k > 0 ? bin <= in.bnd : bin == in.bnd;
        });
        fits = n >= 0;
    }
    Cut cut{0u, INT_MAX};
    if (fits && n <= kRankMost) {
        // composite order: a larger (key, ~id) is ahead
        unsigned long long *ord = reinterpret_cast<unsigned long long *>(&s.wsum[0][0]), *sorted = ord + kRankMost;
        double *wt = reinterpret_cast<double *>(sorted + kRankMost);
        const int i = threadIdx.x, wave = i >> 6, lane = i & 63;
        const bool have = i < n;
        // with top-k the candidates are everything down to the boundary bin
        const int kept = top_k > 0 ? min(n, top_k) : n;
        if (have) ord[i] = ((unsigned long long)order_key(list[i].l) << 32) | (uint32_t)~(uint32_t)list[i].j;
        if (i == 0) end_s = kept - 1;
        __syncthreads();
        if (have) {
            const unsigned long long me = ord[i];
            int at = 0;
            for (int q = 0; q < n; q++) at += ord[q] > me;
            sorted[at] = me;
            wt[at] = at < kept ? soft_weight(list[i].l, mx, t, s.tab) : 0.0;
        }
        __syncthreads();
        // thread i: the i-th member, the weights up to it and before it
        const double w = have ? wt[i] : 0.0;
        const uint32_t key = have ? (uint32_t)(sorted[i] >> 32) : 0u;
        double inc = w;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const double v = __shfl_up(inc, off);
            if (lane >= off) inc += v;
        }
        double exc = __shfl_up(inc, 1);
        if (lane == 0) exc = 0.0;
        // (members of one wave only: the others have nothing to decide)
        double sum = __shfl(inc, 63), base = 0.0;
        if (n > 64) {
            if (lane == 63) waves[wave] = inc;
            __syncthreads();
            sum = 0.0;
            for (int q = 0; q < W; q++) {
                if (q == wave) base = sum;
                sum += waves[q];
            }
        }
        const double before = top_k > 0 ? 0.0 : in.before, total = top_k > 0 ? sum : in.total;
        inc += base;
        exc += base;
        // the boundary is the first key whose members' weights reach top_p (none:
        // the last key); of its members those up to the first one whose running
        // share reaches it are kept, as in radix_cut
        const bool nucleus = top_p > 0.0f && top_p < 1.0f && total > 0.0 && !isinf(total);
        if (nucleus && i < kept && (i + 1 == kept || (uint32_t)(sorted[i + 1] >> 32) != key) &&
            before + inc >= (double)top_p * total)
            atomicMin(&end_s, i);
        __syncthreads();
        const int end = end_s;
        // the first member of the boundary key
        if (i <= end && key == (uint32_t)(sorted[end] >> 32) && (i == 0 || (uint32_t)(sorted[i - 1] >> 32) != key))
            last_s = !nucleus ? end : i - 1 + (int)tie_members(before + exc, w, total, (double)top_p, (uint32_t)(end - i + 1));
        __syncthreads();
        const unsigned long long last = sorted[last_s];
        cut = Cut{(uint32_t)(last >> 32), (int32_t)~(uint32_t)last};
    } else {
        const SelSrc src{p, g.V, fits || direct == 1 ? list : nullptr, fits ? n : g.V, fits && top_k > 0};
        int bin_n = 0;
        if (in.status == kCutBin)
            bin_n = gather<W>(p, g.V, list, s.seg_n,
                              [=](float l) { return bin_of(l, in.map, tg.NB) == in.bnd; });
        cut = radix_cut(src, s, mx, t, in.status == kCutNoTopK ? 0 : top_k, top_p, fits && top_k <= 0, in.before, in.total,
                        direct ? nullptr : list, bin_n, (uint32_t)in.before);
        __syncthreads();
    }
    // the kept weight: candidates (after the bins above them), or the row
    const SelSrc src{p, g.V, fits || direct == 1 ? list : nullptr, fits ? n : g.V, false};
    double sum = 0.0;
    for_each<W>(src, [&](float l, int j) __attribute__((always_inline)) {
        if (j != d && in_cut(order_key(l), j, cut)) sum += soft_weight(l, mx, t, s.tab);
    });
    sum = block_sum<W>(sum, waves);
    if (threadIdx.x == 0) {
        rc.best_v = in.best_v;
        rc.best_i = in.best_i;
        rc.cut = cut;
        rc.rest = sum + (fits && top_k <= 0 ? in.before_rest : 0.0);
        rc.wd = d >= 0 && d < g.V ? weight_of(p[d], d, mx, t, cut, s.tab) : 0.0;
    }
}

// Philox4x32-10 (Salmon et al., SC'11).
__device__ __forceinline__ void philox(uint32_t c[4], uint32_t k0, uint32_t k1) {
    for (int r = 0; r < 10; r++) {
        const uint64_t p0 = (uint64_t)0xD2511F53u * c[0];
        const uint64_t p1 = (uint64_t)0xCD9E8D57u * c[2];
        const uint32_t n0 = (uint32_t)(p1 >> 32) ^ c[1] ^ k0;
        const uint32_t n1 = (uint32_t)p1;
        const uint32_t n2 = (uint32_t)(p0 >> 32) ^ c[3] ^ k1;
        const uint32_t n3 = (uint32_t)p0;
        c[0] = n0; c[1] = n1; c[2] = n2; c[3] = n3;
        k0 += 0x9E3779B9u;
        k1 += 0xBB67AE85u;
    }
}

__device__ __forceinline__ double draw(uint64_t seed, uint64_t step, uint32_t row, uint32_t request,
                                       uint32_t purpose) {
    uint32_t c[4] = {(uint32_t)step, (uint32_t)(step >> 32), request, (row << 8) | (purpose & 0xffu)};
    philox(c, (uint32_t)seed, (uint32_t)(seed >> 32));
    const uint64_t v = ((((uint64_t)c[0]) << 32) | c[1]) >> 11;
    return (double)v * (1.0 / 9007199254740992.0);
}

// Router logits replaced by i.i.d. N(0,1) draws: thread per (row, expert
// pair), one Philox block per pair, Box-Muller on two 53-bit uniforms (u1 in
// (0, 1]).
__global__ __launch_bounds__(256) void router_normal_kernel(float *__restrict__ logits, int rows, int E,
                                                            uint64_t seed, uint32_t layer,
                                                            const uint64_t *__restrict__ step_ptr) {
    const int pairs = (E + 1) / 2;
    const int idx = blockIdx.x * 256 + threadIdx.x;
    if (idx >= rows * pairs) return;
    const int r = idx / pairs, p = idx - r * pairs;
    const uint64_t step = step_ptr ? *step_ptr : 0;
    uint32_t c[4] = {(uint32_t)step, (uint32_t)(step >> 32), layer, ((uint32_t)r << 16) | (uint32_t)p};
    philox(c, (uint32_t)seed, (uint32_t)(seed >> 32));
    const double u1 = (double)(((((uint64_t)c[0]) << 32 | c[1]) >> 11) + 1) * (1.0 / 9007199254740992.0);
    const double u2 = (double)((((uint64_t)c[2]) << 32 | c[3]) >> 11) * (1.0 / 9007199254740992.0);
    const double rad = sqrt(-2.0 * log(u1)), ang = 6.283185307179586 * u2;
    float *row = logits + (uint64_t)r * E;
    row[2 * p] = (float)(rad * cos(ang));
    if (2 * p + 1 < E) row[2 * p + 1] = (float)(rad * sin(ang));
}

// Block-wide inverse CDF inside the chunk [begin, end) of a row: the first index j (j != d,
// weight > 0) whose running weight sum exceeds `target`. Returns -1 when the
// target lies beyond the chunk's own sum (rounding), with *last the last
// positive-weight index of the chunk.
__device__ int scan_chunk(const float *p, int begin, int end, int d, float mx, const Temp &t, const Cut &cut,
                          const ExpEntry *tab, double target, double *shared_prefix, int *shared_pick) {
    const int len = end - begin;
    const int per = (len + 255) / 256;
    const int lo = begin + threadIdx.x * per;
    const int hi = min(lo + per, end);
    double local = 0.0;
    int j = lo;
    for (; j + 7 < hi; j += 8) {  // eight loads in flight, summed in index order
        float l[8];
#pragma unroll
        for (int u = 0; u < 8; u++) l[u] = p[j + u];
#pragma unroll
        for (int u = 0; u < 8; u++)
            if (j + u != d) local += weight_of(l[u], j + u, mx, t, cut, tab);
    }
    for (; j < hi; j++)
        if (j != d) local += weight_of(p[j], j, mx, t, cut, tab);
    shared_prefix[threadIdx.x] = local;
    if (threadIdx.x == 0) *shared_pick = -1;
    __syncthreads();
    if (threadIdx.x == 0) {  // exclusive prefix in thread order, 16 reads in flight at a time
        double run = 0.0;
        for (int t0 = 0; t0 < 256; t0 += 16) {
            double v[16];
#pragma unroll
            for (int i = 0; i < 16; i++) v[i] = shared_prefix[t0 + i];
#pragma unroll
            for (int i = 0; i < 16; i++) {
                shared_prefix[t0 + i] = run;
                run += v[i];
            }
        }
    }
    __syncthreads();
    double run = shared_prefix[threadIdx.x];
    if (run <= target && target < run + local) {
        for (int j = lo; j < hi; j++) {
            if (j == d) continue;
            const double w = weight_of(p[j], j, mx, t, cut, tab);
            if (w <= 0.0) continue;
            run += w;
            if (target < run) {
                *shared_pick = j;
                break;
            }
        }
        if (*shared_pick < 0) {  // rounding at the boundary: last positive weight
            for (int j = hi - 1; j >= lo; j--)
                if (j != d && weight_of(p[j], j, mx, t, cut, tab) > 0.0) {
                    *shared_pick = j;
                    break;
                }
        }
    }
    __syncthreads();
    return *shared_pick;
}

__global__ __launch_bounds__(256) void accept_finalize_kernel(
    const float *__restrict__ logits, Geo g, const int32_t *__restrict__ drafts,
    const Stat *__restrict__ stats, const double *__restrict__ sums,
    const double *__restrict__ wdraft, int stochastic, Temp t, uint64_t seed, uint64_t step,
    uint32_t request_base, int32_t *__restrict__ result, double *__restrict__ debug,
    const uint64_t *__restrict__ step_dev, const int32_t *__restrict__ forced) {
    const int b = blockIdx.x;
    if (step_dev) step = *step_dev;
    const uint32_t request = request_base + (uint32_t)b;
    __shared__ double prefix[256];
    __shared__ ExpEntry tab[16];
    __shared__ int pick;
    __shared__ int decided_next;
    __shared__ int accepted_s;
    __shared__ int argmax0;
    __shared__ Stat row_best_s[256];
    __shared__ double row_rest_s[256];
    __shared__ float row_p0_s[256];  // logit 0 of each row
    __shared__ int row_d_s[256];     // each row's draft (-1 on the bonus row)
    const ExpEntry entry = exp_entry();
    if (threadIdx.x == 0) {
        decided_next = -1;
        accepted_s = 0;
    }
    // Per-row maxima and weight sums: one wave per row, lanes over chunks.
    {
        const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
        for (int row = wave; row <= g.k; row += 4) {
            const Stat *st = stats + ((uint64_t)b * g.R + row) * g.C;
            Stat best{-INFINITY, INT_MAX};
            double rest = 0.0;
            for (int c = lane; c < g.C; c += 64) {
                if (beats(st[c].v, st[c].i, best.v, best.i)) best = st[c];
                if (stochastic) rest += sums[((uint64_t)b * g.R + row) * g.C + c];
            }
            for (int off = 32; off > 0; off >>= 1) {
                const float ov = __shfl_xor(best.v, off);
                const int oi = __shfl_xor(best.i, off);
                if (beats(ov, oi, best.v, best.i)) best = Stat{ov, oi};
                rest += __shfl_xor(rest, off);
            }
            if (lane == 0) {
                row_best_s[row] = best;
                row_rest_s[row] = rest;
                row_p0_s[row] = row_ptr(logits, g, b, row)[0];
                row_d_s[row] = row < g.k ? drafts[(uint64_t)b * g.ds + row] : -1;
            }
        }
    }
    put_exp_entry(tab, entry);
    __syncthreads();
    for (int row = 0; row <= g.k; row++) {
        const float *p = row_ptr(logits, g, b, row);
        __shared__ Stat best_s;
        __shared__ int action;  // 0 accept, 1 done (next decided), 2 resample
        __shared__ double target_s;
        __shared__ int cstar;
        __shared__ float mx_s;
        __shared__ double cs_s[256];  // the row's chunk weight sums, for thread 0's walk below
        if (stochastic)
            for (int c = threadIdx.x; c < g.C && c < 256; c += 256) cs_s[c] = sums[((uint64_t)b * g.R + row) * g.C + c];
        __syncthreads();
        if (threadIdx.x == 0) {
            Stat best = row_best_s[row];
            const float p0 = row_p0_s[row];
            if (p0 != p0) best = Stat{p0, 0};  // argmaxLogit keeps a NaN at index 0
            best_s = best;
            if (row == 0) argmax0 = best.i;
            const int d = row_d_s[row];
            double dbg[4] = {0.0, 0.0, 0.0, (double)best.v};
            action = 1;
            // forced: a prescribed acceptance length replaces the accept test;
            // the token at the first rejected row is still the mode's choice
            const int flen = forced ? forced[b] : -1;
            if (!stochastic) {
                if (row < g.k && (forced ? row < flen : best.i == d)) {
                    action = 0;
                } else {
                    decided_next = best.i;
                }
            } else {
                // The sampler's first candidate: the maximum over valid logits;
                // with none valid, argmaxLogit's answer (sampling.go:83-89).
                Stat sb = row_best_s[row];
                if (sb.v == -INFINITY) sb = best;
                best_s = sb;
                const double *cs = g.C <= 256 ? cs_s : sums + ((uint64_t)b * g.R + row) * g.C;
                const double rest = row_rest_s[row];
                const double wd = (row < g.k && d >= 0 && d < g.V) ? wdraft[(uint64_t)b * g.R + row] : 0.0;
                double total = rest + wd;
                const bool onehot = !(total > 0.0) || isinf(total);
                dbg[2] = total;
                if (row < g.k) {
                    const double pd = onehot ? (d == sb.i ? 1.0 : 0.0) : wd / total;
                    const double u = draw(seed, step, (uint32_t)row, request, 0);
                    dbg[0] = pd;
                    dbg[1] = u;
                    if (forced ? row < flen : u < pd) {
                        action = 0;
                    } else if (onehot || !(rest > 0.0)) {
                        decided_next = sb.i;
                    } else {
                        const double u2 = draw(seed, step, (uint32_t)row, request, 1);
                        const double target = u2 * rest;
                        double run = 0.0;
                        int c = 0;
                        for (; c < g.C - 1; c++) {
                            if (target < run + cs[c]) break;
                            run += cs[c];
                        }
                        target_s = target - run;
                        cstar = c;
                        mx_s = sb.v;
                        action = 2;
                    }
                } else {
                    if (onehot) {
                        decided_next = sb.i;
                    } else {
                        const double u2 = draw(seed, step, (uint32_t)row, request, 1);
                        const double target = u2 * total;
                        double run = 0.0;
                        int c = 0;
                        for (; c < g.C - 1; c++) {
                            if (target < run + cs[c]) break;
                            run += cs[c];
                        }
                        target_s = target - run;
                        cstar = c;
                        mx_s = sb.v;
                        action = 2;
                    }
                }
            }
            if (debug) {
                double *o = debug + (((uint64_t)b * g.R) + row) * 4;
                for (int i = 0; i < 4; i++) o[i] = dbg[i];
            }
        }
        __syncthreads();
        if (action == 0) {
            if (threadIdx.x == 0) accepted_s++;
            __syncthreads();
            continue;
        }
        if (action == 2) {
            const int d = row < g.k ? drafts[(uint64_t)b * g.ds + row] : -1;
            const int begin = cstar * g.L;
            const int j = scan_chunk(p, begin, min(begin + g.L, g.V), d, mx_s, t, Cut{0u, INT_MAX}, tab, target_s, prefix, &pick);
            if (threadIdx.x == 0) decided_next = j >= 0 ? j : best_s.i;
        }
        break;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        int32_t *o = result + (uint64_t)b * 4;
        o[0] = accepted_s;
        o[1] = decided_next;
        o[2] = argmax0;
        o[3] = 0;
    }
}

// What the rows of a request decide (truncated stochastic acceptance):
// the first row that does not accept its draft, and what follows there.
struct Decision {
    int row;       // rows accepted
    int next;      // the next token, or -1: drawn from `row`
    double target; // of the draw: a share of the row's kept weight in index order
    int d;         // draft left out of the draw (-1: none)
};

// Wave 0 of a workgroup: lane l takes rows l, l + 64, ...; every lane
// returns the decision.
__device__ Decision decide(const float *logits, const Geo &g, int b, const int32_t *drafts, uint8_t *area,
                           uint64_t seed, uint64_t step, uint32_t request, const int32_t *forced, double *debug) {
    const int lane = threadIdx.x & 63;
    const int flen = forced ? forced[b] : -1;
    for (int r0 = 0;; r0 += 64) {
        const int row = r0 + lane;
        bool stop = false, onehot = false;
        double rest = 0.0, total = 0.0, pd = 0.0, u = 0.0;
        Stat sb{-INFINITY, INT_MAX};
        float shown = 0.f;
        int d = -1;
        if (row <= g.k) {
            const RowCut &rc = row_cut(area, g, b, row);
            sb = Stat{rc.best_v, rc.best_i};
            rest = rc.rest;
            total = rest + rc.wd;
            onehot = !(total > 0.0) || isinf(total);
            // argmaxLogit keeps a NaN at index 0; the sampler falls back to
            // its answer when no logit is valid (sampling.go:83-89)
            const float p0 = row_ptr(logits, g, b, row)[0];
            shown = p0 != p0 ? p0 : sb.v;
            if (sb.v == -INFINITY && p0 != p0) sb = Stat{p0, 0};
            if (row < g.k) {
                d = drafts[(uint64_t)b * g.ds + row];
                pd = onehot ? (d == sb.i ? 1.0 : 0.0) : rc.wd / total;
                u = draw(seed, step, (uint32_t)row, request, 0);
                stop = !(forced ? row < flen : u < pd);
            } else {
                stop = true;
            }
        }
        const uint64_t m = __ballot(stop);
        const int first = m ? __ffsll((unsigned long long)m) - 1 : 64;
        if (debug && row <= g.k && lane <= first) {
            double *o = debug + ((uint64_t)b * g.R + row) * 4;
            o[0] = pd;
            o[1] = u;
            o[2] = total;
            o[3] = (double)shown;
        }
        if (!m) continue;
        Decision dec{r0 + first, -1, 0.0, -1};
        int next = -1;
        double target = 0.0;
        if (lane == first) {
            if (onehot || (row < g.k && !(rest > 0.0)))
                next = sb.i;
            else
                target = draw(seed, step, (uint32_t)row, request, 1) * (row < g.k ? rest : total);
        }
        dec.next = __shfl(next, first);
        dec.target = __shfl(target, first);
        dec.d = __shfl(d, first);
        return dec;
    }
}

// Kept weight per chunk of the row that a request draws from (RC chunks).
__global__ __launch_bounds__(256) void accept_resample_kernel(const float *__restrict__ logits, Geo g, int RC,
                                                              const int32_t *__restrict__ drafts,
                                                              uint8_t *__restrict__ area, Temp t, uint64_t seed,
                                                              uint64_t step, uint32_t request_base,
                                                              const uint64_t *__restrict__ step_dev,
                                                              const int32_t *__restrict__ forced,
                                                              double *__restrict__ sums) {
    const int c = blockIdx.x, b = blockIdx.y;
    __shared__ int row_s, d_s;
    __shared__ double ws[4];
    __shared__ ExpEntry tab[16];
    const ExpEntry entry = exp_entry();
    if (step_dev) step = *step_dev;
    if (threadIdx.x < 64) {
        const Decision dec = decide(logits, g, b, drafts, area, seed, step, request_base + (uint32_t)b, forced, nullptr);
        if (threadIdx.x == 0) {
            row_s = dec.next < 0 ? dec.row : -1;
            d_s = dec.d;
        }
    }
    put_exp_entry(tab, entry);
    __syncthreads();
    const int row = row_s, d = d_s;
    if (row < 0) return;
    const RowCut &rc = row_cut(area, g, b, row);
    const Cut cut = rc.cut;
    const float mx = rc.best_v;
    const float *p = row_ptr(logits, g, b, row);
    const int begin = (int)((int64_t)g.V * c / RC), end = (int)((int64_t)g.V * (c + 1) / RC);
    double acc = 0.0;
    constexpr int kU = 8;
    for (int j0 = begin + threadIdx.x; j0 < end; j0 += kU * 256) {
        float l[kU];
#pragma unroll
        for (int u = 0; u < kU; u++) l[u] = j0 + u * 256 < end ? p[j0 + u * 256] : NAN;
#pragma unroll
        for (int u = 0; u < kU; u++)
            if (j0 + u * 256 != d) acc += weight_of(l[u], j0 + u * 256, mx, t, cut, tab);
    }
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off);
    if ((threadIdx.x & 63) == 0) ws[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) sums[(uint64_t)b * RC + c] = ws[0] + ws[1] + ws[2] + ws[3];
}

// The draw: the chunk that the target falls into, then the index inside it.
__global__ __launch_bounds__(256) void accept_pick_kernel(const float *__restrict__ logits, Geo g, int RC,
                                                          const int32_t *__restrict__ drafts,
                                                          uint8_t *__restrict__ area,
                                                          const double *__restrict__ sums, Temp t, uint64_t seed,
                                                          uint64_t step, uint32_t request_base,
                                                          const uint64_t *__restrict__ step_dev,
                                                          const int32_t *__restrict__ forced,
                                                          int32_t *__restrict__ result, double *__restrict__ debug) {
    const int b = blockIdx.x, lane = threadIdx.x & 63;
    __shared__ double prefix[256];
    __shared__ int pick, cstar_s;
    __shared__ double target_s;
    __shared__ Decision dec_s;
    __shared__ ExpEntry tab[16];
    const ExpEntry entry = exp_entry();
    if (step_dev) step = *step_dev;
    if (threadIdx.x < 64) {
        // RC <= 64: lane c's chunk; the target's chunk is the last one whose
        // running start it reaches
        const double cs = lane < RC ? sums[(uint64_t)b * RC + lane] : 0.0;
        const Decision dec = decide(logits, g, b, drafts, area, seed, step, request_base + (uint32_t)b, forced, debug);
        double inc = cs;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const double v = __shfl_up(inc, off);
            if (lane >= off) inc += v;
        }
        const uint64_t m = __ballot(lane < RC - 1 && !(dec.target < inc));
        const int c = m == ~0ull ? 63 : __ffsll((unsigned long long)~m) - 1;  // leading chunks that end at or before it
        const double run = __shfl(inc, c ? c - 1 : 0);
        if (lane == 0) {
            dec_s = dec;
            cstar_s = c;
            target_s = dec.target - (c ? run : 0.0);
        }
    }
    put_exp_entry(tab, entry);
    __syncthreads();
    const Decision dec = dec_s;
    int next = dec.next;
    if (next < 0) {
        const RowCut &rc = row_cut(area, g, b, dec.row);
        const int c = cstar_s;
        const int j = scan_chunk(row_ptr(logits, g, b, dec.row), (int)((int64_t)g.V * c / RC),
                                 (int)((int64_t)g.V * (c + 1) / RC), dec.d, rc.best_v, t, rc.cut, tab, target_s, prefix, &pick);
        next = j >= 0 ? j : rc.best_i;
    }
    if (threadIdx.x == 0) {
        // argmaxLogit of row 0 keeps a NaN at index 0
        const float p0 = row_ptr(logits, g, b, 0)[0];
        int32_t *o = result + (uint64_t)b * 4;
        o[0] = dec.row;
        o[1] = next;
        o[2] = p0 != p0 ? 0 : row_cut(area, g, b, 0).best_i;
        o[3] = 0;
    }
}

Geo make_geo(const yuuka_accept_params &p) {
    Geo g;
    g.B = (int)p.batch;
    g.k = (int)p.drafts;
    g.R = g.k + 1;
    g.V = (int)p.vocab;
    g.stride = p.row_stride ? p.row_stride : p.vocab;
    g.ds = g.k;
    int c = (2048 + g.B * g.R - 1) / (g.B * g.R);
    c = c < 1 ? 1 : (c > 256 ? 256 : c);
    int L = (g.V + c - 1) / c;
    L = (L + 3) & ~3;
    g.L = L;
    g.C = (g.V + L - 1) / L;
    return g;
}

// Waves of a cut workgroup (see SelShared).
int cut_waves(int rows) { return rows <= 256 ? 16 : 8; }

// The layout of a row's area. A chunk has a few thousand logits, or the
// workgroups do little but add up the histograms (20 rows of 8200..32000,
// top-p 0.9, with up to 52 chunks of a row: 56 us; now 39..43). The bins take
// at most about half of it, the candidates the rest; few rows have many chunks
// and much room, thousands of rows little (fewer bins, and more of their rows'
// candidates are gathered by the cut's workgroup).
TruncGeo trunc_geo(const Geo &g) {
    TruncGeo t;
    const int rows = g.B * g.R;
    t.NB = g.C >= 8 ? kBins : (g.C >= 4 ? 512 : (g.C >= 2 ? 256 : 128));
    t.HC = std::max(1, std::min({16, g.C / 5, g.V / 8192}));
    t.KC = std::max(1, std::min({64, g.C, (1024 + rows - 1) / rows, g.V / 4096}));
    const uint32_t bytes = (uint32_t)((uint64_t)g.C * kRowArea - sizeof(RowCut));
    t.bins_off = (uint32_t)(g.C * sizeof(Moments));
    t.cnt_off = t.bins_off + (uint32_t)(t.HC * t.NB * 8);
    t.cand_off = t.cnt_off + (uint32_t)(t.KC * 4 * 4);
    // (segments fill unevenly: twice the list's room where there is space)
    t.cap = cand_most(cut_waves(rows));
    t.seg = std::min((int)((bytes - t.cand_off) / sizeof(Member)), 2 * t.cap) / (t.KC * 4);
    return t;
}

}  // namespace

uint64_t accept_scratch_bytes(const yuuka_accept_params &p) {
    const Geo g = make_geo(p);
    const uint64_t n = (uint64_t)g.B * g.R * g.C;
    return ((n * sizeof(Stat) + 255) & ~255ull) + n * sizeof(double) + (uint64_t)g.B * g.R * sizeof(double) + 256 +
           n * kRowArea;
}

hipError_t launch_router_normal(float *logits, int rows, int E, uint64_t seed, uint32_t layer, const uint64_t *step,
                                hipStream_t s) {
    const int n = rows * ((E + 1) / 2);
    if (n > 0) router_normal_kernel<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(logits, rows, E, seed, layer, step);
    return hipGetLastError();
}

hipError_t launch_verify_accept(const float *logits, const int32_t *drafts, int32_t *result,
                                double *debug, const yuuka_accept_params &p, void *scratch,
                                hipStream_t stream, const uint64_t *step_dev, uint32_t draft_stride,
                                const int32_t *forced) {
    Geo g = make_geo(p);
    if (draft_stride) g.ds = (int)draft_stride;
    const uint64_t n = (uint64_t)g.B * g.R * g.C;
    auto *base = static_cast<uint8_t *>(scratch);
    Stat *stats = reinterpret_cast<Stat *>(base);
    double *sums = reinterpret_cast<double *>(base + ((n * sizeof(Stat) + 255) & ~255ull));
    double *wdraft = sums + n;
    const bool stochastic = p.mode == YUUKA_ACCEPT_STOCHASTIC && p.temperature > 0.0f && p.top_k != 1;
    const Temp t = make_temp(stochastic ? p.temperature : 1.0f);
    // top_p 0 means off (sampling.go:46-48); top_k at or above the vocabulary keeps everything.
    const bool top_k_on = p.top_k > 1 && p.top_k < p.vocab;
    const bool top_p_on = p.top_p > 0.0f && p.top_p < 1.0f;
    const bool truncate = stochastic && (top_k_on || top_p_on);
    const dim3 grid((unsigned)g.C, (unsigned)g.R, (unsigned)g.B);
    // 16-byte loads need every row start 16-byte aligned
    const int vec = (reinterpret_cast<uintptr_t>(logits) & 15) == 0 && (g.stride & 3) == 0;
    // one wave per chunk up to 8 logits per lane, else a workgroup per chunk
    const int wpc = g.L <= 512 * 4 ? 1 : 4;
    const dim3 sgrid((unsigned)((g.C + 4 / wpc - 1) / (4 / wpc)), (unsigned)g.R, (unsigned)g.B);
    if (!truncate) {
        accept_stats_kernel<false><<<sgrid, 256, 0, stream>>>(logits, g, stats, vec, wpc, nullptr);
        if (stochastic) accept_weights_kernel<<<grid, 256, 0, stream>>>(logits, g, drafts, stats, t, sums, wdraft);
        accept_finalize_kernel<<<(unsigned)g.B, 256, 0, stream>>>(logits, g, drafts, stats, sums, wdraft,
                                                                 stochastic ? 1 : 0, t, p.seed, p.step, p.request_base,
                                                                 result, debug, step_dev, forced);
        return hipGetLastError();
    }
    uint8_t *area = reinterpret_cast<uint8_t *>((reinterpret_cast<uintptr_t>(wdraft + (uint64_t)g.B * g.R) + 255) &
                                                ~(uintptr_t)255);
    const TruncGeo tg = trunc_geo(g);
    const int tk = top_k_on ? (int)p.top_k : 0;
    const float tp = top_p_on ? p.top_p : 1.0f;
    const dim3 rgrid((unsigned)g.R, (unsigned)g.B);
    const dim3 hgrid((unsigned)tg.HC, (unsigned)g.R, (unsigned)g.B), kgrid((unsigned)tg.KC, (unsigned)g.R, (unsigned)g.B);
    const uint32_t bins_lds = (uint32_t)(kBinWaves * tg.NB) * (top_k_on ? 4u : 8u);
    static const bool attr = [] {  // (once, also with several threads)
        (void)hipFuncSetAttribute(reinterpret_cast<const void *>(accept_cut_kernel<16>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, cand_most(16) * (int)sizeof(Member));
        (void)hipFuncSetAttribute(reinterpret_cast<const void *>(accept_cut_kernel<8>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, cand_most(8) * (int)sizeof(Member));
        (void)hipFuncSetAttribute(reinterpret_cast<const void *>(accept_bins_kernel<false>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, kBinWaves * kBins * 8);
        return true;
    }();
    (void)attr;
    int cand = tg.cap;
    int direct = 0;
    if (g.V <= kDirectMost) direct = g.V <= tg.cap ? 1 : 2;
    else if (top_k_on && !top_p_on && g.V <= kDirectTopK && g.B * g.R <= 256) direct = 2;
    if (direct) {
        accept_stats_kernel<false><<<sgrid, 256, 0, stream>>>(logits, g, stats, vec, wpc, nullptr);
        cand = direct == 1 ? g.V : 0;
    } else if (top_k_on) {
        accept_stats_kernel<true><<<sgrid, 256, 0, stream>>>(logits, g, stats, vec, wpc, area);
        accept_bins_kernel<true><<<hgrid, 64 * kBinWaves, bins_lds, stream>>>(logits, g, tg, drafts, stats, t, area);
        accept_collect_kernel<true><<<kgrid, 256, 0, stream>>>(logits, g, tg, drafts, stats, tk, tp, t, area);
    } else {
        accept_stats_kernel<true><<<sgrid, 256, 0, stream>>>(logits, g, stats, vec, wpc, area);
        accept_bins_kernel<false><<<hgrid, 64 * kBinWaves, bins_lds, stream>>>(logits, g, tg, drafts, stats, t, area);
        accept_collect_kernel<false><<<kgrid, 256, 0, stream>>>(logits, g, tg, drafts, stats, tk, tp, t, area);
    }
    const uint32_t cut_lds = (uint32_t)cand * sizeof(Member);
    if (cut_waves(g.B * g.R) == 16)
        accept_cut_kernel<16><<<rgrid, 64 * 16, cut_lds, stream>>>(logits, g, tg, drafts, stats, tk, tp, t, area, direct);
    else
        accept_cut_kernel<8><<<rgrid, 64 * 8, cut_lds, stream>>>(logits, g, tg, drafts, stats, tk, tp, t, area, direct);
    // chunks of the drawn row: at most 64 (one per lane of pick), and their
    // sums fit the per-chunk sums' place
    const int RC = std::min(64, g.R * g.C);
    accept_resample_kernel<<<dim3((unsigned)RC, (unsigned)g.B), 256, 0, stream>>>(
        logits, g, RC, drafts, area, t, p.seed, p.step, p.request_base, step_dev, forced, sums);
    accept_pick_kernel<<<(unsigned)g.B, 256, 0, stream>>>(logits, g, RC, drafts, area, sums, t, p.seed, p.step,
                                                         p.request_base, step_dev, forced, result, debug);
    return hipGetLastError();
}

}  // namespace yk
