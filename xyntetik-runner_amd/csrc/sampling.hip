// Sampling on the device.
//
// temp <= 0: the first index of the maximum, logits untouched
// (src/sample.c:169-172).  temp > 0, in the reference's order
// (src/sample.c:148-166, :86-127, :302-328):
//   repeat penalty over the recent window (each occurrence counts; exempt ids skipped;
//   a positive logit is divided, another multiplied), z = logit / temp, candidates in
//   the total order "z descending, then id ascending", top-k (softmax over the k kept),
//   top-p (smallest prefix with mass >= top_p, renormalised), min-p (drop p < min_p *
//   p_best, renormalised), then the roulette walk: first candidate whose cumulative
//   mass exceeds the draw r.
// Every cut keeps a prefix of that total order (its key: 32 bits of z, 24 bits of id), so a row
// is never sorted.  Mass is exp(z - z_max) in 40-bit fixed point and added as whole numbers: the
// pick does not depend on the order in which lanes, waves or workgroups add.
//
// A sampled row goes in three steps: its largest and smallest logit (with the penalty applied on
// the way), the mass and number of candidates in each of SM_BINS ranges of z (a histogram in LDS),
// and the cuts: a cut falls into one bin, whose candidates (a few hundred of 128k) are gathered from
// the row and sorted in LDS, and the place inside the bin is exact.  A bin with more than SM_LIST
// candidates (a row of equal logits) is left to a radix selection over the whole row, 7 passes a cut.
// What bounds it: reading a row of 128k logits is 4 us for one compute unit and an exponential for
// each 50 us, so a row's histogram is shared out to up to 8 workgroups where the caller brings room for their
// partial counts; the cuts are a chain of short steps that one workgroup a row walks.
// Where every cut was a radix selection (22 passes over the row for top-p) 64 rows of 128,256 logits
// took 1,150 us; now 54 in three kernels (7 + 17 + 31; 34 with bins of 5 to 256 candidates sorted by a network).
#include "common.h"
#include "no_alloc.h"

#include <mutex>

#define SM_THREADS 1024
#define SM_BINS 2048            // ranges of z a row's candidates are counted in
#define SM_SPAN 28.f            // below z_max - 28 a candidate's mass is 0 (exp(-28) < 2^-40)
#define SM_LIST 2048            // candidates of a cut's bin that are sorted in LDS
#define SM_RANKED 256           // and up to so many by counting the keys below each
#define ROW_SPLITS 32           // workgroups that look for a row's largest and smallest logit

typedef unsigned long long u64;

struct SampleArgs {
    int* out;
    float* logits;
    int ld, V;
    const float* temp;
    const int* top_k;
    const float* top_p;
    const float* min_p;
    const float* repeat_penalty;
    const float* draw;
    const int* recent;      // [W, recent_cap]
    const int* n_recent;    // [W]
    int recent_cap;
    const int* exempt;
    int n_exempt;
    const float* part;          // [W, ROW_SPLITS, 2] from k_pick_extent, or null
    const u64* hist_mass;       // [W, hist_splits, SM_BINS] from k_pick_hist, or null
    const unsigned* hist_count; // the same for the number of candidates (rows with top-k only)
    int hist_splits;
};

__device__ inline uint32_t order_key32(float z) {
    if (z != z) return 0xFFFFFFFFu;          // NaN sorts last
    if (z == 0.f) z = 0.f;                   // -0 and +0 are one value
    uint32_t u = __float_as_uint(z);
    u = (u >> 31) ? ~u : (u | 0x80000000u);  // ascending with z
    return ~u;                               // ascending key = descending z
}

__device__ inline u64 order_key(float z, int id) {
    return ((u64)order_key32(z) << 24) | (u64)(uint32_t)id;
}

// The whole part of e * 2^40 for 0 <= e <= 1.
__device__ inline u64 mass_of(float e) {
    const uint32_t u = __float_as_uint(e);
    const int up = (int)(u >> 23) - 110;            // e = m * 2^(up - 40) with the 24-bit m
    const uint32_t m = (u & 0x7FFFFFu) | 0x800000u;
    return up >= 0 ? (u64)m << up : up > -24 ? (u64)(m >> -up) : 0ull;
}

// z of a key (-0 comes back as +0, whose mass is the same).
__device__ inline float key_z(u64 key) {
    const uint32_t u = ~(uint32_t)(key >> 24);
    return __uint_as_float((u >> 31) ? u & 0x7FFFFFFFu : ~u);
}

// f(value, index) for the candidates [lo, hi) of a row, `step` threads side by side; lo is a multiple of 4.
// 16-byte loads where the row's address allows it, up to 8 of them on their way before the first value is looked at (one
// after the other, a workgroup's pass over 128k logits is 31 trips to memory: k_sample for 64 rows 45 us, now 34), one where
// that is all there is to read (200 sampled rows of 32,000: k_pick_extent 9.6 us with eight, 7.0 with one).
template <int U, typename F>
__device__ __forceinline__ void for_fours(const float* row, int lo, int tail, int tid, int step, F f) {
    for (int i0 = lo + 4 * tid; i0 < tail; i0 += 4 * step * U) {
        float4 v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = i0 + 4 * step * u;
            v[u] = *reinterpret_cast<const float4*>(row + (i < tail ? i : i0));
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = i0 + 4 * step * u;
            if (i < tail) {
                f(v[u].x, i);
                f(v[u].y, i + 1);
                f(v[u].z, i + 2);
                f(v[u].w, i + 3);
            }
        }
    }
}
template <typename F>
__device__ __forceinline__ void for_row(const float* row, int lo, int hi, int tid, int step, F f) {
    int tail = lo;
    if (((uintptr_t)row & 15) == 0) {
        tail = lo + ((hi - lo) & ~3);
        if (tail - lo <= 4 * step) for_fours<1>(row, lo, tail, tid, step, f);
        else for_fours<8>(row, lo, tail, tid, step, f);
    }
    for (int i = tail + tid; i < hi; i += step) f(row[i], i);
}

// The repeat penalty of the tokens in [lo, hi): the thread with a token's first place in the window
// applies it as often as the token occurs, which is what walking the window in order does.
__device__ inline void apply_penalty(const SampleArgs& a, int r, float* row, int lo, int hi) {
    const float rp = a.repeat_penalty ? a.repeat_penalty[r] : 1.f;
    if (rp == 1.f || !a.recent) return;
    const int* rec = a.recent + (size_t)r * a.recent_cap;
    const int n = a.n_recent[r] < a.recent_cap ? a.n_recent[r] : a.recent_cap;
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        const int tok = rec[i];
        if (tok < lo || tok >= hi) continue;
        bool skip = false;
        for (int k = 0; k < a.n_exempt; ++k) skip = skip || a.exempt[k] == tok;
        int times = 0;
        for (int j = 0; j < n; ++j)
            if (rec[j] == tok) { skip = skip || j < i; ++times; }
        if (skip) continue;
        float v = row[tok];
        for (int k = 0; k < times; ++k) v = v > 0.f ? v / rp : v * rp;
        row[tok] = v;
    }
    __syncthreads();
}

// The first pass over a row, by ROW_SPLITS workgroups (one workgroup reads 128k logits in 60 us when it
// waits for every load, bound by their latency): of a greedy row the maximum of each range and the first index
// that has it, of a sampled row the largest and the smallest logit, behind the penalty.
__global__ __launch_bounds__(256) void k_pick_extent(SampleArgs a, float* part) {
    const int r = blockIdx.x, sp = blockIdx.y;
    const int chunk = ((a.V + ROW_SPLITS - 1) / ROW_SPLITS + 3) & ~3;
    const int lo = sp * chunk < a.V ? sp * chunk : a.V, hi = lo + chunk < a.V ? lo + chunk : a.V;
    float* row = a.logits + (size_t)r * a.ld;
    __shared__ float sb[4];
    __shared__ int si[4];
    const int wave = threadIdx.x >> 6;
    float* p = part + ((size_t)r * ROW_SPLITS + sp) * 2;
    if (a.temp[r] > 0.f) {
        apply_penalty(a, r, row, lo, hi);
        float zm = -INFINITY, zn = INFINITY;
        for_row(row, lo, hi, threadIdx.x, 256, [&](float v, int) { zm = v > zm ? v : zm; zn = v < zn && v > -INFINITY ? v : zn; });
        zm = wave_max(zm);
        zn = -wave_max(-zn);
        if ((threadIdx.x & 63) == 0) { sb[wave] = zm; si[wave] = __float_as_int(zn); }
        __syncthreads();
        if (threadIdx.x == 0) {
            for (int w = 1; w < 4; ++w) { zm = fmaxf(zm, sb[w]); zn = fminf(zn, __int_as_float(si[w])); }
            p[0] = zm;
            p[1] = zn;
        }
        return;
    }
    float best = -INFINITY;
    int bi = 0x7fffffff;
    for_row(row, lo, hi, threadIdx.x, 256, [&](float v, int i) { if (v > best || (v == best && i < bi)) { best = v; bi = i; } });
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        float ob = __shfl_xor(best, o, 64);
        int oi = __shfl_xor(bi, o, 64);
        if (ob > best || (ob == best && oi < bi)) { best = ob; bi = oi; }
    }
    if ((threadIdx.x & 63) == 0) { sb[wave] = best; si[wave] = bi; }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < 4; ++w)
            if (sb[w] > best || (sb[w] == best && si[w] < bi)) { best = sb[w]; bi = si[w]; }
        p[0] = best;
        p[1] = __int_as_float(bi);
    }
}

struct RowView {
    const float* row;
    int V;
    float temp;       // candidates carry logit / temp
    float zmax;
    u64 limit;   // keep key <= limit
    float min_e;                // keep exp(z - zmax) >= min_e
};

__device__ inline bool row_item(const RowView& rv, float v, int i, u64& key, u64& mass) {
    float z = v / rv.temp;
    key = order_key(z, i);
    float e = expf(z - rv.zmax);
    if (!(e >= rv.min_e) || key > rv.limit) return false;
    mass = mass_of(e);
    return true;
}

__device__ __forceinline__ u64 block_sum_u64(u64 v, u64* sh) {
    // sh has SM_THREADS / 64 entries
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    __syncthreads();
    if (lane == 0) sh[wave] = v;
    __syncthreads();
    u64 t = 0;
    for (int w = 0; w < SM_THREADS / 64; ++w) t += sh[w];
    return t;
}

// Mass (by_mass) or number of the kept candidates.
__device__ __forceinline__ u64 kept_total(const RowView& rv, bool by_mass, u64* sh) {
    u64 acc = 0;
    for_row(rv.row, 0, rv.V, threadIdx.x, SM_THREADS, [&](float v, int i) __attribute__((always_inline)) {
        u64 key, mass;
        if (row_item(rv, v, i, key, mass)) acc += by_mass ? mass : 1ull;
    });
    return block_sum_u64(acc, sh);
}

// Smallest key B among the kept candidates with F(B) > target, where F(B) is the mass
// (by_mass) or the number of kept candidates with key <= B.  If no key reaches the
// target the largest kept key is returned.
__device__ __forceinline__ u64 radix_select(const RowView& rv, bool by_mass, u64 target,
                                           u64* hist, u64* sh2) {
    u64 prefix = 0, remaining = target;
    for (int shift = 48; shift >= 0; shift -= 8) {
        __syncthreads();
        if (threadIdx.x < 256) hist[threadIdx.x] = 0;
        __syncthreads();
        for_row(rv.row, 0, rv.V, threadIdx.x, SM_THREADS, [&](float v, int i) __attribute__((always_inline)) {
            u64 key, mass;
            if (!row_item(rv, v, i, key, mass)) return;
            if ((key >> (shift + 8)) != (prefix >> (shift + 8))) return;
            u64 w = by_mass ? mass : 1ull;
            if (w) atomicAdd(&hist[(key >> shift) & 255ull], w);
        });
        __syncthreads();
        if (threadIdx.x == 0) {
            u64 cum = 0;
            int sel = -1, last = -1;
            for (int d = 0; d < 256; ++d) {
                u64 h = hist[d];
                if (!h) continue;
                last = d;
                if (cum + h > remaining) { sel = d; break; }
                cum += h;
            }
            if (sel < 0) {            // ran off the end: stay in the last kept bin
                sel = last < 0 ? 0 : last;
                remaining = last < 0 ? 0 : hist[sel] - 1;
            } else {
                remaining -= cum;
            }
            sh2[0] = prefix | ((u64)sel << shift);
            sh2[1] = remaining;
        }
        __syncthreads();
        prefix = sh2[0];
        remaining = sh2[1];
    }
    return prefix;
}

// Bins of a row: bin b holds the candidates with b <= (z_max - z) * scale < b + 1, the last one all below.  z_max - z
// falls and the bins rise with the key, so a prefix of bins is a prefix of the order.  A candidate of -inf (one that is ruled out), which
// has no mass, is in none: with them in the last bin, and the bins stretched over the whole span, a flat row with a third of it ruled out
// went the general way (64 rows of 128,256 1,240 us, now 68).
struct Bins {
    float zmax, scale;
    bool capped;                                    // the row spans more than SM_SPAN: nothing in the last bin has any mass
    __device__ inline int of_distance(float d) const {
        const float b = d * scale;
        return b < (float)(SM_BINS - 1) ? (b > 0.f ? (int)b : 0) : SM_BINS - 1;
    }
    __device__ inline int of(float z) const { return of_distance(zmax - z); }
};

// Of a sampled row: z's maximum and the bins (all threads get the same).  `mx`, `mn`: the largest and the smallest finite logit.
__device__ inline Bins make_bins(float mx, float mn, float temp) {
    Bins b;
    b.zmax = mx / temp;                             // (division by the same number keeps the order)
    const float span = b.zmax - mn / temp;
    b.capped = span >= SM_SPAN;
    b.scale = (float)SM_BINS / fminf(SM_SPAN, span);
    return b;
}

// The largest and smallest logit from the ranges' (lanes 0..31 of every wave hold one each).
__device__ inline void row_extent(const float* part, int r, float& mx, float& mn) {
    const int lane = threadIdx.x & 63;
    const float* p = part + ((size_t)r * ROW_SPLITS + (lane & (ROW_SPLITS - 1))) * 2;
    mx = wave_max(p[0]);
    mn = -wave_max(-p[1]);
}

// Mass and (with `counts`) number of the candidates [lo, hi) by bin, added to `mass` and `count` in LDS.
// (a candidate that is no number or -inf is in no bin)
__device__ __forceinline__ void fill_hist(const float* row, int lo, int hi, float temp, const Bins& bins, bool counts, u64* mass, unsigned* count) {
    for_row(row, lo, hi, threadIdx.x, SM_THREADS, [&](float v, int) __attribute__((always_inline)) {
        const float z = v / temp;
        if (!(z > -INFINITY)) return;
        const int b = bins.of(z);
        const u64 m = mass_of(expf(z - bins.zmax));
        if (m) atomicAdd(&mass[b], m);
        if (counts) atomicAdd(&count[b], 1u);
    });
}

// A share of a row's histogram (grid: rows x shares), written whole: nothing has to be cleared between calls.
__global__ __launch_bounds__(SM_THREADS) void k_pick_hist(SampleArgs a, u64* hist_mass, unsigned* hist_count) {
    __shared__ u64 mass[SM_BINS];
    __shared__ unsigned count[SM_BINS];
    const int r = blockIdx.x, sp = blockIdx.y;
    const float temp = a.temp[r];
    if (!(temp > 0.f)) return;
    float mx, mn;
    row_extent(a.part, r, mx, mn);
    const Bins bins = make_bins(mx, mn, temp);
    if (!(fabsf(bins.zmax) < INFINITY)) return;     // (k_sample reads no histogram of such a row)
    const bool counts = a.top_k && a.top_k[r] > 0 && a.top_k[r] < a.V;
    for (int i = threadIdx.x; i < SM_BINS; i += SM_THREADS) { mass[i] = 0; count[i] = 0; }
    __syncthreads();
    const int chunk = ((a.V + a.hist_splits - 1) / a.hist_splits + 3) & ~3;
    const int lo = sp * chunk < a.V ? sp * chunk : a.V, hi = lo + chunk < a.V ? lo + chunk : a.V;
    fill_hist(a.logits + (size_t)r * a.ld, lo, hi, temp, bins, counts, mass, count);
    __syncthreads();
    const size_t at = ((size_t)r * a.hist_splits + sp) * SM_BINS;
    for (int i = threadIdx.x; i < SM_BINS; i += SM_THREADS) {
        hist_mass[at + i] = mass[i];
        if (counts) hist_count[at + i] = count[i];
    }
}

// Inclusive sums over the workgroup's threads, two values a thread in index order.
template <typename T>
__device__ inline void scan_pairs(T& x0, T& x1, T* sh) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    T t = x0 + x1;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const T u = __shfl_up(t, o, 64);
        if (lane >= o) t += u;
    }
    __syncthreads();
    if (lane == 63) sh[wave] = t;
    __syncthreads();
    T before = 0;
    for (int w = 0; w < wave; ++w) before += sh[w];
    t += before;
    x0 = t - x1;
    x1 = t;
}

// The candidates of some neighbouring bins, sorted, and their inclusive sums of mass.
struct List {
    u64 key[SM_LIST];
    u64 sum[SM_LIST];
    int n;
    int lo, hi;         // the bins
};

// Gather and sort the bins [lo, hi]; false: more candidates than the list holds.
__device__ __forceinline__ bool gather(const float* row, int V, float temp, const Bins& bins, int lo, int hi, List& list) {
    __syncthreads();
    if (threadIdx.x == 0) { list.n = 0; list.lo = lo; list.hi = hi; }
    __syncthreads();
    // logits that may lie in the bins: their z within the bins' edges and a margin far above the rounding of z and of the edges
    const float slack = 1e-4f + 1e-5f * fabsf(bins.zmax);
    const float above = hi == SM_BINS - 1 ? -INFINITY : bins.zmax - (float)(hi + 1) / bins.scale - slack;
    const float below = bins.zmax - (float)lo / bins.scale + slack;
    const float vlo = above * temp - 1e-6f * fabsf(above * temp), vhi = below * temp + 1e-6f * fabsf(below * temp);
    for_row(row, 0, V, threadIdx.x, SM_THREADS, [&](float v, int i) __attribute__((always_inline)) {
        if (!(v >= vlo && v <= vhi)) return;
        const float z = v / temp;
        const int b = bins.of(z);
        if (b < lo || b > hi || !(z > -INFINITY)) return;
        const int at = atomicAdd(&list.n, 1);
        if (at < SM_LIST) list.key[at] = order_key(z, i);
    });
    __syncthreads();
    const int n = list.n;
    if (n > SM_LIST) return false;
    if (n > 4 && n <= SM_RANKED) {
        // few: every key's place is the number of keys below it (no two are equal), counted by as many threads as there are for a key,
        // each over its share (a pair's step of the network below, with its barrier, costs 16 waves as much as 30 comparisons: 256 keys
        // take it 36 steps).  A pick of one row of 8,192 logits in us, by the network and counted: 4 keys 18.0 and 18.0, 8 18.6 and 18.3, 64 21.3 and
        // 19.5, 128 22.9 and 20.9, 256 24.5 and 23.7, but 1 17.3 and 17.6, 300 26.5 and 27.8, 511 26.8 and 33.0.
        unsigned* const place = reinterpret_cast<unsigned*>(list.sum);
        int keys = 64;
        while (keys < n) keys <<= 1;
        const int t = threadIdx.x & (keys - 1), share = threadIdx.x / keys, shares = SM_THREADS / keys;
        const int per = (n + shares - 1) / shares, from = share * per, to = from + per < n ? from + per : n;
        const u64 key = list.key[t < n ? t : 0];
        if (threadIdx.x < keys) place[threadIdx.x] = 0;
        __syncthreads();
        unsigned below_it = 0;
        for (int j = from; j < to; ++j) below_it += list.key[j] < key ? 1u : 0u;
        if (t < n) atomicAdd(&place[t], below_it);
        __syncthreads();
        if (share == 0 && t < n) list.key[place[t]] = key;
        __syncthreads();
        return true;
    }
    int m = 2;
    while (m < n) m <<= 1;
    for (int i = n + threadIdx.x; i < m; i += SM_THREADS) list.key[i] = ~0ull;
    __syncthreads();
    for (int k = 2; k <= m; k <<= 1)                // bitonic, a pair a thread
        for (int j = k >> 1; j > 0; j >>= 1) {
            const int t = threadIdx.x;
            if (t < m / 2) {
                const int i = ((t & ~(j - 1)) << 1) | (t & (j - 1));
                const u64 x = list.key[i], y = list.key[i + j];
                if ((x > y) == ((i & k) == 0)) { list.key[i] = y; list.key[i + j] = x; }
            }
            __syncthreads();
        }
    return true;
}

// The list's sums of mass; a candidate with exp(z - z_max) < min_e or a key over `limit` counts nothing.
__device__ __forceinline__ void sum_list(List& list, float zmax, float min_e, u64 limit, u64* sh) {
    const int i = 2 * threadIdx.x;
    u64 m[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        m[e] = 0;
        if (i + e < list.n) {
            const u64 key = list.key[i + e];
            const float x = expf(key_z(key) - zmax);
            if (x >= min_e && key <= limit) m[e] = mass_of(x);
        }
    }
    scan_pairs(m[0], m[1], sh);
    if (i < list.n) list.sum[i] = m[0];
    if (i + 1 < list.n) list.sum[i + 1] = m[1];
    __syncthreads();
}

// The first index whose inclusive sum exceeds `target` (there is one), the same in all threads.
template <typename T>
__device__ __forceinline__ int first_over(const T* sums, int n, T before, T target, int* sh1) {
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += SM_THREADS)
        if (before + sums[i] > target && (i == 0 || !(before + sums[i - 1] > target))) *sh1 = i;
    __syncthreads();
    return *sh1;
}

// The pick where a cut's bin does not fit the list: every boundary by a radix selection over the row.
__device__ __forceinline__ int sample_by_radix(const SampleArgs& a, int r, const float* row, float temp, float zmax, u64* hist, u64* sh, u64* sh2) {
    RowView rv;
    rv.row = row; rv.V = a.V; rv.temp = temp; rv.zmax = zmax;
    rv.limit = ~0ull; rv.min_e = 0.f;
    const int tk = a.top_k ? a.top_k[r] : 0;
    if (tk > 0 && tk < a.V) rv.limit = radix_select(rv, false, (u64)(tk - 1), hist, sh2);
    const float tp = a.top_p ? a.top_p[r] : 1.f;
    if (tp < 1.f) {
        u64 s_k = kept_total(rv, true, sh);
        u64 want = (u64)((double)(tp > 0.f ? tp : 0.f) * (double)s_k);
        rv.limit = radix_select(rv, true, want > 0 ? want - 1 : 0, hist, sh2);
    }
    const float mp = a.min_p ? a.min_p[r] : 0.f;
    if (mp > 0.f) rv.min_e = mp < 1.f ? mp : 1.f;
    u64 s_keep = kept_total(rv, true, sh);
    u64 target = (u64)((double)a.draw[r] * (double)s_keep);
    if (s_keep > 0 && target >= s_keep) target = s_keep - 1;
    return (int)(radix_select(rv, true, target, hist, sh2) & 0xFFFFFFull);
}

// The pick of a sampled row, from its bins' inclusive sums; -1: a cut's bin does not fit the list.
__device__ __forceinline__ int sample_by_bins(const SampleArgs& a, int r, const float* row, float temp, const Bins& bins, const u64* mass,
                              const unsigned* count, List& list, u64* sh, int* sh1) {
    bool have = false;          // (the same in all threads, as is every cut below)
    auto need = [&](int lo, int hi) {
        if (have && list.lo <= lo && hi <= list.hi) return true;
        have = gather(row, a.V, temp, bins, lo, hi, list);
        if (have) sum_list(list, bins.zmax, 0.f, ~0ull, sh);
        return have;
    };
    auto before = [&]() { return list.lo > 0 ? mass[list.lo - 1] : 0ull; };
    u64 limit = ~0ull, kept = mass[SM_BINS - 1];    // keys up to the limit, and their mass
    int last = SM_BINS - 1;                         // the limit's bin
    const int tk = a.top_k ? a.top_k[r] : 0;
    if (tk > 0 && tk < a.V && count[SM_BINS - 1] >= (unsigned)tk) {
        last = first_over(count, SM_BINS, 0u, (unsigned)(tk - 1), sh1);
        // (a cut among candidates without mass changes nothing; their bin may hold most of the row: 64 peaked rows with top-k 40 987 us, 67 so)
        if (!(bins.capped && last == SM_BINS - 1)) {
            const int lo = count[last] <= SM_LIST ? 0 : last;          // all that is kept at once, where it fits
            if (!need(lo, last)) return -1;
            const int i = tk - 1 - (lo > 0 ? (int)count[lo - 1] : 0);
            limit = list.key[i];
            kept = before() + list.sum[i];
        }
    }
    const float tp = a.top_p ? a.top_p[r] : 1.f;
    if (tp < 1.f) {
        const u64 want = (u64)((double)(tp > 0.f ? tp : 0.f) * (double)kept);
        const u64 target = want > 0 ? want - 1 : 0;
        last = first_over(mass, SM_BINS, 0ull, target, sh1);
        if (!need(last, last)) return -1;
        const int i = first_over(list.sum, list.n, before(), target, sh1);
        limit = list.key[i];
        kept = before() + list.sum[i];
    }
    const float mp = a.min_p ? a.min_p[r] : 0.f;
    int edge = SM_BINS;                             // the first bin where min-p may drop a candidate
    if (mp > 0.f) {
        const float min_e = mp < 1.f ? mp : 1.f;
        // (the cut's distance from z_max, with a margin far above the exponential's rounding)
        edge = bins.of_distance(fmaxf(-logf(min_e) - 1e-3f, 0.f));
        const int past = bins.of_distance(-logf(min_e) + 1e-3f);
        if (last < edge) {
            edge = SM_BINS;
        } else {
            const int to = last < past ? last : past;
            have = gather(row, a.V, temp, bins, edge, to, list);
            if (!have) return -1;
            sum_list(list, bins.zmax, min_e, limit, sh);
            kept = before() + (list.n > 0 ? list.sum[list.n - 1] : 0ull);
            last = to;
        }
    }
    u64 target = (u64)((double)a.draw[r] * (double)kept);
    if (kept > 0 && target >= kept) target = kept - 1;
    const bool full = edge > 0 && (edge == SM_BINS || target < mass[edge - 1]);     // in a bin that min-p leaves whole
    if (full) {
        if (edge < SM_BINS) have = false;           // (the list's sums are those behind min-p)
        const int b = first_over(mass, SM_BINS, 0ull, target, sh1);
        if (!need(b, b)) return -1;
    }
    const int i = first_over(list.sum, list.n, before(), target, sh1);
    return (int)(list.key[i] & 0xFFFFFFull);
}

__global__ __launch_bounds__(SM_THREADS) void k_sample(SampleArgs a) {
    __shared__ u64 mass[SM_BINS];
    __shared__ unsigned count[SM_BINS];
    __shared__ List list;
    __shared__ u64 sh[SM_THREADS / 64];
    __shared__ u64 sh2[2];
    __shared__ float shf[SM_THREADS / 64];
    __shared__ int shi[SM_THREADS / 64];
    const int r = blockIdx.x;
    float* row = a.logits + (size_t)r * a.ld;
    const int V = a.V;
    const float temp = a.temp[r];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;

    if (!(temp > 0.f)) {
        // greedy: first index of the maximum, over the logits or over the ranges' results
        float best = -INFINITY;
        int bi = 0x7fffffff;
        if (a.part) {
            if (threadIdx.x < ROW_SPLITS) {
                const float* p = a.part + ((size_t)r * ROW_SPLITS + threadIdx.x) * 2;
                best = p[0];
                bi = __float_as_int(p[1]);
            }
        } else {
            for (int i = threadIdx.x; i < V; i += SM_THREADS) {
                float v = row[i];
                if (v > best || (v == best && i < bi)) { best = v; bi = i; }
            }
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            float ob = __shfl_xor(best, o, 64);
            int oi = __shfl_xor(bi, o, 64);
            if (ob > best || (ob == best && oi < bi)) { best = ob; bi = oi; }
        }
        if (lane == 0) { shf[wave] = best; shi[wave] = bi; }
        __syncthreads();
        if (threadIdx.x == 0) {
            for (int w = 1; w < SM_THREADS / 64; ++w)
                if (shf[w] > best || (shf[w] == best && shi[w] < bi)) { best = shf[w]; bi = shi[w]; }
            a.out[r] = bi == 0x7fffffff ? 0 : bi;
        }
        return;
    }

    float mx = -INFINITY, mn = INFINITY;
    if (a.part) {
        row_extent(a.part, r, mx, mn);
    } else {
        apply_penalty(a, r, row, 0, V);
        for_row(row, 0, V, threadIdx.x, SM_THREADS, [&](float v, int) { mx = v > mx ? v : mx; mn = v < mn && v > -INFINITY ? v : mn; });
        mx = wave_max(mx);
        mn = -wave_max(-mn);
        if (lane == 0) { shf[wave] = mx; shi[wave] = __float_as_int(mn); }
        __syncthreads();
        for (int w = 0; w < SM_THREADS / 64; ++w) { mx = fmaxf(mx, shf[w]); mn = fminf(mn, __int_as_float(shi[w])); }
    }
    const Bins bins = make_bins(mx, mn, temp);
    if (!(fabsf(bins.zmax) < INFINITY)) {           // nothing has any mass
        if (threadIdx.x == 0) a.out[r] = 0;
        return;
    }

    // the bins' sums: two bins a thread
    const bool counts = a.top_k && a.top_k[r] > 0 && a.top_k[r] < V;
    const int b0 = 2 * threadIdx.x;
    u64 m0 = 0, m1 = 0;
    unsigned c0 = 0, c1 = 0;
    if (a.hist_mass) {
        for (int s0 = 0; s0 < a.hist_splits; s0 += 8) {      // (eight shares' loads side by side)
            ulonglong2 m[8];
            uint2 c[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const size_t at = ((size_t)r * a.hist_splits + (s0 + u < a.hist_splits ? s0 + u : s0)) * SM_BINS + b0;
                m[u] = *reinterpret_cast<const ulonglong2*>(a.hist_mass + at);
                c[u] = counts ? *reinterpret_cast<const uint2*>(a.hist_count + at) : make_uint2(0, 0);
            }
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (s0 + u < a.hist_splits) { m0 += m[u].x; m1 += m[u].y; c0 += c[u].x; c1 += c[u].y; }
        }
    } else {
        mass[b0] = mass[b0 + 1] = 0;
        count[b0] = count[b0 + 1] = 0;
        __syncthreads();
        fill_hist(row, 0, V, temp, bins, counts, mass, count);
        __syncthreads();
        m0 = mass[b0]; m1 = mass[b0 + 1];
        c0 = count[b0]; c1 = count[b0 + 1];
    }
    scan_pairs(m0, m1, sh);
    scan_pairs(c0, c1, (unsigned*)sh);
    mass[b0] = m0; mass[b0 + 1] = m1;
    count[b0] = c0; count[b0 + 1] = c1;
    __syncthreads();
    int pick = sample_by_bins(a, r, row, temp, bins, mass, count, list, sh, shi);
    if (pick < 0) pick = sample_by_radix(a, r, row, temp, bins.zmax, mass, sh, sh2);
    if (threadIdx.x == 0) a.out[r] = pick;
}

static int sample_launch(int* out, float* logits, int W, int V, int ld, const float* temp, const int* top_k,
                         const float* top_p, const float* min_p, const float* repeat_penalty,
                         const float* draw, const int* recent, const int* n_recent, int recent_cap,
                         const int* exempt, int n_exempt, float* part_ws, u64* hist_ws, int hist_splits, hipStream_t stream) {
    XR_REQUIRE(W >= 0 && V > 0 && ld >= V, "sample: bad sizes W=%d V=%d ld=%d", W, V, ld);
    XR_REQUIRE(V <= (1 << 24), "sample: vocabulary %d exceeds 2^24", V);
    XR_REQUIRE(out && logits && temp && draw, "sample: null operand");
    XR_REQUIRE(!recent || (n_recent && recent_cap > 0), "sample: a recent window without its length");
    if (W == 0) return XR_OK;
    SampleArgs a;
    a.out = out; a.logits = logits; a.ld = ld; a.V = V; a.temp = temp; a.top_k = top_k; a.top_p = top_p;
    a.min_p = min_p; a.repeat_penalty = repeat_penalty; a.draw = draw; a.recent = recent;
    a.n_recent = n_recent; a.recent_cap = recent_cap; a.exempt = exempt; a.n_exempt = exempt ? n_exempt : 0;
    a.part = part_ws;
    a.hist_mass = nullptr; a.hist_count = nullptr; a.hist_splits = 0;
    if (part_ws) {          // [W, ROW_SPLITS, 2] floats
        k_pick_extent<<<dim3(W, ROW_SPLITS), 256, 0, stream>>>(a, part_ws);
        XR_CHECK_LAUNCH("sample_extent");
    }
    if (part_ws && hist_ws && hist_splits > 0) {     // [W, splits, SM_BINS] masses, then as many counts
        a.hist_mass = hist_ws;
        a.hist_count = (const unsigned*)(hist_ws + (size_t)W * hist_splits * SM_BINS);
        a.hist_splits = hist_splits;
        k_pick_hist<<<dim3(W, hist_splits), SM_THREADS, 0, stream>>>(a, hist_ws, (unsigned*)a.hist_count);
        XR_CHECK_LAUNCH("sample_hist");
    }
    k_sample<<<W, SM_THREADS, 0, stream>>>(a);
    XR_CHECK_LAUNCH("sample");
    return XR_OK;
}

extern "C" int xr_sample(int* out, float* logits, int W, int V, int ld, const float* temp, const int* top_k,
                         const float* top_p, const float* min_p, const float* repeat_penalty,
                         const float* draw, const int* recent, const int* n_recent, int recent_cap,
                         const int* exempt, int n_exempt, float* greedy_ws, hipStream_t stream) {
    return sample_launch(out, logits, W, V, ld, temp, top_k, top_p, min_p, repeat_penalty, draw, recent, n_recent,
                         recent_cap, exempt, n_exempt, greedy_ws, nullptr, 0, stream);
}

// The same with a work area of W * splits * 3 * SM_BINS * 4 bytes for the sampled rows' histograms, each shared out to
// `splits` workgroups.
extern "C" int xr_sample_split(int* out, float* logits, int W, int V, int ld, const float* temp, const int* top_k,
                               const float* top_p, const float* min_p, const float* repeat_penalty,
                               const float* draw, const int* recent, const int* n_recent, int recent_cap,
                               const int* exempt, int n_exempt, float* greedy_ws, void* hist_ws, long long hist_bytes,
                               int splits, hipStream_t stream) {
    XR_REQUIRE(greedy_ws && hist_ws && splits > 0 && splits <= 32, "sample_split: no work area or %d splits", splits);
    XR_REQUIRE(((uintptr_t)hist_ws & 15) == 0 && hist_bytes >= (long long)W * splits * SM_BINS * 12, "sample_split: a work area of %lld bytes for %d rows in %d parts",
               hist_bytes, W, splits);
    return sample_launch(out, logits, W, V, ld, temp, top_k, top_p, min_p, repeat_penalty, draw, recent, n_recent,
                         recent_cap, exempt, n_exempt, greedy_ws, (u64*)hist_ws, splits, stream);
}

// ------------------------------------------------------------------------------ no allocation
// The same pick with the first pass's work area in an array of the library's own (no_alloc.h).
// In host code the array's name is only a handle: its device address is asked for once per
// device and kept, and the kernels get that address as they get the caller's work area above.
#define XR_MAX_DEVICES 64
static __device__ __align__(256) float scratch[(size_t)XR_SAMPLE_STATIC_MAX_ROWS * ROW_SPLITS * 2];
static float* scratch_ptr[XR_MAX_DEVICES];       // the array's address on each device, once resolved
static std::mutex scratch_lock;

static int scratch_on_current_device(float** ptr) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) (void)hipGetLastError();
    XR_REQUIRE(e == hipSuccess, "sample_static: no current device: %s", hipGetErrorString(e));
    XR_REQUIRE(dev >= 0 && dev < XR_MAX_DEVICES, "sample_static: device %d is beyond the %d this library keeps an address for", dev, XR_MAX_DEVICES);
    std::lock_guard<std::mutex> hold(scratch_lock);
    if (!scratch_ptr[dev]) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) (void)hipGetLastError();
        XR_REQUIRE(e == hipSuccess && p, "sample_static: the work area's address on device %d: %s", dev, hipGetErrorString(e));
        scratch_ptr[dev] = (float*)p;
    }
    *ptr = scratch_ptr[dev];
    return XR_OK;
}

extern "C" int xr_sample_static_init() {
    float* p = nullptr;
    return scratch_on_current_device(&p);
}

extern "C" int xr_sample_static(int* out, float* logits, int W, int V, int ld, const float* temp, const int* top_k,
                                const float* top_p, const float* min_p, const float* repeat_penalty,
                                const float* draw, const int* recent, const int* n_recent, int recent_cap,
                                const int* exempt, int n_exempt, hipStream_t stream) {
    XR_REQUIRE(W <= XR_SAMPLE_STATIC_MAX_ROWS, "sample_static: %d rows, the library's work area holds %d (use xr_sample with a work area of the caller's)",
               W, XR_SAMPLE_STATIC_MAX_ROWS);
    float* ws = nullptr;
    const int rc = scratch_on_current_device(&ws);
    if (rc != XR_OK) return rc;
    return sample_launch(out, logits, W, V, ld, temp, top_k, top_p, min_p, repeat_penalty, draw, recent, n_recent,
                         recent_cap, exempt, n_exempt, ws, nullptr, 0, stream);
}
