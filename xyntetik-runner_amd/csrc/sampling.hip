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
// What bounds it: the logits come twice from the caches and an exponential for each is 5 us; the rest is chains of short dependent steps.
// So a row is shared out to up to 8 workgroups where the caller brings room, and the last of them goes on alone, a step as short as it can be: it adds up the
// histograms and says which bins the cuts can fall into (k_pick_hist), and among the candidates that all found there it picks (k_pick_rows).
// 64 rows of 128,256 logits, top-p: 1,150 us where every cut was a radix selection (22 passes over the row), 54 in three kernels with one workgroup a row for the
// cuts, which read the row again for each (7 + 16 + 30), now 44 (7 + 17 + 19; the sums of the bins moved from the third to the second).
#include "common.h"
#include "no_alloc.h"

#include <mutex>

#define SM_THREADS 1024
#define SM_BINS 2048            // ranges of z a row's candidates are counted in
#define SM_SPAN 28.f            // below z_max - 28 a candidate's mass is 0 (exp(-28) < 2^-40)
#define SM_LIST 2048            // candidates of a cut's bin that are sorted in LDS
#define SM_RANKED 256           // and up to so many by counting the keys below each
#define PENALTY_LDS 512         // recent tokens that a workgroup keeps in LDS
#define ROW_SPLITS 32           // workgroups that look for a row's largest and smallest logit
#define SM_FEW 256              // threads that pick among few candidates of a row that many workgroups shared
#define SM_CUTS 4               // runs of bins that a pick may look into
#define SM_FOUND 2048           // candidates of all of them that are kept for a row

typedef unsigned long long u64;

// What the workgroups of a row tell each other.
struct RowNotes {
    int arrived[2];             // workgroups that have left their histogram, their candidates
    int n_found;
    int n_cuts;                 // runs of bins to look into; -1: nothing has any mass
    int lo[SM_CUTS], hi[SM_CUTS];
    float vlo[SM_CUTS], vhi[SM_CUTS];       // logits outside are in no bin of the run
    float zmax, scale;
    int capped, pad;
};
static_assert(sizeof(RowNotes) == 96, "a row's notes are 96 bytes");

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
    // the work area of k_pick_hist and k_pick_rows
    u64* hist_mass;             // [W, hist_splits, SM_BINS]
    unsigned* hist_count;       // the same for the number of candidates (rows with top-k only)
    u64* mass;                  // [W, SM_BINS] sums over the row of the bins up to each
    unsigned* count;            // the same
    u64* found;                 // [W, SM_FOUND] keys of the candidates in the runs of bins
    RowNotes* notes;            // [W]
    int hist_splits;
};

// A row's options.  The kernels bring them into LDS beside their first loads: read where they are needed, each is a trip to memory that
// nothing covers (four of them in the walk from cut to cut).
struct Options {
    int top_k;
    float top_p, min_p, draw;
    __device__ inline void load(const SampleArgs& a, int r) {
        top_k = a.top_k ? a.top_k[r] : 0;
        top_p = a.top_p ? a.top_p[r] : 1.f;
        min_p = a.min_p ? a.min_p[r] : 0.f;
        draw = a.draw[r];
    }
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

// The whole part of e * 2^40 for 0 <= e <= 1 (its upper 9 bits, then the 32 below; every step is exact).
__device__ inline u64 mass_of(float e) {
    const float t = e * 256.f;
    const uint32_t hi = (uint32_t)t;
    return (u64)hi << 32 | (u64)(uint32_t)((t - (float)hi) * 4294967296.f);
}

// Words that the workgroups of a row hand each other, past the caches of one XCD.
__device__ inline void store_agent(u64* p, u64 v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ inline void store_agent(unsigned* p, unsigned v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
template <typename T> __device__ inline T load_agent(const T* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
// Whether this workgroup is the last of `n` to come here; what each stored before (by store_agent) is then there for it.  Nobody waits.
__device__ inline bool last_to_arrive(int* counter, int n, int* sh1) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // this wave's own stores
    __syncthreads();
    if (threadIdx.x == 0) *sh1 = __hip_atomic_fetch_add(counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == n - 1;
    __syncthreads();
    return *sh1 != 0;
}

// z of a key (-0 comes back as +0, whose mass is the same).
__device__ inline float key_z(u64 key) {
    const uint32_t u = ~(uint32_t)(key >> 24);
    return __uint_as_float((u >> 31) ? u & 0x7FFFFFFFu : ~u);
}

// f(value, index) for the candidates [lo, hi) of a row, `step` threads side by side; lo is a multiple of 4.
// 16-byte loads where the row's address allows it, up to 8 of them on their way before the first value is looked at (one
// after the other, a workgroup's pass over 128k logits is 31 trips to memory: k_sample for 64 rows 45 us, now 34), one where
// that is all there is to read (200 sampled rows of 32,000: k_pick_extent 9.6 us with eight, 7.0 with one).  Where f is long (U = 0): a loop that
// is not unrolled, two loads ahead; a workgroup that walks its share once waits for every line of code as it waits for every line of data.
template <int U, typename P, typename F>
__device__ __forceinline__ void for_fours(const float* row, int lo, int tail, int tid, int step, P prepare, F f) {
    int i0 = lo + 4 * tid;
    if constexpr (U == 0) {
        auto at = [&](int i) __attribute__((always_inline)) { return *reinterpret_cast<const float4*>(row + (i < tail ? i : i0)); };
        float4 a = make_float4(0.f, 0.f, 0.f, 0.f), b = a;
        if (i0 < tail) { a = at(i0); b = at(i0 + 4 * step); }
        prepare();
#pragma unroll 1
        for (; i0 < tail; i0 += 4 * step) {
            const float4 c = at(i0 + 8 * step);
            f(a.x, i0);
            f(a.y, i0 + 1);
            f(a.z, i0 + 2);
            f(a.w, i0 + 3);
            a = b;
            b = c;
        }
        return;
    }
    float4 v[U ? U : 1];
    auto load = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = i0 + 4 * step * u;
            v[u] = *reinterpret_cast<const float4*>(row + (i < tail ? i : i0));
        }
    };
    if (i0 < tail) load();
    prepare();
    while (i0 < tail) {
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
        i0 += 4 * step * U;
        if (i0 < tail) load();
    }
}
// `prepare` (what `f` needs, by all threads) runs while the first loads are on their way.
template <int U = 8, typename P, typename F>
__device__ __forceinline__ void for_row_after(const float* row, int lo, int hi, int tid, int step, P prepare, F f) {
    int tail = lo;
    if (((uintptr_t)row & 15) == 0) {
        tail = lo + ((hi - lo) & ~3);
        if (tail - lo <= 4 * step) for_fours<1>(row, lo, tail, tid, step, prepare, f);
        else for_fours<U>(row, lo, tail, tid, step, prepare, f);
    } else {
        prepare();
    }
    for (int i = tail + tid; i < hi; i += step) f(row[i], i);
}
template <int U = 8, typename F>
__device__ __forceinline__ void for_row(const float* row, int lo, int hi, int tid, int step, F f) {
    for_row_after<U>(row, lo, hi, tid, step, [] {}, f);
}

// The repeat penalty of the tokens in [lo, hi): the thread with a token's first place in the window
// applies it as often as the token occurs, which is what walking the window in order does.
__device__ inline void apply_penalty(const SampleArgs& a, int r, float* row, int lo, int hi) {
    const float rp = a.repeat_penalty ? a.repeat_penalty[r] : 1.f;
    if (rp == 1.f || !a.recent) return;
    const int* rec = a.recent + (size_t)r * a.recent_cap;
    const int n = a.n_recent[r] < a.recent_cap ? a.n_recent[r] : a.recent_cap;
    // (the window in LDS: every token walks all of it, and read from memory step by step the windows of 64 rows were 40 us of their 120)
    __shared__ int window[PENALTY_LDS];
    const bool staged = n <= PENALTY_LDS;
    if (staged)
        for (int i = threadIdx.x; i < n; i += blockDim.x) window[i] = rec[i];
    __syncthreads();
    auto walk = [&](const int* rec) __attribute__((always_inline)) {
        for (int i = threadIdx.x; i < n; i += blockDim.x) {
            const int tok = rec[i];
            if (tok < lo || tok >= hi) continue;
            bool skip = false;
            for (int k = 0; k < a.n_exempt; ++k) skip = skip || a.exempt[k] == tok;
            int times = 0;
#pragma unroll 8
            for (int j = 0; j < n; ++j) {
                const bool same = rec[j] == tok;
                skip = skip | (same & (j < i));
                times += same ? 1 : 0;
            }
            if (skip) continue;
            float v = row[tok];
            for (int k = 0; k < times; ++k) v = v > 0.f ? v / rp : v * rp;
            row[tok] = v;
        }
    };
    if (staged) walk(window);
    else walk(rec);
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
    if (a.notes && sp == 0 && threadIdx.x < sizeof(RowNotes) / 4) reinterpret_cast<int*>(a.notes + r)[threadIdx.x] = 0;
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

template <int NT>
__device__ __forceinline__ u64 block_sum_u64(u64 v, u64* sh) {
    // sh has NT / 64 entries
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    __syncthreads();
    if (lane == 0) sh[wave] = v;
    __syncthreads();
    u64 t = 0;
    for (int w = 0; w < NT / 64; ++w) t += sh[w];
    return t;
}

// Mass (by_mass) or number of the kept candidates.
template <int U, int NT>
__device__ __forceinline__ u64 kept_total(const RowView& rv, bool by_mass, u64* sh) {
    u64 acc = 0;
    for_row<U>(rv.row, 0, rv.V, threadIdx.x, NT, [&](float v, int i) __attribute__((always_inline)) {
        u64 key, mass;
        if (row_item(rv, v, i, key, mass)) acc += by_mass ? mass : 1ull;
    });
    return block_sum_u64<NT>(acc, sh);
}

// Smallest key B among the kept candidates with F(B) > target, where F(B) is the mass
// (by_mass) or the number of kept candidates with key <= B.  If no key reaches the
// target the largest kept key is returned.
template <int U, int NT>
__device__ __forceinline__ u64 radix_select(const RowView& rv, bool by_mass, u64 target,
                                           u64* hist, u64* sh2) {
    u64 prefix = 0, remaining = target;
    for (int shift = 48; shift >= 0; shift -= 8) {
        __syncthreads();
        if (threadIdx.x < 256) hist[threadIdx.x] = 0;
        __syncthreads();
        for_row<U>(rv.row, 0, rv.V, threadIdx.x, NT, [&](float v, int i) __attribute__((always_inline)) {
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
    bool ordinary;                                  // `quotient` may stand for the division (see there)
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
    b.ordinary = fmaxf(fabsf(mx), fabsf(mn)) < 0x1p60f && temp > 0x1p-20f && temp < 0x1p20f && span > 0x1p-20f;
    return b;
}

// v / temp with inv = 1 / temp rounded, in five instructions for the division's ten: v inv is within two units of the last place, one step of Newton's brings
// it within one, and from there q + (v - q temp) inv rounds as the quotient does (the remainder is exact).  |v| below 2^-60, where a remainder may be lost, does not matter
// in a row whose z span more than 2^-20: neither its bin nor its mass depends on its last place.  (-inf and what is no number give no number, as
// a candidate that is in no bin.)
__device__ __forceinline__ float quotient(float v, float temp, float inv) {
    float q = v * inv;
    q = fmaf(fmaf(-temp, q, v), inv, q);
    return fmaf(fmaf(-temp, q, v), inv, q);
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
template <int U, bool PLAIN, typename P>
__device__ __forceinline__ void fill_hist(const float* row, int lo, int hi, float temp, const Bins& bins, bool counts, u64* mass, unsigned* count, P prepare,
                                          const bool& skip) {
    const float inv = 1.0f / temp;
    for_row_after<U>(row, lo, hi, threadIdx.x, SM_THREADS, prepare, [&](float v, int) __attribute__((always_inline)) {
        if (skip) return;
        const float z = PLAIN ? v / temp : quotient(v, temp, inv);
        if (!(z > -INFINITY)) return;
        const int b = bins.of(z);
        const u64 m = mass_of(expf(z - bins.zmax));
        if (m) atomicAdd(&mass[b], m);
        if (counts) atomicAdd(&count[b], 1u);
    });
}

// A lane's value from another lane of its wave (DPP), zero where there is none.
template <int CTRL, int ROWS> __device__ __forceinline__ unsigned from_lane(unsigned v) {
    return (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xF, false);
}
template <int CTRL, int ROWS> __device__ __forceinline__ u64 from_lane(u64 v) {
    return (u64)from_lane<CTRL, ROWS>((unsigned)(v >> 32)) << 32 | from_lane<CTRL, ROWS>((unsigned)v);
}
// Inclusive sums over 16 lanes: shifts by 1, 2, 4 and 8 lanes inside a row of 16.
template <typename T> __device__ __forceinline__ T scan_16(T t) {
    t += from_lane<0x111, 0xF>(t);
    t += from_lane<0x112, 0xF>(t);
    t += from_lane<0x114, 0xF>(t);
    t += from_lane<0x118, 0xF>(t);
    return t;
}
// Inclusive sums over the workgroup's threads, two values a thread in index order.  (Shuffles go through LDS, and the waves' sums added
// one after the other are 15 reads in a row: a histogram's sums 2.4 us, 1.5 so.)
template <int NT = SM_THREADS, typename T>
__device__ __forceinline__ void scan_pairs(T& x0, T& x1, T* sh) {
    static_assert(NT <= 1024, "16 waves");
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    T t = scan_16(x0 + x1);
    t += from_lane<0x142, 0xA>(t);          // the last lane of rows 0 and 2 to rows 1 and 3,
    t += from_lane<0x143, 0xC>(t);          // that of row 1 to rows 2 and 3
    __syncthreads();
    if (lane == 63) sh[wave] = t;
    __syncthreads();
    const T s = scan_16((lane & 15) < NT / 64 ? sh[lane & 15] : (T)0);
    T before = 0;
    if (wave > 0) {
        if constexpr (sizeof(T) == 8)
            before = (T)(unsigned)__builtin_amdgcn_readlane((int)((u64)s >> 32), wave - 1) << 32 | (unsigned)__builtin_amdgcn_readlane((int)(u64)s, wave - 1);
        else before = (T)__builtin_amdgcn_readlane((int)s, wave - 1);
    }
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

// Logits that may lie in the bins [lo, hi]: their z within the bins' edges and a margin far above the rounding of z and of the edges.
__device__ inline void logit_range(const Bins& bins, float temp, int lo, int hi, float& vlo, float& vhi) {
    const float slack = 1e-4f + 1e-5f * fabsf(bins.zmax);
    const float above = hi == SM_BINS - 1 ? -INFINITY : bins.zmax - (float)(hi + 1) / bins.scale - slack;
    const float below = bins.zmax - (float)lo / bins.scale + slack;
    vlo = above * temp - 1e-6f * fabsf(above * temp);
    vhi = below * temp + 1e-6f * fabsf(below * temp);
}

// Candidates that the row's workgroups found, in LDS, and the runs of bins they are all of; `n` < 0: none.
struct Found {
    const u64* key;
    int n;
    const RowNotes* notes;
    __device__ inline bool covers(int lo, int hi) const {
        bool in = false;
        if (n >= 0)
            for (int c = 0; c < notes->n_cuts; ++c) in = in || (notes->lo[c] <= lo && hi <= notes->hi[c]);
        return in;
    }
};

// Gather and sort the bins [lo, hi], from what was found or from the row; false: more candidates than the list holds.
template <int U, int NT>
__device__ __forceinline__ bool gather(const float* row, int V, float temp, const Bins& bins, const Found& found, int lo, int hi, List& list) {
    __syncthreads();
    if (threadIdx.x == 0) { list.n = 0; list.lo = lo; list.hi = hi; }
    __syncthreads();
    if (found.covers(lo, hi)) {
        for (int i = threadIdx.x; i < found.n; i += NT) {
            const u64 key = found.key[i];
            const int b = bins.of(key_z(key));
            if (b < lo || b > hi) continue;
            const int at = atomicAdd(&list.n, 1);
            if (at < SM_LIST) list.key[at] = key;
        }
    } else {
        float vlo, vhi;
        logit_range(bins, temp, lo, hi, vlo, vhi);
        for_row<U>(row, 0, V, threadIdx.x, NT, [&](float v, int i) __attribute__((always_inline)) {
            if (!(v >= vlo && v <= vhi)) return;
            const float z = v / temp;
            const int b = bins.of(z);
            if (b < lo || b > hi || !(z > -INFINITY)) return;
            const int at = atomicAdd(&list.n, 1);
            if (at < SM_LIST) list.key[at] = order_key(z, i);
        });
    }
    __syncthreads();
    const int n = list.n;
    if (n > SM_LIST || n > 2 * NT) return false;
    if (n > 4 && n <= SM_RANKED) {
        // few: every key's place is the number of keys below it (no two are equal), counted by as many threads as there are for a key,
        // each over its share (a pair's step of the network below, with its barrier, costs 16 waves as much as 30 comparisons: 256 keys
        // take it 36 steps).  A pick of one row of 8,192 logits in us, by the network and counted: 4 keys 18.0 and 18.0, 8 18.6 and 18.3, 64 21.3 and
        // 19.5, 128 22.9 and 20.9, 256 24.5 and 23.7, but 1 17.3 and 17.6, 300 26.5 and 27.8, 511 26.8 and 33.0.
        unsigned* const place = reinterpret_cast<unsigned*>(list.sum);
        int keys = 64;
        while (keys < n) keys <<= 1;
        const int t = threadIdx.x & (keys - 1), share = threadIdx.x / keys, shares = NT / keys;
        const int per = ((n + shares - 1) / shares + 7) & ~7, from = share * per;      // (eight comparisons' reads side by side)
        const u64 key = list.key[t < n ? t : 0];
        if (threadIdx.x < keys) place[threadIdx.x] = 0;
        for (int i = n + threadIdx.x; i < shares * per; i += NT) list.key[i] = ~0ull;
        __syncthreads();
        unsigned below_it = 0;
#pragma unroll 1
        for (int j = from; j < from + per; j += 8) {
            u64 other[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) other[e] = list.key[j + e];
#pragma unroll
            for (int e = 0; e < 8; ++e) below_it += other[e] < key ? 1u : 0u;
        }
        if (t < n) atomicAdd(&place[t], below_it);
        __syncthreads();
        if (share == 0 && t < n) list.key[place[t]] = key;
        __syncthreads();
        return true;
    }
    int m = 2;
    while (m < n) m <<= 1;
    for (int i = n + threadIdx.x; i < m; i += NT) list.key[i] = ~0ull;
    __syncthreads();
    for (int k = 2; k <= m; k <<= 1)                // bitonic, a pair a thread
        for (int j = k >> 1; j > 0; j >>= 1) {
            for (int t = threadIdx.x; t < m / 2; t += NT) {
                const int i = ((t & ~(j - 1)) << 1) | (t & (j - 1));
                const u64 x = list.key[i], y = list.key[i + j];
                if ((x > y) == ((i & k) == 0)) { list.key[i] = y; list.key[i + j] = x; }
            }
            __syncthreads();
        }
    return true;
}

// The list's sums of mass; a candidate with exp(z - z_max) < min_e or a key over `limit` counts nothing.
template <int NT>
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
    scan_pairs<NT>(m[0], m[1], sh);
    if (i < list.n) list.sum[i] = m[0];
    if (i + 1 < list.n) list.sum[i + 1] = m[1];
    __syncthreads();
}

// The first index whose inclusive sum exceeds `target` (at most n - 1, n up to SM_BINS), the same in all threads: every wave looks at
// the ends of 64 blocks, then into one.  (No barrier: all threads at once need one before and after.)
template <typename T>
__device__ __forceinline__ int first_over(const T* sums, int n, T before, T target) {
    constexpr int BLOCK = SM_BINS / 64;
    static_assert(SM_LIST <= SM_BINS && BLOCK <= 64, "a lane a block");
    const int lane = threadIdx.x & 63;
    const int end = lane * BLOCK + BLOCK - 1;
    const int block = __ffsll((unsigned long long)__ballot(end >= n || before + sums[end] > target)) - 1;
    const int none = n > 0 ? n - 1 : 0;
    if (block < 0) return none;
    const int i = block * BLOCK + (lane < BLOCK ? lane : BLOCK - 1);
    const int at = __ffsll((unsigned long long)__ballot(i >= n || before + sums[i] > target)) - 1;
    const int found = block * BLOCK + (at < 0 ? 0 : at);
    return found < n ? found : none;
}

// The runs of bins that sample_by_bins may gather, from the sums of the bins alone.  Inside a cut's bin the cut's place is not known yet,
// so the mass that is kept lies between those of the bins before it and with it, and what follows from it (a share of it, or the draw's
// place) in the bins between two.  More runs or longer ones than needed cost time only, and a run that is missed is gathered from the row.
__device__ __forceinline__ void plan_cuts(const SampleArgs& a, int r, const Options& opt, const Bins& bins, const u64* mass, const unsigned* count) {
    int lo[SM_CUTS], hi[SM_CUTS], n = 0;
    auto add = [&](int l, int h) {
#pragma unroll
        for (int c = 0; c < SM_CUTS; ++c)
            if (c == n) { lo[c] = l; hi[c] = h; }
        ++n;
    };
    auto up_to = [&](int b) { return b > 0 ? mass[b - 1] : 0ull; };
    u64 least = mass[SM_BINS - 1], most = least;        // the mass that is kept
    int last = SM_BINS - 1;                             // the limit's bin, at most
    const int tk = opt.top_k;
    if (tk > 0 && tk < a.V && count[SM_BINS - 1] >= (unsigned)tk) {
        last = first_over(count, SM_BINS, 0u, (unsigned)(tk - 1));
        if (!(bins.capped && last == SM_BINS - 1)) {
            add(count[last] <= SM_LIST ? 0 : last, last);
            least = up_to(last);
            most = mass[last];
        }
    }
    const float tp = opt.top_p;
    if (tp < 1.f) {
        const double share = tp > 0.f ? (double)tp : 0.0;
        const u64 w0 = (u64)(share * (double)least), w1 = (u64)(share * (double)most);
        const int first = first_over(mass, SM_BINS, 0ull, w0 > 0 ? w0 - 1 : 0ull);
        last = first_over(mass, SM_BINS, 0ull, w1 > 0 ? w1 - 1 : 0ull);
        add(first, last);
        least = up_to(first);
        most = mass[last];
    }
    const float mp = opt.min_p;
    if (mp > 0.f) {
        const float min_e = mp < 1.f ? mp : 1.f;
        const int edge = bins.of_distance(fmaxf(-logf(min_e) - 1e-3f, 0.f)), past = bins.of_distance(-logf(min_e) + 1e-3f);
        if (last >= edge) {
            add(edge, last < past ? last : past);
            least = least < up_to(edge) ? least : up_to(edge);
            const u64 whole = mass[last < past ? last : past];      // (what lies behind the cut's bins goes: min-p alone, 20 rows of 128,256 logits 62 us a pick with all
            most = most < whole ? most : whole;                      // that mass left to the draw, whose run of bins then held more than the list takes)
        }
    }
    const double draw = (double)opt.draw;
    const u64 t0 = (u64)(draw * (double)least);
    u64 t1 = (u64)(draw * (double)most);
    if (most > 0 && t1 >= most) t1 = most - 1;
    add(first_over(mass, SM_BINS, 0ull, t0 < t1 ? t0 : t1), first_over(mass, SM_BINS, 0ull, t1));
    if (threadIdx.x == 0) {
        RowNotes* notes = a.notes + r;
#pragma unroll
        for (int c = 0; c < SM_CUTS; ++c)
            if (c < n) {
                notes->lo[c] = lo[c];
                notes->hi[c] = hi[c];
                logit_range(bins, a.temp[r], lo[c], hi[c], notes->vlo[c], notes->vhi[c]);
            }
        notes->n_cuts = n;
        notes->zmax = bins.zmax;
        notes->scale = bins.scale;
        notes->capped = bins.capped;
    }
}

// The pick where a cut's bin does not fit the list: every boundary by a radix selection over the row.
template <int U, int NT>
__device__ __forceinline__ int sample_by_radix(const SampleArgs& a, int r, const float* row, float temp, float zmax, u64* hist, u64* sh, u64* sh2) {
    RowView rv;
    rv.row = row; rv.V = a.V; rv.temp = temp; rv.zmax = zmax;
    rv.limit = ~0ull; rv.min_e = 0.f;
    const int tk = a.top_k ? a.top_k[r] : 0;
    if (tk > 0 && tk < a.V) rv.limit = radix_select<U, NT>(rv, false, (u64)(tk - 1), hist, sh2);
    const float tp = a.top_p ? a.top_p[r] : 1.f;
    if (tp < 1.f) {
        u64 s_k = kept_total<U, NT>(rv, true, sh);
        u64 want = (u64)((double)(tp > 0.f ? tp : 0.f) * (double)s_k);
        rv.limit = radix_select<U, NT>(rv, true, want > 0 ? want - 1 : 0, hist, sh2);
    }
    const float mp = a.min_p ? a.min_p[r] : 0.f;
    if (mp > 0.f) rv.min_e = mp < 1.f ? mp : 1.f;
    u64 s_keep = kept_total<U, NT>(rv, true, sh);
    u64 target = (u64)((double)a.draw[r] * (double)s_keep);
    if (s_keep > 0 && target >= s_keep) target = s_keep - 1;
    return (int)(radix_select<U, NT>(rv, true, target, hist, sh2) & 0xFFFFFFull);
}

// The pick of a sampled row, from its bins' inclusive sums; -1: a cut's bin does not fit the list.
template <int U, int NT>
__device__ __forceinline__ int sample_by_bins(const SampleArgs& a, const Options& opt, const float* row, float temp, const Bins& bins, const Found& found,
                              const u64* mass, const unsigned* count, List& list, u64* sh) {
    bool have = false;          // (the same in all threads, as is every cut below)
    u64 limit = ~0ull, kept = mass[SM_BINS - 1];    // keys up to the limit, and their mass
    int last = SM_BINS - 1;                         // the limit's bin
    int edge = SM_BINS;                             // the first bin where min-p may drop a candidate
    // One turn a cut: its bins and what is looked for in them, the list of their candidates, the place in the list.  (A loop, not four copies
    // of the list's code: a workgroup that walks a copy once waits for its code line by line.)
#pragma unroll 1
    for (int cut = 0; cut < 4; ++cut) {
        int lo = 0, hi = -1, rank = 0;
        u64 target = 0, under = ~0ull;
        float min_e = 0.f;
        if (cut == 0) {
            const int tk = opt.top_k;
            if (tk > 0 && tk < a.V && count[SM_BINS - 1] >= (unsigned)tk) {
                last = first_over(count, SM_BINS, 0u, (unsigned)(tk - 1));
                // (a cut among candidates without mass changes nothing; their bin may hold most of the row: 64 peaked rows with top-k 40 987 us, 67 so)
                if (!(bins.capped && last == SM_BINS - 1)) {
                    lo = count[last] <= SM_LIST ? 0 : last;            // all that is kept at once, where it fits
                    hi = last;
                    rank = tk - 1 - (lo > 0 ? (int)count[lo - 1] : 0);
                }
            }
        } else if (cut == 1) {
            const float tp = opt.top_p;
            if (tp < 1.f) {
                const u64 want = (u64)((double)(tp > 0.f ? tp : 0.f) * (double)kept);
                target = want > 0 ? want - 1 : 0;
                lo = hi = last = first_over(mass, SM_BINS, 0ull, target);
            }
        } else if (cut == 2) {
            const float mp = opt.min_p;
            if (mp > 0.f) {
                min_e = mp < 1.f ? mp : 1.f;
                // (the cut's distance from z_max, with a margin far above the exponential's rounding)
                const int first = bins.of_distance(fmaxf(-logf(min_e) - 1e-3f, 0.f));
                const int past = bins.of_distance(-logf(min_e) + 1e-3f);
                if (last >= first) {
                    lo = edge = first;
                    hi = last < past ? last : past;
                    under = limit;
                    have = false;
                }
            }
        } else {
            target = (u64)((double)opt.draw * (double)kept);
            if (kept > 0 && target >= kept) target = kept - 1;
            if (edge > 0 && (edge == SM_BINS || target < mass[edge - 1])) {     // in a bin that min-p leaves whole
                if (edge < SM_BINS) have = false;           // (the list's sums are those behind min-p)
                lo = hi = first_over(mass, SM_BINS, 0ull, target);
            } else {
                lo = list.lo;
                hi = list.hi;
            }
        }
        if (hi < lo) continue;
        if (!(have && list.lo <= lo && hi <= list.hi)) {
            have = gather<U, NT>(row, a.V, temp, bins, found, lo, hi, list);
            if (!have) return -1;
            sum_list<NT>(list, bins.zmax, min_e, under, sh);
        }
        const u64 before = list.lo > 0 ? mass[list.lo - 1] : 0ull;
        if (cut == 2) {
            kept = before + (list.n > 0 ? list.sum[list.n - 1] : 0ull);
            last = hi;
            continue;
        }
        const int i = cut == 0 ? rank : first_over(list.sum, list.n, before, target);
        if (cut == 3) return (int)(list.key[i] & 0xFFFFFFull);
        limit = list.key[i];
        kept = before + list.sum[i];
    }
    return -1;
}

// A greedy row's pick from the first pass's ranges (`part`) or over the logits: the first index of the maximum.
__device__ __forceinline__ void pick_greedy(const SampleArgs& a, int r, const float* row, float* shf, int* shi) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    float best = -INFINITY;
    int bi = 0x7fffffff;
    if (a.part) {
        if (threadIdx.x < ROW_SPLITS) {
            const float* p = a.part + ((size_t)r * ROW_SPLITS + threadIdx.x) * 2;
            best = p[0];
            bi = __float_as_int(p[1]);
        }
    } else {
        for (int i = threadIdx.x; i < a.V; i += SM_THREADS) {
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
}

// A share of a row's histogram (grid: rows x shares).  The last of the row's workgroups adds the shares up and leaves the sums of the
// bins and the runs of bins to look into; or (PICK) it picks, reading the row again for every cut, which for a row that is not long is less than a kernel's
// boundary and what the workgroups tell each other a second time.
template <bool PICK>
__global__ __launch_bounds__(SM_THREADS, 8) void k_pick_hist(SampleArgs a) {
    __shared__ u64 mass[SM_BINS];
    __shared__ unsigned count[SM_BINS];
    __shared__ u64 sh[SM_THREADS / 64];
    __shared__ int shi[2];
    __shared__ Bins shared_bins;
    __shared__ Options options;
    const int r = blockIdx.x, sp = blockIdx.y;
    const float temp = a.temp[r];
    if (!(temp > 0.f)) {
        if (PICK && sp == 0) pick_greedy(a, r, a.logits + (size_t)r * a.ld, (float*)sh, (int*)(sh + SM_THREADS / 128));
        return;
    }
    const bool counts = a.top_k && a.top_k[r] > 0 && a.top_k[r] < a.V;
    const int chunk = ((a.V + a.hist_splits - 1) / a.hist_splits + 3) & ~3;
    const int lo = sp * chunk < a.V ? sp * chunk : a.V, hi = lo + chunk < a.V ? lo + chunk : a.V;
    float* row = a.logits + (size_t)r * a.ld;
    Bins bins;
    auto prepare = [&] {
        for (int i = threadIdx.x; i < SM_BINS; i += SM_THREADS) { mass[i] = 0; count[i] = 0; }
        if (threadIdx.x < 64) {             // (by every wave, the divisions alone take a compute unit's 32 waves 1 us)
            float mx, mn;
            row_extent(a.part, r, mx, mn);
            const Bins b = make_bins(mx, mn, temp);
            if (threadIdx.x == 0) { shared_bins = b; options.load(a, r); }
        }
        __syncthreads();
        bins = shared_bins;
    };
    // (an unusual row is left for the plain division; its loads are then for nothing)
    bool unusual = false;
    fill_hist<0, false>(row, lo, hi, temp, bins, counts, mass, count, [&] { prepare(); unusual = !bins.ordinary; }, unusual);
    if (unusual && fabsf(bins.zmax) < INFINITY) fill_hist<0, true>(row, lo, hi, temp, bins, counts, mass, count, [] {}, false);
    if (!(fabsf(bins.zmax) < INFINITY)) {           // (no histogram of such a row is read)
        if (sp == 0 && threadIdx.x == 0) {
            if (PICK) a.out[r] = 0;
            else a.notes[r].n_cuts = -1;
        }
        return;
    }
    __syncthreads();
    const size_t at = ((size_t)r * a.hist_splits + sp) * SM_BINS;
    for (int i = threadIdx.x; i < SM_BINS; i += SM_THREADS) {
        store_agent(a.hist_mass + at + i, mass[i]);
        if (counts) store_agent(a.hist_count + at + i, count[i]);
    }
    if (!last_to_arrive(&a.notes[r].arrived[0], a.hist_splits, shi)) return;

    const int b0 = 2 * threadIdx.x;
    u64 m0 = 0, m1 = 0;
    unsigned c0 = 0, c1 = 0;
    for (int s0 = 0; s0 < a.hist_splits; s0 += 4) {      // (four shares' loads side by side)
        u64 m[4][2];
        unsigned c[4][2];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const size_t from = ((size_t)r * a.hist_splits + (s0 + u < a.hist_splits ? s0 + u : s0)) * SM_BINS + b0;
            m[u][0] = load_agent(a.hist_mass + from);
            m[u][1] = load_agent(a.hist_mass + from + 1);
            c[u][0] = counts ? load_agent(a.hist_count + from) : 0;
            c[u][1] = counts ? load_agent(a.hist_count + from + 1) : 0;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (s0 + u < a.hist_splits) { m0 += m[u][0]; m1 += m[u][1]; c0 += c[u][0]; c1 += c[u][1]; }
    }
    scan_pairs(m0, m1, sh);
    if (counts) scan_pairs(c0, c1, (unsigned*)sh);
    mass[b0] = m0; mass[b0 + 1] = m1;
    count[b0] = c0; count[b0 + 1] = c1;
    if constexpr (PICK) {
        __shared__ List list;
        __shared__ u64 sh2[2];
        __syncthreads();
        int pick = sample_by_bins<4, SM_THREADS>(a, options, row, temp, bins, Found{nullptr, -1, nullptr}, mass, count, list, sh);
        if (pick < 0) pick = sample_by_radix<4, SM_THREADS>(a, r, row, temp, bins.zmax, mass, sh, sh2);
        if (threadIdx.x == 0) a.out[r] = pick;
        return;
    }
    const size_t to = (size_t)r * SM_BINS + b0;
    *reinterpret_cast<ulonglong2*>(a.mass + to) = make_ulonglong2(m0, m1);
    if (counts) *reinterpret_cast<uint2*>(a.count + to) = make_uint2(c0, c1);
    __syncthreads();
    if (threadIdx.x < 64) plan_cuts(a, r, options, bins, mass, count);
}

// One workgroup a row: greedy rows, and sampled rows of short vocabularies and of callers that bring no work area.  (Five waves a SIMD: with the registers of four, a
// unit's second workgroup began a whole one later, 300 greedy rows of 1,000 logits 7.2 us for 6.1; room for eight spills, 64 sampled rows 15.5 us for 12.9.)
__global__ __launch_bounds__(SM_THREADS, 5) void k_sample(SampleArgs a) {
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
    if (!(temp > 0.f)) { pick_greedy(a, r, row, shf, shi); return; }

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
    mass[b0] = mass[b0 + 1] = 0;
    count[b0] = count[b0 + 1] = 0;
    __syncthreads();
    if (bins.ordinary) fill_hist<0, false>(row, 0, V, temp, bins, counts, mass, count, [] {}, false);
    else fill_hist<0, true>(row, 0, V, temp, bins, counts, mass, count, [] {}, false);
    __syncthreads();
    u64 m0 = mass[b0], m1 = mass[b0 + 1];
    unsigned c0 = count[b0], c1 = count[b0 + 1];
    scan_pairs(m0, m1, sh);
    scan_pairs(c0, c1, (unsigned*)sh);
    mass[b0] = m0; mass[b0 + 1] = m1;
    count[b0] = c0; count[b0 + 1] = c1;
    __syncthreads();
    Options options;
    options.load(a, r);
    int pick = sample_by_bins<8, SM_THREADS>(a, options, row, temp, bins, Found{nullptr, -1, nullptr}, mass, count, list, sh);
    if (pick < 0) pick = sample_by_radix<8, SM_THREADS>(a, r, row, temp, bins.zmax, mass, sh, sh2);
    if (threadIdx.x == 0) a.out[r] = pick;
}

// The rest of a long vocabulary's rows (grid: rows x shares of a row): every workgroup leaves the candidates of its share that lie in the
// planned runs of bins, and the row's last one picks among them.
__global__ __launch_bounds__(SM_THREADS, 8) void k_pick_rows(SampleArgs a) {
    __shared__ u64 mass[SM_BINS];
    __shared__ unsigned count[SM_BINS];
    __shared__ List list;
    __shared__ u64 found[SM_FOUND];
    __shared__ u64 sh[SM_THREADS / 64];
    __shared__ u64 sh2[2];
    __shared__ float shf[SM_THREADS / 64];
    __shared__ int shi[SM_THREADS / 64];
    __shared__ int n_mine, at_mine;
    __shared__ RowNotes notes;
    __shared__ Options options;
    const int r = blockIdx.x, sp = blockIdx.y;
    float* row = a.logits + (size_t)r * a.ld;
    const float temp = a.temp[r];
    if (!(temp > 0.f)) {
        if (sp == 0) pick_greedy(a, r, row, shf, shi);
        return;
    }
    const RowNotes& told = a.notes[r];
    int n_cuts;
    Bins bins;
    float vlo[SM_CUTS], vhi[SM_CUTS];
    const int shares = gridDim.y;
    const int chunk = ((a.V + shares - 1) / shares + 3) & ~3;
    const int lo = sp * chunk < a.V ? sp * chunk : a.V, hi = lo + chunk < a.V ? lo + chunk : a.V;
    for_row_after<0>(row, lo, hi, threadIdx.x, SM_THREADS, [&] {
        n_cuts = told.n_cuts;
        bins.zmax = told.zmax; bins.scale = told.scale; bins.capped = told.capped; bins.ordinary = false;
#pragma unroll
        for (int c = 0; c < SM_CUTS; ++c) {
            vlo[c] = c < n_cuts ? told.vlo[c] : INFINITY;
            vhi[c] = c < n_cuts ? told.vhi[c] : -INFINITY;
        }
        if (threadIdx.x == 0) {
            n_mine = 0;
            notes = told;
            options.load(a, r);
        }
        __syncthreads();
    }, [&](float v, int i) __attribute__((always_inline)) {
        bool near = false;
#pragma unroll
        for (int c = 0; c < SM_CUTS; ++c) near |= (v >= vlo[c]) & (v <= vhi[c]);
        if (!near) return;
        const float z = v / temp;
        if (!(z > -INFINITY)) return;
        const int b = bins.of(z);
        bool in = false;
        for (int c = 0; c < n_cuts; ++c) in = in || (b >= notes.lo[c] && b <= notes.hi[c]);
        if (!in) return;
        const int at = atomicAdd(&n_mine, 1);
        if (at < SM_FOUND) found[at] = order_key(z, i);
    });
    if (n_cuts < 0) {                               // nothing has any mass
        if (sp == 0 && threadIdx.x == 0) a.out[r] = 0;
        return;
    }
    __syncthreads();
    const int n = n_mine < SM_FOUND ? n_mine : SM_FOUND;
    // (a count over the list's room tells that candidates are missing)
    if (threadIdx.x == 0 && n_mine > 0) at_mine = __hip_atomic_fetch_add(&a.notes[r].n_found, n_mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (n > 0)
        for (int i = threadIdx.x; i < n; i += SM_THREADS)
            if (at_mine + i < SM_FOUND) store_agent(a.found + (size_t)r * SM_FOUND + at_mine + i, found[i]);
    if (!last_to_arrive(&a.notes[r].arrived[1], shares, shi)) return;

    const bool counts = options.top_k > 0 && options.top_k < a.V;
    const int n_all = load_agent(&a.notes[r].n_found);
    const int b0 = 2 * threadIdx.x;
    const size_t from = (size_t)r * SM_BINS + b0;
    const ulonglong2 m = *reinterpret_cast<const ulonglong2*>(a.mass + from);
    const uint2 c = counts ? *reinterpret_cast<const uint2*>(a.count + from) : make_uint2(0, 0);
    for (int i = threadIdx.x; i < n_all && i < SM_FOUND; i += SM_THREADS) found[i] = load_agent(a.found + (size_t)r * SM_FOUND + i);
    mass[b0] = m.x; mass[b0 + 1] = m.y;
    count[b0] = c.x; count[b0 + 1] = c.y;
    __syncthreads();
    const Found all = Found{found, n_all <= SM_FOUND ? n_all : -1, &notes};
    // (for a few hundred candidates 16 waves that meet at every step take longer than four: one row 6.5 us, 5.4 so.  A barrier does not wait for a wave that has ended.)
    int pick;
    if (all.n >= 0 && all.n <= 2 * SM_FEW) {
        if (threadIdx.x >= SM_FEW) return;
        pick = sample_by_bins<2, SM_FEW>(a, options, row, temp, bins, all, mass, count, list, sh);
        if (pick < 0) pick = sample_by_radix<2, SM_FEW>(a, r, row, temp, bins.zmax, mass, sh, sh2);
    } else {
        pick = sample_by_bins<2, SM_THREADS>(a, options, row, temp, bins, all, mass, count, list, sh);
        if (pick < 0) pick = sample_by_radix<2, SM_THREADS>(a, r, row, temp, bins.zmax, mass, sh, sh2);
    }
    if (threadIdx.x == 0) a.out[r] = pick;
}

static int sample_launch(int* out, float* logits, int W, int V, int ld, const float* temp, const int* top_k,
                         const float* top_p, const float* min_p, const float* repeat_penalty,
                         const float* draw, const int* recent, const int* n_recent, int recent_cap,
                         const int* exempt, int n_exempt, float* part_ws, void* hist_ws, int hist_splits, int row_splits, hipStream_t stream) {
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
    a.hist_mass = nullptr; a.hist_count = nullptr; a.mass = nullptr; a.count = nullptr; a.found = nullptr; a.notes = nullptr; a.hist_splits = hist_splits;
    if (part_ws && hist_ws) {
        // per row: masses of every share, their sums, candidates, notes, then the numbers of every share and their sums
        const size_t bins = (size_t)W * SM_BINS;
        a.hist_mass = (u64*)hist_ws;
        a.mass = a.hist_mass + bins * hist_splits;
        a.found = a.mass + bins;
        a.notes = (RowNotes*)(a.found + (size_t)W * SM_FOUND);
        a.hist_count = (unsigned*)(a.notes + W);
        a.count = a.hist_count + bins * hist_splits;
    }
    if (part_ws) {          // [W, ROW_SPLITS, 2] floats
        k_pick_extent<<<dim3(W, ROW_SPLITS), 256, 0, stream>>>(a, part_ws);
        XR_CHECK_LAUNCH("sample_extent");
    }
    if (a.notes) {
        if (row_splits == 0) k_pick_hist<true><<<dim3(W, hist_splits), SM_THREADS, 0, stream>>>(a);
        else k_pick_hist<false><<<dim3(W, hist_splits), SM_THREADS, 0, stream>>>(a);
        XR_CHECK_LAUNCH("sample_hist");
        if (row_splits == 0) return XR_OK;
        k_pick_rows<<<dim3(W, row_splits), SM_THREADS, 0, stream>>>(a);
        XR_CHECK_LAUNCH("sample_rows");
        return XR_OK;
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
                         recent_cap, exempt, n_exempt, greedy_ws, nullptr, 0, 0, stream);
}

// The same with a work area for the sampled rows: their histograms are shared out to `splits` workgroups a row, their candidates to
// `row_splits` (0: none, the histogram's last workgroup picks).  Its bytes a row:
static long long sample_work_bytes(int splits) { return (long long)(splits + 1) * SM_BINS * 12 + SM_FOUND * 8 + (long long)sizeof(RowNotes); }

extern "C" int xr_sample_split(int* out, float* logits, int W, int V, int ld, const float* temp, const int* top_k,
                               const float* top_p, const float* min_p, const float* repeat_penalty,
                               const float* draw, const int* recent, const int* n_recent, int recent_cap,
                               const int* exempt, int n_exempt, float* greedy_ws, void* hist_ws, long long hist_bytes,
                               int splits, int row_splits, hipStream_t stream) {
    XR_REQUIRE(greedy_ws && hist_ws && splits > 0 && splits <= 32 && row_splits >= 0 && row_splits <= 64, "sample_split: no work area or %d and %d splits", splits, row_splits);
    XR_REQUIRE(((uintptr_t)hist_ws & 15) == 0 && hist_bytes >= W * sample_work_bytes(splits), "sample_split: a work area of %lld bytes for %d rows in %d parts",
               hist_bytes, W, splits);
    return sample_launch(out, logits, W, V, ld, temp, top_k, top_p, min_p, repeat_penalty, draw, recent, n_recent,
                         recent_cap, exempt, n_exempt, greedy_ws, hist_ws, splits, row_splits, stream);
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
                         recent_cap, exempt, n_exempt, ws, nullptr, 0, 0, stream);
}
