// Attention over the paged cache with 32-bit arithmetic only: the attention of the
// true 32-bit path, for prompt portions and decoded tokens alike, any head size up
// to 256.  k_attention_ref: one wave per (token, query head), any type.  k_attention_f32: 32-bit operands on the
// matrix cores, a workgroup per 32 rows of a request and key/value head (below); same options, same result up to rounding.
//
// For the token at position p of its request and query head h (key/value head
// h / (H/Hk), contiguous groups): s_t = (q . K_t) * scale for t in [lo, p], causal by
// the loop bound, lo = max(0, p - window + 1) for a windowed layer
// (src/model.c:3553-3573, :6326); softmax with the maximum taken out
// (src/model.c:3409-3415); out = sum_t p_t V_t (:3576-3587).  The
// softmax runs over blocks of 64 keys with a running maximum and sum, which gives the
// same value up to rounding.  With `slopes` (one number a query head) a bias that grows with the distance is
// taken off every score: s_t = (q . K_t) * scale - slope_h * (p - t).
// Other masks: `chunk` > 0: lo = p - p mod chunk (a position reads its own chunk of positions, counted from 0);
// `keep` > 0: the keys [0, keep) are read as well wherever lo lies.  `sinks` (one number a query head): the
// softmax's denominator also holds exp(sink_h) (of the sink as it is: no scale, no cap), an entry that has no key and no value.  Values may have another
// size than keys (Dv; cache layout K [page][kv_head][slot][D], V [page][kv_head][Dv][slot]).
// With `cap` > 0 a scaled score s counts as cap * tanh(s / cap), before a slope's bias.  A head's output is multiplied by
// `out_scale` and, with `gate` (a number a token and head), by sigmoid(gate); output rows are ld_out apart.
#include "common.h"

#define AR_MAX_D 256

template <typename T>
__global__ __launch_bounds__(64) void k_attention_ref(
    T* __restrict__ out, const T* __restrict__ q, const T* __restrict__ kc, const T* __restrict__ vc,
    const int* __restrict__ positions, const int* __restrict__ req_of_token,
    const int* __restrict__ block_table, int table_stride, int H, int Hk, int D, int Dv, int page_shift,
    int page_mask, int page_size, float scale, int window, int chunk, int keep, const float* __restrict__ slopes,
    const float* __restrict__ sinks, float cap, const float* __restrict__ gate, int ld_gate, float out_scale, int ld_out) {
    __shared__ float qs[AR_MAX_D];
    const int t = blockIdx.x, h = blockIdx.y, lane = threadIdx.x;
    const int pos = positions[t];
    const int req = req_of_token[t];
    const int kvh = h / (H / Hk);
    const int lo = chunk > 0 ? pos - pos % chunk : (window > 0 && pos - window + 1 > 0) ? pos - window + 1 : 0;
    const int kept = keep < lo ? keep : lo;         // kept keys [0, kept) lie below the row's own range
    const T* qrow = q + ((size_t)t * H + h) * D;
    for (int d = lane; d < D; d += 64) qs[d] = ld<T>(qrow, d);
    __syncthreads();
    const int* bt = block_table + (size_t)req * table_stride;
    const float slope = slopes ? slopes[h] : 0.f;

    float m = -INFINITY, l = 0.f;
    float acc[AR_MAX_D / 64];
#pragma unroll
    for (int dd = 0; dd < AR_MAX_D / 64; ++dd) acc[dd] = 0.f;

    for (int seg = kept > 0 ? 0 : 1; seg < 2; ++seg)
    for (int k0 = seg ? lo : 0, last = seg ? pos : kept - 1; k0 <= last; k0 += 64) {
        const int key = k0 + lane;
        const bool valid = key <= last;
        float s = -INFINITY;
        if (valid) {
            const int page = bt[key >> page_shift];
            const int off = key & page_mask;
            const T* kr = kc + (((size_t)page * Hk + kvh) * page_size + off) * D;
            float dot = 0.f;
            for (int d = 0; d < D; ++d) dot = fmaf(qs[d], ld<T>(kr, d), dot);
            s = dot * scale;
            if (cap > 0.f) s = cap * tanhf(s / cap);
            s -= slope * (float)(pos - key);
        }
        const float mn = fmaxf(m, wave_max(s));
        const float p = valid ? expf(s - mn) : 0.f;
        const float corr = m == -INFINITY ? 0.f : expf(m - mn);
        l = l * corr + wave_sum(p);
#pragma unroll
        for (int dd = 0; dd < AR_MAX_D / 64; ++dd) acc[dd] *= corr;
        const int nk = (last - k0 + 1) < 64 ? (last - k0 + 1) : 64;
        for (int j = 0; j < nk; ++j) {
            const float pj = __shfl(p, j, 64);
            const int kj = k0 + j;
            const int page = bt[kj >> page_shift];
            const int off = kj & page_mask;
            const T* vb = vc + ((size_t)page * Hk + kvh) * Dv * page_size + off;
#pragma unroll
            for (int dd = 0; dd < AR_MAX_D / 64; ++dd) {
                const int d = lane + 64 * dd;
                if (d < Dv) acc[dd] = fmaf(pj, ld<T>(vb, (size_t)d * page_size), acc[dd]);
            }
        }
        m = mn;
    }
    if (sinks) {            // one more entry of the denominator, with nothing to add to the output
        const float sk = sinks[h];
        const float mn = fmaxf(m, sk);
        const float corr = expf(m - mn);
        l = l * corr + expf(sk - mn);
#pragma unroll
        for (int dd = 0; dd < AR_MAX_D / 64; ++dd) acc[dd] *= corr;
    }
    T* orow = out + (size_t)t * ld_out + (size_t)h * Dv;
    const float f = gate ? out_scale / (1.0f + expf(-gate[(size_t)t * ld_gate + h])) : out_scale;
#pragma unroll
    for (int dd = 0; dd < AR_MAX_D / 64; ++dd) {
        const int d = lane + 64 * dd;
        if (d < Dv) st<T>(orow, d, acc[dd] / l * f);
    }
}

// The same for 32-bit operands with the two products on the matrix cores (v_mfma_f32_16x16x4_f32: 32-bit operands, products
// and sums).  A workgroup of four waves takes 32 rows (token x head of the group, token major) of one request and key/value
// head and walks the keys they see in tiles of 64: keys and values through LDS, wave w the scores of keys 16 w .. 16 w + 15,
// the softmax eight lanes a row, then wave w every fourth 16 channels of the output.  An MFMA step takes one
// column from each quarter of the wave; a lane reads the four columns of its quarter at once and feeds four steps.
// Keys that no row of the workgroup sees are never read (their pages may be gone) and count as zeros.  A tile whose values are not
// all finite is added key by key, so that such a value shows in the rows that see it and in no other.
// One wave a (token, head) walked the keys lane by lane, every lane a row of its own: 401 tokens, 32 heads of 64 took
// 900 us and with this kernel 90, a decoded token of a tiny model 12 and 7.  Bound by the chain of a tile's steps in the workgroups that see
// most keys: with a softmax row a wave at a time (eight rows one after another, each with twelve exchanges) and every tile's keys read
// when the tile before was done, 90 us; all rows' softmax at once and the next tile fetched meanwhile 60; its pieces' places by a product
// instead of divisions, and the row blocks that see most keys first 55; the pages looked up a step ahead 48.  Lone tokens with a wave a row (eight lanes
// a row had made heads of 16 and 32 slower than before all this) and heads of up to 32 with two pieces a thread, 650 keys: heads of 16 30.2 us, 33.4 and 24.5, of 32 38.9, 43.1
// and 30.7, of 64 (584 keys) 50.5, 45.3 and 36.8.
#define AF_ROWS 32
#define AF_KEYS 64
#define AF_MAX_D 128
#define AF_LD_S (AF_KEYS + 4)
typedef float f32x4 __attribute__((ext_vector_type(4)));

struct AttnF32 {
    float* out;
    const float* q;
    const float* kc;
    const float* vc;
    const int* positions;
    const int* cu_q;
    const int* block_table;
    const float* slopes;
    const float* sinks;
    const float* gate;
    int table_stride, H, Hk, D, Dv, page_shift, page_mask, page_size, window, chunk, keep, ld_gate, ld_out;
    float scale, cap, out_scale;
};

static inline int af_ld(int d) { return ((d + 15) & ~15) + 4; }
static inline size_t af_lds_bytes(int D, int Dv) {
    return sizeof(float) * ((size_t)(AF_ROWS + AF_KEYS) * af_ld(D) + (size_t)((Dv + 15) & ~15) * AF_LD_S + AF_ROWS * AF_LD_S);
}

// PIECES: 16-byte pieces of a tile's keys, and of its values, a thread: heads of up to 16 PIECES channels, or (FULL) keys of so many exactly.
template <int PIECES, bool FULL>
__global__ __launch_bounds__(256) void k_attention_f32(AttnF32 a) {
    constexpr int CS = (PIECES + 3) / 4;                // 16 channels of the output a wave
    extern __shared__ __align__(16) float lds[];
    __shared__ int row_pos[AF_ROWS], row_lo[AF_ROWS];
    __shared__ float row_corr[AF_ROWS], row_l[AF_ROWS], row_m[AF_ROWS];
    __shared__ int odd_tile;                            // the last tile of keys with a value that is not finite
    const int b = blockIdx.z, kvh = blockIdx.y, G = a.H / a.Hk;
    const int t0 = a.cu_q[b], nq = a.cu_q[b + 1] - t0;
    const int r0 = (int)(gridDim.x - 1 - blockIdx.x) * AF_ROWS;     // of the request's nq * G rows; the last ones, which see most keys, first
    const int n_rows = nq * G - r0 < AF_ROWS ? nq * G - r0 : AF_ROWS;
    if (n_rows <= 0) return;
    const int D16 = (a.D + 15) & ~15, Dv16 = (a.Dv + 15) & ~15, ldd = D16 + 4;
    float* Q = lds;
    float* Kt = Q + AF_ROWS * ldd;
    float* Vt = Kt + AF_KEYS * ldd;
    float* S = Vt + Dv16 * AF_LD_S;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int* bt = a.block_table + (size_t)b * a.table_stride;

    if (tid < AF_ROWS) {
        const int r = tid < n_rows ? tid : n_rows - 1;  // (rows past the end repeat the last; nothing of them is written)
        const int pos = a.positions[t0 + (r0 + r) / G];
        row_pos[tid] = pos;
        row_lo[tid] = a.chunk > 0 ? pos - pos % a.chunk : (a.window > 0 && pos - a.window + 1 > 0) ? pos - a.window + 1 : 0;
        row_m[tid] = -INFINITY;
        row_l[tid] = 0.f;
        if (tid == 0) odd_tile = -1;
    }
    for (int i = tid; i < AF_ROWS * D16 / 4; i += 256) {
        const int r = i / (D16 / 4), d = (i - r * (D16 / 4)) * 4;
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (r < n_rows && d < a.D)
            v = *reinterpret_cast<const float4*>(a.q + ((size_t)(t0 + (r0 + r) / G) * a.H + kvh * G + (r0 + r) % G) * a.D + d);
        *reinterpret_cast<float4*>(Q + r * ldd + d) = v;
    }
    __syncthreads();
    // positions rise with the rows, and so do the first keys
    const int lo_min = row_lo[0], lo_max = row_lo[AF_ROWS - 1], hi = row_pos[AF_ROWS - 1] + 1;
    const int kept_max = a.keep < lo_max ? a.keep : lo_max;     // first keys that stay readable behind the window
    f32x4 acc[2][CS];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int c = 0; c < CS; ++c) acc[i][c] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int l16 = lane & 15, quad = lane >> 4;
    const int tiles = n_rows > 16 ? 2 : 1;

    // A tile's pieces are fetched into registers while the tile before is worked on, and its keys' pages are looked up before that: a piece's
    // place is two reads, one behind the other.
    // (i / (D16 / 4) for i up to 2,047 and D16 / 4 up to 32, as a product: the remainder's share of 2^16 stays below one)
    const int ck = D16 / 4;
    const uint32_t inv_ck = (65536u + (uint32_t)ck - 1u) / (uint32_t)ck;
    float4 pk[PIECES], pv[PIECES];
    int page_k[PIECES], page_v[PIECES];                     // -1: nothing is read
    auto pages = [&](int seg, int k0) {
        const int from = seg ? lo_min : 0, to = seg ? hi : kept_max;
#pragma unroll
        for (int u = 0; u < PIECES; ++u) {
            const int i = u * 256 + tid, j = (int)(((uint32_t)i * inv_ck) >> 16), jv = i % (AF_KEYS / 4) * 4;
            const bool k_in = i < AF_KEYS * ck && (i - j * ck) * 4 < a.D && k0 + j >= from && k0 + j < to;
            const bool v_in = i / (AF_KEYS / 4) < a.Dv && k0 + jv + 3 >= from && k0 + jv < to;
            page_k[u] = k_in ? bt[(k0 + j) >> a.page_shift] : -1;
            page_v[u] = v_in ? bt[(k0 + jv) >> a.page_shift] : -1;      // (four keys of a channel lie in one page, side by side)
        }
    };
    auto fetch = [&](int k0) {
#pragma unroll
        for (int u = 0; u < PIECES; ++u) {
            const int i = u * 256 + tid, j = (int)(((uint32_t)i * inv_ck) >> 16), jv = i % (AF_KEYS / 4) * 4;
            pk[u] = pv[u] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (page_k[u] >= 0)
                pk[u] = *reinterpret_cast<const float4*>(a.kc + (((size_t)page_k[u] * a.Hk + kvh) * a.page_size + ((k0 + j) & a.page_mask)) * a.D + (i - j * ck) * 4);
            if (page_v[u] >= 0)
                pv[u] = *reinterpret_cast<const float4*>(a.vc + (((size_t)page_v[u] * a.Hk + kvh) * a.Dv + i / (AF_KEYS / 4)) * a.page_size + ((k0 + jv) & a.page_mask));
        }
    };
    int seg = kept_max > 0 ? 0 : 1, k0 = (seg ? lo_min : 0) & ~(AF_KEYS - 1);
    pages(seg, k0);
    fetch(k0);
    for (;;) {
        const int from = seg ? lo_min : 0, to = seg ? hi : kept_max;
        int seg_next = seg, k0_next = k0 + AF_KEYS;
        if (k0_next >= to && seg == 0) { seg_next = 1; k0_next = lo_min & ~(AF_KEYS - 1); }
        const bool more = k0_next < (seg_next ? hi : kept_max);
        if (more) pages(seg_next, k0_next);
        {
            __syncthreads();                            // the tile before has been read
#pragma unroll
            for (int u = 0; u < PIECES; ++u) {
                const int i = u * 256 + tid;
                if (i < AF_KEYS * D16 / 4) {
                    const int j = (int)(((uint32_t)i * inv_ck) >> 16), d = (i - j * ck) * 4;
                    *reinterpret_cast<float4*>(Kt + j * ldd + d) = pk[u];
                }
                if (i < Dv16 * (AF_KEYS / 4)) {
                    const int d = i / (AF_KEYS / 4), j = (i - d * (AF_KEYS / 4)) * 4, key = k0 + j;
                    float4 v = pv[u];
                    if (key < from || key >= to) v.x = 0.f;
                    if (key + 1 < from || key + 1 >= to) v.y = 0.f;
                    if (key + 2 < from || key + 2 >= to) v.z = 0.f;
                    if (key + 3 < from || key + 3 >= to) v.w = 0.f;
                    const float n = 0.f * v.x + 0.f * v.y + 0.f * v.z + 0.f * v.w;      // (0, or no number where one of them is not finite)
                    if (n != n) odd_tile = 2 * k0 + seg;
                    *reinterpret_cast<float4*>(Vt + d * AF_LD_S + j) = v;
                }
            }
            __syncthreads();
            if (more) fetch(k0_next);
            {   // scores: a lane has key 16 wave + lane % 16 and rows 4 (lane / 16) + e of each 16
                f32x4 s[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
                const float* kp = Kt + (16 * wave + l16) * ldd + 4 * quad;
                const float* qp = Q + l16 * ldd + 4 * quad;
                auto step = [&](int d) {                // (the two sums in turn: a product waits for the one before it in its own sum)
                    const float4 fk = *reinterpret_cast<const float4*>(kp + d);
                    const float4 f0 = *reinterpret_cast<const float4*>(qp + d);
                    const float4 f1 = *reinterpret_cast<const float4*>(qp + 16 * ldd + d);
#pragma unroll
                    for (int x = 0; x < 4; ++x) {
                        s[0] = __builtin_amdgcn_mfma_f32_16x16x4f32((&f0.x)[x], (&fk.x)[x], s[0], 0, 0, 0);
                        s[1] = __builtin_amdgcn_mfma_f32_16x16x4f32((&f1.x)[x], (&fk.x)[x], s[1], 0, 0, 0);
                    }
                };
                if (tiles == 1) {
                    for (int d = 0; d < D16; d += 16) {
                        const float4 fk = *reinterpret_cast<const float4*>(kp + d);
                        const float4 f0 = *reinterpret_cast<const float4*>(qp + d);
#pragma unroll
                        for (int x = 0; x < 4; ++x) s[0] = __builtin_amdgcn_mfma_f32_16x16x4f32((&f0.x)[x], (&fk.x)[x], s[0], 0, 0, 0);
                    }
                } else if constexpr (FULL) {
#pragma unroll
                    for (int d = 0; d < 16 * PIECES; d += 16) step(d);
                } else {
                    for (int d = 0; d < D16; d += 16) step(d);
                }
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int e = 0; e < 4; ++e) S[(16 * i + 4 * quad + e) * AF_LD_S + 16 * wave + l16] = s[i][e];
            }
            __syncthreads();
            // softmax: eight lanes a row, all rows at a time; a lane has keys 4 j .. 4 j + 3 of either half of the tile.  Up to four rows a wave each, a key a lane:
            // one exponential behind the other is what eight keys a lane wait for.  Either way a row's exponentials are added up in one order.
            // (What rows that do not exist have in S is their own results' alone, which are not stored.)
            if (n_rows <= 4) {
                const int r = wave, key = k0 + lane;
                if (r < n_rows) {
                    const int pos = row_pos[r], lo = row_lo[r];
                    const bool valid = key >= from && key < to && (seg ? key >= lo && key <= pos : key < a.keep && key < lo);
                    float y = S[r * AF_LD_S + lane] * a.scale;
                    if (a.cap > 0.f) y = a.cap * tanhf(y / a.cap);
                    if (a.slopes) y -= a.slopes[kvh * G + (r0 + r) % G] * (float)(pos - key);
                    y = valid ? y : -INFINITY;
                    const float m = row_m[r], mn = fmaxf(m, wave_max(y));
                    const float p = valid ? expf(y - mn) : 0.f;
                    S[r * AF_LD_S + lane] = p;
                    float sum = p;
#pragma unroll
                    for (int o : {1, 2, 32, 16, 8, 4}) sum += __shfl_xor(sum, o, 64);
                    if (lane == 0) {
                        const float corr = m == -INFINITY ? 0.f : expf(m - mn);
                        row_corr[r] = corr;
                        row_l[r] = row_l[r] * corr + sum;
                        row_m[r] = mn;
                    }
                }
            } else {
                const int r = tid >> 3, j = tid & 7;
                float* const row = S + r * AF_LD_S + 4 * j;
                if (r < n_rows) {
                    const int pos = row_pos[r], lo = row_lo[r];
                    const float slope = a.slopes ? a.slopes[kvh * G + (r0 + r) % G] : 0.f;
                    float v[8];
                    bool valid[8];
#pragma unroll
                    for (int x = 0; x < 8; ++x) {
                        const int key = k0 + 4 * j + (x & 3) + (x >> 2) * (AF_KEYS / 2);
                        valid[x] = key >= from && key < to && (seg ? key >= lo && key <= pos : key < a.keep && key < lo);
                        float y = row[(x & 3) + (x >> 2) * (AF_KEYS / 2)] * a.scale;
                        if (a.cap > 0.f) y = a.cap * tanhf(y / a.cap);
                        if (a.slopes) y -= slope * (float)(pos - key);
                        v[x] = valid[x] ? y : -INFINITY;
                    }
                    const float m = row_m[r];
                    float mn = v[0];
#pragma unroll
                    for (int x = 1; x < 8; ++x) mn = fmaxf(mn, v[x]);
#pragma unroll
                    for (int o = 4; o > 0; o >>= 1) mn = fmaxf(mn, __shfl_xor(mn, o, 64));
                    mn = fmaxf(m, mn);
#pragma unroll
                    for (int x = 0; x < 8; ++x) v[x] = valid[x] ? expf(v[x] - mn) : 0.f;
                    float sum = ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
#pragma unroll
                    for (int o = 4; o > 0; o >>= 1) sum += __shfl_xor(sum, o, 64);
                    *reinterpret_cast<float4*>(row) = make_float4(v[0], v[1], v[2], v[3]);
                    *reinterpret_cast<float4*>(row + AF_KEYS / 2) = make_float4(v[4], v[5], v[6], v[7]);
                    if (j == 0) {
                        const float corr = m == -INFINITY ? 0.f : expf(m - mn);
                        row_corr[r] = corr;
                        row_l[r] = row_l[r] * corr + sum;
                        row_m[r] = mn;
                    }
                } else if (r < 16 * tiles) {
                    *reinterpret_cast<float4*>(row) = make_float4(0.f, 0.f, 0.f, 0.f);
                    *reinterpret_cast<float4*>(row + AF_KEYS / 2) = make_float4(0.f, 0.f, 0.f, 0.f);
                }
            }
            __syncthreads();
            float corr[2][4];
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) corr[i][e] = row_corr[16 * i + 4 * quad + e];
#pragma unroll
            for (int c = 0; c < CS; ++c) {
                const int d0 = 16 * (wave + 4 * c);
                if (d0 >= Dv16) continue;
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[i][c][e] *= corr[i][e];
                if (odd_tile == 2 * k0 + seg) {         // 0 times it is no 0: a row adds the keys that it sees, one by one
                    for (int i = 0; i < tiles; ++i)
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const int r = 16 * i + 4 * quad + e, lo = row_lo[r], last = seg ? row_pos[r] : min(a.keep, lo) - 1;
                            float sum = 0.f;
                            for (int j = 0; j < AF_KEYS; ++j)
                                if (k0 + j >= (seg ? lo : 0) && k0 + j <= last) sum = fmaf(S[r * AF_LD_S + j], Vt[(d0 + l16) * AF_LD_S + j], sum);
                            if (i) acc[1][c][e] += sum; else acc[0][c][e] += sum;
                        }
                    continue;
                }
                const float* vp = Vt + (d0 + l16) * AF_LD_S + 4 * quad;
                const float* pp = S + l16 * AF_LD_S + 4 * quad;
                if (tiles == 1) {
#pragma unroll
                    for (int k = 0; k < AF_KEYS; k += 16) {
                        const float4 fv = *reinterpret_cast<const float4*>(vp + k);
                        const float4 f0 = *reinterpret_cast<const float4*>(pp + k);
#pragma unroll
                        for (int x = 0; x < 4; ++x) acc[0][c] = __builtin_amdgcn_mfma_f32_16x16x4f32((&f0.x)[x], (&fv.x)[x], acc[0][c], 0, 0, 0);
                    }
                } else {
#pragma unroll
                    for (int k = 0; k < AF_KEYS; k += 16) {
                        const float4 fv = *reinterpret_cast<const float4*>(vp + k);
                        const float4 f0 = *reinterpret_cast<const float4*>(pp + k);
                        const float4 f1 = *reinterpret_cast<const float4*>(pp + 16 * AF_LD_S + k);
#pragma unroll
                        for (int x = 0; x < 4; ++x) {
                            acc[0][c] = __builtin_amdgcn_mfma_f32_16x16x4f32((&f0.x)[x], (&fv.x)[x], acc[0][c], 0, 0, 0);
                            acc[1][c] = __builtin_amdgcn_mfma_f32_16x16x4f32((&f1.x)[x], (&fv.x)[x], acc[1][c], 0, 0, 0);
                        }
                    }
                }
            }
        }
        if (!more) break;
        seg = seg_next;
        k0 = k0_next;
    }
    __syncthreads();
    // a lane has channel lane % 16 of its 16 and rows 4 (lane / 16) + e
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int r = 16 * i + 4 * quad + e;
            if (r >= n_rows) continue;
            const int t = t0 + (r0 + r) / G, h = kvh * G + (r0 + r) % G;
            float l = row_l[r], corr = 1.f;
            if (a.sinks) {                              // one more entry of the denominator, with nothing to add to the output
                const float sk = a.sinks[h], mn = fmaxf(row_m[r], sk);
                corr = expf(row_m[r] - mn);
                l = l * corr + expf(sk - mn);
            }
            const float f = a.gate ? a.out_scale / (1.0f + expf(-a.gate[(size_t)t * a.ld_gate + h])) : a.out_scale;
#pragma unroll
            for (int c = 0; c < CS; ++c) {
                const int d = 16 * (wave + 4 * c) + l16;
                if (d < a.Dv) a.out[(size_t)t * a.ld_out + (size_t)h * a.Dv + d] = acc[i][c][e] * corr / l * f;
            }
        }
}

// 32-bit operands, `B` requests with up to `max_q` tokens in the step (rows [cu_q[b], cu_q[b + 1]) are request b's, at rising positions).
extern "C" int xr_attention_f32(float* out, const float* q, const float* k_cache, const float* v_cache, const int* positions,
                                const int* cu_q, const int* block_table, int table_stride, int B, int max_q, int H, int Hk, int D,
                                int Dv, int page_size, float scale, int window, int chunk, int keep, const float* slopes,
                                const float* sinks, float cap, const float* gate, int ld_gate, float out_scale, int ld_out,
                                hipStream_t stream) {
    XR_REQUIRE(ld_out >= H * Dv && (!gate || ld_gate >= H), "attention: output rows %d apart, gate rows %d apart for %d heads of %d", ld_out, ld_gate, H, Dv);
    XR_REQUIRE(cap >= 0.f, "attention: soft cap %g of the scores is negative", (double)cap);
    XR_REQUIRE(B >= 0 && max_q >= 0 && H > 0 && Hk > 0 && H % Hk == 0, "attention: bad sizes B=%d of up to %d tokens, %d heads over %d", B, max_q, H, Hk);
    XR_REQUIRE(D > 0 && D <= AF_MAX_D && D % 4 == 0 && Dv > 0 && Dv <= AF_MAX_D, "attention: head size %d (a multiple of 4) or value size %d exceeds %d", D, Dv, AF_MAX_D);
    XR_REQUIRE(((uintptr_t)q | (uintptr_t)k_cache | (uintptr_t)v_cache) % 16 == 0, "attention: operands are not 16-byte aligned");
    const int shift = ilog2_exact(page_size);
    XR_REQUIRE(shift >= 2, "attention: page size %d is no power of two of at least 4", page_size);
    XR_REQUIRE(window >= 0 && chunk >= 0 && keep >= 0, "attention: window %d, chunk %d or kept keys %d are negative", window, chunk, keep);
    XR_REQUIRE(B <= 65535 && Hk <= 65535, "attention: %d requests, %d key/value heads", B, Hk);
    if (B == 0 || max_q == 0) return XR_OK;
    AttnF32 a{out, q, k_cache, v_cache, positions, cu_q, block_table, slopes, sinks, gate, table_stride, H, Hk, D, Dv, shift,
              page_size - 1, page_size, window, chunk, keep, ld_gate, ld_out, scale, cap, out_scale};
    const size_t bytes = af_lds_bytes(D, Dv);
    dim3 grid((unsigned)(((long long)max_q * (H / Hk) + AF_ROWS - 1) / AF_ROWS), Hk, B);
    auto run = [&](auto kernel) {
        if (bytes > 65536) {
            // (the largest there is, whatever this call needs: smaller heads of another thread would take it back)
            const hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)af_lds_bytes(AF_MAX_D, AF_MAX_D));
            if (e != hipSuccess) (void)hipGetLastError();
            XR_REQUIRE(e == hipSuccess, "attention: %zu bytes of LDS: %s", bytes, hipGetErrorString(e));
        }
        kernel<<<grid, 256, bytes, stream>>>(a);
        XR_CHECK_LAUNCH("attention_f32");
        return XR_OK;
    };
    const int widest = D > Dv ? D : Dv;
    const int keys = (D + 15) / 16;
    if (widest <= 16) return run(k_attention_f32<1, true>);
    if (widest <= 32) return keys == 2 ? run(k_attention_f32<2, true>) : run(k_attention_f32<2, false>);
    if (widest <= 64) return keys == 4 ? run(k_attention_f32<4, true>) : run(k_attention_f32<4, false>);
    return keys == 8 ? run(k_attention_f32<8, true>) : run(k_attention_f32<8, false>);
}

extern "C" int xr_attention_ref(void* out, const void* q, const void* k_cache, const void* v_cache,
                                const int* positions, const int* req_of_token, const int* block_table,
                                int table_stride, int T, int H, int Hk, int D, int Dv, int page_size, float scale,
                                int window, int chunk, int keep, int dtype, const float* slopes, const float* sinks,
                                float cap, const float* gate, int ld_gate, float out_scale, int ld_out, hipStream_t stream) {
    XR_REQUIRE(ld_out >= H * Dv && (!gate || ld_gate >= H), "attention: output rows %d apart, gate rows %d apart for %d heads of %d", ld_out, ld_gate, H, Dv);
    XR_REQUIRE(cap >= 0.f, "attention: soft cap %g of the scores is negative", (double)cap);
    XR_REQUIRE(T >= 0 && H > 0 && Hk > 0 && D > 0, "attention: bad sizes T=%d H=%d Hk=%d D=%d", T, H, Hk, D);
    XR_REQUIRE(H % Hk == 0, "attention: %d query heads are not a multiple of %d key/value heads", H, Hk);
    XR_REQUIRE(D <= AR_MAX_D && Dv > 0 && Dv <= AR_MAX_D, "attention: head size %d or value size %d exceeds %d", D, Dv, AR_MAX_D);
    XR_REQUIRE(chunk >= 0 && keep >= 0, "attention: chunk %d or kept keys %d are negative", chunk, keep);
    int shift = ilog2_exact(page_size);
    XR_REQUIRE(shift >= 0, "attention: page size %d is not a power of two", page_size);
    XR_REQUIRE(window >= 0, "attention: window %d is negative", window);
    if (T == 0) return XR_OK;
    dim3 grid(T, H);
    if (dtype == XR_F32)
        k_attention_ref<float><<<grid, 64, 0, stream>>>((float*)out, (const float*)q, (const float*)k_cache,
                                                        (const float*)v_cache, positions, req_of_token, block_table,
                                                        table_stride, H, Hk, D, Dv, shift, page_size - 1, page_size, scale, window, chunk, keep, slopes, sinks, cap, gate, ld_gate, out_scale, ld_out);
    else if (dtype == XR_BF16)
        k_attention_ref<bf16_t><<<grid, 64, 0, stream>>>((bf16_t*)out, (const bf16_t*)q, (const bf16_t*)k_cache,
                                                         (const bf16_t*)v_cache, positions, req_of_token, block_table,
                                                         table_stride, H, Hk, D, Dv, shift, page_size - 1, page_size, scale, window, chunk, keep, slopes, sinks, cap, gate, ld_gate, out_scale, ld_out);
    else { xr_set_error("attention: bad dtype %d", dtype); return XR_BAD_ARG; }
    XR_CHECK_LAUNCH("attention_ref");
    return XR_OK;
}
