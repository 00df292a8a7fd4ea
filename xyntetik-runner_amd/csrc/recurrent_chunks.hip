// Retention and the gated delta rule over long portions, in chunks of 64 rows on the matrix cores with 32-bit operands,
// products and sums (v_mfma_f32_16x16x4_f32; q . k in 64 bits, v_mfma_f64_16x16x4_f64).  The recurrences and the state are those of recurrent_kernels.hip:
//
//   retention:   S <- g S + k v^T;                                  o = S^T q
//   delta rule:  S <- g S;  u = beta (v - S^T k);  S <- S + k u^T;  o = S^T q
//
// (The chunked form of the delta rule, with its triangular inverse: S. Yang, B. Wang, Y. Zhang, Y. Shen, Y. Kim, "Parallelizing Linear
// Transformers with the Delta Rule over Sequence Length", 2024; with decays: S. Yang, J. Kautz, A. Hatamizadeh, "Gated Delta Networks", 2024.)
// A chunk begins with the state S0.  With L_i the sum of log g up to row i of the chunk (inclusive):
//
//   u_i = v_i                                                                            (retention)
//   u_i = beta_i (v_i - exp(L_i) S0^T k_i - sum_(j < i) exp(L_i - L_j) (k_i . k_j) u_j)  (delta rule)
//   o_i = exp(L_i) S0^T q_i + sum_(j <= i) exp(L_i - L_j) (q_i . k_j) u_j
//   S   = exp(L_63) S0 + sum_j exp(L_63 - L_j) k_j u_j^T
//
// What does not need S0 is made for all chunks side by side (k_chunk_mats): P_ij = exp(L_i - L_j) (q_i . k_j), j <= i, and for
// the delta rule the inverse T of the unit lower triangular I + beta_i exp(L_i - L_j) (k_i . k_j), so that
// U = T (beta (V - exp(L) K S0)) is a product.  k_chunk_run then walks a request's chunks, a workgroup per head and 16
// columns of the state (columns never meet), the state in LDS: three to five small products a chunk.  Rows past a portion's
// end are zeros with beta 0 and no decay.  L is formed and subtracted in 64 bits; a decay of nothing counts as exp(-100).  A portion
// that comes to something not finite, or has a negative decay, runs again token by token, a workgroup its 16 columns.
// Bound by the chain of chunks, a chunk 4.5 us of the delta rule, 3.0 of retention: 1.7 and 1.1 of them the products of a SIMD's two waves, the rest the
// barriers and trips to LDS between them (neither K's columns from LDS instead of memory nor rows asked for two chunks ahead made it faster).  2,048 tokens, 32 heads of 128 x 128: k_chunk_run 143 us and k_chunk_mats 70 for the
// delta rule, 95 and 37 for retention (k_chunk_mats 77 and 39 with a row of blocks a wave, one to four of them; 57 and 24 of these with q . k in 32 bits); with four waves that staged every operand in LDS, at
// barriers that waited for the next chunk's loads too, and a branch a number for the activation 189 and 138; 700 tokens, 16 heads 47 and 34 (67 and 51);
// token by token (k_recurrence) 634, and retention in two passes over chunks of 256 side by side 520.
#include "common.h"

typedef float rc_f32x4 __attribute__((ext_vector_type(4)));
typedef double rc_f64x4 __attribute__((ext_vector_type(4)));
#define RC_L 64                 // rows of a chunk
#define RC_LDM (RC_L + 4)       // LDS floats between rows of a 64 x 64 matrix
#define RC_C 16                 // columns of the state a workgroup takes
#define RC_VEC (3 * RC_L)       // a chunk's exp(L_i), exp(L_63 - L_i) and beta_i

struct ChunkArgs {
    float* out;                 // [T, H, Dv]
    const float* q;             // [T, ld]: G heads of D
    const float* k;
    const float* v;             // [T, ld]: H heads of Dv
    const float* beta;          // [T, ld_b]
    const float* gate;          // [T, ld_g]: g (delta rule)
    const float* decay;         // [H]: g (retention)
    float* state;               // [slots, H, D / 16, Dv, 16]
    float* mats;                // [places, H, 1 or 2, 64, 64]: P (and T) of every chunk
    float* vecs;                // [places, H, RC_VEC]
    const int* cu_q;
    const int* slots;
    const int* reqs;            // the portions that run so: (request, place of its first chunk) of each
    int H, G, Dv, ld, ld_g, ld_b;
    float q_scale, k_scale;
};

// (ACT: SiLU first.  Decided at run time, it was a branch for every number: a third of the chunks' time.)
template <bool ACT> __device__ inline float rc_act(float x, float scale) { return (ACT ? x / (1.0f + expf(-x)) : x) * scale; }
template <bool ACT> __device__ inline float4 rc_act4(float4 x, float scale) {
    return make_float4(rc_act<ACT>(x.x, scale), rc_act<ACT>(x.y, scale), rc_act<ACT>(x.z, scale), rc_act<ACT>(x.w, scale));
}
__device__ inline float4 rc_ld4(const float* p) { return *reinterpret_cast<const float4*>(p); }
__device__ inline void rc_st4(float* p, float4 v) { *reinterpret_cast<float4*>(p) = v; }
// 16 columns of a product: four steps, one from each element of the lanes' four
__device__ inline rc_f32x4 rc_mfma4(float4 a, float4 b, rc_f32x4 c) {
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, b.x, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, b.y, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.z, b.z, c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a.w, b.w, c, 0, 0, 0);
}

// The same in 64 bits (of a result a lane has the rows lane / 16 + 4 e of column lane % 16)
__device__ inline rc_f64x4 rc_mfma4(float4 a, float4 b, rc_f64x4 c) {
    c = __builtin_amdgcn_mfma_f64_16x16x4f64((double)a.x, (double)b.x, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f64_16x16x4f64((double)a.y, (double)b.y, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f64_16x16x4f64((double)a.z, (double)b.z, c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f64_16x16x4f64((double)a.w, (double)b.w, c, 0, 0, 0);
}

// 16 rows (a lane's pieces of its row in registers) times 16 columns of the state: four chains of products side by side
template <int J>
__device__ inline rc_f32x4 times_state(const float4 (&x)[J], const float* state) {
    float4 y[J];
#pragma unroll
    for (int j = 0; j < J; ++j) y[j] = rc_ld4(state + j * RC_C * 20);
    __builtin_amdgcn_sched_barrier(0);                  // (every operand is read before them, not two at a time)
    rc_f32x4 s[4] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int j = 0; j < J; ++j) s[j & 3] = rc_mfma4(x[j], y[j], s[j & 3]);
    return (s[0] + s[1]) + (s[2] + s[3]);
}
// a barrier for what lies in LDS: loads on their way to registers stay there
__device__ inline void rc_meet() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}
__device__ inline float4 rc_mul4(float4 a, float4 b) { return make_float4(a.x * b.x, a.y * b.y, a.z * b.z, a.w * b.w); }

template <int D, bool DELTA, bool ACT>
__global__ __launch_bounds__(256) void k_chunk_mats(ChunkArgs a) {
    constexpr int LD = D + 4;
    extern __shared__ __align__(16) float lds[];
    float* Q = lds;                                     // [64][LD]
    float* K = Q + RC_L * LD;
    float* A = K + RC_L * LD;                           // (delta) [64][RC_LDM]: the strict lower triangle
    float* T = A + RC_L * RC_LDM;                       // (delta) its inverse
    __shared__ double L[RC_L];
    __shared__ float beta[RC_L];
    const int b = a.reqs[2 * blockIdx.z], h = blockIdx.y, chunk = blockIdx.x;
    const int row_b = a.cu_q[b], n = a.cu_q[b + 1] - row_b;
    if (chunk * RC_L >= n) return;
    const int row0 = row_b + chunk * RC_L, rows = n - chunk * RC_L < RC_L ? n - chunk * RC_L : RC_L;
    const size_t place = (size_t)(a.reqs[2 * blockIdx.z + 1] + chunk) * a.H + h;
    float* mats = a.mats + place * (DELTA ? 2 : 1) * RC_L * RC_L;
    const int kvh = h / (a.H / a.G);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l16 = lane & 15, quad = lane >> 4;
#pragma unroll
    for (int e = 0; e < RC_L * D / 1024; ++e) {
        const int i = tid + e * 256, r = i / (D / 4), c = i % (D / 4) * 4;
        float4 fq = make_float4(0.f, 0.f, 0.f, 0.f), fk = fq;
        if (r < rows) {
            const size_t at = (size_t)(row0 + r) * a.ld + (size_t)kvh * D + c;
            fq = rc_act4<ACT>(rc_ld4(a.q + at), a.q_scale);
            fk = rc_act4<ACT>(rc_ld4(a.k + at), a.k_scale);
        }
        rc_st4(Q + r * LD + c, fq);
        rc_st4(K + r * LD + c, fk);
    }
    if (tid < RC_L) {
        double s = 0.0;
        float bt = 0.f;
        if (tid < rows) {
            const float g = DELTA ? a.gate[(size_t)(row0 + tid) * a.ld_g + h] : a.decay[h];
            s = g == 0.f ? -100.0 : log((double)g);     // (no number for a negative decay: such a portion runs token by token)
            s = s < -100.0 ? -100.0 : s;
            if (DELTA) bt = a.beta[(size_t)(row0 + tid) * a.ld_b + h];
        }
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const double t = __shfl_up(s, o, 64);
            if (lane >= o) s += t;
        }
        const double last = __shfl(s, 63, 64);
        L[tid] = s;
        beta[tid] = bt;
        float* vec = a.vecs + place * RC_VEC;
        vec[tid] = expf((float)s);
        vec[RC_L + tid] = expf((float)(last - s));
        vec[2 * RC_L + tid] = bt;
    }
    __syncthreads();
    for (int blk = wave; blk < 10; blk += 4) {          // the triangle's ten blocks, two or three a wave: rows 16 rt .., columns 16 ct ..
        const int rt = blk < 1 ? 0 : blk < 3 ? 1 : blk < 6 ? 2 : 3, ct = blk - rt * (rt + 1) / 2;
        // q . k in 64 bits, k . k in four chains of 32: with one chain of 128 sums each the errors of the results were twice those
        // of the recurrence token by token, and with these they are as large or smaller (retention's half)
        rc_f64x4 s = {0.0, 0.0, 0.0, 0.0};
        rc_f32x4 t[4] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int d = 0; d < D; d += 16) {
            const float4 fb = rc_ld4(K + (16 * ct + l16) * LD + d + 4 * quad);
            s = rc_mfma4(rc_ld4(Q + (16 * rt + l16) * LD + d + 4 * quad), fb, s);
            if (DELTA) t[d / 16 & 3] = rc_mfma4(rc_ld4(K + (16 * rt + l16) * LD + d + 4 * quad), fb, t[d / 16 & 3]);
        }
        const rc_f32x4 kk = (t[0] + t[1]) + (t[2] + t[3]);
        const int j = 16 * ct + l16;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int i = 16 * rt + 4 * e + quad;
            mats[i * RC_L + j] = j <= i ? (float)(s[e] * expf((float)(L[i] - L[j]))) : 0.f;
            if (DELTA) {
                const int r = 16 * rt + 4 * quad + e;
                A[r * RC_LDM + j] = j < r ? beta[r] * expf((float)(L[r] - L[j])) * kk[e] : 0.f;
            }
        }
    }
    if (!DELTA) return;
    __syncthreads();
    {   // a block of the diagonal a wave, a column a lane: x_i = e_i - sum_(m < i) A_im x_m
        float x[16];
        const float* blk = A + 16 * wave * RC_LDM + 16 * wave;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            float v = l16 == i ? 1.f : 0.f;
#pragma unroll
            for (int m = 0; m < i; ++m) v = fmaf(-blk[i * RC_LDM + m], x[m], v);
            x[i] = v;
        }
        if (lane < 16)
#pragma unroll
            for (int i = 0; i < 16; ++i) T[(16 * wave + i) * RC_LDM + 16 * wave + l16] = x[i];
    }
    __syncthreads();
    for (int off = 1; off < 4; ++off) {                 // T_ij = -T_ii sum_(j <= m < i) A_im T_mj, block diagonal by block diagonal
        if (wave >= off) {
            const int i = wave, j = wave - off;
            rc_f32x4 s = {0.f, 0.f, 0.f, 0.f};
            for (int m = j; m < i; ++m) {
                const float* tp = T + (16 * m + 4 * quad) * RC_LDM + 16 * j + l16;
                s = rc_mfma4(rc_ld4(A + (16 * i + l16) * RC_LDM + 16 * m + 4 * quad),
                             make_float4(tp[0], tp[RC_LDM], tp[2 * RC_LDM], tp[3 * RC_LDM]), s);
            }
            // (a result's layout, a lane four rows of a column, is an operand's)
            rc_f32x4 t = {0.f, 0.f, 0.f, 0.f};
            t = rc_mfma4(rc_ld4(T + (16 * i + l16) * RC_LDM + 16 * i + 4 * quad), make_float4(s[0], s[1], s[2], s[3]), t);
#pragma unroll
            for (int e = 0; e < 4; ++e) T[(16 * i + 4 * quad + e) * RC_LDM + 16 * j + l16] = -t[e];
        }
        __syncthreads();
    }
#pragma unroll
    for (int e = 0; e < RC_L * RC_L / 1024; ++e) {      // (blocks above the diagonal are never read)
        const int i = tid + e * 256, r = i / (RC_L / 4), c = i % (RC_L / 4) * 4;
        if (c / 16 <= r / 16) rc_st4(mats + RC_L * RC_L + r * RC_L + c, rc_ld4(T + r * RC_LDM + c));
    }
}

// Waves 0 to 3 carry the state on, waves 4 to 7 read it out: wave w and wave 7 - w have the same 16 rows of a chunk, so that a SIMD's two
// waves, w and w + 4, have as many blocks of T and P together as any other's.  Whatever is used by one wave alone (rows of Q and K, the
// triangles P and T, K once more by columns) goes from memory to its registers as the instructions want it, asked for as soon as
// the chunk before has used its own; through LDS go the state, the right side and U.
template <int D, bool DELTA, bool ACT>
__global__ __launch_bounds__(512) void k_chunk_run(ChunkArgs a) {
    constexpr int LD = D + 4, J = D / 16, JP = (J + 3) / 4, MATS = DELTA ? 2 : 1, BUFS = DELTA ? 1 : 2;
    __shared__ __align__(16) float S[BUFS][J][RC_C][20];    // the state's columns, 16 rows side by side (retention: this chunk's and the next one's)
    __shared__ __align__(16) float R[DELTA ? RC_C : 1][RC_LDM], U[DELTA ? RC_C : 1][RC_LDM], W[DELTA ? RC_C : 1][RC_LDM];   // by column: right side, u_i, u_i exp(L_63 - L_i)
    __shared__ int odd;                                 // something came out that is not finite
    // Workgroup i runs on XCD i % 8: the column workgroups of a head, which read the same rows and matrices, go to one XCD
    // (where the heads come in eights), so that its L2 serves all but the first of them.
    const int shares = a.Dv / RC_C, id = blockIdx.x, b = a.reqs[2 * blockIdx.y];
    const bool eights = a.H % 8 == 0;
    const int h = eights ? (id >> 3) / shares * 8 + (id & 7) : id / shares, c0 = (eights ? (id >> 3) % shares : id % shares) * RC_C;
    const int row_b = a.cu_q[b], n = a.cu_q[b + 1] - row_b;
    if (n <= 0) return;
    const int kvh = h / (a.H / a.G), chunks = (n + RC_L - 1) / RC_L;
    const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, quad = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), w16 = wave < 4 ? wave : 7 - wave;
    const int i0 = 16 * w16 + 4 * quad;                 // this lane's rows of a product whose rows are the chunk's
    const size_t place0 = (size_t)a.reqs[2 * blockIdx.y + 1] * a.H + h;
    float* st = a.state + (((size_t)a.slots[b] * a.H + h) * J * a.Dv + c0) * 16;
    for (int i = tid; i < J * RC_C * 4; i += 512) {
        const int j = i / (RC_C * 4), c = i / 4 % RC_C, r = i % 4 * 4;
        rc_st4(&S[0][j][c][r], rc_ld4(st + ((size_t)j * a.Dv + c) * 16 + r));
    }
    if (tid == 0) odd = 0;
    __syncthreads();

    // Where a chunk's operands lie: a base that all lanes share, which moves from chunk to chunk in scalar registers, and a lane's bytes from there.  A
    // row past the portion's end is read from its last row, and dropped where it is used.
    const uint32_t ldb = (uint32_t)a.ld * 4u;
    auto rows_at = [&](const float* x, int chunk) { return reinterpret_cast<const char*>(x + (size_t)(row_b + chunk * RC_L) * a.ld); };
    auto vec_at = [&](int chunk) { return a.vecs + (place0 + (size_t)chunk * a.H) * RC_VEC; };
    auto mats_at = [&](int chunk) { return a.mats + (place0 + (size_t)chunk * a.H) * MATS * RC_L * RC_L; };
    auto row_pieces = [&](float4 (&x)[J], const float* base, int chunk) {
        const char* p = rows_at(base, chunk);
        const uint32_t off = (uint32_t)min(16 * w16 + l16, n - 1 - chunk * RC_L) * ldb + (uint32_t)(kvh * D + 4 * quad) * 4u;
#pragma unroll
        for (int j = 0; j < J; ++j) x[j] = *reinterpret_cast<const float4*>(p + off + 64 * j);
    };
    const uint32_t tri_off = (uint32_t)((16 * w16 + l16) * RC_L + 4 * quad);
    auto triangle = [&](float4 (&x)[4], const float* mat) {      // (all four blocks, used or not: how many loads are on their way has to be known)
#pragma unroll
        for (int m = 0; m < 4; ++m) x[m] = rc_ld4(mat + tri_off + 16 * m);
    };
    // rows 16 m + 4 quad .. of a column (i: 4 m and which of the four rows)
    auto columns = [&](auto& x, const float* base, int chunk, uint32_t col, auto put) {
        const char* p = rows_at(base, chunk);
        const uint32_t off = (uint32_t)(4 * quad) * ldb + col;
        if (n - chunk * RC_L >= RC_L) {
#pragma unroll
            for (int i = 0; i < RC_L / 4; ++i) put(x, i, p + (size_t)((uint32_t)(i / 4 * 16 + i % 4) * ldb), off);
        } else {
#pragma unroll
            for (int i = 0; i < RC_L / 4; ++i) put(x, i, p, (uint32_t)min(i / 4 * 16 + 4 * quad + i % 4, n - 1 - chunk * RC_L) * ldb + col);
        }
    };
    auto put_one = [](float4& x, int e, const char* p, uint32_t off) { (e == 0 ? x.x : e == 1 ? x.y : e == 2 ? x.z : x.w) = *reinterpret_cast<const float*>(p + off); };
    auto v_columns = [&](float4 (&x)[4], int chunk) {
        columns(x, a.v, chunk, (uint32_t)(h * a.Dv + c0 + l16) * 4u, [&](float4 (&y)[4], int i, const char* p, uint32_t off) { put_one(y[i / 4], i % 4, p, off); });
    };
    // what is used of it: the activation's, times the scale, and nothing past the end
    auto used_row = [&](float4 (&x)[J], float scale, int chunk) {
        if (ACT || scale != 1.f) {
#pragma unroll
            for (int j = 0; j < J; ++j) x[j] = rc_act4<ACT>(x[j], scale);
        }
        if (n - chunk * RC_L < RC_L) {
            const bool in = 16 * w16 + l16 < n - chunk * RC_L;
#pragma unroll
            for (int j = 0; j < J; ++j) x[j] = make_float4(in ? x[j].x : 0.f, in ? x[j].y : 0.f, in ? x[j].z : 0.f, in ? x[j].w : 0.f);
        }
    };
    auto used_columns = [&](float4 (&x)[4], float scale, int chunk) {      // rows 16 m + 4 quad ..
        if (ACT || scale != 1.f) {
#pragma unroll
            for (int m = 0; m < 4; ++m) x[m] = rc_act4<ACT>(x[m], scale);
        }
        if (n - chunk * RC_L < RC_L) {
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                const int rows = n - chunk * RC_L - 16 * m - 4 * quad;
                x[m] = make_float4(rows > 0 ? x[m].x : 0.f, rows > 1 ? x[m].y : 0.f, rows > 2 ? x[m].z : 0.f, rows > 3 ? x[m].w : 0.f);
            }
        }
    };

    float none = 0.f;                                   // 0, or no number once a read-out or the state was not finite
    auto has = [&](int t) { return J % 4 == 0 || wave + 4 * t < J; };
    float4 own[JP];                                     // waves 0 to 3: rows 16 j + 4 quad .. of column l16 of the state, j = wave, wave + 4
    if (wave < 4) {
        float4 kr[J], kc[JP][4], tri[4], v[4], grow[4], beta, fall;
        float all = 0.f;
        auto load_columns = [&](int chunk) {
            columns(kc, a.k, chunk, (uint32_t)(kvh * D + 16 * wave + l16) * 4u, [&](float4 (&y)[JP][4], int i, const char* p, uint32_t off) {
#pragma unroll
                for (int t = 0; t < JP; ++t)
                    if (has(t)) put_one(y[t][i / 4], i % 4, p, off + 256 * t);
            });
        };
        // (delta: this lane's rows of V, beta, exp(L) and exp(L_63 - L); retention: V and exp(L_63 - L) of all rows, as an operand of its product)
        auto load_rest = [&](int chunk) {
            const float* vec = vec_at(chunk);
            all = vec[RC_L - 1];
            if (DELTA) {
                const char* p = rows_at(a.v, chunk);
#pragma unroll
                for (int e = 0; e < 4; ++e) put_one(v[0], e, p, (uint32_t)min(i0 + e, n - 1 - chunk * RC_L) * ldb + (uint32_t)(h * a.Dv + c0 + l16) * 4u);
                grow[0] = rc_ld4(vec + RC_L + i0);
                fall = rc_ld4(vec + i0);
                beta = rc_ld4(vec + 2 * RC_L + i0);
            } else {
                v_columns(v, chunk);
#pragma unroll
                for (int m = 0; m < 4; ++m) grow[m] = rc_ld4(vec + RC_L + 16 * m + 4 * quad);
            }
        };
#pragma unroll
        for (int t = 0; t < JP; ++t)
            if (has(t)) own[t] = rc_ld4(st + ((size_t)(wave + 4 * t) * a.Dv + l16) * 16 + 4 * quad);
        if (DELTA) {
            row_pieces(kr, a.k, 0);
            triangle(tri, mats_at(0) + RC_L * RC_L);
        }
        load_rest(0);
        load_columns(0);
        for (int chunk = 0; chunk < chunks; ++chunk) {
            const int next = chunk + 1 < chunks ? chunk + 1 : chunk;
            const float all_now = all;
            float4 w[4];
            if (DELTA) {
                used_row(kr, a.k_scale, chunk);
                const rc_f32x4 x = times_state<J>(kr, &S[0][0][l16][4 * quad]);          // K S0
                row_pieces(kr, a.k, next);
                const float4 vv = rc_act4<ACT>(v[0], 1.f);     // (past the end beta is 0)
                rc_st4(&R[l16][i0], make_float4(beta.x * (vv.x - fall.x * x[0]), beta.y * (vv.y - fall.y * x[1]),
                                                beta.z * (vv.z - fall.z * x[2]), beta.w * (vv.w - fall.w * x[3])));
                rc_meet();
                rc_f32x4 u = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int m = 0; m < 4; ++m)
                    if (m <= w16) u = rc_mfma4(tri[m], rc_ld4(&R[l16][16 * m + 4 * quad]), u);
                triangle(tri, mats_at(next) + RC_L * RC_L);
                const float4 uu = make_float4(u[0], u[1], u[2], u[3]);
                rc_st4(&U[l16][i0], uu);
                rc_st4(&W[l16][i0], rc_mul4(uu, grow[0]));
                load_rest(next);
                rc_meet();                              // U and W are there, and the state of the chunk's start is read
#pragma unroll
                for (int m = 0; m < 4; ++m) w[m] = rc_ld4(&W[l16][16 * m + 4 * quad]);
            } else {
                used_columns(v, 1.f, chunk);
#pragma unroll
                for (int m = 0; m < 4; ++m) w[m] = rc_mul4(v[m], grow[m]);
                load_rest(next);
            }
#pragma unroll
            for (int t = 0; t < JP; ++t) {              // 16 rows of the state: its own decayed, and K^T W
                if (!has(t)) break;
                rc_f32x4 s[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
                used_columns(kc[t], a.k_scale, chunk);
#pragma unroll
                for (int m = 0; m < 4; ++m) s[m & 1] = rc_mfma4(kc[t][m], w[m], s[m & 1]);
                const rc_f32x4 x = s[0] + s[1];
                own[t] = make_float4(fmaf(own[t].x, all_now, x[0]), fmaf(own[t].y, all_now, x[1]), fmaf(own[t].z, all_now, x[2]), fmaf(own[t].w, all_now, x[3]));
                rc_st4(&S[DELTA ? 0 : (chunk + 1) & 1][wave + 4 * t][l16][4 * quad], own[t]);
            }
            load_columns(next);
            rc_meet();                                  // the state is written, and U read
        }
#pragma unroll
        for (int t = 0; t < JP; ++t)
            if (has(t)) none += 0.f * own[t].x + 0.f * own[t].y + 0.f * own[t].z + 0.f * own[t].w;
    } else {
        float4 q[J], tri[4], v[4], fall;
        row_pieces(q, a.q, 0);
        fall = rc_ld4(vec_at(0) + i0);
        triangle(tri, mats_at(0));
        if (!DELTA) v_columns(v, 0);
        for (int chunk = 0; chunk < chunks; ++chunk) {
            const int next = chunk + 1 < chunks ? chunk + 1 : chunk, row0 = row_b + chunk * RC_L, rows = n - chunk * RC_L;
            used_row(q, a.q_scale, chunk);
            rc_f32x4 o = times_state<J>(q, &S[DELTA ? 0 : chunk & 1][0][l16][4 * quad]);          // Q S0
            row_pieces(q, a.q, next);
            o[0] *= fall.x; o[1] *= fall.y; o[2] *= fall.z; o[3] *= fall.w;
            fall = rc_ld4(vec_at(next) + i0);
            if (DELTA) {
                rc_meet();
                rc_meet();
            }
            rc_f32x4 p[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
            if (!DELTA) used_columns(v, 1.f, chunk);
#pragma unroll
            for (int m = 0; m < 4; ++m)
                if (m <= w16) p[m & 1] = rc_mfma4(tri[m], DELTA ? rc_ld4(&U[l16][16 * m + 4 * quad]) : v[m], p[m & 1]);
            triangle(tri, mats_at(next));
            if (!DELTA) v_columns(v, next);
            o += p[0] + p[1];
            {
                float* to = a.out + ((size_t)(row0 + 16 * w16) * a.H + h) * a.Dv + c0;
                const uint32_t off = (uint32_t)(4 * quad * a.H * a.Dv + l16), row = (uint32_t)(a.H * a.Dv);
                if (rows >= RC_L) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) *(to + (size_t)(e * row) + off) = o[e];
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (i0 + e < rows) *(to + (size_t)(e * row) + off) = o[e];
                }
            }
            none += 0.f * o[0] + 0.f * o[1] + 0.f * o[2] + 0.f * o[3];
            rc_meet();
        }
    }
    if (none != none) odd = 1;
    __syncthreads();
    if (!odd) {
        if (wave < 4)
#pragma unroll
            for (int t = 0; t < JP; ++t)
                if (has(t)) rc_st4(st + ((size_t)(wave + 4 * t) * a.Dv + l16) * 16 + 4 * quad, own[t]);
        return;
    }
    // Not finite somewhere (a state that once is stays so): the portion again from its first state, token by token.  0 times an
    // infinity or a NaN is no 0, so that above it shows in rows before its own, too; and a negative decay has no logarithm.
    extern __shared__ __align__(16) float lds[];
    float* Q = lds;                                     // [64][LD]
    float* K = Q + RC_L * LD;
    float* V = K + RC_L * LD;                           // [64][17]
    const int c = tid >> 4 & 15, r = tid & 15;          // waves 0 to 3: 16 lanes a column, rows r, r + 16, ..
    float s[J];
#pragma unroll
    for (int j = 0; j < J; ++j) s[j] = st[((size_t)j * a.Dv + c) * 16 + r];
    __syncthreads();                                    // (all have read the state before some write it)
    for (int chunk = 0; chunk < chunks; ++chunk) {
        const int row0 = row_b + chunk * RC_L, rows = n - chunk * RC_L < RC_L ? n - chunk * RC_L : RC_L;
        for (int i = tid; i < rows * (D / 4); i += 512) {
            const int y = i / (D / 4), x = i % (D / 4) * 4;
            const size_t at = (size_t)(row0 + y) * a.ld + (size_t)kvh * D + x;
            rc_st4(Q + y * LD + x, rc_act4<ACT>(rc_ld4(a.q + at), a.q_scale));
            rc_st4(K + y * LD + x, rc_act4<ACT>(rc_ld4(a.k + at), a.k_scale));
        }
        for (int i = tid; i < rows * RC_C; i += 512)
            V[i / RC_C * (RC_C + 1) + i % RC_C] = rc_act<ACT>(a.v[(size_t)(row0 + i / RC_C) * a.ld + (size_t)h * a.Dv + c0 + i % RC_C], 1.f);
        __syncthreads();
        for (int i = 0; i < rows && wave < 4; ++i) {
            const float g = DELTA ? a.gate[(size_t)(row0 + i) * a.ld_g + h] : a.decay[h];
            const float* k = K + i * LD + r;
            const float* q = Q + i * LD + r;
            float u = V[i * (RC_C + 1) + c], o = 0.f;
            if (DELTA) {
                float d = 0.f;
#pragma unroll
                for (int j = 0; j < J; ++j) d = fmaf(s[j], k[16 * j], d);
#pragma unroll
                for (int m = 8; m > 0; m >>= 1) d += __shfl_xor(d, m, 64);
                u = a.beta[(size_t)(row0 + i) * a.ld_b + h] * (u - g * d);
            }
#pragma unroll
            for (int j = 0; j < J; ++j) {
                s[j] = fmaf(g, s[j], k[16 * j] * u);
                o = fmaf(s[j], q[16 * j], o);
            }
#pragma unroll
            for (int m = 8; m > 0; m >>= 1) o += __shfl_xor(o, m, 64);
            if (r == 0) a.out[((size_t)(row0 + i) * a.H + h) * a.Dv + c0 + c] = o;
        }
        __syncthreads();
    }
    if (wave < 4)
#pragma unroll
        for (int j = 0; j < J; ++j) st[((size_t)j * a.Dv + c) * 16 + r] = s[j];
}

#define RC_UNITS 256            // compute units
template <int D, bool DELTA> constexpr bool RC_STAGED = D <= (DELTA ? 48 : 80);
// The same with four waves a workgroup, which stage a chunk's operands in LDS and each do all of 16 rows: for small heads and more workgroups than compute
// units.  Two of these run on a unit, whose products then wait for each other's trips to LDS; k_chunk_run has the registers for one of its own, and fetches K's columns number by
// number: a shorter chain and more loads.  (It without fetching ahead, two a unit: no faster.)  Both, k_chunk_run and these, us with k_chunk_mats: retention, 8 portions of 1,024 rows,
// 32 heads of 64 x 64 (1,024 workgroups) 200 and 165, 16 of 80 x 64 (512) 122 and 106, 4 of 512 rows, 16 heads of 48 x 96 (384) 48 and 38; the delta rule, of 48 x 96
// 61.5 and 57.  Heads of 96 and more have no room for two; one workgroup a unit and fewer go faster with k_chunk_run (one portion of 2,048 rows, 32 heads of 64: 81, staged 107)
// unless q, k and v are to pass an activation: every wave there makes the numbers it reads, K's once more by columns, here each is made once (2,048 rows, 8 heads of 48 x 96 140 us and 116, 32 of 64 163 and 151).
template <int D, bool DELTA, bool ACT>
__global__ __launch_bounds__(256) void k_chunk_run_staged(ChunkArgs a) {
    constexpr int LD = D + 4, J = D / 16, NQ = RC_L * D / 1024, NM = RC_L * RC_L / 1024, MATS = DELTA ? 2 : 1;
    extern __shared__ __align__(16) float lds[];
    float* Q = lds;                                     // [64][LD]
    float* K = Q + RC_L * LD;
    float* P = K + RC_L * LD;                           // [64][RC_LDM]
    float* T = P + RC_L * RC_LDM;                       // (delta) [64][RC_LDM]
    __shared__ __align__(16) float S[J][RC_C][20];      // the state's columns, 16 rows side by side
    __shared__ __align__(16) float U[RC_C][RC_LDM], W[RC_C][RC_LDM];     // by column: u_i; (delta) the right side; u_i exp(L_63 - L_i)
    __shared__ float V[RC_L][RC_C + 1];
    __shared__ float vec[RC_VEC];
    __shared__ int odd;                                 // something came out that is not finite
    // Workgroup i runs on XCD i % 8: the column workgroups of a head, which read the same rows and matrices, go to one XCD
    // (where the heads come in eights), so that its L2 serves all but the first of them.
    const int shares = a.Dv / RC_C, id = blockIdx.x, b = a.reqs[2 * blockIdx.y];
    const bool eights = a.H % 8 == 0;
    const int h = eights ? (id >> 3) / shares * 8 + (id & 7) : id / shares, c0 = (eights ? (id >> 3) % shares : id % shares) * RC_C;
    const int row_b = a.cu_q[b], n = a.cu_q[b + 1] - row_b;
    if (n <= 0) return;
    const int kvh = h / (a.H / a.G);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l16 = lane & 15, quad = lane >> 4;
    const int place0 = a.reqs[2 * blockIdx.y + 1];
    float* st = a.state + (((size_t)a.slots[b] * a.H + h) * J * a.Dv + c0) * 16;
    for (int i = tid; i < J * RC_C * 4; i += 256) {
        const int j = i / (RC_C * 4), c = i / 4 % RC_C, r = i % 4 * 4;
        rc_st4(&S[j][c][r], rc_ld4(st + ((size_t)j * a.Dv + c) * 16 + r));
    }
    // a chunk's operands come into registers while the chunk before it is worked on
    float4 rq[NQ], rk[NQ], rm[MATS * NM], rv;
    float rvec = 0.f;
    auto fetch = [&](int chunk) {
        const int row0 = row_b + chunk * RC_L, rows = n - chunk * RC_L;
        const size_t place = (size_t)(place0 + chunk) * a.H + h;
#pragma unroll
        for (int e = 0; e < NQ; ++e) {
            const int i = tid + e * 256, r = i / (D / 4), c = i % (D / 4) * 4;
            const size_t at = (size_t)(row0 + (r < rows ? r : 0)) * a.ld + (size_t)kvh * D + c;
            rq[e] = rc_ld4(a.q + at);
            rk[e] = rc_ld4(a.k + at);
            if (r >= rows) rq[e] = rk[e] = make_float4(0.f, 0.f, 0.f, 0.f);
        }
        const float* mats = a.mats + place * MATS * RC_L * RC_L;
#pragma unroll
        for (int e = 0; e < MATS * NM; ++e) {
            const int i = tid + e * 256, r = i / (RC_L / 4) % RC_L, c = i % (RC_L / 4) * 4;
            rm[e] = c / 16 <= r / 16 ? rc_ld4(mats + (size_t)i * 4) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
        const int r = tid / 4, c = tid % 4 * 4;
        rv = rc_ld4(a.v + (size_t)(row0 + (r < rows ? r : 0)) * a.ld + (size_t)h * a.Dv + c0 + c);
        if (r >= rows) rv = make_float4(0.f, 0.f, 0.f, 0.f);
        if (tid < RC_VEC) rvec = a.vecs[place * RC_VEC + tid];
    };
    auto stage = [&]() {                                // the fetched chunk to LDS
#pragma unroll
        for (int e = 0; e < NQ; ++e) {
            const int i = tid + e * 256, r = i / (D / 4), c = i % (D / 4) * 4;
            rc_st4(Q + r * LD + c, rc_act4<ACT>(rq[e], a.q_scale));
            rc_st4(K + r * LD + c, rc_act4<ACT>(rk[e], a.k_scale));
        }
#pragma unroll
        for (int e = 0; e < MATS * NM; ++e) {
            const int i = tid + e * 256, r = i / (RC_L / 4), c = i % (RC_L / 4) * 4;
            rc_st4(P + r * RC_LDM + c, rm[e]);          // (T lies behind P)
        }
        {
            const int r = tid / 4, c = tid % 4 * 4;
            const float4 x = rc_act4<ACT>(rv, 1.f);
            V[r][c] = x.x; V[r][c + 1] = x.y; V[r][c + 2] = x.z; V[r][c + 3] = x.w;
        }
        if (tid < RC_VEC) vec[tid] = rvec;
    };
    auto rows_times_state = [&](const float* rows, const float* state) {
        float4 x[J];
#pragma unroll
        for (int j = 0; j < J; ++j) x[j] = rc_ld4(rows + (16 * wave + l16) * LD + 4 * quad + 16 * j);
        return times_state<J>(x, state);
    };
    if (tid == 0) odd = 0;
    float none = 0.f;                                   // 0, or no number once a read-out was not finite
    fetch(0);
    for (int chunk = 0; chunk * RC_L < n; ++chunk) {
        const int row0 = row_b + chunk * RC_L, rows = n - chunk * RC_L;
        __syncthreads();                                // the chunk before has been read, the state is written
        stage();
        __syncthreads();
        if ((chunk + 1) * RC_L < n) fetch(chunk + 1);
        const int i0 = 16 * wave + 4 * quad;            // this lane's rows of a product whose rows are the chunk's
        rc_f32x4 u;
        if (DELTA) {
            const rc_f32x4 x = rows_times_state(K, &S[0][l16][4 * quad]);       // K S0
            float r[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) r[e] = vec[2 * RC_L + i0 + e] * (V[i0 + e][l16] - vec[i0 + e] * x[e]);
            rc_st4(&W[l16][i0], make_float4(r[0], r[1], r[2], r[3]));
            __syncthreads();
            u = rc_f32x4{0.f, 0.f, 0.f, 0.f};
            for (int m = 0; m <= wave; ++m) u = rc_mfma4(rc_ld4(T + (16 * wave + l16) * RC_LDM + 16 * m + 4 * quad), rc_ld4(&W[l16][16 * m + 4 * quad]), u);
            __syncthreads();                            // W is read, and written again below
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) u[e] = V[i0 + e][l16];
        }
        rc_st4(&U[l16][i0], make_float4(u[0], u[1], u[2], u[3]));
        rc_st4(&W[l16][i0], make_float4(u[0] * vec[RC_L + i0], u[1] * vec[RC_L + i0 + 1], u[2] * vec[RC_L + i0 + 2], u[3] * vec[RC_L + i0 + 3]));
        rc_f32x4 o = rows_times_state(Q, &S[0][l16][4 * quad]);         // Q S0
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] *= vec[i0 + e];
        __syncthreads();                                // U and W are there, and the state of the chunk's start is read
        rc_f32x4 p[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int m = 0; m < RC_L / 16; ++m)
            if (m <= wave) p[m & 1] = rc_mfma4(rc_ld4(P + (16 * wave + l16) * RC_LDM + 16 * m + 4 * quad), rc_ld4(&U[l16][16 * m + 4 * quad]), p[m & 1]);
        o += p[0] + p[1];
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (i0 + e < rows) a.out[((size_t)(row0 + i0 + e) * a.H + h) * a.Dv + c0 + l16] = o[e];
        none += 0.f * o[0] + 0.f * o[1] + 0.f * o[2] + 0.f * o[3];
        const float all = vec[RC_L - 1];                // exp(L_63)
        for (int j = wave; j < J; j += 4) {             // 16 rows of the state: its own decayed, and K^T W
            const float4 s0 = rc_ld4(&S[j][l16][4 * quad]);
            rc_f32x4 s[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
            for (int m = 0; m < RC_L / 16; ++m) {
                const float* kp = K + (16 * m + 4 * quad) * LD + 16 * j + l16;
                s[m & 1] = rc_mfma4(make_float4(kp[0], kp[LD], kp[2 * LD], kp[3 * LD]), rc_ld4(&W[l16][16 * m + 4 * quad]), s[m & 1]);
            }
            const rc_f32x4 t = s[0] + s[1];
            rc_st4(&S[j][l16][4 * quad], make_float4(fmaf(s0.x, all, t[0]), fmaf(s0.y, all, t[1]), fmaf(s0.z, all, t[2]), fmaf(s0.w, all, t[3])));
        }
    }
    __syncthreads();
    for (int i = tid; i < J * RC_C * 4; i += 256) {
        const float4 x = rc_ld4(&S[i / (RC_C * 4)][i / 4 % RC_C][i % 4 * 4]);
        none += 0.f * x.x + 0.f * x.y + 0.f * x.z + 0.f * x.w;
    }
    if (none != none) odd = 1;
    __syncthreads();
    if (!odd) {
        for (int i = tid; i < J * RC_C * 4; i += 256) {
            const int j = i / (RC_C * 4), c = i / 4 % RC_C, r = i % 4 * 4;
            rc_st4(st + ((size_t)j * a.Dv + c) * 16 + r, rc_ld4(&S[j][c][r]));
        }
        return;
    }
    // Not finite somewhere (a state that once is stays so): the portion again from its first state, token by token.  0 times an
    // infinity or a NaN is no 0, so that above it shows in rows before its own, too; and a negative decay has no logarithm.
    const int c = tid >> 4, r = tid & 15;               // 16 lanes a column, rows r, r + 16, ..
    float s[J];
#pragma unroll
    for (int j = 0; j < J; ++j) s[j] = st[((size_t)j * a.Dv + c) * 16 + r];
    for (int chunk = 0; chunk * RC_L < n; ++chunk) {
        const int row0 = row_b + chunk * RC_L, rows = n - chunk * RC_L < RC_L ? n - chunk * RC_L : RC_L;
        fetch(chunk);
        __syncthreads();
        stage();
        __syncthreads();
        for (int i = 0; i < rows; ++i) {
            const float g = DELTA ? a.gate[(size_t)(row0 + i) * a.ld_g + h] : a.decay[h];
            const float* k = K + i * LD + r;
            const float* q = Q + i * LD + r;
            float u = V[i][c], o = 0.f;
            if (DELTA) {
                float d = 0.f;
#pragma unroll
                for (int j = 0; j < J; ++j) d = fmaf(s[j], k[16 * j], d);
#pragma unroll
                for (int m = 8; m > 0; m >>= 1) d += __shfl_xor(d, m, 64);
                u = vec[2 * RC_L + i] * (u - g * d);
            }
#pragma unroll
            for (int j = 0; j < J; ++j) {
                s[j] = fmaf(g, s[j], k[16 * j] * u);
                o = fmaf(s[j], q[16 * j], o);
            }
#pragma unroll
            for (int m = 8; m > 0; m >>= 1) o += __shfl_xor(o, m, 64);
            if (r == 0) a.out[((size_t)(row0 + i) * a.H + h) * a.Dv + c0 + c] = o;
        }
    }
#pragma unroll
    for (int j = 0; j < J; ++j) st[((size_t)j * a.Dv + c) * 16 + r] = s[j];
}

template <int D, bool DELTA, bool ACT>
static int launch_chunks(const ChunkArgs& a, int B, int max_q, hipStream_t stream) {
    const int one = 2 * RC_L * (D + 4) * 4, mats = one + (DELTA ? 2 : 0) * RC_L * RC_LDM * 4, columns = a.Dv / RC_C * a.H;
    const bool staged = RC_STAGED<D, DELTA> && (ACT || (long long)columns * B > RC_UNITS);
    constexpr bool always = RC_STAGED<D, DELTA> && ACT;
    const int run = one + (staged ? (DELTA ? 2 : 1) * RC_L * RC_LDM : RC_L * (RC_C + 1)) * 4;
    const auto k_run = staged ? k_chunk_run_staged<RC_STAGED<D, DELTA> ? D : 48, DELTA, ACT> : k_chunk_run<D, DELTA, ACT && !always>;
    const void* kernels[2] = {(const void*)k_chunk_mats<D, DELTA, ACT>, (const void*)k_run};
    const int bytes[2] = {mats, run};
    for (int i = 0; i < 2; ++i)
        if (bytes[i] > 65536) {
            const hipError_t e = hipFuncSetAttribute(kernels[i], hipFuncAttributeMaxDynamicSharedMemorySize, bytes[i]);
            if (e != hipSuccess) (void)hipGetLastError();
            XR_REQUIRE(e == hipSuccess, "recurrence in chunks: %d bytes of LDS: %s", bytes[i], hipGetErrorString(e));
        }
    k_chunk_mats<D, DELTA, ACT><<<dim3((max_q + RC_L - 1) / RC_L, a.H, B), 256, mats, stream>>>(a);
    XR_CHECK_LAUNCH("chunk_mats");
    k_run<<<dim3(columns, B), staged ? 256 : 512, run, stream>>>(a);
    XR_CHECK_LAUNCH("chunk_run");
    return XR_OK;
}

// `n_reqs` portions of up to `max_q` rows: reqs [n_reqs][2] are the request and the place of its first chunk; they take `places` chunks
// of 64 rows together, one after another.

extern "C" int xr_recurrence_chunks(float* out, const float* q, const float* k, const float* v, const float* beta, const float* gate,
                                    const float* decay, float* state, const int* cu_q, const int* slots, const int* reqs, float* scratch,
                                    long long scratch_floats, int places, int n_reqs, int max_q, int H, int G, int D, int Dv, int ld, int ld_g, int ld_b, int delta, int act,
                                    float q_scale, float k_scale, hipStream_t stream) {
    XR_REQUIRE(places >= 0 && n_reqs >= 0 && max_q >= 0 && H > 0 && G > 0 && H % G == 0, "recurrence in chunks: %d heads over %d key heads", H, G);
    XR_REQUIRE(D % 16 == 0 && D > 32 && D <= 128 && Dv > 0 && Dv % RC_C == 0, "recurrence in chunks: key size %d (48 to 128), value size %d: in steps of 16", D, Dv);
    XR_REQUIRE(out && q && k && v && state && cu_q && slots && reqs && scratch, "recurrence in chunks: a pointer is missing");
    XR_REQUIRE(delta ? (beta && gate && ld_b >= H && ld_g >= H) : decay != nullptr, "recurrence in chunks: the gates are missing");
    XR_REQUIRE(ld % 4 == 0 && (((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)state | (uintptr_t)scratch) & 15) == 0,
               "recurrence in chunks: rows that are not 16-byte aligned (%d apart)", ld);
    XR_REQUIRE(act == 0 || act == 1, "recurrence in chunks: activation %d of q, k and v (0: none, 1: SiLU)", act);
    XR_REQUIRE((long long)ld * RC_L * 4 < (1ll << 32) && (long long)H * Dv * RC_L < (1ll << 31), "recurrence in chunks: rows %d apart", ld);
    XR_REQUIRE(n_reqs <= 65535 && H <= 65535, "recurrence in chunks: %d requests, %d heads", n_reqs, H);
    const long long mats = (long long)places * H * (delta ? 2 : 1) * RC_L * RC_L;
    XR_REQUIRE(scratch_floats >= mats + (long long)places * H * RC_VEC, "recurrence in chunks: a scratch of %lld floats for %d chunks", scratch_floats, places);
    if (n_reqs == 0 || max_q == 0) return XR_OK;
    ChunkArgs a{out, q, k, v, beta, gate, decay, state, scratch, scratch + mats, cu_q, slots, reqs,
                H, G, Dv, ld, ld_g, ld_b, q_scale, k_scale};
#define RCA(DD, ACT) (delta ? launch_chunks<DD, true, ACT>(a, n_reqs, max_q, stream) : launch_chunks<DD, false, ACT>(a, n_reqs, max_q, stream))
#define RC(DD) case DD: return act ? RCA(DD, true) : RCA(DD, false)
    switch (D) { RC(48); RC(64); RC(80); RC(96); RC(112); RC(128); }
#undef RC
#undef RCA
    return XR_BAD_ARG;
}
