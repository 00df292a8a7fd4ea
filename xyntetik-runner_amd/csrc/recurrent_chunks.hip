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
// Bound by the chain of chunks, a chunk (5.7 us of the delta rule, 4.1 of retention) by five barriers, the trips to LDS between
// them and, a third of it, its products.  2,048 tokens, 32 heads of 128 x 128: k_chunk_run 182 us and k_chunk_mats 74 for the
// delta rule, 130 and 34 for retention (k_chunk_mats 57 and 24 with q . k in 32 bits); token by token (k_recurrence) 634, and
// retention in two passes over chunks of 256 side by side 520.
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
    int H, G, Dv, ld, ld_g, ld_b, act;
    float q_scale, k_scale;
};

__device__ inline float rc_act(float x, int act, float scale) { return (act ? x / (1.0f + expf(-x)) : x) * scale; }
__device__ inline float4 rc_act4(float4 x, int act, float scale) {
    return make_float4(rc_act(x.x, act, scale), rc_act(x.y, act, scale), rc_act(x.z, act, scale), rc_act(x.w, act, scale));
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

// 16 rows (a lane's at `rows`) times 16 columns of the state: four chains of products side by side, every operand read before them
template <int J>
__device__ inline rc_f32x4 times_state(const float* rows, const float* state) {
    float4 x[J], y[J];
#pragma unroll
    for (int j = 0; j < J; ++j) { x[j] = rc_ld4(rows + 16 * j); y[j] = rc_ld4(state + j * RC_C * 20); }
    rc_f32x4 s[4] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int j = 0; j < J; ++j) s[j & 3] = rc_mfma4(x[j], y[j], s[j & 3]);
    return (s[0] + s[1]) + (s[2] + s[3]);
}

template <int D, bool DELTA>
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
            fq = rc_act4(rc_ld4(a.q + at), a.act, a.q_scale);
            fk = rc_act4(rc_ld4(a.k + at), a.act, a.k_scale);
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
    for (int ct = 0; ct <= wave; ++ct) {                // rows 16 wave .., columns 16 ct ..
        // q . k in 64 bits, k . k in four chains of 32: with one chain of 128 sums each the errors of the results were twice those
        // of the recurrence token by token, and with these they are as large or smaller (retention's half)
        rc_f64x4 s = {0.0, 0.0, 0.0, 0.0};
        rc_f32x4 t[4] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int d = 0; d < D; d += 16) {
            const float4 fb = rc_ld4(K + (16 * ct + l16) * LD + d + 4 * quad);
            s = rc_mfma4(rc_ld4(Q + (16 * wave + l16) * LD + d + 4 * quad), fb, s);
            if (DELTA) t[d / 16 & 3] = rc_mfma4(rc_ld4(K + (16 * wave + l16) * LD + d + 4 * quad), fb, t[d / 16 & 3]);
        }
        const rc_f32x4 kk = (t[0] + t[1]) + (t[2] + t[3]);
        const int j = 16 * ct + l16;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int i = 16 * wave + 4 * e + quad;
            mats[i * RC_L + j] = j <= i ? (float)(s[e] * expf((float)(L[i] - L[j]))) : 0.f;
            if (DELTA) {
                const int r = 16 * wave + 4 * quad + e;
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

template <int D, bool DELTA>
__global__ __launch_bounds__(256) void k_chunk_run(ChunkArgs a) {
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
            rc_st4(Q + r * LD + c, rc_act4(rq[e], a.act, a.q_scale));
            rc_st4(K + r * LD + c, rc_act4(rk[e], a.act, a.k_scale));
        }
#pragma unroll
        for (int e = 0; e < MATS * NM; ++e) {
            const int i = tid + e * 256, r = i / (RC_L / 4), c = i % (RC_L / 4) * 4;
            rc_st4(P + r * RC_LDM + c, rm[e]);          // (T lies behind P)
        }
        {
            const int r = tid / 4, c = tid % 4 * 4;
            const float4 x = rc_act4(rv, a.act, 1.f);
            V[r][c] = x.x; V[r][c + 1] = x.y; V[r][c + 2] = x.z; V[r][c + 3] = x.w;
        }
        if (tid < RC_VEC) vec[tid] = rvec;
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
            const rc_f32x4 x = times_state<J>(K + (16 * wave + l16) * LD + 4 * quad, &S[0][l16][4 * quad]);       // K S0
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
        rc_f32x4 o = times_state<J>(Q + (16 * wave + l16) * LD + 4 * quad, &S[0][l16][4 * quad]);         // Q S0
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

template <int D, bool DELTA>
static int launch_chunks(const ChunkArgs& a, int B, int max_q, hipStream_t stream) {
    const int one = 2 * RC_L * (D + 4) * 4, mats = one + (DELTA ? 2 : 0) * RC_L * RC_LDM * 4, run = one + (DELTA ? 2 : 1) * RC_L * RC_LDM * 4;
    const void* kernels[2] = {(const void*)k_chunk_mats<D, DELTA>, (const void*)k_chunk_run<D, DELTA>};
    const int bytes[2] = {mats, run};
    for (int i = 0; i < 2; ++i)
        if (bytes[i] > 65536) {
            const hipError_t e = hipFuncSetAttribute(kernels[i], hipFuncAttributeMaxDynamicSharedMemorySize, bytes[i]);
            if (e != hipSuccess) (void)hipGetLastError();
            XR_REQUIRE(e == hipSuccess, "recurrence in chunks: %d bytes of LDS: %s", bytes[i], hipGetErrorString(e));
        }
    k_chunk_mats<D, DELTA><<<dim3((max_q + RC_L - 1) / RC_L, a.H, B), 256, mats, stream>>>(a);
    XR_CHECK_LAUNCH("chunk_mats");
    k_chunk_run<D, DELTA><<<dim3(a.Dv / RC_C * a.H, B), 256, run, stream>>>(a);
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
    XR_REQUIRE(n_reqs <= 65535 && H <= 65535, "recurrence in chunks: %d requests, %d heads", n_reqs, H);
    const long long mats = (long long)places * H * (delta ? 2 : 1) * RC_L * RC_L;
    XR_REQUIRE(scratch_floats >= mats + (long long)places * H * RC_VEC, "recurrence in chunks: a scratch of %lld floats for %d chunks", scratch_floats, places);
    if (n_reqs == 0 || max_q == 0) return XR_OK;
    ChunkArgs a{out, q, k, v, beta, gate, decay, state, scratch, scratch + mats, cu_q, slots, reqs,
                H, G, Dv, ld, ld_g, ld_b, act, q_scale, k_scale};
#define RC(DD) case DD: return delta ? launch_chunks<DD, true>(a, n_reqs, max_q, stream) : launch_chunks<DD, false>(a, n_reqs, max_q, stream)
    switch (D) { RC(48); RC(64); RC(80); RC(96); RC(112); RC(128); }
#undef RC
    return XR_BAD_ARG;
}
