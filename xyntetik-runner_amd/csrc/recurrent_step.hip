// A decoded token of a linear recurrence in one kernel: what lies between the input product's 32-bit rows and the output
// product's, for steps in which every request brings one row.
//
//   retention:   q, k rotated (channel j with j + rot/2), k scaled;  S <- decay_h S + k v^T;               o = S^T q
//   delta rule:  q, k to unit length, q scaled;  beta = sigmoid(b);  g = exp(-exp(A_log) softplus(a + dt_bias));
//                S <- g S;  u = beta (v - S^T k);  S <- S + k u^T;                                         o = S^T q
//   then  o / sqrt(mean(o^2) + eps) * w * act(gate)  per head.
//
// What bounds it is the chain of kernels: preparing rows, the recurrence and the norm are 3 to 7 us each beside the 64 KB that a head's
// state of 128 x 128 moves twice.  A workgroup of 1,024 threads takes a whole head of a request, so that its norm is at hand: 16
// lanes a column, as k_recurrence lays the state out ([J][Dv][16], S[16 j + r][c] at (j Dv + c) 16 + r), its columns 64 at a time; the state's
// loads are on their way while the rows are prepared.  A decode step of 8 requests of the Suripel shape of width 2,048: retention's four kernels
// behind its product 17.0 us a layer, 7.8 so, the delta rule's three behind its convolution 13.1, 8.3; whole steps of 1 to 64 requests 2 to 6% less.
#include "common.h"

#define STEP_RETENTION 0
#define STEP_DELTA 1
#define STEP_MAX_D 128
#define STEP_MAX_DV 128

struct StepArgs {
    void* out;               // [B, ld_out]
    const float* q;          // [B, ld]: G heads of D
    const float* k;
    const float* v;          // H heads of Dv
    float* state;            // [slots][H][J][Dv][16]
    const int* slots;
    const int* positions;
    const float* inv_freq;   // [rot / 2] (retention)
    const float* decay;      // [H] (retention)
    const float* beta;       // [B, ld_b] at head 0, before the sigmoid (delta rule)
    const float* a;          // [B, ld_b] at head 0 (delta rule)
    const float* a_log;      // [H]
    const float* dt_bias;    // [H]
    const float* gate;       // [B, ld_g]: H heads of Dv
    const float* w;          // [Dv], [H * Dv] (w_full) or null
    int H, G, D, Dv, ld, ld_b, ld_g, ld_out, rot, w_full, gate_act;
    float q_scale, k_scale, unit_eps, eps;
};

template <int CTRL> __device__ inline float row_permute(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, true));
}
__device__ inline float sum_of_16(float v) {
    v += row_permute<0x128>(v);     // row_ror:8
    v += row_permute<0x124>(v);     // row_ror:4
    v += row_permute<0x4E>(v);      // quad_perm [2,3,0,1]
    v += row_permute<0xB1>(v);      // quad_perm [1,0,3,2]
    return v;
}

template <int MODE, typename TO>
__global__ __launch_bounds__(1024) void k_recurrence_step(StepArgs a) {
    constexpr int DPER = STEP_MAX_D / 16, NC = STEP_MAX_DV / 64;
    __shared__ float qf[STEP_MAX_D], kf[STEP_MAX_D];        // channel 16 j + r at r DPER + j, zeros from D on
    __shared__ float of[STEP_MAX_DV];
    __shared__ float beta_s, decay_s;
    const int h = blockIdx.x, t = blockIdx.y, tid = threadIdx.x;
    const int wave = tid >> 6, lane = tid & 63;
    const int r = tid & 15, c0 = tid >> 4;
    const int g = h / (a.H / a.G);
    const int J = (a.D + 15) >> 4;
    float* sp = a.state + ((size_t)a.slots[t] * a.H + h) * J * a.Dv * 16;
    float S[NC][DPER], vv[NC];
#pragma unroll
    for (int n = 0; n < NC; ++n) {
        const int c = c0 + 64 * n;
#pragma unroll
        for (int j = 0; j < DPER; ++j) S[n][j] = (c < a.Dv && j < J) ? sp[((size_t)j * a.Dv + c) * 16 + r] : 0.f;
        vv[n] = c < a.Dv ? a.v[(size_t)t * a.ld + (size_t)h * a.Dv + c] : 0.f;
    }
    auto place = [](int d) { return (d & 15) * DPER + (d >> 4); };
    if (wave < 2) {                  // a wave the queries, a wave the keys
        const float* row = (wave ? a.k : a.q) + (size_t)t * a.ld + (size_t)g * a.D;
        float* to = wave ? kf : qf;
        const float scale = wave ? a.k_scale : a.q_scale;
        if (MODE == STEP_RETENTION) {
            const int half = a.rot >> 1;
            const float pos = half ? (float)a.positions[t] : 0.f;
            for (int j = lane; j < half; j += 64) {
                const float x = pos * a.inv_freq[j];
                const float c = cosf(x), s = sinf(x);
                const float u = row[j], v = row[j + half];
                to[place(j)] = (u * c - v * s) * scale;
                to[place(j + half)] = (v * c + u * s) * scale;
            }
            for (int d = a.rot + lane; d < a.D; d += 64) to[place(d)] = row[d] * scale;
        } else {
            float x[STEP_MAX_D / 64], ss = 0.f;
#pragma unroll
            for (int i = 0; i < STEP_MAX_D / 64; ++i) {
                x[i] = lane + 64 * i < a.D ? row[lane + 64 * i] : 0.f;
                ss += x[i] * x[i];
            }
            const float f = scale / sqrtf(wave_sum(ss) + a.unit_eps);
#pragma unroll
            for (int i = 0; i < STEP_MAX_D / 64; ++i)
                if (lane + 64 * i < a.D) to[place(lane + 64 * i)] = x[i] * f;
        }
        for (int d = a.D + lane; d < STEP_MAX_D; d += 64) to[place(d)] = 0.f;
    } else if (wave == 2 && lane == 0) {
        if (MODE == STEP_DELTA) {
            const size_t i = (size_t)t * a.ld_b + h;
            beta_s = 1.0f / (1.0f + expf(-a.beta[i]));
            const float z = a.a[i] + a.dt_bias[h];
            const float sp_ = z > 20.0f ? z : log1pf(expf(z));
            decay_s = expf(-expf(a.a_log[h]) * sp_);
        } else {
            decay_s = a.decay[h];
        }
    }
    // the gate and the norm's weight, by the wave that will need them
    float gt[NC], wt[NC];
#pragma unroll
    for (int n = 0; n < NC; ++n) {
        const int c = lane + 64 * n;
        const bool in = wave == 0 && c < a.Dv;
        gt[n] = in ? a.gate[(size_t)t * a.ld_g + (size_t)h * a.Dv + c] : 0.f;
        wt[n] = in && a.w ? a.w[(a.w_full ? (size_t)h * a.Dv : 0) + c] : 1.f;
    }
    __syncthreads();
    const float dec = decay_s, bt = MODE == STEP_DELTA ? beta_s : 0.f;
    float q[DPER], k[DPER];
#pragma unroll
    for (int j = 0; j < DPER; j += 4) {
        const float4 x = *reinterpret_cast<const float4*>(qf + r * DPER + j), y = *reinterpret_cast<const float4*>(kf + r * DPER + j);
        q[j] = x.x; q[j + 1] = x.y; q[j + 2] = x.z; q[j + 3] = x.w;
        k[j] = y.x; k[j + 1] = y.y; k[j + 2] = y.z; k[j + 3] = y.w;
    }
#pragma unroll
    for (int n = 0; n < NC; ++n) {
        const int c = c0 + 64 * n;
        float u = vv[n];
        if (MODE == STEP_DELTA) {
            float d0 = 0.f, d1 = 0.f;
#pragma unroll
            for (int j = 0; j < DPER; j += 2) { d0 = fmaf(S[n][j], k[j], d0); d1 = fmaf(S[n][j + 1], k[j + 1], d1); }
            u = bt * (u - dec * sum_of_16(d0 + d1));            // S^T k of the decayed state = g (S^T k)
        }
        float o0 = 0.f, o1 = 0.f;
#pragma unroll
        for (int j = 0; j < DPER; j += 2) {
            S[n][j] = fmaf(dec, S[n][j], k[j] * u);
            S[n][j + 1] = fmaf(dec, S[n][j + 1], k[j + 1] * u);
            o0 = fmaf(S[n][j], q[j], o0);
            o1 = fmaf(S[n][j + 1], q[j + 1], o1);
        }
        const float o = sum_of_16(o0 + o1);
        if (c < a.Dv) {
            if (r == 0) of[c] = o;
#pragma unroll
            for (int j = 0; j < DPER; ++j)
                if (j < J) sp[((size_t)j * a.Dv + c) * 16 + r] = S[n][j];
        }
    }
    __syncthreads();
    if (wave > 0) return;
    float x[NC], ss = 0.f;
#pragma unroll
    for (int n = 0; n < NC; ++n) {
        x[n] = lane + 64 * n < a.Dv ? of[lane + 64 * n] : 0.f;
        ss += x[n] * x[n];
    }
    const float rinv = 1.0f / sqrtf(wave_sum(ss) / (float)a.Dv + a.eps);
#pragma unroll
    for (int n = 0; n < NC; ++n) {
        const int c = lane + 64 * n;
        if (c >= a.Dv) continue;
        const float sg = 1.0f / (1.0f + expf(-gt[n]));
        st<TO>((TO*)a.out, (size_t)t * a.ld_out + (size_t)h * a.Dv + c, x[n] * rinv * wt[n] * (a.gate_act ? sg : gt[n] * sg));
    }
}

extern "C" int xr_recurrence_step(void* out, const float* q, const float* k, const float* v, float* state, const int* slots, const int* positions,
                                  const float* inv_freq, const float* decay, const float* beta, const float* a, const float* a_log,
                                  const float* dt_bias, const float* gate, const float* w, int B, int H, int G, int D, int Dv, int ld, int ld_b,
                                  int ld_g, int rot, int w_full, int gate_act, float q_scale, float k_scale, float unit_eps, float eps,
                                  int delta, int dtype, hipStream_t stream) {
    XR_REQUIRE(B >= 0 && B < 65536 && H > 0 && G > 0 && H % G == 0, "recurrence_step: bad sizes B=%d H=%d G=%d", B, H, G);
    XR_REQUIRE(D > 32 && D <= STEP_MAX_D && Dv > 0 && Dv <= STEP_MAX_DV, "recurrence_step: heads of %d by %d (33 to %d by 1 to %d)", D, Dv, STEP_MAX_D, STEP_MAX_DV);
    XR_REQUIRE(out && q && k && v && state && slots && gate, "recurrence_step: null operand");
    XR_REQUIRE(delta ? (beta && a && a_log && dt_bias) : decay != nullptr, "recurrence_step: no decays");
    XR_REQUIRE(rot >= 0 && rot <= D && rot % 2 == 0 && (rot == 0 || (!delta && inv_freq && positions)), "recurrence_step: rotary width %d", rot);
    XR_REQUIRE(dtype == XR_F32 || dtype == XR_BF16, "recurrence_step: bad dtype %d", dtype);
    if (B == 0) return XR_OK;
    StepArgs s;
    s.out = out; s.q = q; s.k = k; s.v = v; s.state = state; s.slots = slots; s.positions = positions; s.inv_freq = inv_freq; s.decay = decay;
    s.beta = beta; s.a = a; s.a_log = a_log; s.dt_bias = dt_bias; s.gate = gate; s.w = w;
    s.H = H; s.G = G; s.D = D; s.Dv = Dv; s.ld = ld; s.ld_b = ld_b; s.ld_g = ld_g; s.ld_out = H * Dv; s.rot = rot; s.w_full = w_full; s.gate_act = gate_act;
    s.q_scale = q_scale; s.k_scale = k_scale; s.unit_eps = unit_eps; s.eps = eps;
    const dim3 grid(H, B);
    if (delta) {
        if (dtype == XR_F32) k_recurrence_step<STEP_DELTA, float><<<grid, 1024, 0, stream>>>(s);
        else k_recurrence_step<STEP_DELTA, bf16_t><<<grid, 1024, 0, stream>>>(s);
    } else {
        if (dtype == XR_F32) k_recurrence_step<STEP_RETENTION, float><<<grid, 1024, 0, stream>>>(s);
        else k_recurrence_step<STEP_RETENTION, bf16_t><<<grid, 1024, 0, stream>>>(s);
    }
    XR_CHECK_LAUNCH("recurrence_step");
    return XR_OK;
}
