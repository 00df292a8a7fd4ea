// Row-wise and time-wise operations around the sequence mixers: layer norm, a short causal
// convolution over time with its carried inputs, the PolyNorm activation, a rotation of 32-bit
// projections in place, the gated norm of a recurrent mixer's read-out, and what a gated delta
// rule needs of its projections (unit vectors, write strengths, decays).
//
// All arithmetic is 32-bit; T is the storage type of what comes in or goes out.  A step's rows
// are the tokens of its requests one after another: request b owns rows cu_q[b] .. cu_q[b+1]-1
// and the state row slots[b].
#include "common.h"

// ---------------------------------------------------------------- layer norm
// y = (x - mean) / sqrt(var + eps) * w, var = mean((x - mean)^2); no bias.  One workgroup a row.
// NW waves a row: 4 where there are rows enough to fill the chip, 16 for the few rows of a
// decode step, whose time is the latency of one workgroup's passes over its row.
template <int NW> __device__ inline float block_sum(float v, float* part) {
    v = wave_sum(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
    __syncthreads();
    float t = 0.f;
#pragma unroll
    for (int i = 0; i < NW; ++i) t += part[i];
    return t;
}
#define FEW_ROWS 128
__device__ inline void st4(float* p, float4 v) { *reinterpret_cast<float4*>(p) = v; }
__device__ inline void st4(bf16_t* p, float4 v) { *reinterpret_cast<uint2*>(p) = make_uint2(pack_bf16x2(v.x, v.y), pack_bf16x2(v.z, v.w)); }

template <typename TO, int NW>
__global__ __launch_bounds__(64 * NW) void k_layernorm(TO* __restrict__ out, const float* __restrict__ x,
                                                      const float* __restrict__ w, const int* __restrict__ rows,
                                                      int E, int ldx, float eps) {
    __shared__ float part[NW];
    const int r = blockIdx.x;
    const int src = rows ? rows[r] : r;
    const float* xr = x + (size_t)src * ldx;
    float s = 0.f;
    for (int i = threadIdx.x; i < E; i += 64 * NW) s += xr[i];
    const float mean = block_sum<NW>(s, part) / (float)E;
    float ss = 0.f;
    for (int i = threadIdx.x; i < E; i += 64 * NW) {
        const float d = xr[i] - mean;
        ss += d * d;
    }
    const float rinv = 1.0f / sqrtf(block_sum<NW>(ss, part) / (float)E + eps);
    TO* o = out + (size_t)r * E;
    for (int i = threadIdx.x; i < E; i += 64 * NW) st<TO>(o, i, (xr[i] - mean) * rinv * (w ? w[i] : 1.f));
}

// The same with a row read once: a lane's PER values (the same ones, added in the same order: the same bits) stay in registers
// from the sum to the scaling.  2,048 rows of 4,096 to 32 bits: 13 us, 22 where it was read three times.
template <typename TO, int NW, int PER>
__global__ __launch_bounds__(64 * NW) void k_layernorm_rows(TO* __restrict__ out, const float* __restrict__ x,
                                                           const float* __restrict__ w, const int* __restrict__ rows,
                                                           int E, int ldx, float eps) {
    __shared__ float part[NW];
    const int r = blockIdx.x;
    const float* xr = x + (size_t)(rows ? rows[r] : r) * ldx;
    float v[PER], g[PER];
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        const int i = threadIdx.x + u * 64 * NW;
        v[u] = i < E ? xr[i] : 0.f;
        g[u] = w && i < E ? w[i] : 1.f;
    }
    float s = 0.f;
#pragma unroll
    for (int u = 0; u < PER; ++u) s += v[u];
    const float mean = block_sum<NW>(s, part) / (float)E;
    float ss = 0.f;
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        const float d = v[u] - mean;
        if (threadIdx.x + u * 64 * NW < E) ss += d * d;
    }
    const float rinv = 1.0f / sqrtf(block_sum<NW>(ss, part) / (float)E + eps);
    TO* o = out + (size_t)r * E;
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        const int i = threadIdx.x + u * 64 * NW;
        if (i < E) st<TO>(o, i, (v[u] - mean) * rinv * g[u]);
    }
}

// Rows whose width is a multiple of 4 (up to 4 * 64 NW * NV), to bfloat16: a thread keeps its float4 pieces in registers
// from the sum to the scaling, so that a row is read once.  (32-bit rows stay with the kernel above: k_layernorm_conv sums
// in its order, and a step of single rows must give the same bits with and without it.)
template <int NW, int NV>
__global__ __launch_bounds__(64 * NW) void k_layernorm_v4(bf16_t* __restrict__ out, const float* __restrict__ x,
                                                         const float* __restrict__ w, const int* __restrict__ rows,
                                                         int E, int ldx, float eps) {
    __shared__ float part[NW];
    const int r = blockIdx.x;
    const int src = rows ? rows[r] : r;
    const float4* xr = reinterpret_cast<const float4*>(x + (size_t)src * ldx);
    const float4* w4 = reinterpret_cast<const float4*>(w);
    const int n4 = E >> 2;
    float4 v[NV], g[NV];
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int c = threadIdx.x + i * 64 * NW;
        v[i] = c < n4 ? xr[c] : make_float4(0.f, 0.f, 0.f, 0.f);
        g[i] = (w && c < n4) ? w4[c] : make_float4(1.f, 1.f, 1.f, 1.f);
        s += v[i].x + v[i].y + v[i].z + v[i].w;
    }
    const float mean = block_sum<NW>(s, part) / (float)E;
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        if (threadIdx.x + i * 64 * NW >= n4) continue;
        v[i].x -= mean; v[i].y -= mean; v[i].z -= mean; v[i].w -= mean;
        ss += v[i].x * v[i].x + v[i].y * v[i].y + v[i].z * v[i].z + v[i].w * v[i].w;
    }
    const float rinv = 1.0f / sqrtf(block_sum<NW>(ss, part) / (float)E + eps);
    bf16_t* o = out + (size_t)r * E;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int c = threadIdx.x + i * 64 * NW;
        if (c < n4)
            *reinterpret_cast<uint2*>(o + 4 * c) = make_uint2(pack_bf16x2(v[i].x * rinv * g[i].x, v[i].y * rinv * g[i].y),
                                                              pack_bf16x2(v[i].z * rinv * g[i].z, v[i].w * rinv * g[i].w));
    }
}

extern "C" int xr_layernorm(void* out, const float* x, const float* w, const int* rows, int R, int E, int ldx,
                            float eps, int out_dtype, hipStream_t stream) {
    XR_REQUIRE(R >= 0 && E > 0 && ldx >= E, "layernorm: bad sizes R=%d E=%d ldx=%d", R, E, ldx);
    XR_REQUIRE(eps >= 0.f, "layernorm: eps %g is negative", eps);
    XR_REQUIRE(out_dtype == XR_F32 || out_dtype == XR_BF16, "layernorm: bad dtype %d", out_dtype);
    if (R == 0) return XR_OK;
    const bool few = R <= FEW_ROWS && E >= 1024;
    const bool vec = E % 4 == 0 && ldx % 4 == 0 && ((uintptr_t)x % 16) == 0 && ((uintptr_t)out % 16) == 0 && ((uintptr_t)w % 16) == 0 &&
                     E <= 4 * 256 * 8;
    if (vec && out_dtype == XR_BF16) {
        bf16_t* o = (bf16_t*)out;
        if (few && E <= 4096) k_layernorm_v4<16, 1><<<R, 1024, 0, stream>>>(o, x, w, rows, E, ldx, eps);
        else if (few) k_layernorm_v4<16, 2><<<R, 1024, 0, stream>>>(o, x, w, rows, E, ldx, eps);
        else if (E <= 4 * 256 * 2) k_layernorm_v4<4, 2><<<R, 256, 0, stream>>>(o, x, w, rows, E, ldx, eps);
        else if (E <= 4 * 256 * 4) k_layernorm_v4<4, 4><<<R, 256, 0, stream>>>(o, x, w, rows, E, ldx, eps);
        else k_layernorm_v4<4, 8><<<R, 256, 0, stream>>>(o, x, w, rows, E, ldx, eps);
    } else if (out_dtype == XR_F32) {
        if (few) k_layernorm<float, 16><<<R, 1024, 0, stream>>>((float*)out, x, w, rows, E, ldx, eps);
        else if (E <= 256 * 8) k_layernorm_rows<float, 4, 8><<<R, 256, 0, stream>>>((float*)out, x, w, rows, E, ldx, eps);
        else if (E <= 256 * 16) k_layernorm_rows<float, 4, 16><<<R, 256, 0, stream>>>((float*)out, x, w, rows, E, ldx, eps);
        else if (E <= 256 * 32) k_layernorm_rows<float, 4, 32><<<R, 256, 0, stream>>>((float*)out, x, w, rows, E, ldx, eps);
        else k_layernorm<float, 4><<<R, 256, 0, stream>>>((float*)out, x, w, rows, E, ldx, eps);
    } else {
        if (few) k_layernorm<bf16_t, 16><<<R, 1024, 0, stream>>>((bf16_t*)out, x, w, rows, E, ldx, eps);
        else k_layernorm<bf16_t, 4><<<R, 256, 0, stream>>>((bf16_t*)out, x, w, rows, E, ldx, eps);
    }
    XR_CHECK_LAUNCH("layernorm");
    return XR_OK;
}

// ---------------------------------------------------------------- short causal convolution over time
// y_t[c] = sum_j w[c][j] * u_(t - taps + 1 + j)[c]  (+ bias[c]) (+ u_t[c] with `residual`), then the activation.
// Inputs before a portion's first row come from the request's state row, which holds its last
// taps - 1 inputs, oldest first, and is zero for a request that begins.  Who reads a request's state rewrites it: in a
// step where every request brings one row (`fuse`) a row's own thread, else the threads of the request's first rows
// (k_causal_conv_rows); a kernel of its own (k_conv_state) only where taps are so many that several workgroups read it.
#define CONV_MAX_TAPS 16
#define XR_CONV_NONE 0
#define XR_CONV_SILU 1

template <typename TU, typename TO>
__global__ __launch_bounds__(256) void k_causal_conv(TO* __restrict__ out, const TU* __restrict__ u,
                                                     const float* __restrict__ w, const float* __restrict__ bias, TU* state,
                                                     const int* __restrict__ cu_q, const int* __restrict__ slots,
                                                     const int* __restrict__ req_of_token, int C, int taps, int ld_u,
                                                     int ld_out, int residual, int act, int fuse) {
    const int t = blockIdx.y;
    const int c = blockIdx.x * 256 + threadIdx.x;
    if (c >= C) return;
    const int b = req_of_token[t];
    const int row0 = cu_q[b];
    const int i = t - row0;
    TU* srow = state + (size_t)slots[b] * (taps - 1) * C;
    float acc = 0.f;
    for (int j = 0; j < taps; ++j) {
        const int s = i - (taps - 1) + j;
        const float val = s >= 0 ? ld<TU>(u, (size_t)(row0 + s) * ld_u + c) : ld<TU>(srow, (size_t)(taps - 1 + s) * C + c);
        acc = fmaf(w[(size_t)c * taps + j], val, acc);
        // one row a request: input j of this row is state entry j, which moves one place down
        if (fuse && j > 0) st<TU>(srow, (size_t)(j - 1) * C + c, val);
    }
    if (bias) acc += bias[c];
    if (residual) acc += ld<TU>(u, (size_t)t * ld_u + c);
    if (act == XR_CONV_SILU) acc = acc / (1.0f + expf(-acc));
    st<TO>(out, (size_t)t * ld_out + c, acc);
}

// A lane's sum with another lane's number (DPP), where there is one.
template <int CTRL, int ROWS> __device__ __forceinline__ int plus_lane(int v) { return v + __builtin_amdgcn_update_dpp(0, v, CTRL, ROWS, 0xF, false); }

// A step's rows in blocks of R, none of which holds rows of two requests: block `blk` is block k of request b, which has n rows from row0 on and
// its carried inputs at `slot`.  At most (T + B (R - 1)) / R blocks; false for those past the last.  (Every lane of a wave takes part; requests without rows
// have no block.  All a workgroup needs to know before its first row is one round of loads and a scan between lanes: with the request looked for by
// shuffles, and what it has loaded again behind that, 8 requests of 7 rows took 1.1 us longer.)
struct RowBlock { int b, k, row0, n, slot; };
template <int R> __device__ inline bool rows_of_block(const int* __restrict__ cu_q, const int* __restrict__ slots, int B, int blk, RowBlock& x) {
    if (B == 1) {
        x.b = 0; x.k = blk; x.row0 = cu_q[0]; x.n = cu_q[1] - x.row0; x.slot = slots[0];
        return blk * R < x.n;
    }
    const int lane = threadIdx.x & 63;
    for (int b0 = 0; b0 < B; b0 += 64) {
        const int b = b0 + lane < B ? b0 + lane : B - 1;
        const int row0 = cu_q[b], n = b0 + lane < B ? cu_q[b + 1] - row0 : 0, slot = slots[b], own = (n + R - 1) / R;
        int upto = plus_lane<0x111, 0xF>(own);          // shifts by 1, 2, 4 and 8 lanes inside a row of 16,
        upto = plus_lane<0x112, 0xF>(upto);
        upto = plus_lane<0x114, 0xF>(upto);
        upto = plus_lane<0x118, 0xF>(upto);
        upto = plus_lane<0x142, 0xA>(upto);             // the last lane of rows 0 and 2 to rows 1 and 3,
        upto = plus_lane<0x143, 0xC>(upto);             // that of row 1 to rows 2 and 3
        const int total = __builtin_amdgcn_readlane(upto, 63);
        if (blk < total) {
            const int at = __ffsll((unsigned long long)__ballot(upto > blk)) - 1;
            x.b = b0 + at;
            x.k = blk - __builtin_amdgcn_readlane(upto - own, at);
            x.row0 = __builtin_amdgcn_readlane(row0, at);
            x.n = __builtin_amdgcn_readlane(n, at);
            x.slot = __builtin_amdgcn_readlane(slot, at);
            return true;
        }
        blk -= total;
    }
    return false;
}

// Steps of several rows a request: a thread takes up to CONV_ROWS consecutive rows of its channel, all of one request, so that
// every input is read once; what a row needs before its first input (its request, the request's first row and state row) are loads
// that wait for each other, once a block and not once a row.  The first block of a request is the only one that reads its state (up to
// CONV_ROWS + 1 taps), and writes it anew.  Bound by memory and, for few rows, by that chain.  (Four channels a thread with 16-byte loads was slower:
// 34 us for 26 at 2,048 rows of 2,048 channels.)  2,048 rows of 8,192 channels 24.2 us, and k_conv_state's 4.7 behind it are saved; 17 rows of 2,048
// channels with 5 taps 4.2 (a row a thread and k_conv_state 4.9), 8 requests of 7 rows with 4 taps 4.2 (4.9), 200 rows of 8,192 with 9 taps 7.6 (18).
#define CONV_ROWS 8
// Rows i0 to i0 + CONV_ROWS - 1 of channel c of a request (those that exist; the others' results mean nothing), before the activation; in the
// request's first block also its new carried inputs.  All inputs of the rows are read before the first product, for up to TM taps and for rows that are fewer than a
// block, too (input by input, a row after the other, 17 rows of 2,048 channels with 16 taps took 14.7 us, with 5 6.8).
template <int TM, typename TU>
__device__ __forceinline__ void conv_rows(float (&y)[CONV_ROWS], const TU* __restrict__ u, const float* __restrict__ w, float bias, TU* state, const RowBlock& x,
                                          int i0, int c, int C, int taps, int ld_u, int residual) {
    TU* const srow = state + (size_t)x.slot * (taps - 1) * C;
    const TU* const col = u + (size_t)x.row0 * ld_u + c;
    const int none = TM - taps;                     // places of the window that fewer taps leave unread
    float wt[TM], v[CONV_ROWS + TM - 1];
    // (a channel's weights in whole pieces: number by number the lanes' loads lie `taps` apart, 600 rows of 300 requests, 8,192 channels, 16 taps 128 us; so 83, 2,048 rows of one 79 and 41)
    if (TM % 4 == 0 && taps % 4 == 0 && ((uintptr_t)w & 15) == 0) {
#pragma unroll
        for (int j = 0; j + 3 < TM; j += 4) {
            const float4 f = j >= none ? *reinterpret_cast<const float4*>(w + (size_t)c * taps + j - none) : make_float4(0.f, 0.f, 0.f, 0.f);
            wt[j] = f.x; wt[j + 1] = f.y; wt[j + 2] = f.z; wt[j + 3] = f.w;
        }
    } else {
#pragma unroll
        for (int j = 0; j < TM; ++j) wt[j] = j >= none ? w[(size_t)c * taps + j - none] : 0.f;
    }
#pragma unroll
    for (int m = 0; m < CONV_ROWS + TM - 1; ++m) {
        const int s = i0 + m - (TM - 1);
        v[m] = m < none ? 0.f : s >= 0 ? ld<TU>(col, (size_t)(s < x.n ? s : x.n - 1) * ld_u) : ld<TU>(srow, (size_t)(taps - 1 + s) * C + c);
    }
    const bool carries = i0 == 0 && taps > 1 && taps - 1 <= CONV_ROWS;
    constexpr int KEEP = TM - 1 < CONV_ROWS ? TM - 1 : CONV_ROWS;
    TU keep[KEEP];
    if (carries) {
#pragma unroll
        for (int m = 0; m < KEEP; ++m) {
            const int s = x.n - (taps - 1) + m;
            if (m < taps - 1) keep[m] = s >= 0 ? col[(size_t)s * ld_u] : srow[(size_t)(m + x.n) * C + c];
        }
    }
#pragma unroll
    for (int r = 0; r < CONV_ROWS; ++r) y[r] = 0.f;
#pragma unroll
    for (int j = 0; j < TM; ++j) {
        if (j < none) continue;
#pragma unroll
        for (int r = 0; r < CONV_ROWS; ++r) y[r] = fmaf(wt[j], v[r + j], y[r]);
    }
#pragma unroll
    for (int r = 0; r < CONV_ROWS; ++r) {
        y[r] += bias;
        if (residual) y[r] += v[r + TM - 1];
    }
    if (carries) {
#pragma unroll
        for (int m = 0; m < KEEP; ++m)
            if (m < taps - 1) srow[(size_t)m * C + c] = keep[m];
    }
}

template <int TM, typename TU, typename TO>
__global__ __launch_bounds__(256) void k_causal_conv_rows(TO* __restrict__ out, const TU* __restrict__ u,
                                                          const float* __restrict__ w, const float* __restrict__ bias, TU* state,
                                                          const int* __restrict__ cu_q, const int* __restrict__ slots, int B, int C,
                                                          int taps, int ld_u, int ld_out, int residual, int act) {
    RowBlock x;
    if (!rows_of_block<CONV_ROWS>(cu_q, slots, B, (int)(blockIdx.z * gridDim.y + blockIdx.y), x)) return;
    const int c = blockIdx.x * 256 + threadIdx.x;
    if (c >= C) return;
    const int i0 = x.k * CONV_ROWS;
    float y[CONV_ROWS];
    conv_rows<TM, TU>(y, u, w, bias ? bias[c] : 0.f, state, x, i0, c, C, taps, ld_u, residual);
#pragma unroll
    for (int r = 0; r < CONV_ROWS; ++r) {
        if (i0 + r >= x.n) break;
        st<TO>(out, (size_t)(x.row0 + i0 + r) * ld_out + c, act == XR_CONV_SILU ? y[r] / (1.0f + expf(-y[r])) : y[r]);
    }
}

// The blocks of a step's rows over y and z of a grid, however many they are.
static bool conv_rows_grid(int C, int T, int B, dim3& grid) {
    const long long blocks = ((long long)T + (long long)B * (CONV_ROWS - 1)) / CONV_ROWS, z = (blocks + 65534) / 65535;
    if (blocks > 1 << 27) return false;
    grid = dim3((C + 255) / 256, (unsigned)((blocks + z - 1) / z), (unsigned)z);
    return true;
}

// The convolution of a mixer's queries, keys and values (no bias, no activation) with the store behind it: queries go to q_out, keys and values to the cache pages
// of their positions (K [page][kv head][place][D], V [page][kv head][Dv][place]; Hk 0: none).  A thread's rows of a value are places side by side, one store where they are
// whole and aligned (store8), where a kernel of its own stored 2 bytes a lane 128 apart.  2,048 rows, 6,144 and 4,096 channels:
// 20.9 us on average, as two kernels 21.3 + 17.0; 700 rows of half the width 8.3 (6.5 + 7.9).
__device__ inline void store8(float* p, const float (&y)[CONV_ROWS]) {
    reinterpret_cast<float4*>(p)[0] = make_float4(y[0], y[1], y[2], y[3]);
    reinterpret_cast<float4*>(p)[1] = make_float4(y[4], y[5], y[6], y[7]);
}
__device__ inline void store8(bf16_t* p, const float (&y)[CONV_ROWS]) {
    *reinterpret_cast<uint4*>(p) = make_uint4(pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3]), pack_bf16x2(y[4], y[5]), pack_bf16x2(y[6], y[7]));
}
template <int TM, typename T>
__global__ __launch_bounds__(256) void k_conv_rows_store(T* __restrict__ q_out, T* __restrict__ kc, T* __restrict__ vc, const float* __restrict__ u, int ld,
                                                         const float* __restrict__ w, float* state, const int* __restrict__ cu_q,
                                                         const int* __restrict__ slots, int taps, const int* __restrict__ starts,
                                                         const int* __restrict__ block_table, int table_stride, int B, int Q, int Hk, int D, int Dv,
                                                         int page_shift, int page_mask, int page_size, int wide) {
    RowBlock x;
    if (!rows_of_block<CONV_ROWS>(cu_q, slots, B, (int)(blockIdx.z * gridDim.y + blockIdx.y), x)) return;
    const int C = Q + Hk * (D + Dv), c = blockIdx.x * 256 + threadIdx.x;
    if (c >= C) return;
    const int i0 = x.k * CONV_ROWS, n = x.n, pos = starts[x.b] + i0;
    float y[CONV_ROWS];
    conv_rows<TM, float>(y, u, w, 0.f, state, x, i0, c, C, taps, ld, 0);
    if (c < Q) {
#pragma unroll
        for (int r = 0; r < CONV_ROWS; ++r)
            if (i0 + r < n) st<T>(q_out, (size_t)(x.row0 + i0 + r) * Q + c, y[r]);
        return;
    }
    const int* bt = block_table + (size_t)x.b * table_stride;
    const bool key = c - Q < Hk * D;
    const int i = key ? c - Q : c - Q - Hk * D, size = key ? D : Dv, h = i / size, d = i - h * size;
    if (wide && !key && i0 + CONV_ROWS <= n && pos % CONV_ROWS == 0) {
        store8(vc + (((size_t)bt[pos >> page_shift] * Hk + h) * Dv + d) * page_size + (pos & page_mask), y);
        return;
    }
#pragma unroll
    for (int r = 0; r < CONV_ROWS; ++r) {
        if (i0 + r >= n) break;
        const int page = bt[(pos + r) >> page_shift], off = (pos + r) & page_mask;
        if (key) st<T>(kc, (((size_t)page * Hk + h) * page_size + off) * D + d, y[r]);
        else st<T>(vc, (((size_t)page * Hk + h) * Dv + d) * page_size + off, y[r]);
    }
}

extern "C" int xr_conv_rows_store(void* q_out, void* k_cache, void* v_cache, const float* u, int ld, const float* w, float* state, const int* cu_q,
                                  const int* slots, int taps, const int* starts, const int* block_table, int table_stride, int T, int B, int H,
                                  int Hk, int D, int Dv, int page_size, int dtype, hipStream_t stream) {
    XR_REQUIRE(T >= 0 && B >= 0 && H > 0 && Hk >= 0 && D > 0 && Dv > 0 && taps > 1 && taps - 1 <= CONV_ROWS, "conv_rows_store: bad sizes T=%d B=%d H=%d Hk=%d D=%d Dv=%d taps=%d",
               T, B, H, Hk, D, Dv, taps);
    const int C = H * D + Hk * (D + Dv), shift = ilog2_exact(page_size);
    XR_REQUIRE(shift >= 0 && ld >= C, "conv_rows_store: page size %d, rows %d apart for %d channels", page_size, ld, C);
    XR_REQUIRE(q_out && u && w && state && cu_q && slots && starts && (Hk == 0 || (k_cache && v_cache && block_table)), "conv_rows_store: null operand");
    XR_REQUIRE(dtype == XR_F32 || dtype == XR_BF16, "conv_rows_store: bad dtype %d", dtype);
    if (T == 0 || B == 0) return XR_OK;
    dim3 grid;
    XR_REQUIRE(conv_rows_grid(C, T, B, grid), "conv_rows_store: %d rows of %d requests", T, B);
    const int wide = page_size % CONV_ROWS == 0 && ((uintptr_t)v_cache & 15) == 0;      // (a value's eight places are 16 bytes or 32 behind one another)
#define CRS(T_) (taps <= 4 ? k_conv_rows_store<4, T_> : k_conv_rows_store<CONV_ROWS + 1, T_>)<<<grid, 256, 0, stream>>>((T_*)q_out, (T_*)k_cache, (T_*)v_cache, u, ld, w, state, cu_q, slots, taps, starts, block_table, \
                                                               table_stride, B, H * D, Hk, D, Dv, shift, page_size - 1, page_size, wide)
    if (dtype == XR_F32) CRS(float);
    else CRS(bf16_t);
#undef CRS
    XR_CHECK_LAUNCH("conv_rows_store");
    return XR_OK;
}

template <typename TU>
__global__ __launch_bounds__(256) void k_conv_state(TU* __restrict__ state, const TU* __restrict__ u,
                                                    const int* __restrict__ cu_q, const int* __restrict__ slots,
                                                    int C, int taps, int ld_u) {
    const int b = blockIdx.y;
    const int c = blockIdx.x * 256 + threadIdx.x;
    if (c >= C) return;
    const int row0 = cu_q[b], n = cu_q[b + 1] - row0;
    if (n <= 0) return;
    TU* srow = state + (size_t)slots[b] * (taps - 1) * C;
    TU keep[CONV_MAX_TAPS];
#pragma unroll
    for (int m = 0; m < CONV_MAX_TAPS; ++m) {
        if (m >= taps - 1) break;
        const int s = n - (taps - 1) + m;
        keep[m] = s >= 0 ? u[(size_t)(row0 + s) * ld_u + c] : srow[(size_t)(m + n) * C + c];
    }
#pragma unroll
    for (int m = 0; m < CONV_MAX_TAPS; ++m) {
        if (m >= taps - 1) break;
        srow[(size_t)m * C + c] = keep[m];
    }
}

extern "C" int xr_causal_conv(void* out, const void* u, const float* w, const float* bias, void* state, const int* cu_q, const int* slots,
                              const int* req_of_token, int T, int B, int C, int taps, int ld_u, int ld_out,
                              int u_dtype, int out_dtype, int residual, int act, int one_row_each, hipStream_t stream) {
    XR_REQUIRE(T >= 0 && B >= 0 && C > 0 && ld_u >= C && ld_out >= C, "causal_conv: bad sizes T=%d B=%d C=%d ld_u=%d ld_out=%d",
               T, B, C, ld_u, ld_out);
    XR_REQUIRE(taps >= 1 && taps <= CONV_MAX_TAPS, "causal_conv: %d taps (1 to %d)", taps, CONV_MAX_TAPS);
    XR_REQUIRE(act == XR_CONV_NONE || act == XR_CONV_SILU, "causal_conv: activation code %d", act);
    XR_REQUIRE(out != u, "causal_conv: the result cannot overwrite its input");
    XR_REQUIRE(taps == 1 || state != nullptr, "causal_conv: a convolution of %d taps needs its state", taps);
    XR_REQUIRE(!one_row_each || T == B, "causal_conv: %d rows of %d requests are not one row each", T, B);
    if (T == 0 || B == 0) return XR_OK;
    const int fuse = one_row_each && taps > 1 ? 1 : 0;
    dim3 grid((C + 255) / 256, T), sgrid((C + 255) / 256, B), rgrid;
    // Taps whose carried inputs a kernel of its own moves on: few rows go a row a thread, more of them side by side (17 rows of
    // 2,048 channels, 16 taps 9.5 us and 8.1 a row a thread; 200 rows of 8,192 16.4 and more than 25)
    const bool pair = taps - 1 > CONV_ROWS && T < 64;
    XR_REQUIRE(one_row_each ? T <= 65535 : conv_rows_grid(C, T, B, rgrid) && (taps - 1 <= CONV_ROWS || B <= 65535), "causal_conv: %d rows of %d requests", T, B);
#define CC(TU, TO)                                                                                                   \
    do {                                                                                                             \
        if (one_row_each) {                                                                                          \
            k_causal_conv<TU, TO><<<grid, 256, 0, stream>>>((TO*)out, (const TU*)u, w, bias, (TU*)state, cu_q, slots, \
                                                            req_of_token, C, taps, ld_u, ld_out, residual, act, fuse); \
            break;                                                                                                   \
        }                                                                                                            \
        if (pair) {                                                                                                  \
            k_causal_conv<TU, TO><<<grid, 256, 0, stream>>>((TO*)out, (const TU*)u, w, bias, (TU*)state, cu_q, slots, \
                                                            req_of_token, C, taps, ld_u, ld_out, residual, act, 0);  \
        } else                                                                                                       \
        (taps <= 4 ? k_causal_conv_rows<4, TU, TO> : taps <= CONV_ROWS + 1 ? k_causal_conv_rows<CONV_ROWS + 1, TU, TO> : k_causal_conv_rows<CONV_MAX_TAPS, TU, TO>)<<<rgrid, 256, 0, stream>>>((TO*)out, (const TU*)u, w, bias, (TU*)state, cu_q, slots, B, C, taps, \
                                                              ld_u, ld_out, residual, act);                          \
        if (taps - 1 > CONV_ROWS)                                                                                    \
            k_conv_state<TU><<<sgrid, 256, 0, stream>>>((TU*)state, (const TU*)u, cu_q, slots, C, taps, ld_u);       \
    } while (0)
    if (u_dtype == XR_F32 && out_dtype == XR_F32) CC(float, float);
    else if (u_dtype == XR_F32 && out_dtype == XR_BF16) CC(float, bf16_t);
    else if (u_dtype == XR_BF16 && out_dtype == XR_BF16) CC(bf16_t, bf16_t);
    else if (u_dtype == XR_BF16 && out_dtype == XR_F32) CC(bf16_t, float);
    else { xr_set_error("causal_conv: bad dtypes %d %d", u_dtype, out_dtype); return XR_BAD_ARG; }
#undef CC
    XR_CHECK_LAUNCH("causal_conv");
    return XR_OK;
}

// ---------------------------------------------------------------- mixes of a row with the row before it
// out[t][s][c] = h[t][c] + (h[t-1][c] - h[t][c]) * mu[s][c] for n mixes s ("token shift"); the row before a
// portion's first row is the request's state row (zero for a request that begins), which afterwards holds
// the portion's last row.  As for the convolution above, a second kernel rewrites the state once every row
// has been read, and in a step of one row a request (`fuse`) the row's own thread does.
template <typename TO>
__global__ __launch_bounds__(256) void k_token_shift(TO* __restrict__ out, const float* __restrict__ h,
                                                     const float* __restrict__ mu, float* state,
                                                     const int* __restrict__ cu_q, const int* __restrict__ slots,
                                                     const int* __restrict__ req_of_token, int E, int n, int ld_h, int fuse) {
    const int t = blockIdx.y;
    const int c = blockIdx.x * 256 + threadIdx.x;
    if (c >= E) return;
    const int b = req_of_token[t];
    const bool first = t == cu_q[b];
    float* srow = state + (size_t)slots[b] * E;
    const float cur = h[(size_t)t * ld_h + c];
    const float before = first ? srow[c] : h[(size_t)(t - 1) * ld_h + c];
    const float d = before - cur;
    for (int s = 0; s < n; ++s) st<TO>(out, ((size_t)t * n + s) * E + c, fmaf(d, mu[(size_t)s * E + c], cur));
    if (fuse) srow[c] = cur;
}

__global__ __launch_bounds__(256) void k_shift_state(float* __restrict__ state, const float* __restrict__ h,
                                                     const int* __restrict__ cu_q, const int* __restrict__ slots, int E, int ld_h) {
    const int b = blockIdx.y;
    const int c = blockIdx.x * 256 + threadIdx.x;
    if (c >= E) return;
    const int end = cu_q[b + 1];
    if (end <= cu_q[b]) return;
    state[(size_t)slots[b] * E + c] = h[(size_t)(end - 1) * ld_h + c];
}

extern "C" int xr_token_shift(void* out, const float* h, const float* mu, float* state, const int* cu_q, const int* slots,
                              const int* req_of_token, int T, int B, int E, int n, int ld_h, int out_dtype, int one_row_each,
                              hipStream_t stream) {
    XR_REQUIRE(T >= 0 && B >= 0 && E > 0 && n > 0 && ld_h >= E, "token_shift: bad sizes T=%d B=%d E=%d n=%d ld=%d", T, B, E, n, ld_h);
    XR_REQUIRE(out && h && mu && state && cu_q && slots && req_of_token, "token_shift: a pointer is missing");
    XR_REQUIRE(!one_row_each || T == B, "token_shift: %d rows of %d requests are not one row each", T, B);
    XR_REQUIRE(out_dtype == XR_F32 || out_dtype == XR_BF16, "token_shift: bad dtype %d", out_dtype);
    if (T == 0 || B == 0) return XR_OK;
    const int fuse = one_row_each ? 1 : 0;
    const dim3 grid((E + 255) / 256, T), sgrid((E + 255) / 256, B);
    if (out_dtype == XR_F32) k_token_shift<float><<<grid, 256, 0, stream>>>((float*)out, h, mu, state, cu_q, slots, req_of_token, E, n, ld_h, fuse);
    else k_token_shift<bf16_t><<<grid, 256, 0, stream>>>((bf16_t*)out, h, mu, state, cu_q, slots, req_of_token, E, n, ld_h, fuse);
    if (!fuse) k_shift_state<<<sgrid, 256, 0, stream>>>(state, h, cu_q, slots, E, ld_h);
    XR_CHECK_LAUNCH("token_shift");
    return XR_OK;
}

// Layer norm and the convolution behind it in one kernel, for a step in which every request
// brings one row: row b is request b's, its convolution reads the request's carried inputs and
// the row itself, and the thread that owns a channel moves that channel's carried inputs on.
//   h = layernorm(x);  y = h + sum_j cw[:, j] * (carried_j, ..., h);  carried <- (carried_1.., h)
template <typename TO, int NW>
__global__ __launch_bounds__(64 * NW) void k_layernorm_conv(TO* __restrict__ out, const float* __restrict__ x,
                                                           const float* __restrict__ w, const float* __restrict__ cw,
                                                           float* state, const int* __restrict__ slots, int E, int ldx,
                                                           int taps, float eps) {
    __shared__ float part[NW];
    const int r = blockIdx.x;
    const float* xr = x + (size_t)r * ldx;
    float s = 0.f;
    for (int i = threadIdx.x; i < E; i += 64 * NW) s += xr[i];
    const float mean = block_sum<NW>(s, part) / (float)E;
    float ss = 0.f;
    for (int i = threadIdx.x; i < E; i += 64 * NW) {
        const float d = xr[i] - mean;
        ss += d * d;
    }
    const float rinv = 1.0f / sqrtf(block_sum<NW>(ss, part) / (float)E + eps);
    float* srow = state + (size_t)slots[r] * (taps - 1) * E;
    TO* o = out + (size_t)r * E;
    for (int i = threadIdx.x; i < E; i += 64 * NW) {
        const float h = (xr[i] - mean) * rinv * (w ? w[i] : 1.f);
        float acc = 0.f;
        for (int j = 0; j < taps - 1; ++j) {
            const float val = srow[(size_t)j * E + i];
            acc = fmaf(cw[(size_t)i * taps + j], val, acc);
            if (j > 0) srow[(size_t)(j - 1) * E + i] = val;
        }
        acc = fmaf(cw[(size_t)i * taps + taps - 1], h, acc);
        if (taps > 1) srow[(size_t)(taps - 2) * E + i] = h;
        st<TO>(o, i, acc + h);
    }
}

// The same for four taps with everything fetched before the row's sums (a lane's PER channels: the row, its weights and taps, the
// carried inputs; the same bits): a carried input's store kept the next one's load waiting, three trips to memory a channel
// behind the two sums.  Eight rows of 2,048: 4.4 us, 7.1 with the stores between the loads.
template <typename TO, int NW, int PER>
__global__ __launch_bounds__(64 * NW) void k_layernorm_conv4(TO* __restrict__ out, const float* __restrict__ x,
                                                            const float* __restrict__ w, const float* __restrict__ cw,
                                                            float* state, const int* __restrict__ slots, int E, int ldx, float eps) {
    __shared__ float part[NW];
    const int r = blockIdx.x;
    const float* xr = x + (size_t)r * ldx;
    float* srow = state + (size_t)slots[r] * 3 * E;
    float v[PER], g[PER], c[PER][3];
    float4 t[PER];
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        const int i = threadIdx.x + u * 64 * NW, at = i < E ? i : 0;
        v[u] = i < E ? xr[at] : 0.f;
        g[u] = w ? w[at] : 1.f;
        t[u] = *reinterpret_cast<const float4*>(cw + (size_t)at * 4);
#pragma unroll
        for (int j = 0; j < 3; ++j) c[u][j] = srow[(size_t)j * E + at];
    }
    float s = 0.f;
#pragma unroll
    for (int u = 0; u < PER; ++u) s += v[u];
    const float mean = block_sum<NW>(s, part) / (float)E;
    float ss = 0.f;
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        const float d = v[u] - mean;
        if (threadIdx.x + u * 64 * NW < E) ss += d * d;
    }
    const float rinv = 1.0f / sqrtf(block_sum<NW>(ss, part) / (float)E + eps);
    TO* o = out + (size_t)r * E;
#pragma unroll
    for (int u = 0; u < PER; ++u) {
#pragma clang fp contract(off)      // (h is rounded before it is added, as where the norm's kernel stores it)
        const int i = threadIdx.x + u * 64 * NW;
        if (i >= E) continue;
        const float h = (v[u] - mean) * rinv * g[u];
        float acc = fmaf(t[u].x, c[u][0], 0.f);
        acc = fmaf(t[u].y, c[u][1], acc);
        acc = fmaf(t[u].z, c[u][2], acc);
        acc = fmaf(t[u].w, h, acc);
        srow[i] = c[u][1];
        srow[(size_t)E + i] = c[u][2];
        srow[(size_t)2 * E + i] = h;
        st<TO>(o, i, acc + h);
    }
}

template <typename TO>
static bool launch_layernorm_conv4(TO* out, const float* x, const float* w, const float* cw, float* state, const int* slots, int R, int E,
                                   int ldx, int taps, float eps, hipStream_t stream) {
    if (taps != 4 || ((uintptr_t)cw % 16) || E < 1024 || E > 1024 * 8 || R > FEW_ROWS) return false;
    if (E <= 1024 * 2) k_layernorm_conv4<TO, 16, 2><<<R, 1024, 0, stream>>>(out, x, w, cw, state, slots, E, ldx, eps);
    else if (E <= 1024 * 4) k_layernorm_conv4<TO, 16, 4><<<R, 1024, 0, stream>>>(out, x, w, cw, state, slots, E, ldx, eps);
    else k_layernorm_conv4<TO, 16, 8><<<R, 1024, 0, stream>>>(out, x, w, cw, state, slots, E, ldx, eps);
    return true;
}

extern "C" int xr_layernorm_conv(void* out, const float* x, const float* w, const float* cw, float* state,
                                 const int* slots, int R, int E, int ldx, int taps, float eps, int out_dtype,
                                 hipStream_t stream) {
    XR_REQUIRE(R >= 0 && E > 0 && ldx >= E, "layernorm_conv: bad sizes R=%d E=%d ldx=%d", R, E, ldx);
    XR_REQUIRE(taps >= 1 && taps <= CONV_MAX_TAPS && cw && slots && (taps == 1 || state), "layernorm_conv: %d taps, or an operand is missing", taps);
    XR_REQUIRE(out_dtype == XR_F32 || out_dtype == XR_BF16, "layernorm_conv: bad dtype %d", out_dtype);
    if (R == 0) return XR_OK;
    const bool few = R <= FEW_ROWS && E >= 1024;
    if (out_dtype == XR_F32) {
        if (launch_layernorm_conv4<float>((float*)out, x, w, cw, state, slots, R, E, ldx, taps, eps, stream)) {}
        else if (few) k_layernorm_conv<float, 16><<<R, 1024, 0, stream>>>((float*)out, x, w, cw, state, slots, E, ldx, taps, eps);
        else k_layernorm_conv<float, 4><<<R, 256, 0, stream>>>((float*)out, x, w, cw, state, slots, E, ldx, taps, eps);
    } else {
        if (launch_layernorm_conv4<bf16_t>((bf16_t*)out, x, w, cw, state, slots, R, E, ldx, taps, eps, stream)) {}
        else if (few) k_layernorm_conv<bf16_t, 16><<<R, 1024, 0, stream>>>((bf16_t*)out, x, w, cw, state, slots, E, ldx, taps, eps);
        else k_layernorm_conv<bf16_t, 4><<<R, 256, 0, stream>>>((bf16_t*)out, x, w, cw, state, slots, E, ldx, taps, eps);
    }
    XR_CHECK_LAUNCH("layernorm_conv");
    return XR_OK;
}

// Layer norm and the convolution behind it (2 to 4 taps) for steps of several rows a request: a workgroup takes LNC_ROWS rows of one request and the
// three before them, a thread 4 channels of all eight, which stay in its registers from the one read through both sums to the convolution: the
// normed rows never go to memory.  A request's first workgroup alone reads the carried inputs; with no rows before its own it takes the portion's last three
// in their place, which become the new ones.  Neighbouring workgroups, which share three rows, run on one XCD.  Bound by memory: a row comes 8 / LNC_ROWS
// times, from L2 all but once, and goes once; and by a workgroup's two sums, one behind the other.  2,048 rows of 4,096 23 us, where k_layernorm_rows, k_causal_conv_rows and
// k_conv_state took 32; 700 rows of 2,048 6.9 (13.3), 33 rows of 4,096 9.3 (9.7; with loads that waited for one another 10.1, and weights of two taps loaded one by one 12.2).  A wave a row for the sums and every row read again for the convolution: 40.8.
// (Up to 4,096 channels: with 8 a thread the registers do not suffice.)
#define LNC_ROWS 5
#define LNC_HELD (LNC_ROWS + 3)

// The workgroup's sums of eight numbers a thread, the lane % 8-th of them in a lane: halves of the numbers change lanes, so that ten
// exchanges serve all eight.  (Whoever made its eight means and deviations in every thread would spend more on them than on its rows.)
template <int NW> __device__ inline float sums_of_8(float (&s)[8], float (*part)[16]) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int w = 4, bit = 32; w > 0; w >>= 1, bit >>= 1) {
        const bool up = lane & bit;
#pragma unroll
        for (int i = 0; i < w; ++i) {
            const float keep = up ? s[i + w] : s[i], send = up ? s[i] : s[i + w];
            s[i] = keep + __shfl_xor(send, bit, 64);
        }
    }
    float t = s[0];
    t += __shfl_xor(t, 4, 64);
    t += __shfl_xor(t, 2, 64);
    t += __shfl_xor(t, 1, 64);
    __syncthreads();
    if ((lane & 7) == 0) part[lane >> 3][wave] = t;
    __syncthreads();
    float u = 0.f;
#pragma unroll
    for (int w = 0; w < NW; w += 4) {
        const float4 p = *reinterpret_cast<const float4*>(&part[lane & 7][w]);
        u += (p.x + p.y) + (p.z + p.w);
    }
    return u;
}
__device__ inline float of_lane(float v, int lane) { return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), lane)); }
__device__ inline float4 pick(bool first, float4 a, float4 b) {
    return make_float4(first ? a.x : b.x, first ? a.y : b.y, first ? a.z : b.z, first ? a.w : b.w);
}

// The weights of four channels that lie behind one another, taps from the right, in as many 16-byte pieces as there are taps.
template <int N> __device__ __forceinline__ void tap_weights(float (&wt)[4][4], const float* cw) {
    float f[4 * N];
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const float4 t = reinterpret_cast<const float4*>(cw)[i];
        f[4 * i] = t.x; f[4 * i + 1] = t.y; f[4 * i + 2] = t.z; f[4 * i + 3] = t.w;
    }
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
        for (int j = 0; j < 4; ++j) wt[d][j] = j + N >= 4 ? f[d * N + j + N - 4] : 0.f;
}

template <typename TO, int NW, int TAPS>
__global__ __launch_bounds__(64 * NW, 4) void k_layernorm_conv_rows(TO* __restrict__ out, const float* __restrict__ x,
                                                                 const float* __restrict__ w, const float* __restrict__ cw,
                                                                 float* state, const int* __restrict__ cu_q,
                                                                 const int* __restrict__ slots, int B, int E, int ldx, float eps) {
#pragma clang fp contract(off)      // (a normed row is rounded before it is added, as where the norm's kernel stores it)
    __shared__ __align__(16) float part[8][16];
    RowBlock blk;
    const int share = (int)gridDim.x >> 3;              // (the grid is a multiple of 8: an XCD takes an eighth of the blocks, in order)
    if (!rows_of_block<LNC_ROWS>(cu_q, slots, B, ((int)blockIdx.x & 7) * share + ((int)blockIdx.x >> 3), blk)) return;
    const int row0 = blk.row0, n = blk.n, k = blk.k, i0 = k * LNC_ROWS;
    const int c = threadIdx.x * 4;
    const int cs = c < E ? c : 0;
    float4 h[LNC_HELD];                                 // the rows; then without their mean, normed, as the convolution reads them
    auto row_of = [&](int m) { return k == 0 && m < 3 ? n - 3 + m : i0 - 3 + m; };
#pragma unroll
    for (int m = 0; m < LNC_HELD; ++m) {                // (from some row and column in any case, so that no load waits for another)
        const int i = row_of(m);
        h[m] = *reinterpret_cast<const float4*>(x + (size_t)(row0 + (i < 0 ? 0 : i < n ? i : n - 1)) * ldx + cs);
    }
    const float4 gw = w ? *reinterpret_cast<const float4*>(w + cs) : make_float4(1.f, 1.f, 1.f, 1.f);
    float wt[4][4];                                 // channel, tap (the last is the row itself)
    tap_weights<TAPS>(wt, cw + (size_t)cs * TAPS);
#pragma unroll
    for (int m = 0; m < LNC_HELD; ++m) {
        const bool in = c < E && row_of(m) >= 0 && row_of(m) < n;
        h[m] = pick(in, h[m], make_float4(0.f, 0.f, 0.f, 0.f));
    }
    float s[8];
#pragma unroll
    for (int m = 0; m < 8; ++m) s[m] = (h[m].x + h[m].y) + (h[m].z + h[m].w);
    const float mean = sums_of_8<NW>(s, part) / (float)E;
#pragma unroll
    for (int m = 0; m < 8; ++m) {
        const float mu = of_lane(mean, m);
        float4& d = h[m];
        d.x -= mu; d.y -= mu; d.z -= mu; d.w -= mu;
        s[m] = c < E ? fmaf(d.x, d.x, d.y * d.y) + fmaf(d.z, d.z, d.w * d.w) : 0.f;
    }
    const float rinv = 1.0f / sqrtf(sums_of_8<NW>(s, part) / (float)E + eps);
#pragma unroll
    for (int m = 0; m < 8; ++m) s[m] = of_lane(rinv, m);        // (here, where all lanes are: below, rinv would be made in those that go on)
    float* const srow = state + (size_t)blk.slot * (TAPS - 1) * E;
    if (c >= E) return;
#pragma unroll
    for (int m = 0; m < LNC_HELD; ++m) h[m] = make_float4(h[m].x * s[m] * gw.x, h[m].y * s[m] * gw.y, h[m].z * s[m] * gw.z, h[m].w * s[m] * gw.w);
    if (k == 0) {
        // (rows -3 to -1 are carried inputs TAPS - 4 to TAPS - 2, if there are so many; new input m of 3 is row n - 3 + m, or an old one)
        float4 old[3], last[3];
#pragma unroll
        for (int m = 0; m < 3; ++m)
            old[m] = m + TAPS >= 4 ? *reinterpret_cast<const float4*>(srow + (size_t)(m + TAPS - 4) * E + c) : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int m = 0; m < 3; ++m) last[m] = pick(n >= 3 - m, h[m], pick(m + n == 1, old[1], old[2]));      // (n < 3 - m, n >= 1: m + n is 1 or 2)
#pragma unroll
        for (int m = 0; m < 3; ++m) h[m] = old[m];
#pragma unroll
        for (int m = 0; m < 3; ++m)
            if (m + TAPS >= 4) *reinterpret_cast<float4*>(srow + (size_t)(m + TAPS - 4) * E + c) = last[m];
    }
#pragma unroll
    for (int r = 0; r < LNC_ROWS; ++r) {
        float y[4];
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            auto at = [&](int m) { return d == 0 ? h[m].x : d == 1 ? h[m].y : d == 2 ? h[m].z : h[m].w; };
            float acc = 0.f;
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (j + TAPS >= 4) acc = fmaf(wt[d][j], at(r + j), acc);
            y[d] = acc + at(r + 3);
        }
        if (i0 + r < n) st4(out + (size_t)(row0 + i0 + r) * E + c, make_float4(y[0], y[1], y[2], y[3]));
    }
}

// Row b's request brings rows cu_q[b] .. cu_q[b + 1] - 1 of the T; its carried inputs are row slots[b] of state [., taps - 1, E].
extern "C" int xr_layernorm_conv_rows(void* out, const float* x, const float* w, const float* cw, float* state, const int* cu_q, const int* slots,
                                      int T, int B, int E, int ldx, int taps, float eps, int out_dtype, hipStream_t stream) {
    XR_REQUIRE(T >= 0 && B >= 0 && E > 0 && E % 4 == 0 && E <= 4096 && ldx >= E && ldx % 4 == 0, "layernorm_conv: bad sizes T=%d B=%d E=%d ldx=%d", T, B, E, ldx);
    XR_REQUIRE(taps >= 2 && taps <= 4 && x && cw && state && cu_q && slots && out, "layernorm_conv: %d taps (2 to 4), or an operand is missing", taps);
    XR_REQUIRE((((uintptr_t)out | (uintptr_t)x | (uintptr_t)w | (uintptr_t)state | (uintptr_t)cw) & 15) == 0, "layernorm_conv: operands must be 16-byte aligned");
    XR_REQUIRE(out_dtype == XR_F32 || out_dtype == XR_BF16, "layernorm_conv: bad dtype %d", out_dtype);
    if (T == 0 || B == 0) return XR_OK;
    const unsigned blocks = (unsigned)(((long long)T + (long long)B * (LNC_ROWS - 1)) / LNC_ROWS + 7) / 8 * 8;
#define LNC(TO, NW) (taps == 4 ? k_layernorm_conv_rows<TO, NW, 4> : taps == 3 ? k_layernorm_conv_rows<TO, NW, 3> : k_layernorm_conv_rows<TO, NW, 2>)<<<blocks, 64 * NW, 0, stream>>>((TO*)out, x, w, cw, state, cu_q, slots, B, E, ldx, eps)
#define LNCS(TO) do { if (E <= 2048) LNC(TO, 8); else LNC(TO, 16); } while (0)
    if (out_dtype == XR_F32) LNCS(float);
    else LNCS(bf16_t);
#undef LNCS
#undef LNC
    XR_CHECK_LAUNCH("layernorm_conv_rows");
    return XR_OK;
}

// ---------------------------------------------------------------- PolyNorm
// y = a N(z) + b N(z^2) + c N(z^3) + e, powers element by element, N(v) = v / sqrt(mean(v^2) + eps)
// over the row.  One workgroup a row: the three sums in one pass, the result in a second.
template <typename TZ, typename TO, int NW>
__global__ __launch_bounds__(64 * NW) void k_polynorm(TO* __restrict__ out, const TZ* __restrict__ z,
                                                     const float* __restrict__ coef, int F, int ld_z, float eps) {
    __shared__ float part[NW];
    const TZ* zr = z + (size_t)blockIdx.x * ld_z;
    float s2 = 0.f, s4 = 0.f, s6 = 0.f;
    for (int i = threadIdx.x; i < F; i += 64 * NW) {
        const float v = ld<TZ>(zr, i), v2 = v * v, v3 = v2 * v;
        s2 += v2;
        s4 += v2 * v2;
        s6 += v3 * v3;
    }
    const float inv = 1.0f / (float)F;
    const float r1 = coef[0] / sqrtf(block_sum<NW>(s2, part) * inv + eps);
    const float r2 = coef[1] / sqrtf(block_sum<NW>(s4, part) * inv + eps);
    const float r3 = coef[2] / sqrtf(block_sum<NW>(s6, part) * inv + eps);
    const float e = coef[3];
    TO* o = out + (size_t)blockIdx.x * F;
    for (int i = threadIdx.x; i < F; i += 64 * NW) {
        const float v = ld<TZ>(zr, i), v2 = v * v;
        st<TO>(o, i, v * r1 + v2 * r2 + v2 * v * r3 + e);
    }
}

// The same where rows come in aligned fours: a row is read once and stays in registers (N4 fours a lane) between its sums and its
// values, the three sums meet at one barrier.  Bound by memory: 2,048 rows of 21,504 (264 MB) in 50 us,
// 100 where a row was read twice, once for its sums and once for its values.
__device__ inline float4 ld4(const float* p) { return *reinterpret_cast<const float4*>(p); }
__device__ inline float4 ld4(const bf16_t* p) {
    const uint2 u = *reinterpret_cast<const uint2*>(p);
    return make_float4(__uint_as_float(u.x << 16), __uint_as_float(u.x & 0xffff0000u), __uint_as_float(u.y << 16), __uint_as_float(u.y & 0xffff0000u));
}

// AGAIN: squares and cubes are made again.  Kept from the sums, they take two registers more a value, and a compute unit then has room for one row of more
// than 8,192 numbers instead of two or more; where it has one to work on anyway, making them again is the longer way.
template <typename TZ, typename TO, int NW, int N4, bool AGAIN>
__global__ __launch_bounds__(64 * NW) void k_polynorm_v4(TO* __restrict__ out, const TZ* __restrict__ z, const float* __restrict__ coef,
                                                         int F, int ld_z, float eps) {
    __shared__ float part[3][NW];
    const TZ* zr = z + (size_t)blockIdx.x * ld_z;
    float4 v[N4];
#pragma unroll
    for (int u = 0; u < N4; ++u) {
        const int i = (threadIdx.x + u * 64 * NW) * 4;
        v[u] = i < F ? ld4(zr + i) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
    float s2 = 0.f, s4 = 0.f, s6 = 0.f;
    auto add = [&](float x) {
        const float x2 = x * x, x3 = x2 * x;
        s2 += x2;
        s4 += x2 * x2;
        s6 += x3 * x3;
    };
#pragma unroll
    for (int u = 0; u < N4; ++u) { add(v[u].x); add(v[u].y); add(v[u].z); add(v[u].w); }
    s2 = wave_sum(s2);
    s4 = wave_sum(s4);
    s6 = wave_sum(s6);
    if ((threadIdx.x & 63) == 0) { part[0][threadIdx.x >> 6] = s2; part[1][threadIdx.x >> 6] = s4; part[2][threadIdx.x >> 6] = s6; }
    __syncthreads();
    s2 = s4 = s6 = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) { s2 += part[0][w]; s4 += part[1][w]; s6 += part[2][w]; }
    const float inv = 1.0f / (float)F;
    const float r1 = coef[0] / sqrtf(s2 * inv + eps), r2 = coef[1] / sqrtf(s4 * inv + eps), r3 = coef[2] / sqrtf(s6 * inv + eps), e = coef[3];
    auto value = [&](float x) { const float x2 = x * x; return x * r1 + x2 * r2 + x2 * x * r3 + e; };
    TO* o = out + (size_t)blockIdx.x * F;
    if constexpr (AGAIN)
#pragma unroll
    for (int u = 0; u < N4; ++u) asm volatile("" : "+v"(v[u].x), "+v"(v[u].y), "+v"(v[u].z), "+v"(v[u].w));
#pragma unroll
    for (int u = 0; u < N4; ++u) {
        const int i = (threadIdx.x + u * 64 * NW) * 4;
        if (i < F) st4(o + i, make_float4(value(v[u].x), value(v[u].y), value(v[u].z), value(v[u].w)));
    }
}

// More rows than compute units, each of more than 8,192 numbers, make their powers again (us without and with it, in bfloat16:
// 257 rows of 10,752 7.4 and 6.2, of 21,504 9.6 and 8.0, 2,048 rows of them 30 and 22, 42 and 32; 64 rows of 16,384 4.8 and 5.1, 2,048 of 8,192 19.9 and 20.9)
#define POLY_AGAIN_ROWS 256
template <typename TZ, typename TO>
static bool launch_polynorm_v4(TO* out, const TZ* z, const float* coef, int T, int F, int ld_z, float eps, hipStream_t stream) {
    if (F % 4 || ld_z % 4 || ((uintptr_t)z % 16) || ((uintptr_t)out % 16) || F > 16 * 64 * 4 * 8) return false;
    const bool again = T > POLY_AGAIN_ROWS;
#define PV(NW, N4) k_polynorm_v4<TZ, TO, NW, N4, false><<<T, 64 * NW, 0, stream>>>(out, z, coef, F, ld_z, eps)
#define PA(NW, N4) do { if (again) k_polynorm_v4<TZ, TO, NW, N4, true><<<T, 64 * NW, 0, stream>>>(out, z, coef, F, ld_z, eps); else PV(NW, N4); } while (0)
    // four waves a row where they hold it; 16 where rows are few (every lane's loads are a trip to memory) or long
    if (F <= 4 * 256 * 4 && !(T <= FEW_ROWS && F >= 1024)) PV(4, 4);
    else if (F <= 16 * 256 * 2) PV(16, 2);
    else if (F <= 16 * 256 * 4) PA(16, 4);
    else if (F <= 16 * 256 * 6) PA(16, 6);
    else PA(16, 8);
#undef PA
#undef PV
    return true;
}

extern "C" int xr_polynorm(void* out, const void* z, const float* coef, int T, int F, int ld_z, float eps, int z_dtype,
                           int out_dtype, hipStream_t stream) {
    XR_REQUIRE(T >= 0 && F > 0 && ld_z >= F, "polynorm: bad sizes T=%d F=%d ld=%d", T, F, ld_z);
    if (T == 0) return XR_OK;
    const bool few = T <= FEW_ROWS && F >= 1024;
#define PN(TZ, TO)                                                                                                        \
    do {                                                                                                                  \
        if (launch_polynorm_v4<TZ, TO>((TO*)out, (const TZ*)z, coef, T, F, ld_z, eps, stream)) break;                     \
        if (few) k_polynorm<TZ, TO, 16><<<T, 1024, 0, stream>>>((TO*)out, (const TZ*)z, coef, F, ld_z, eps);              \
        else k_polynorm<TZ, TO, 4><<<T, 256, 0, stream>>>((TO*)out, (const TZ*)z, coef, F, ld_z, eps);                    \
    } while (0)
    if (z_dtype == XR_F32 && out_dtype == XR_F32) PN(float, float);
    else if (z_dtype == XR_F32 && out_dtype == XR_BF16) PN(float, bf16_t);
    else if (z_dtype == XR_BF16 && out_dtype == XR_BF16) PN(bf16_t, bf16_t);
    else { xr_set_error("polynorm: bad dtypes %d %d", z_dtype, out_dtype); return XR_BAD_ARG; }
#undef PN
    XR_CHECK_LAUNCH("polynorm");
    return XR_OK;
}

// ---------------------------------------------------------------- rotation of 32-bit projections in place
// For every head of x [T, heads, D] (row stride ld): channel j < rot/2 pairs with j + rot/2,
// angle = position * inv_freq[j] as a 32-bit product; then every channel times `scale`.
__global__ __launch_bounds__(64) void k_rotate_rows(float* __restrict__ x, const int* __restrict__ positions,
                                                    const float* __restrict__ inv_freq, int D, int rot, int ld, float scale) {
    const int t = blockIdx.x, h = blockIdx.y;
    float* row = x + (size_t)t * ld + (size_t)h * D;
    const float pos = (float)positions[t];
    const int half = rot >> 1;
    for (int j = threadIdx.x; j < half; j += 64) {
        const float a = pos * inv_freq[j];
        const float c = cosf(a), s = sinf(a);
        const float u = row[j], v = row[j + half];
        row[j] = (u * c - v * s) * scale;
        row[j + half] = (v * c + u * s) * scale;
    }
    if (scale != 1.0f)
        for (int d = rot + threadIdx.x; d < D; d += 64) row[d] *= scale;
}

extern "C" int xr_rotate_rows(float* x, const int* positions, const float* inv_freq, int T, int heads, int D, int rot,
                              int ld, float scale, hipStream_t stream) {
    XR_REQUIRE(T >= 0 && heads > 0 && D > 0 && ld >= heads * D, "rotate_rows: bad sizes T=%d heads=%d D=%d ld=%d", T, heads, D, ld);
    XR_REQUIRE(rot >= 0 && rot <= D && rot % 2 == 0, "rotate_rows: rotary width %d does not fit head size %d", rot, D);
    XR_REQUIRE(rot == 0 || inv_freq != nullptr, "rotate_rows: no frequency table");
    if (T == 0 || (rot == 0 && scale == 1.0f)) return XR_OK;
    k_rotate_rows<<<dim3(T, heads), 64, 0, stream>>>(x, positions, inv_freq, D, rot, ld, scale);
    XR_CHECK_LAUNCH("rotate_rows");
    return XR_OK;
}

// Queries and keys of a token with the same number of heads in one launch; angles are made once a workgroup, not once a head.  Bound by memory, and for few
// tokens by a thread's chain of heads: so a token's 2 x heads heads are shared out to gridDim.y workgroups, which make its angles each.  2,048 tokens, 32 heads of
// 128: 22 us, as two launches of k_rotate_rows 38; 8 tokens 2.8, as two launches 4.1, with one workgroup a token 5.4.
#define ROT_PAIR_FILL 512
__global__ __launch_bounds__(256) void k_rotate_pair(float* __restrict__ x, float* __restrict__ y, const int* __restrict__ positions,
                                                     const float* __restrict__ inv_freq, int heads, int D, int half, int ld, float scale_x, float scale_y) {
    extern __shared__ float2 turn[];                    // [half]
    const int t = blockIdx.x;
    const float pos = (float)positions[t];
    for (int j = threadIdx.x; j < half; j += 256) {
        const float a = pos * inv_freq[j];
        turn[j] = make_float2(cosf(a), sinf(a));
    }
    __syncthreads();
    const int share = (2 * heads + (int)gridDim.y - 1) / (int)gridDim.y, from = (int)blockIdx.y * share, to = min(from + share, 2 * heads);
    const int rest = D - 2 * half;
    for (int which = 0; which < 2; ++which) {
        const int lo = max(from - which * heads, 0), hi = min(to - which * heads, heads);       // this workgroup's heads of x, of y
        float* row = (which ? y : x) + (size_t)t * ld + (size_t)lo * D;
        const float scale = which ? scale_y : scale_x;
        for (int i = threadIdx.x; i < (hi - lo) * half; i += 256) {
            const int h = i / half, j = i - h * half;
            const float c = turn[j].x, s = turn[j].y;
            float* at = row + (size_t)h * D + j;
            const float u = at[0], v = at[half];
            at[0] = (u * c - v * s) * scale;
            at[half] = (v * c + u * s) * scale;
        }
        if (scale != 1.0f && rest > 0)
            for (int i = threadIdx.x; i < (hi - lo) * rest; i += 256) row[(size_t)(i / rest) * D + 2 * half + i % rest] *= scale;
    }
}

extern "C" int xr_rotate_pair(float* x, float* y, const int* positions, const float* inv_freq, int T, int heads, int D, int rot, int ld, float scale_x,
                              float scale_y, hipStream_t stream) {
    XR_REQUIRE(T >= 0 && heads > 0 && D > 0 && ld >= heads * D, "rotate_pair: bad sizes T=%d heads=%d D=%d ld=%d", T, heads, D, ld);
    XR_REQUIRE(rot >= 0 && rot <= D && rot % 2 == 0 && rot <= 4096, "rotate_pair: rotary width %d does not fit head size %d", rot, D);
    XR_REQUIRE(x && y && positions && (rot == 0 || inv_freq), "rotate_pair: null operand");
    if (T == 0) return XR_OK;
    const int half = rot / 2;
    if (half == 0) {
        const int a = xr_rotate_rows(x, positions, inv_freq, T, heads, D, rot, ld, scale_x, stream);
        return a != XR_OK ? a : xr_rotate_rows(y, positions, inv_freq, T, heads, D, rot, ld, scale_y, stream);
    }
    // so many workgroups a token that a thread has one pair of each of two heads' rows, while all fit the compute units twice over
    int shares = 1;
    const long long most = (long long)heads * (half > D - 2 * half ? half : D - 2 * half);
    while (2 * shares <= 2 * heads && 2LL * shares * T <= ROT_PAIR_FILL && most > 256LL * shares) shares *= 2;
    k_rotate_pair<<<dim3(T, shares), 256, half * sizeof(float2), stream>>>(x, y, positions, inv_freq, heads, D, half, ld, scale_x, scale_y);
    XR_CHECK_LAUNCH("rotate_pair");
    return XR_OK;
}

// ---------------------------------------------------------------- gated norm of a read-out
// out[t][h][d] = o[t][h][d] / sqrt(mean_d(o^2) + eps) * w * act(gate[t][h][d]); w may be absent, is one
// weight a channel of a head that the heads share (w [Dv]) or, with w_full, one a channel of the row
// (w [H * Dv]); act is SiLU (gate_act 0) or the sigmoid (1).  A norm over all heads together is
// H = 1 with Dv the whole row.  One wave per (token, head).  With gate_first the gate comes before the norm:
// u = o * act(gate), out = u / sqrt(mean_d(u^2) + eps) * w.  Everything is multiplied by `scale` at last; output rows are
// ld_out apart.
#define XR_GATE_SILU 0
#define XR_GATE_SIGMOID 1
__device__ inline float norm_gate(float g, int gate_act) {
    const float sg = 1.0f / (1.0f + expf(-g));
    return gate_act == XR_GATE_SIGMOID ? sg : g * sg;
}
template <typename TO>
__global__ __launch_bounds__(64) void k_gated_rmsnorm(TO* __restrict__ out, const float* __restrict__ o,
                                                      const float* __restrict__ gate, const float* __restrict__ w,
                                                      int H, int Dv, int ld_g, float eps, int w_full, int gate_act,
                                                      int gate_first, float scale, int ld_out) {
    const int t = blockIdx.x, h = blockIdx.y;
    const float* orow = o + ((size_t)t * H + h) * Dv;
    const float* grow = gate + (size_t)t * ld_g + (size_t)h * Dv;
    const float* wrow = w ? (w_full ? w + (size_t)h * Dv : w) : nullptr;
    float ss = 0.f;
    for (int d = threadIdx.x; d < Dv; d += 64) {
        const float u = gate_first ? orow[d] * norm_gate(grow[d], gate_act) : orow[d];
        ss += u * u;
    }
    const float rinv = scale / sqrtf(wave_sum(ss) / (float)Dv + eps);
    TO* dst = out + (size_t)t * ld_out + (size_t)h * Dv;
    for (int d = threadIdx.x; d < Dv; d += 64)
        st<TO>(dst, d, orow[d] * rinv * (wrow ? wrow[d] : 1.f) * norm_gate(grow[d], gate_act));
}

// The same with a workgroup of 256 a (token, head), for long rows (all heads normed together).
template <typename TO>
__global__ __launch_bounds__(256) void k_gated_rmsnorm_wide(TO* __restrict__ out, const float* __restrict__ o,
                                                           const float* __restrict__ gate, const float* __restrict__ w,
                                                           int H, int Dv, int ld_g, float eps, int w_full, int gate_act,
                                                           int gate_first, float scale, int ld_out) {
    __shared__ float part[4];
    const int t = blockIdx.x, h = blockIdx.y;
    const float* orow = o + ((size_t)t * H + h) * Dv;
    const float* grow = gate + (size_t)t * ld_g + (size_t)h * Dv;
    const float* wrow = w ? (w_full ? w + (size_t)h * Dv : w) : nullptr;
    float ss = 0.f;
    for (int d = threadIdx.x; d < Dv; d += 256) {
        const float u = gate_first ? orow[d] * norm_gate(grow[d], gate_act) : orow[d];
        ss += u * u;
    }
    ss = wave_sum(ss);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = ss;
    __syncthreads();
    const float rinv = scale / sqrtf(((part[0] + part[1]) + (part[2] + part[3])) / (float)Dv + eps);
    TO* dst = out + (size_t)t * ld_out + (size_t)h * Dv;
    for (int d = threadIdx.x; d < Dv; d += 256)
        st<TO>(dst, d, orow[d] * rinv * (wrow ? wrow[d] : 1.f) * norm_gate(grow[d], gate_act));
}

// Rows of up to 64 * 4 * NV channels that come in fours: a wave a (token, head) keeps its float4 pieces in registers from the
// sum to the store, and every gate is made once.
// PAIR (up to 128 channels): two heads a wave, so that no lane is idle; their sums are those of a wave whose other half adds zeros.  2,048 tokens, 32 heads of
// 128: 27 us -> 17, 700 of 16 heads 6.8 -> 5.6.
template <typename TO, int NV, bool PAIR = false>
__global__ __launch_bounds__(256) void k_gated_rmsnorm_v4(TO* __restrict__ out, const float* __restrict__ o,
                                                         const float* __restrict__ gate, const float* __restrict__ w,
                                                         int TH, int H, int Dv, int ld_g, float eps, int w_full, int gate_act,
                                                         int gate_first, float scale, int ld_out) {
    const int th = PAIR ? blockIdx.x * 8 + (threadIdx.x >> 5) : blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & (PAIR ? 31 : 63);
    if (th >= TH) return;
    const int t = th / H, h = th - t * H, n4 = Dv >> 2;
    const float4* o4 = reinterpret_cast<const float4*>(o + (size_t)th * Dv);
    const float4* g4 = reinterpret_cast<const float4*>(gate + (size_t)t * ld_g + (size_t)h * Dv);
    const float4* w4 = reinterpret_cast<const float4*>(w ? (w_full ? w + (size_t)h * Dv : w) : nullptr);
    float4 u[NV];
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int c = lane + 64 * i;
        u[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (c >= n4) continue;
        const float4 x = o4[c], g = g4[c];
        u[i] = make_float4(x.x * norm_gate(g.x, gate_act), x.y * norm_gate(g.y, gate_act), x.z * norm_gate(g.z, gate_act), x.w * norm_gate(g.w, gate_act));
        const float4 y = gate_first ? u[i] : x;
        ss += y.x * y.x + y.y * y.y + y.z * y.z + y.w * y.w;
    }
#pragma unroll
    for (int m = PAIR ? 16 : 32; m > 0; m >>= 1) ss += __shfl_xor(ss, m, 64);
    const float f = scale / sqrtf(ss / (float)Dv + eps);
    TO* dst = out + (size_t)t * ld_out + (size_t)h * Dv;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int c = lane + 64 * i;
        if (c >= n4) continue;
        const float4 g = w ? w4[c] : make_float4(1.f, 1.f, 1.f, 1.f);
        const float4 y = make_float4(u[i].x * f * g.x, u[i].y * f * g.y, u[i].z * f * g.z, u[i].w * f * g.w);
        if constexpr (sizeof(TO) == 4) *reinterpret_cast<float4*>((float*)dst + 4 * c) = y;
        else *reinterpret_cast<uint2*>((bf16_t*)dst + 4 * c) = make_uint2(pack_bf16x2(y.x, y.y), pack_bf16x2(y.z, y.w));
    }
}

extern "C" int xr_gated_rmsnorm(void* out, const float* o, const float* gate, const float* w, int T, int H, int Dv,
                                int ld_g, float eps, int out_dtype, int w_full, int gate_act, int gate_first, float scale,
                                int ld_out, hipStream_t stream) {
    XR_REQUIRE(ld_out >= H * Dv, "gated_rmsnorm: output rows of %d are %d apart", H * Dv, ld_out);
    XR_REQUIRE(T >= 0 && H > 0 && Dv > 0 && ld_g >= H * Dv, "gated_rmsnorm: bad sizes T=%d H=%d Dv=%d ld=%d", T, H, Dv, ld_g);
    XR_REQUIRE(gate_act == XR_GATE_SILU || gate_act == XR_GATE_SIGMOID, "gated_rmsnorm: unknown gate activation %d", gate_act);
    if (T == 0) return XR_OK;
    // (bfloat16 only: results in 32 bits keep the order of sums they had)
    const bool v4 = out_dtype == XR_BF16 && Dv % 4 == 0 && Dv >= 128 && Dv <= 1024 && ld_g % 4 == 0 && ld_out % 4 == 0 && ((uintptr_t)out % 8) == 0 &&
                    ((uintptr_t)o % 16) == 0 && ((uintptr_t)gate % 16) == 0 && ((uintptr_t)w % 16) == 0;
    if (v4) {
        const int TH = T * H, blocks = (TH + 3) / 4;
        bf16_t* ob = (bf16_t*)out;
        if (Dv <= 128) k_gated_rmsnorm_v4<bf16_t, 1, true><<<(TH + 7) / 8, 256, 0, stream>>>(ob, o, gate, w, TH, H, Dv, ld_g, eps, w_full, gate_act, gate_first, scale, ld_out);
        else if (Dv <= 256) k_gated_rmsnorm_v4<bf16_t, 1><<<blocks, 256, 0, stream>>>(ob, o, gate, w, TH, H, Dv, ld_g, eps, w_full, gate_act, gate_first, scale, ld_out);
        else if (Dv <= 512) k_gated_rmsnorm_v4<bf16_t, 2><<<blocks, 256, 0, stream>>>(ob, o, gate, w, TH, H, Dv, ld_g, eps, w_full, gate_act, gate_first, scale, ld_out);
        else k_gated_rmsnorm_v4<bf16_t, 4><<<blocks, 256, 0, stream>>>(ob, o, gate, w, TH, H, Dv, ld_g, eps, w_full, gate_act, gate_first, scale, ld_out);
        XR_CHECK_LAUNCH("gated_rmsnorm");
        return XR_OK;
    }
    const bool wide = Dv > 256;       // (the sums' order differs between the two kernels, not between calls of one size)
    if (out_dtype == XR_F32 && wide) k_gated_rmsnorm_wide<float><<<dim3(T, H), 256, 0, stream>>>((float*)out, o, gate, w, H, Dv, ld_g, eps, w_full, gate_act, gate_first, scale, ld_out);
    else if (out_dtype == XR_BF16 && wide) k_gated_rmsnorm_wide<bf16_t><<<dim3(T, H), 256, 0, stream>>>((bf16_t*)out, o, gate, w, H, Dv, ld_g, eps, w_full, gate_act, gate_first, scale, ld_out);
    else if (out_dtype == XR_F32) k_gated_rmsnorm<float><<<dim3(T, H), 64, 0, stream>>>((float*)out, o, gate, w, H, Dv, ld_g, eps, w_full, gate_act, gate_first, scale, ld_out);
    else if (out_dtype == XR_BF16) k_gated_rmsnorm<bf16_t><<<dim3(T, H), 64, 0, stream>>>((bf16_t*)out, o, gate, w, H, Dv, ld_g, eps, w_full, gate_act, gate_first, scale, ld_out);
    else { xr_set_error("gated_rmsnorm: bad dtype %d", out_dtype); return XR_BAD_ARG; }
    XR_CHECK_LAUNCH("gated_rmsnorm");
    return XR_OK;
}

// ---------------------------------------------------------------- an activation on 32-bit rows
// x[t][c] <- act(x[t][c]) for the first W columns of rows of stride ld, in place; or, with `out`, into
// contiguous rows [T, W] of the type the next product reads.  act 1 = SiLU, 2 = tanh.
#define XR_ACT_ROWS_TANH 2
#define XR_ACT_ROWS_RELU2 3
template <typename TO>
__global__ void k_act_rows(float* __restrict__ x, TO* __restrict__ out, int W, int ld, size_t n, int act) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const size_t t = i / W;
    float* p = x + t * ld + (i - t * W);
    const float v = *p;
    const float r = fmaxf(v, 0.f);
    const float y = act == XR_ACT_ROWS_TANH ? tanhf(v) : act == XR_ACT_ROWS_RELU2 ? r * r : v / (1.0f + expf(-v));
    if (out) st<TO>(out, i, y);
    else *p = y;
}

extern "C" int xr_act_rows(float* x, int T, int W, int ld, int act, void* out, int out_dtype, hipStream_t stream) {
    XR_REQUIRE(T >= 0 && W > 0 && ld >= W, "act_rows: bad sizes T=%d W=%d ld=%d", T, W, ld);
    XR_REQUIRE(act == XR_CONV_SILU || act == XR_ACT_ROWS_TANH || act == XR_ACT_ROWS_RELU2, "act_rows: activation %d is not built (1 = SiLU, 2 = tanh, 3 = relu squared)", act);
    XR_REQUIRE(!out || out_dtype == XR_F32 || out_dtype == XR_BF16, "act_rows: output type %d", out_dtype);
    const size_t n = (size_t)T * W;
    if (n == 0) return XR_OK;
    const unsigned blocks = (unsigned)((n + 255) / 256);
    if (out && out_dtype == XR_BF16) k_act_rows<bf16_t><<<blocks, 256, 0, stream>>>(x, (bf16_t*)out, W, ld, n, act);
    else k_act_rows<float><<<blocks, 256, 0, stream>>>(x, (float*)out, W, ld, n, act);
    XR_CHECK_LAUNCH("act_rows");
    return XR_OK;
}

// ---------------------------------------------------------------- what a gated delta rule reads
// In place on 32-bit rows (queries and keys of row stride ld, b and a of row stride ld_g): every query and key head becomes a unit vector
// x / sqrt(sum(x^2) + unit_eps), queries also times q_scale; the write strength of head h becomes
// sigmoid(b), its decay exp(-exp(a_log[h]) * softplus(a + dt_bias[h])).
__global__ __launch_bounds__(64) void k_delta_prepare(float* __restrict__ q, float* __restrict__ k, float* __restrict__ b,
                                                      float* __restrict__ a, const float* __restrict__ a_log,
                                                      const float* __restrict__ dt_bias, int G, int H, int D, int ld,
                                                      int ld_g, float q_scale, float unit_eps) {
    const int t = blockIdx.x, y = blockIdx.y;
    if (y < 2 * G) {
        float* row = (y < G ? q : k) + (size_t)t * ld + (size_t)(y < G ? y : y - G) * D;
        float ss = 0.f;
        for (int d = threadIdx.x; d < D; d += 64) ss += row[d] * row[d];
        const float f = (y < G ? q_scale : 1.0f) / sqrtf(wave_sum(ss) + unit_eps);
        for (int d = threadIdx.x; d < D; d += 64) row[d] *= f;
        return;
    }
    for (int h = threadIdx.x; h < H; h += 64) {
        const size_t i = (size_t)t * ld_g + h;
        b[i] = 1.0f / (1.0f + expf(-b[i]));
        if (!a) continue;           // (the decays are made elsewhere: one a key channel, say)
        const float z = a[i] + dt_bias[h];
        const float sp = z > 20.0f ? z : log1pf(expf(z));
        a[i] = expf(-expf(a_log[h]) * sp);
    }
}

extern "C" int xr_delta_prepare(float* q, float* k, float* b, float* a, const float* a_log, const float* dt_bias, int T,
                                int G, int H, int D, int ld, int ld_g, float q_scale, float unit_eps, hipStream_t stream) {
    XR_REQUIRE(T >= 0 && G > 0 && H > 0 && D > 0 && ld >= G * D && ld_g >= H, "delta_prepare: bad sizes T=%d G=%d H=%d D=%d ld=%d ld_g=%d",
               T, G, H, D, ld, ld_g);
    if (T == 0) return XR_OK;
    k_delta_prepare<<<dim3(T, 2 * G + 1), 64, 0, stream>>>(q, k, b, a, a_log, dt_bias, G, H, D, ld, ld_g, q_scale, unit_eps);
    XR_CHECK_LAUNCH("delta_prepare");
    return XR_OK;
}
