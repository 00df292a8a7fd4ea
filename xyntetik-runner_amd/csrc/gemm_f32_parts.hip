// Matrix products of 32-bit operands, out[M,N] = a[M,K] * w[N,K]^T (+ bias), on the matrix cores' bfloat16 instructions, which do sixteen
// products in the time the 32-bit ones (k_gemm_f32) do one.  Every number is three bfloat16 parts that add up to it exactly (8 bits a
// part, rounded to nearest, each with its sign: 24 bits), and a product of two numbers the six largest of the nine products of
// their parts; the three left out are 2^-24 of it at most together (x = y = 1.00389862, whose products all miss as much; 2^-27.4 in root mean
// square of normal ones).  Part 0 times part 0, which a bfloat16 instruction makes exactly
// and adds up in 32 bits, sixteen columns at a time, is summed in runs of PFOLD slabs and the runs' sums with what each addition loses; the
// smaller products have a sum of their own over all of K, where 2^-8 of the size their rounding does not count.  That is fewer
// roundings than a 32-bit instruction's, two columns at a time: root mean square error against 64 bits, in units of the result's, 401 x
// 2048 x 2048 9.1e-8 (k_gemm_f32 2.1e-7), 401 x 2048 x 8192 9.0e-8 (2.1e-7), positive numbers 3.9e-8 (4.8e-8) and 3.1e-8 (3.4e-8), numbers
// of very different size (times exp(3 N(0,1))) 1.2e-7 (1.9e-7) and 1.1e-7 (1.5e-7).  A row's result does not depend on the tile.
//
// A workgroup makes a tile of BM x BN from slabs of PK columns: 32-bit pieces from memory into registers, PF slabs ahead; their parts into LDS, three
// planes, two slabs; fragments from there.  Splitting once a workgroup and not once a wave is what makes the vector units' share (5.5
// instructions a number) smaller than the matrix cores'.  The instructions of the half slab in use, of the reads of the next half and of the
// next slab's parts are interleaved by hand (first, second: without that 871 us became 973 in the four-wave 128 x 128 tile), with one
// barrier a slab, behind the parts.  Bound by the matrix cores at the clock that the power leaves (products and LDS reads alone 544 us of
// 751 at 2048 x 16384 x 2048, 160 the parts, 40 the loads' way through the caches).  us, k_gemm_f32 and so: 2048 x 16384 x 2048 1,101 and
// 766 (179 TFLOP/s, of 157 that 32-bit instructions could reach), 401 x 16384 x 2048 262 and 192, 401 x 2048 x 8192 149 and 102, 2048 x 2048 x
// 8192 554 and 361, 100 x 4096 x 14336 156 and 93, 17 x 2048 x 8192 56 and 22.  Left out: four waves with 64 x 64 each (512 registers, one wave a
// SIMD; 928 us for 751), four slabs on their way (fewer workgroups fit: 5 to 20% slower), pieces of 8 numbers a lane (5%).
#include <type_traits>

#include "common.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

#define PK 32           // columns of a slab
#define PCH (PK / 8)    // pieces of 8 numbers a row of a slab
#define PFOLD 8         // slabs of a run (16: no faster by more than 3%, and positive numbers lose the little they are ahead)

__device__ inline bf16x8 frag(uint4 v) {
    union { uint4 u; bf16x8 b; } c;
    c.u = v;
    return c.b;
}

// Two numbers in three pairs of parts: x = part 0 + part 1 + part 2, each the nearest bfloat16 to what the parts before it leave.  (A number
// that rounds to infinity, or is none, leaves a NaN.)
__device__ inline void parts_of(float x, float y, uint32_t (&p)[3]) {
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        p[i] = pack_bf16x2(x, y);
        if (i < 2) {
            x -= __uint_as_float(p[i] << 16);
            y -= __uint_as_float(p[i] & 0xffff0000u);
        }
    }
}

// The largest of a >= 0 and of x and y without their signs: NaN if one of them is (one v_maximum3_f32).
__device__ inline float larger(float a, float x, float y) {
    return __builtin_elementwise_maximum(__builtin_elementwise_maximum(a, fabsf(x)), fabsf(y));
}

// GM x GN waves, each TM x TN tiles of 32 x 32; MW: waves a SIMD there must be registers for.  ranges > 1: K is cut into ranges of range_slabs
// slabs (an even number, as K / PK is), and a range's sum goes to `partial` [range][M][N] in two parts.  Item i of the grid runs on XCD i % 8,
// and an XCD takes an eighth of the items, row tiles first, so that a weight tile comes from memory for one XCD.
template <typename TO, bool ACC, int GM, int GN, int TM, int TN, int MW, int PF>
__global__ __launch_bounds__(64 * GM * GN, MW) void k_gemm_f32_parts(TO* __restrict__ out, const float* __restrict__ a, const float* __restrict__ w,
                                                     const float* __restrict__ bias, int M, int N, int K, int lda, int ldo, int ranges,
                                                     int range_slabs, float2* __restrict__ partial) {
    constexpr int WAVES = GM * GN, THREADS = 64 * WAVES, BM = GM * TM * 32, BN = GN * TN * 32, ROWS = BM + BN;
    static_assert(PF == 2 && PFOLD % PF == 0, "slabs come in pairs");
    static_assert(ROWS * 2 * PCH % THREADS == 0 && PCH == 4, "every thread has as many pieces, eight of them side by side a row's");
    constexpr int UNITS = ROWS * 2 * PCH / THREADS; // pieces a thread moves of every slab
    extern __shared__ __align__(16) uint4 lds[];            // [2 slabs][3 parts][ROWS][PCH], a row's pieces turned by a quarter of its number; [ROWS] numbers
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN, items = tiles_m * tiles_n * ranges;
    const int item = (int)(blockIdx.x & 7) * ((items + 7) >> 3) + (int)(blockIdx.x >> 3);
    if (item >= items || (int)(blockIdx.x >> 3) >= ((items + 7) >> 3)) return;
    const int m0 = item % tiles_m * BM, n0 = item / tiles_m % tiles_n * BN, range = item / (tiles_m * tiles_n);
    const int wm = wave / GN * (TM * 32), wn = wave % GN * (TN * 32);
    const int slab0 = range * range_slabs, slabs = min(K / PK - slab0, range_slabs);
    auto turn = [](int r) { return (r >> 2) & (PCH - 1); };

    // this thread's pieces: 4 numbers of a row (of the last row that exists where it does not: its results are not stored), the same of every RU-th
    constexpr int RU = THREADS / (2 * PCH);
    static_assert(BM % RU == 0 && RU % 16 == 0, "a piece is the activations' or the weights' for all threads, and turned alike");
    const int r0 = tid / (2 * PCH), c0 = tid % (2 * PCH), dst = (r0 * PCH + ((c0 >> 1) ^ turn(r0))) * 2 + (c0 & 1);
    const float* src[UNITS];
#pragma unroll
    for (int u = 0; u < UNITS; ++u) {
        const int r = u * RU + r0;
        src[u] = (u * RU < BM ? a + (size_t)min(m0 + r, M - 1) * lda : w + (size_t)min(n0 + r - BM, N - 1) * K) + (size_t)slab0 * PK + c0 * 4;
    }
    float4 ahead[PF][UNITS];                                // the next slabs' pieces, on their way
    float top[UNITS] = {};                                  // the largest number of this thread's pieces of a row so far, without its sign
    auto fetch = [&](int slot, int s) {
        const int at = min(s, slabs - 1) * PK;              // (past the end the last slab once more: it is not multiplied)
#pragma unroll
        for (int u = 0; u < UNITS; ++u) ahead[slot][u] = *reinterpret_cast<const float4*>(src[u] + at);
    };
    auto stash = [&](int slot, int buf) {
        uint2* const to = reinterpret_cast<uint2*>(lds) + buf * 3 * ROWS * PCH * 2;
#pragma unroll
        for (int u = 0; u < UNITS; ++u) {
            const float4 x = ahead[slot][u];
            uint32_t p[2][3];
            parts_of(x.x, x.y, p[0]);
            parts_of(x.z, x.w, p[1]);
            top[u] = larger(larger(top[u], x.x, x.y), x.z, x.w);
#pragma unroll
            for (int i = 0; i < 3; ++i) to[i * ROWS * PCH * 2 + dst + u * RU * PCH * 2] = make_uint2(p[0][i], p[1][i]);
        }
    };
    auto meet = [&]() {                                     // LDS alone is waited for: the slabs on their way stay there
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    };

    // run: part 0 times part 0, a run's; tot: the runs' sum; low: the other parts' products of all K, and what tot has lost
    constexpr int VA = (UNITS * 23 + 6 * TM * TN - 1) / (6 * TM * TN);
    f32x16 run[TM][TN], tot[TM][TN], low[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) run[i][j] = tot[i][j] = low[i][j] = f32x16{};
    const int row = lane & 31;
    bf16x8 fa[2][TM][3], fw[2][TN][3];                      // the operands of the 16 columns in use and of the next 16
    auto read = [&](int set, int buf, int kk) {
        const uint4* const A = lds + buf * 3 * ROWS * PCH;
        const int c = kk + (lane >> 5);
#pragma unroll
        for (int p = 0; p < 3; ++p) {
#pragma unroll
            for (int i = 0; i < TM; ++i) { const int r = wm + 32 * i + row; fa[set][i][p] = frag(A[p * ROWS * PCH + r * PCH + (c ^ turn(r))]); }
#pragma unroll
            for (int j = 0; j < TN; ++j) { const int r = BM + wn + 32 * j + row; fw[set][j][p] = frag(A[p * ROWS * PCH + r * PCH + (c ^ turn(r))]); }
        }
    };
    auto products = [&](int set) {
        auto mul = [&](f32x16 (&acc)[TM][TN], int pa, int pw) {
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[set][i][pa], fw[set][j][pw], acc[i][j], 0, 0, 0);
        };
        mul(run, 0, 0);
        mul(low, 1, 0);
        mul(low, 0, 1);
        mul(low, 1, 1);
        mul(low, 2, 0);
        mul(low, 0, 2);
    };
    constexpr int MM = 6 * TM * TN, RD = 3 * (TM + TN);     // products and reads of 16 columns
    auto fold = [&]() {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const float x = run[i][j][e], t = tot[i][j][e] + x;
                    low[i][j][e] += x - (t - tot[i][j][e]);
                    tot[i][j][e] = t;
                    run[i][j][e] = 0.f;
                }
    };
    // Half a slab's products beside the reads of its other half and the parts of the next slab, half beside the reads of that one
    auto first = [&](int slot, int buf) {
        __builtin_amdgcn_sched_barrier(0);
        read(1, buf, 2);
        stash(slot, buf ^ 1);
        products(0);
#pragma unroll
        for (int i = 0; i < MM; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
            if (i < RD) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x2, VA, 0);
            if (i >= MM - 3 * UNITS) __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
        }
#pragma unroll
        for (int u = 0; u < UNITS; ++u) asm volatile("" : "+v"(top[u]));       // made here: left for later, the pieces would have to stay, too
        __builtin_amdgcn_sched_barrier(0);
        meet();
        __builtin_amdgcn_sched_barrier(0);
    };
    auto second = [&](int slot, int s, int buf) {
        fetch(slot, s);
        read(0, buf ^ 1, 0);
        products(1);
#pragma unroll
        for (int i = 0; i < MM; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
            if (i < RD) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            else __builtin_amdgcn_sched_group_barrier(0x20, 1, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll
    for (int i = 0; i < PF; ++i) fetch(i, i);
    stash(0, 0);
    fetch(0, PF);
    meet();
    read(0, 0, 0);
    for (int s = 0; s < slabs; s += PF) {
#pragma unroll
        for (int u = 0; u < PF; ++u) {
            first((u + 1) % PF, u & 1);
            second((u + 1) % PF, s + u + 1 + PF, u & 1);
        }
        if ((s + PF) % PFOLD == 0) fold();
    }
    fold();

    // Results that are not finite, or so small that what parts have lost may count, are made again from 32-bit products, a wave's 32 x 32 at a time:
    // an infinity stays one, whatever it meets, and an overflow happens where it did.  (The part of a number that is below 2^-126 is lost: over K columns
    // up to K 2^-125 times the largest number of the row and of the weight row that meet, `most` here.  Where that is above 2^-27 of a result, or a result is
    // below 2^-60 and products of parts may be too small for 32 bits, it is made again; a zero is one where one of the rows has nothing else.)  The others of
    // the 32 x 32 stay as they are: a result depends on its own row and column alone.  (Where every tile is made again, a product takes three times as long.)
    float* const tops = reinterpret_cast<float*>(lds + 2 * 3 * ROWS * PCH);
#pragma unroll
    for (int u = 0; u < UNITS; ++u) {
        float t = top[u];
#pragma unroll
        for (int o = 4; o > 0; o >>= 1) t = larger(t, __shfl_xor(t, o), 0.f);
        if (c0 == 0) tops[u * RU + r0] = t;
    }
    meet();
    const float lost_share = (float)(slabs * PK) * 0x1p-98f;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int n = n0 + wn + 32 * j + row, mb = m0 + wm + 32 * i + 4 * (lane >> 5);
            const float top_w = tops[BM + wn + 32 * j + row];
            float least = 1.f, largest = 0.f;
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const float v = fabsf(tot[i][j][e] + low[i][j][e]);
                least = __builtin_elementwise_minimum(least, v);
                largest = larger(largest, v, 0.f);
            }
            const bool usual = least >= 0x1p-60f && largest <= 3.402823466e38f && lost_share * larger(top_w, tops[wm + 32 * i + row], 0.f) <= 0x1p-60f;
            if (!__any(!usual)) continue;
            uint32_t bad = 0;                               // a bit for each of the lane's 16
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const float v = fabsf(tot[i][j][e] + low[i][j][e]), top_a = tops[wm + 32 * i + 4 * (lane >> 5) + 8 * (e >> 2) + (e & 3)];
                const float most = larger(top_a, top_w, 0.f);
                const bool fine = v <= 3.402823466e38f && ((v >= 0x1p-60f && v >= lost_share * most) || top_a == 0.f || top_w == 0.f);
                if (n < N && mb + 8 * (e >> 2) + (e & 3) < M && !fine) bad |= 1u << e;
                asm volatile("" : "+v"(bad));               // (a bit and not a mask of lanes each)
            }
            if (__any(bad != 0)) {
                const float* const x = a + (size_t)min(m0 + wm + 32 * i + row, M - 1) * lda + 4 * (lane >> 5);
                const float* const y = w + (size_t)min(n, N - 1) * K + 4 * (lane >> 5);
                f32x16 acc{}, t{}, lost{};
                for (int k = slab0 * PK; k < (slab0 + slabs) * PK; k += 8) {
                    const float4 u = *reinterpret_cast<const float4*>(x + k), v = *reinterpret_cast<const float4*>(y + k);
                    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(u.x, v.x, acc, 0, 0, 0);
                    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(u.y, v.y, acc, 0, 0, 0);
                    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(u.z, v.z, acc, 0, 0, 0);
                    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(u.w, v.w, acc, 0, 0, 0);
                    if (k % 128 == 120 || k + 8 == (slab0 + slabs) * PK)
#pragma unroll
                        for (int e = 0; e < 16; ++e) {
                            const float z = acc[e] - lost[e], s = t[e] + z;
                            lost[e] = __builtin_amdgcn_fmed3f((s - t[e]) - z, -1e32f, 1e32f);
                            t[e] = s;
                            acc[e] = 0.f;
                        }
                }
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    tot[i][j][e] = bad >> e & 1 ? t[e] : tot[i][j][e];
                    low[i][j][e] = bad >> e & 1 ? -lost[e] : low[i][j][e];
                }
            }
        }
    // a lane has column lane % 32 and rows 8 (e / 4) + 4 (lane / 32) + e % 4 of a tile
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        const int n = n0 + wn + 32 * j + row;
        if (n >= N) continue;
        const float add = bias && ranges == 1 ? bias[n] : 0.f;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int m = m0 + wm + 32 * i + 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3);
                if (m >= M) continue;
                if (ranges > 1) {
                    partial[((size_t)range * M + m) * N + n] = make_float2(tot[i][j][e], low[i][j][e]);
                    continue;
                }
                const size_t at = (size_t)m * ldo + n;
                float v = tot[i][j][e] + low[i][j][e];
                if (bias) v += add;
                if (ACC) v += ld<TO>(out, at);
                st<TO>(out, at, v);
            }
    }
}

// The ranges' sums, added in their order with what each addition loses (Knuth's two-sum).
template <typename TO, bool ACC>
__global__ __launch_bounds__(256) void k_gemm_f32_ranges(TO* __restrict__ out, const float2* __restrict__ partial, const float* __restrict__ bias,
                                                         int M, int N, int ldo, int ranges) {
    const size_t q = (size_t)blockIdx.x * 256 + threadIdx.x, mn = (size_t)M * N;
    if (q >= mn) return;
    const int m = (int)(q / N), n = (int)(q % N);
    float tot = 0.f, low = 0.f;
    for (int r0 = 0; r0 < ranges; r0 += 8) {
        float2 p[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) p[i] = r0 + i < ranges ? partial[(size_t)(r0 + i) * mn + q] : make_float2(0.f, 0.f);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float x = p[i].x, t = tot + x, z = t - tot;
            low += ((tot - (t - z)) + (x - z)) + p[i].y;
            tot = t;
        }
    }
    const float sum = tot + low;
    float v = fabsf(tot) <= 3.402823466e38f ? sum : tot;    // (what an infinite sum loses is no number)
    if (bias) v += bias[n];
    const size_t at = (size_t)m * ldo + n;
    if (ACC) v += ld<TO>(out, at);
    st<TO>(out, at, v);
}

// Columns that a range of `ranges` has, in slabs, and the ranges that leaves.
static int parts_range(int K, int& ranges) {
    const int pairs = K / (2 * PK), per = (pairs + ranges - 1) / ranges;
    ranges = (pairs + per - 1) / per;
    return 2 * per;
}

template <int GM, int GN, int TM, int TN, int MW, int PF>
static int launch_parts(void* out, const float* a, const float* w, const float* bias, int M, int N, int K, int lda, int ldo, int out_dtype,
                        int accumulate, int ranges, float2* partial, hipStream_t stream) {
    constexpr int BM = GM * TM * 32, BN = GN * TN * 32, smem = 2 * 3 * (BM + BN) * PK * 2 + (BM + BN) * 4;
    const int per = parts_range(K, ranges);
    const long long items = (long long)((M + BM - 1) / BM) * ((N + BN - 1) / BN) * ranges;
    XR_REQUIRE(items < (1ll << 28), "gemm: %lld tiles", items);
    const unsigned blocks = 8 * (unsigned)((items + 7) / 8);
    // `which`: the kernel's number (that adds to its output and that stores it are of one type, and so share this function's statics)
    auto run = [&](auto kernel, auto finish, auto* to, int which) {
        static bool attr_set[3] = {};
        if (!attr_set[which]) {
            const hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, smem);
            if (e != hipSuccess) {
                (void)hipGetLastError();             // or the next launch's check would report this refusal
                xr_set_error("gemm: cannot reserve %d bytes of LDS: %s", smem, hipGetErrorString(e));
                return XR_LAUNCH;
            }
            attr_set[which] = true;
        }
        kernel<<<blocks, 64 * GM * GN, smem, stream>>>(to, a, w, bias, M, N, K, lda, ldo, ranges, per, partial);
        XR_CHECK_LAUNCH("gemm_f32_parts");
        if (ranges > 1) {
            finish<<<(unsigned)(((size_t)M * N + 255) / 256), 256, 0, stream>>>(to, partial, bias, M, N, ldo, ranges);
            XR_CHECK_LAUNCH("gemm_f32_ranges");
        }
        return XR_OK;
    };
    if (out_dtype == XR_BF16) return run(k_gemm_f32_parts<bf16_t, false, GM, GN, TM, TN, MW, PF>, k_gemm_f32_ranges<bf16_t, false>, (bf16_t*)out, 0);
    if (accumulate) return run(k_gemm_f32_parts<float, true, GM, GN, TM, TN, MW, PF>, k_gemm_f32_ranges<float, true>, (float*)out, 1);
    return run(k_gemm_f32_parts<float, false, GM, GN, TM, TN, MW, PF>, k_gemm_f32_ranges<float, false>, (float*)out, 2);
}

#define XR_PARTS_TILES 4
struct PartsTile { int bm, bn, most; double slab, waves, tile; };     // `most`: workgroups a compute unit has room for
// `slab`, `tile`: microseconds of a slab and of a tile's beginning and end with one workgroup a compute unit; w at once take (w + `waves`) / (1 + `waves`)
// times as long as one
static const PartsTile parts_tiles[XR_PARTS_TILES] = {{32, 128, 2, 0.570, 0.460, 0.569}, {64, 64, 3, 0.516, 0.493, 0.112},
                                                      {64, 128, 2, 0.917, 0.655, 1.661}, {128, 128, 1, 1.081, 0.0, 2.966}};

// The time of a product in tiles of kind t and `ranges` ranges, us: the fullest compute unit's workgroups and the mean's, each its slabs, more of them at
// once at a better rate; the weights' arrival; the kernel that adds ranges up.  Fitted to 4,466 timed launches (14 products, N 512 to 128,256, K 768
// to 14,336, 17 to 2,048 rows, weights from memory): off by 6%, and its choice 1.0% slower than the best (14.5% at most).
static double parts_us(int M, int N, int K, int t, int ranges) {
    const PartsTile& p = parts_tiles[t];
    const int slabs = parts_range(K, ranges);
    const long long items = (long long)((M + p.bm - 1) / p.bm) * ((N + p.bn - 1) / p.bn) * ranges;
    const double most = (double)((items + 255) / 256), mean = items > 256 ? items / 256.0 : 1.0, at_once = most < p.most ? most : p.most;
    const double work = (0.858 * most + 0.142 * mean) * (slabs * p.slab + p.tile) * (at_once + p.waves) / (at_once * (1 + p.waves));
    const double add = ranges > 1 ? 1.318 + (double)M * N * 8 * (ranges + 0.5) / 3.13e6 : 0.0;
    return work + (double)N * K * 4 / 19.0e6 + add + 7.5;
}

double xr_f32_tiles_us(int M, int N, int K);       // gemm_ref.hip: k_gemm_f32's time as its own model has it

// Whether a 32-bit product of more than 16 rows is faster in parts: 0, or 1 + its tile + XR_PARTS_TILES * (ranges - 1).  Taken where this model's
// time is a tenth below the other kernel's (whose model leaves out 3 us of a launch): of the 245 timed products (M, N, K) 23% faster on average (24%
// with the better of the two everywhere), five more than 3% slower (8% at most); 183 drawn ones (64 to 60,000 weight rows) 31%, four
// 3 to 5% slower.  Few columns stay with k_gemm_f32: there is no gain.
extern "C" int xr_gemm_f32_parts_plan(int M, int N, int K) {
    if (M <= 16 || K < 512 || K % (2 * PK) != 0 || N < 1 || (long long)M * N > (1ll << 31)) return 0;
    static const int tried[] = {1, 2, 3, 4, 6, 8, 12, 16, 24};
    double best = 1e30;
    int plan = 0;
    for (int t = 0; t < XR_PARTS_TILES; ++t) {
        const PartsTile& p = parts_tiles[t];
        const long long tiles = (long long)((M + p.bm - 1) / p.bm) * ((N + p.bn - 1) / p.bn);
        for (int want : tried) {
            int r = want;
            if (r > 1 && (tiles * r > (t == 3 ? 1100 : 2200) || parts_range(K, r) < 4)) break;
            const double us = parts_us(M, N, K, t, r);
            if (us < best) best = us, plan = 1 + t + XR_PARTS_TILES * (r - 1);
        }
    }
    return best < 0.9 * (xr_f32_tiles_us(M, N, K) + 3.0) ? plan : 0;
}
extern "C" int xr_gemm_f32_parts_ranges(int plan) { return plan > 0 ? (plan - 1) / XR_PARTS_TILES + 1 : 0; }

// plan: xr_gemm_f32_parts_plan's, or another of its form; partial: room for xr_gemm_f32_parts_ranges M N pairs of floats (one range: null).
extern "C" int xr_gemm_f32_parts(void* out, const float* a, const float* w, const float* bias, int M, int N, int K, int lda, int ldo,
                                 int out_dtype, int accumulate, int plan, void* partial, hipStream_t stream) {
    XR_REQUIRE(M > 0 && N > 0 && K > 0 && K % (2 * PK) == 0, "gemm: bad sizes M=%d N=%d K=%d (K a multiple of %d)", M, N, K, 2 * PK);
    XR_REQUIRE(lda >= K && ldo >= N, "gemm: row strides lda=%d ldo=%d are shorter than K=%d N=%d", lda, ldo, K, N);
    XR_REQUIRE(lda % 4 == 0 && (((uintptr_t)a | (uintptr_t)w) % 16) == 0, "gemm: operands that are not 16-byte aligned rows");
    XR_REQUIRE(out_dtype == XR_F32 || (out_dtype == XR_BF16 && !accumulate), "gemm: bad output type %d", out_dtype);
    XR_REQUIRE(plan > 0, "gemm: no plan %d", plan);
    const int tile = (plan - 1) % XR_PARTS_TILES, ranges = (plan - 1) / XR_PARTS_TILES + 1;
    XR_REQUIRE(ranges == 1 || (partial && (uintptr_t)partial % 8 == 0), "gemm: no room for the sums of %d ranges", ranges);
    float2* const p = (float2*)partial;
    if (tile == 0) return launch_parts<1, 4, 1, 1, 2, 2>(out, a, w, bias, M, N, K, lda, ldo, out_dtype, accumulate, ranges, p, stream);
    if (tile == 1) return launch_parts<2, 2, 1, 1, 3, 2>(out, a, w, bias, M, N, K, lda, ldo, out_dtype, accumulate, ranges, p, stream);
    if (tile == 2) return launch_parts<2, 2, 1, 2, 2, 2>(out, a, w, bias, M, N, K, lda, ldo, out_dtype, accumulate, ranges, p, stream);
    return launch_parts<2, 4, 2, 1, 2, 2>(out, a, w, bias, M, N, K, lda, ldo, out_dtype, accumulate, ranges, p, stream);
}
