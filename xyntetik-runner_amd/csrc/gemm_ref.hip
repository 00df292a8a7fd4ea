// Matrix product out[M,N] = a[M,K] * w[N,K]^T (+ bias) in true 32 bits: the matrix product of the 32-bit
// path, and (k_gemm_ref, FMA only, any types and alignment) the yardstick of the bfloat16 MFMA kernels.
// Weights are [n_out][n_in] row-major as the reference keeps them
// (src/model.c:193-205).  A row's result does not depend on the rows beside it, but the order
// of its sum over k depends on how many rows the product has: with more than 16 rows the tile
// kernels (k_gemm_f32 on the matrix cores, k_gemm_ref where operands are not 16-byte aligned or not 32-bit)
// sum in two levels, with up to 16 the kernel further down
// (k_gemv_ref) gives every lane every 64th group of four columns and adds the lanes' sums in a
// tree.  A token's 32-bit result therefore differs in its last bits between a step of 16 rows and
// one of 17 (both stay within 1e-6 of the exact product at K = 14,336), and between steps of so many rows that
// k_gemm_f32 takes another number of waves for a tile (a run is then 128 columns of every second slice of 32).
// The tile kernels' two levels: runs of RBK * RB_FOLD = 128 columns are summed one after another, and the runs'
// sums are added up with a compensated (Kahan) sum.  One running 32-bit sum over the 14,336
// columns of a wide feed-forward loses about 1e-5 of the result to rounding, which at such
// widths is as much as a real fault may be; summed this way a product is about ten times closer
// to the exact one, so the 32-bit path can be held to the tolerance that small models are.
#include "common.h"
#include "async_copy.h"

#define RBM 64
#define RBN 64
#define RBK 16
#define RB_FOLD 8

// A run's sum into the sum of the runs, by Kahan's compensated addition.  What is lost is at most half a unit of the last place,
// 1e31: the bounds only act where the sum is infinite, whose next compensation would make it NaN (2048 x 16384 x 2048 takes 1,161
// us without them, 1,170 with).
__device__ inline void fold_run(float& acc, float& tot, float& lost) {
    const float y = acc - lost, t = tot + y;
    lost = __builtin_amdgcn_fmed3f((t - tot) - y, -1e32f, 1e32f);
    tot = t;
    acc = 0.f;
}

template <typename TI, typename TO, bool ACC>
__global__ __launch_bounds__(256) void k_gemm_ref(TO* __restrict__ out, const TI* __restrict__ a,
                                                   const TI* __restrict__ w, const float* __restrict__ bias,
                                                   int M, int N, int K, int lda, int ldo) {
    __shared__ float As[RBK][RBM + 4];
    __shared__ float Ws[RBK][RBN + 4];
    int m0 = blockIdx.y * RBM, n0 = blockIdx.x * RBN;
    int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
    float acc[4][4], tot[4][4], lost[4][4];      // the run's sum, the sum of the runs, what that sum has lost
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = tot[i][j] = lost[i][j] = 0.f;
    auto fold = [&]() {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) fold_run(acc[i][j], tot[i][j], lost[i][j]);
    };

    int slice = 0;
    for (int k0 = 0; k0 < K; k0 += RBK, ++slice) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            int idx = threadIdx.x + e * 256;
            int r = idx >> 4, kk = idx & 15;
            int gm = m0 + r, gn = n0 + r, gk = k0 + kk;
            As[kk][r] = (gm < M && gk < K) ? ld<TI>(a, (size_t)gm * lda + gk) : 0.f;
            Ws[kk][r] = (gn < N && gk < K) ? ld<TI>(w, (size_t)gn * K + gk) : 0.f;
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < RBK; ++kk) {
            float av[4], wv[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) av[i] = As[kk][ty * 4 + i];
#pragma unroll
            for (int j = 0; j < 4; ++j) wv[j] = Ws[kk][tx * 4 + j];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(av[i], wv[j], acc[i][j]);
        }
        __syncthreads();
        if (slice % RB_FOLD == RB_FOLD - 1) fold();
    }
    fold();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        int gm = m0 + ty * 4 + i;
        if (gm >= M) continue;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            int gn = n0 + tx * 4 + j;
            if (gn >= N) continue;
            float v = tot[i][j];
            if (bias) v += bias[gn];
            size_t o = (size_t)gm * ldo + gn;
            if (ACC) v += ld<TO>(out, o);
            st<TO>(out, o, v);
        }
    }
}

// The same sums on the matrix cores (v_mfma_f32_32x32x2_f32: 32-bit operands, products and sums), 16-byte pieces copied
// straight into LDS.  A workgroup of four waves, two by two, makes a tile of BM x BN from slices of 32 columns, STAGES - 1 of
// them on their way while one is used: a slice's products take a wave 1,000 to 2,000 cycles, less than a trip to memory
// (with the next slice alone ahead of the products, through registers, 401 x 2048 x 8192 took 213 us and 2048 x 16384 x 2048 1,237).
// An MFMA step takes two columns, one from each half of the wave; which two does not matter as long as both operands agree,
// so a lane reads four columns at once (its half's) and feeds four steps with them.  A row's eight pieces lie turned by
// half its number, so that the reads of 16 rows meet no bank twice.  Workgroup i runs on XCD i % 8, and an XCD takes an
// eighth of the tiles, row tiles first: a weight tile comes from memory for one XCD (401 x 128256 x 2048, 1 GB of weights, read
// them four times with the column tiles first).
// Bound by the matrix cores' 32-bit rate (157 TFLOP/s): 2048 x 16384 x 2048 at 112 to 119 TFLOP/s, 401 x 128256 x 2048 at 100 to 105
// (84 before), 401 x 2048 x 8192 at 79 (63; 224 tiles for 256 compute units); the FMA kernel above reached 18 to 25.
typedef float f32x16 __attribute__((ext_vector_type(16)));
#define FBK 32

// KG 2 (few tiles): two sets of four waves make the same tile, each from every second slice, and add their sums up at the end:
// two waves a SIMD, one of which works while the other waits for its reads.
template <typename TO, bool ACC, int BM, int BN, int STAGES, int KG>
__global__ __launch_bounds__(256 * KG, 2) void k_gemm_f32(TO* __restrict__ out, const float* __restrict__ a, const float* __restrict__ w,
                                                     const float* __restrict__ bias, int M, int N, int K, int lda, int ldo) {
    constexpr int TM = BM / 64, TN = BN / 64;           // 32 x 32 tiles a wave
    constexpr int ROWS = BM + BN, CH = FBK / 4;         // rows of a slice (activations, then weights), pieces of a row
    constexpr int LOADS = ROWS * CH / 256;              // copies a lane and stage (KG slices)
    static_assert(BM % 32 == 0 && LOADS * STAGES < 64, "whole copy instructions, and a count that fits the counter");
    extern __shared__ __align__(16) float4 lds[];       // [STAGES][KG][ROWS][CH]
    const int tid = threadIdx.x, lane = tid & 63, wave8 = __builtin_amdgcn_readfirstlane(tid >> 6), wave = wave8 & 3, set = wave8 >> 2;
    const int tiles_m = (M + BM - 1) / BM, tiles = tiles_m * ((N + BN - 1) / BN);
    const int tile = (int)(blockIdx.x & 7) * ((tiles + 7) >> 3) + (int)(blockIdx.x >> 3);
    if (tile >= tiles) return;
    const int m0 = tile % tiles_m * BM, n0 = tile / tiles_m * BN;
    const int wm = (wave >> 1) * (BM / 2), wn = (wave & 1) * (BN / 2);
    auto turn = [](int r) { return (r >> 1) & (CH - 1); };
    // this lane's pieces of a slice: 8 rows a copy instruction
    const float* src[LOADS];
    int col[LOADS];
    const float* zero_src = reinterpret_cast<const float*>(xr_zero_chunk);
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
        const int all = (i * 4 * KG + wave8) * 8 + (lane >> 3), r = all % ROWS;
        col[i] = ((lane & (CH - 1)) ^ turn(r)) * 4 + all / ROWS * FBK;
        const int m = m0 + r, n = n0 + r - BM;
        src[i] = r < BM ? (m < M ? a + (size_t)m * lda + col[i] : nullptr) : (n < N ? w + (size_t)n * K + col[i] : nullptr);
    }
    const uint32_t lds_wave = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)lds + (uint32_t)(wave8 * 64 * 16));
    auto copy = [&](int stage) {                        // (pieces that do not exist are zeros)
        const uint32_t dst = lds_wave + (uint32_t)(stage % STAGES * KG * ROWS * CH * 16);
#pragma unroll
        for (int i = 0; i < LOADS; ++i)
            lds_dma16(src[i] && stage * KG * FBK + col[i] < K ? src[i] + (size_t)stage * KG * FBK : zero_src, dst + i * KG * 256 * 16);
    };
    f32x16 acc[TM][TN], tot[TM][TN], lost[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = tot[i][j][e] = lost[i][j][e] = 0.f;
    auto fold = [&]() {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    float x = acc[i][j][e], t = tot[i][j][e], l = lost[i][j][e];
                    fold_run(x, t, l);
                    acc[i][j][e] = x; tot[i][j][e] = t; lost[i][j][e] = l;
                }
    };
    const int row = lane & 31, half = (lane >> 5) * 4;
    const int n_stages = (K + KG * FBK - 1) / (KG * FBK);
#pragma unroll
    for (int st = 0; st < STAGES - 1; ++st) copy(st);
    for (int stage = 0; stage < n_stages; ++stage) {
        wait_vmcnt<LOADS * (STAGES - 2)>();             // this wave's share of the stage has landed
        __builtin_amdgcn_s_barrier();                   // every wave's has, and nobody reads the stage before any more
        copy(stage + STAGES - 1);
        const float4* As = lds + (stage % STAGES * KG + set) * ROWS * CH;
        const float4* Ws = As + BM * CH;
#pragma unroll
        for (int kk = 0; kk < CH; kk += 2) {
            const int c = kk + (lane >> 5);
            float4 fa[TM], fw[TN];
#pragma unroll
            for (int i = 0; i < TM; ++i) { const int r = wm + 32 * i + row; fa[i] = As[r * CH + (c ^ turn(r))]; }
#pragma unroll
            for (int j = 0; j < TN; ++j) { const int r = wn + 32 * j + row; fw[j] = Ws[r * CH + (c ^ turn(r))]; }
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32((&fa[i].x)[s], (&fw[j].x)[s], acc[i][j], 0, 0, 0);
        }
        if ((stage + 1) % (RBK * RB_FOLD / FBK) == 0) fold();
    }
    wait_vmcnt<0>();                                    // the trailing copies of zeros
    fold();
    if constexpr (KG == 2) {                            // the second set's sums, and what they lack
        static_assert(2 * TM * TN * 4 * 1024 <= STAGES * KG * ROWS * FBK, "room for both");
        __syncthreads();
        float* other = reinterpret_cast<float*>(lds) + wave * 2 * TM * TN * 1024 + lane;
        if (set == 1)
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int e = 0; e < 16; ++e) {
                        other[((i * TN + j) * 32 + e) * 64] = tot[i][j][e];
                        other[((i * TN + j) * 32 + 16 + e) * 64] = lost[i][j][e];
                    }
        __syncthreads();
        if (set == 1) return;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    // the two sums, what that addition loses (exactly: Knuth's two-sum), and what both lack, rounded once (an
                    // infinite sum's loss is no number: the bounds make it one, as in fold_run).  One more run of the first
                    // set instead rounds the second's sum on the way: 17 x 2048 x 14336 of one sign 0.56 units of 2^-24 off, 0.42 so.
                    const float x = tot[i][j][e], y = other[((i * TN + j) * 32 + e) * 64], t = x + y, z = t - x;
                    const float lacks = ((x - (t - z)) + (y - z)) - (lost[i][j][e] + other[((i * TN + j) * 32 + 16 + e) * 64]);
                    tot[i][j][e] = t + __builtin_amdgcn_fmed3f(lacks, -1e32f, 1e32f);
                }
    }
    // a lane has column lane % 32 and rows 8 (e / 4) + 4 (lane / 32) + e % 4 of a tile
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        const int n = n0 + wn + 32 * j + row;
        if (n >= N) continue;
        const float add = bias ? bias[n] : 0.f;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int m = m0 + wm + 32 * i + 8 * (e >> 2) + half + (e & 3);
                if (m >= M) continue;
                const size_t at = (size_t)m * ldo + n;
                float v = tot[i][j][e];
                if (bias) v += add;
                if (ACC) v += ld<TO>(out, at);
                st<TO>(out, at, v);
            }
    }
}

template <int BM, int BN, int STAGES, int KG>
static int launch_gemm_f32(void* out, const float* a, const float* w, const float* bias, int M, int N, int K, int lda, int ldo,
                           int out_dtype, int accumulate, hipStream_t stream) {
    const long long tiles = (long long)((M + BM - 1) / BM) * ((N + BN - 1) / BN);
    XR_REQUIRE(tiles < (1ll << 28), "gemm: %lld tiles", tiles);
    const unsigned blocks = 8 * (unsigned)((tiles + 7) / 8);
    constexpr int smem = STAGES * KG * (BM + BN) * FBK * 4;
    auto run = [&](auto kernel, auto* to) {
        if (smem > 65536) {
            const hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, smem);
            if (e != hipSuccess) (void)hipGetLastError();
            XR_REQUIRE(e == hipSuccess, "gemm: cannot reserve %d bytes of LDS: %s", smem, hipGetErrorString(e));
        }
        kernel<<<blocks, 256 * KG, smem, stream>>>(to, a, w, bias, M, N, K, lda, ldo);
        return XR_OK;
    };
    if (out_dtype == XR_BF16) return run(k_gemm_f32<bf16_t, false, BM, BN, STAGES, KG>, (bf16_t*)out);
    if (accumulate) return run(k_gemm_f32<float, true, BM, BN, STAGES, KG>, (float*)out);
    return run(k_gemm_f32<float, false, BM, BN, STAGES, KG>, (float*)out);
}

// Up to 16 rows of 32-bit operands (decoded tokens): the product is bound by how fast the weights
// arrive, and the tile kernel above, 64 weight rows a workgroup, leaves most of the chip idle then
// (a decode step of the Llama-3.1-8B shape took 136 ms).  Here a wave takes COLS weight rows: a lane
// sums, for every row of `a` and each of them, the columns 4 l .. 4 l + 3 (mod 256) in ascending
// order by FMA, and the lanes' sums are added in a fixed tree.  A row's result does not depend
// on the rows beside it; it differs from the tile kernel's by the order of the sum only.
// All sums go through the tree at once: at the first step a lane hands half of its sums to the lane 32 further and
// takes over the other half, and so on, until a lane holds the whole sum of one (row, weight row) or what is left of few sums
// goes on as a plain tree.  The additions are those of a tree a sum, in the same order.  (2048 x 2048, 16 rows: 13 us with 2 weight
// rows a wave and one tree, 46 us with 8 weight rows and a tree of six steps for each of 128 sums.)
template <int N>
__device__ inline void tree_sums(float (&v)[N], int lane, int& mine) {
    mine = 0;
    int o = 32;
#pragma unroll
    for (int n = N; n > 1; n >>= 1) {
        if (o > 0) {
            const bool up = lane & o;
            mine = 2 * mine + (up ? 1 : 0);
#pragma unroll
            for (int i = 0; i < n / 2; ++i) {
                // (both values first: a choice between two elements in place is an index that is not known, which
                // costs a choice among all elements: 32 sums took 2,000 selects and 4 us)
                const float low = v[i], high = v[n / 2 + i];
                v[i] = (up ? high : low) + __shfl_xor(up ? low : high, o, 64);
            }
            o >>= 1;
        }
    }
    for (; o > 0; o >>= 1) v[0] += __shfl_xor(v[0], o, 64);
}

template <int MT, int COLS, typename TO, bool ACC>
__global__ __launch_bounds__(256) void k_gemv_ref(TO* __restrict__ out, const float* __restrict__ a,
                                                   const float* __restrict__ w, const float* __restrict__ bias,
                                                   int M, int N, int K, int lda, int ldo) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int n0 = (blockIdx.x * 4 + wave) * COLS;
    if (n0 >= N) return;
    float acc[COLS][MT];
#pragma unroll
    for (int c = 0; c < COLS; ++c)
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[c][m] = 0.f;
    for (int k = lane * 4; k < K; k += 256) {
        float4 av[MT];
#pragma unroll
        for (int m = 0; m < MT; ++m)
            av[m] = m < M ? *reinterpret_cast<const float4*>(a + (size_t)m * lda + k) : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int c = 0; c < COLS; ++c) {
            const int n = n0 + c;
            const float4 wv = n < N ? *reinterpret_cast<const float4*>(w + (size_t)n * K + k) : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                float t = acc[c][m];
                t = fmaf(av[m].x, wv.x, t);
                t = fmaf(av[m].y, wv.y, t);
                t = fmaf(av[m].z, wv.z, t);
                t = fmaf(av[m].w, wv.w, t);
                acc[c][m] = t;
            }
        }
    }
    // 64 sums at a time (a lane ends with one), or all of them where they are fewer
    constexpr int ALL = COLS * MT, GROUP = ALL < 64 ? ALL : 64;
#pragma unroll
    for (int g0 = 0; g0 < ALL; g0 += GROUP) {
        float v[GROUP];
#pragma unroll
        for (int i = 0; i < GROUP; ++i) v[i] = acc[(g0 + i) / MT][(g0 + i) % MT];
        int mine;
        tree_sums<GROUP>(v, lane, mine);
        const int n = n0 + (g0 + mine) / MT, m = (g0 + mine) % MT;
        if ((lane & (64 / GROUP - 1)) == 0 && m < M && n < N) {
            float s = v[0];
            if (bias) s += bias[n];
            const size_t at = (size_t)m * ldo + n;
            if (ACC) s += ld<TO>(out, at);
            st<TO>(out, at, s);
        }
    }
}

template <int MT, int COLS>
static void launch_gemv_cols(void* out, const float* a, const float* w, const float* bias, int M, int N, int K,
                             int lda, int ldo, int out_dtype, int accumulate, hipStream_t stream) {
    const unsigned blocks = (unsigned)((N + 4 * COLS - 1) / (4 * COLS));
    if (out_dtype == XR_BF16) k_gemv_ref<MT, COLS, bf16_t, false><<<blocks, 256, 0, stream>>>((bf16_t*)out, a, w, bias, M, N, K, lda, ldo);
    else if (accumulate) k_gemv_ref<MT, COLS, float, true><<<blocks, 256, 0, stream>>>((float*)out, a, w, bias, M, N, K, lda, ldo);
    else k_gemv_ref<MT, COLS, float, false><<<blocks, 256, 0, stream>>>((float*)out, a, w, bias, M, N, K, lda, ldo);
}

// Weight rows a wave: more share the reads of `a` and cost fewer sums, fewer spread over more compute units.  One row: 2.  More
// rows: 2 for as long as weight rows are few, then 4, and 8 where K is long enough to keep them busy (or rows are 16).  Times in us
// with 2, 4 and 8, weights from memory: 4096 x 4096, 8 rows 19, 22, 29; 8192 x 2048, 16 rows 32, 22, 28; 14336 x 4096, 16 rows 105, 76, 61;
// 16384 x 2048, 3 rows 27, 27, 35; 28672 x 4096, 8 rows 132, 102, 101.
template <int MT>
static int gemv_cols(int N, int K) {
    if (MT == 1 || N < (MT == 4 ? 16384 : MT == 8 ? 6144 : 4096)) return 2;
    return (K >= 4096 && N >= 8192) || (MT == 16 && N >= 16384) ? 8 : 4;
}

template <int MT>
static void launch_gemv_ref(void* out, const float* a, const float* w, const float* bias, int M, int N, int K,
                            int lda, int ldo, int out_dtype, int accumulate, hipStream_t stream) {
    const int cols = gemv_cols<MT>(N, K);
    if (cols == 8) launch_gemv_cols<MT, 8>(out, a, w, bias, M, N, K, lda, ldo, out_dtype, accumulate, stream);
    else if (cols == 4) launch_gemv_cols<MT, 4>(out, a, w, bias, M, N, K, lda, ldo, out_dtype, accumulate, stream);
    else launch_gemv_cols<MT, 2>(out, a, w, bias, M, N, K, lda, ldo, out_dtype, accumulate, stream);
}

// accumulate != 0: out (float) += product.
extern "C" int xr_gemm_ref(void* out, const void* a, const void* w, const float* bias, int M, int N, int K,
                           int lda, int ldo, int in_dtype, int out_dtype, int accumulate, hipStream_t stream) {
    XR_REQUIRE(M >= 0 && N > 0 && K > 0, "gemm: bad sizes M=%d N=%d K=%d", M, N, K);
    XR_REQUIRE(lda >= K && ldo >= N, "gemm: row strides lda=%d ldo=%d are shorter than K=%d N=%d", lda, ldo, K, N);
    XR_REQUIRE(!accumulate || out_dtype == XR_F32, "gemm: accumulation needs a 32-bit output");
    if (M == 0) return XR_OK;
    if (in_dtype == XR_F32 && (out_dtype == XR_F32 || out_dtype == XR_BF16) && K % 4 == 0 && lda % 4 == 0 &&
        ((uintptr_t)a % 16) == 0 && ((uintptr_t)w % 16) == 0) {
        const float* af = (const float*)a;
        const float* wf = (const float*)w;
        if (M > 16) {
            // 64 x 128 tiles read three quarters of what 64 x 64 ones read from L2, but two of their workgroups fill a compute
            // unit: they are taken where there are at least that many (larger tiles with their three sums a value spill)
            const long long tiles = (long long)((M + 63) / 64) * ((N + 127) / 128);
            // (with no more 64 x 64 tiles than compute units, eight waves a tile: 401 x 2048 x 8192 195 us with four, 171 with eight)
            const long long small = (long long)((M + 63) / 64) * ((N + 63) / 64);
            const int rc = tiles >= 512 ? launch_gemm_f32<64, 128, 3, 1>(out, af, wf, bias, M, N, K, lda, ldo, out_dtype, accumulate, stream)
                         : small > 256  ? launch_gemm_f32<64, 64, 4, 1>(out, af, wf, bias, M, N, K, lda, ldo, out_dtype, accumulate, stream)
                                        : launch_gemm_f32<64, 64, 3, 2>(out, af, wf, bias, M, N, K, lda, ldo, out_dtype, accumulate, stream);
            if (rc != XR_OK) return rc;
            XR_CHECK_LAUNCH("gemm_f32");
            return XR_OK;
        }
        if (M == 1) launch_gemv_ref<1>(out, af, wf, bias, M, N, K, lda, ldo, out_dtype, accumulate, stream);
        else if (M <= 4) launch_gemv_ref<4>(out, af, wf, bias, M, N, K, lda, ldo, out_dtype, accumulate, stream);
        else if (M <= 8) launch_gemv_ref<8>(out, af, wf, bias, M, N, K, lda, ldo, out_dtype, accumulate, stream);
        else launch_gemv_ref<16>(out, af, wf, bias, M, N, K, lda, ldo, out_dtype, accumulate, stream);
        XR_CHECK_LAUNCH("gemv_ref");
        return XR_OK;
    }
    dim3 grid((N + RBN - 1) / RBN, (M + RBM - 1) / RBM);
#define G(TI, TO, ACC) k_gemm_ref<TI, TO, ACC><<<grid, 256, 0, stream>>>((TO*)out, (const TI*)a, (const TI*)w, bias, M, N, K, lda, ldo)
    if (in_dtype == XR_F32 && out_dtype == XR_F32) { if (accumulate) G(float, float, true); else G(float, float, false); }
    else if (in_dtype == XR_BF16 && out_dtype == XR_F32) { if (accumulate) G(bf16_t, float, true); else G(bf16_t, float, false); }
    else if (in_dtype == XR_BF16 && out_dtype == XR_BF16) G(bf16_t, bf16_t, false);
    else if (in_dtype == XR_F32 && out_dtype == XR_BF16) G(float, bf16_t, false);
    else { xr_set_error("gemm: bad dtypes in=%d out=%d", in_dtype, out_dtype); return XR_BAD_ARG; }
#undef G
    XR_CHECK_LAUNCH("gemm_ref");
    return XR_OK;
}
