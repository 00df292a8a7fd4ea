// Matrix product out[M,N] = a[M,K] * w[N,K]^T (+ bias) in true 32 bits: the matrix product of the 32-bit
// path (but for products of many rows or columns, which gemm_f32_parts.hip makes), and (k_gemm_ref, FMA only, any types and alignment) the yardstick of the bfloat16 MFMA kernels.
// Weights are [n_out][n_in] row-major as the reference keeps them
// (src/model.c:193-205).  A row's result does not depend on the rows beside it, but the order
// of its sum over k depends on how many rows the product has: with more than 16 rows the tile
// kernels (k_gemm_f32 on the matrix cores, k_gemm_ref where operands are not 16-byte aligned or not 32-bit)
// sum in two levels, with up to 16 the kernel further down
// (k_gemv_ref) gives every lane every 64th group of four columns and adds the lanes' sums in a
// tree, and with up to 4 rows (xr_gemv_extra) norms them on the way, so that the norm's factor comes behind the sum instead of before
// it.  A token's 32-bit result therefore differs in its last bits between steps of 4 rows and 5, of 16 rows and
// 17 (all stay within 1e-6 of the exact product at K = 14,336), and between steps of so many rows that
// k_gemm_f32 takes another number of waves for a tile (a run is then 128 columns of every second or fourth slice of 32, or 64 of every second).
// The tile kernels' two levels: runs of RBK * RB_FOLD = 128 columns (64 in one tile, see f32_tile) are summed one after another, and the runs'
// sums are added up with a compensated (Kahan) sum.  One running 32-bit sum over the 14,336
// columns of a wide feed-forward loses about 1e-5 of the result to rounding, which at such
// widths is as much as a real fault may be; summed this way a product is about ten times closer
// to the exact one, so the 32-bit path can be held to the tolerance that small models are.
#include <type_traits>

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
// straight into LDS.  A workgroup makes a tile of BM x BN from slices of 32 columns, STAGES - 1 of
// them on their way while one is used (a slice's products take a wave 1,000 to 2,000 cycles).
// An MFMA step takes two columns, one from each half of the wave; which two does not matter as long as both operands agree,
// so a lane reads four columns at once (its half's) and feeds four steps with them.  A row's eight pieces lie turned by
// half its number, so that the reads of 16 rows meet no bank twice.  Workgroup i runs on XCD i % 8, and an XCD takes an
// eighth of the tiles, row tiles first: a weight tile comes from memory for one XCD (401 x 128256 x 2048, 1 GB of weights, read
// them four times with the column tiles first).
// Bound by the matrix cores' 32-bit rate (157 TFLOP/s; 153 is what the card's library gets of it on 8192 x 8192 x 8192) and the sums of
// runs: 2048 x 16384 x 2048 at 131 TFLOP/s, 401 x 128256 x 2048 at 126, 401 x 2048 x 8192 at 95 (416 rows of tiles, 3.25 tiles of
// 32 x 32 a compute unit where four are the fullest one's); the FMA kernel above reached 18 to 25.
typedef float f32x16 __attribute__((ext_vector_type(16)));
#define FBK 32

// GM x GN waves make a tile, each its 32 x 32 tiles.  KG > 1 (few tiles): KG sets of so many waves make the same tile, each from every
// KG-th slice, and add their sums up at the end.  The products of one wave do not overlap its own sums of runs, nor its waits for reads
// and for the other waves, so what keeps the matrix cores busy is waves: two stages of 64 x 64 or 32 x 64 in LDS leave room for four and
// more a SIMD.  (2048 x 16384 x 2048: three stages of 64 x 128, two waves a SIMD, 1,302 us; with a run's four stages unrolled, so that no
// sums move between registers, 1,187; two stages of 64 x 64 and four waves 1,070.  Without the sums of runs 1,034, and they cannot go.)
// WHOLE: K is whole stages.  A row that does not exist is then read from the last one that does (its results are not stored), so
// that a copy is a base in scalar registers and a fixed offset a lane; else a lane's pieces beyond the matrices are zeros.
// RUN: a run's stages.
template <typename TO, bool ACC, int GM, int GN, int BM, int BN, int STAGES, int KG, bool WHOLE, int RUN = RBK * RB_FOLD / FBK>
__global__ __launch_bounds__(64 * GM * GN * KG, 4) void k_gemm_f32(TO* __restrict__ out, const float* __restrict__ a, const float* __restrict__ w,
                                                     const float* __restrict__ bias, int M, int N, int K, int lda, int ldo) {
    constexpr int WAVES = GM * GN;                      // of a set
    constexpr int TM = BM / 32 / GM, TN = BN / 32 / GN; // 32 x 32 tiles a wave
    constexpr int ROWS = BM + BN, CH = FBK / 4;         // rows of a slice (activations, then weights), pieces of a row
    constexpr int LOADS = ROWS * CH / (64 * WAVES);     // copies a lane and stage (KG slices)
    static_assert(ROWS * CH % (64 * WAVES) == 0 && BM % 32 == 0 && LOADS * STAGES < 64, "whole copy instructions, and a count that fits the counter");
    extern __shared__ __align__(16) float4 lds[];       // [STAGES][KG][ROWS][CH]
    const int tid = threadIdx.x, lane = tid & 63, wave8 = __builtin_amdgcn_readfirstlane(tid >> 6), wave = wave8 % WAVES, set = wave8 / WAVES;
    const int tiles_m = (M + BM - 1) / BM, tiles = tiles_m * ((N + BN - 1) / BN);
    const int tile = (int)(blockIdx.x & 7) * ((tiles + 7) >> 3) + (int)(blockIdx.x >> 3);
    if (tile >= tiles) return;
    const int m0 = tile % tiles_m * BM, n0 = tile / tiles_m * BN;
    const int wm = wave / GN * (BM / GM), wn = wave % GN * (BN / GN);
    auto turn = [](int r) { return (r >> 1) & (CH - 1); };
    const int n_stages = (K + KG * FBK - 1) / (KG * FBK);
    // this lane's pieces of a slice: 8 rows a copy instruction, the first of a stage activations and weights by turns of ROWS / 8
    const float* src[LOADS];
    int col[LOADS];
    uint32_t off[LOADS];
    const float* zero_src = reinterpret_cast<const float*>(xr_zero_chunk);
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
        const int all = (i * WAVES * KG + wave8) * 8 + (lane >> 3), r = all % ROWS;
        col[i] = ((lane & (CH - 1)) ^ turn(r)) * 4 + all / ROWS * FBK;
        const int m = m0 + r, n = n0 + r - BM;
        if constexpr (WHOLE)
            off[i] = r < BM ? (uint32_t)((m < M ? r : M - 1 - m0) * (size_t)lda + col[i]) * 4u : (uint32_t)((n < N ? r - BM : N - 1 - n0) * (size_t)K + col[i]) * 4u;
        else
            src[i] = r < BM ? (m < M ? a + (size_t)m * lda + col[i] : nullptr) : (n < N ? w + (size_t)n * K + col[i] : nullptr);
    }
    const float* a_tile = a + (size_t)m0 * lda;
    const float* w_tile = w + (size_t)n0 * K;
    const uint32_t lds_wave = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)lds + (uint32_t)(wave8 * 64 * 16));
    auto copy = [&](int stage) {
        const uint32_t dst = lds_wave + (uint32_t)(stage % STAGES * KG * ROWS * CH * 16);
        if constexpr (WHOLE) {
            const int s = stage < n_stages ? stage : n_stages - 1;       // (past the end the last stage once more: as many copies on their way)
            const float* const a_now = a_tile + (size_t)s * KG * FBK;
            const float* const w_now = w_tile + (size_t)s * KG * FBK;
#pragma unroll
            for (int i = 0; i < LOADS; ++i) {
                const bool act = (i * WAVES * KG + wave8) * 8 % ROWS < BM;
                lds_dma16_base(act ? a_now : w_now, off[i], dst + i * KG * WAVES * 64 * 16);
            }
        } else {                                                         // (pieces that do not exist are zeros)
#pragma unroll
            for (int i = 0; i < LOADS; ++i)
                lds_dma16(src[i] && stage * KG * FBK + col[i] < K ? src[i] + (size_t)stage * KG * FBK : zero_src, dst + i * KG * WAVES * 64 * 16);
        }
    };
    f32x16 acc[TM][TN], tot[TM][TN], lost[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) tot[i][j][e] = lost[i][j][e] = 0.f;
    auto fold = [&]() {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    float x = acc[i][j][e], t = tot[i][j][e], l = lost[i][j][e];
                    fold_run(x, t, l);
                    tot[i][j][e] = t; lost[i][j][e] = l;
                }
    };
    const int row = lane & 31, half = (lane >> 5) * 4;
#pragma unroll
    for (int st = 0; st < STAGES - 1; ++st) copy(st);
    auto products = [&](const float4* As, auto first) {
        const float4* Ws = As + BM * CH;
        // (the operands of the next four steps are read while these are multiplied, into a second set of registers: the compiler keeps
        // one set, and a read then waits for the products before it and they for the read)
        float4 fa[2][TM], fw[2][TN];
        auto read = [&](int kk, int set_) {
            const int c = kk + (lane >> 5);
#pragma unroll
            for (int i = 0; i < TM; ++i) { const int r = wm + 32 * i + row; fa[set_][i] = As[r * CH + (c ^ turn(r))]; }
#pragma unroll
            for (int j = 0; j < TN; ++j) { const int r = wn + 32 * j + row; fw[set_][j] = Ws[r * CH + (c ^ turn(r))]; }
        };
        read(0, 0);
#pragma unroll
        for (int kk = 0; kk < CH; kk += 2) {
            const int now = (kk >> 1) & 1;
            if (kk + 2 < CH) read(kk + 2, now ^ 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j) {
                        const bool begins = decltype(first)::value && kk == 0 && s == 0;
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32((&fa[now][i].x)[s], (&fw[now][j].x)[s], begins ? f32x16{} : acc[i][j], 0, 0, 0);
                    }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    for (int run = 0; run < n_stages; run += RUN) {
#pragma unroll
        for (int u = 0; u < RUN; ++u) {
            const int stage = run + u;
            if (u > 0 && stage >= n_stages) break;
            wait_vmcnt<LOADS * (STAGES - 2)>();         // this wave's share of the stage has landed
            __builtin_amdgcn_s_barrier();               // every wave's has, and nobody reads the stage before any more
            copy(stage + STAGES - 1);
            const float4* As = lds + (stage % STAGES * KG + set) * ROWS * CH;
            if (u == 0) products(As, std::true_type{});
            else products(As, std::false_type{});
        }
        fold();
    }
    wait_vmcnt<0>();                                    // the trailing copies
    if constexpr (KG > 1) {                             // the other sets' sums, and what they lack
        static_assert(2 * TM * TN * WAVES * (KG - 1) * 1024 <= STAGES * KG * ROWS * FBK, "room for all of them");
        __syncthreads();
        float* const theirs = reinterpret_cast<float*>(lds) + wave * 2 * TM * TN * 1024 + lane;
        constexpr int SET = WAVES * 2 * TM * TN * 1024;
        if (set > 0)
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int e = 0; e < 16; ++e) {
                        theirs[(set - 1) * SET + ((i * TN + j) * 32 + e) * 64] = tot[i][j][e];
                        theirs[(set - 1) * SET + ((i * TN + j) * 32 + 16 + e) * 64] = lost[i][j][e];
                    }
        __syncthreads();
        if (set > 0) return;
        // The sets' sums one after another, what each addition loses (exactly: Knuth's two-sum), and what all of them lack,
        // rounded once (an infinite sum's loss is no number: the bounds make it one, as in fold_run).  One more run of the
        // first set instead rounds another's sum on the way: 17 x 2048 x 14336 of one sign 0.56 units of 2^-24 off, 0.42 so.
#pragma unroll 1
        for (int o = 0; o < KG - 1; ++o)
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int e = 0; e < 16; ++e) {
                        const float x = tot[i][j][e], y = theirs[o * SET + ((i * TN + j) * 32 + e) * 64], t = x + y, z = t - x;
                        lost[i][j][e] -= ((x - (t - z)) + (y - z)) - theirs[o * SET + ((i * TN + j) * 32 + 16 + e) * 64];
                        tot[i][j][e] = t;
                    }
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) tot[i][j][e] += __builtin_amdgcn_fmed3f(-lost[i][j][e], -1e32f, 1e32f);
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

template <int GM, int GN, int BM, int BN, int STAGES, int KG, int RUN = RBK * RB_FOLD / FBK>
static int launch_gemm_f32(void* out, const float* a, const float* w, const float* bias, int M, int N, int K, int lda, int ldo,
                           int out_dtype, int accumulate, hipStream_t stream) {
    const long long tiles = (long long)((M + BM - 1) / BM) * ((N + BN - 1) / BN);
    XR_REQUIRE(tiles < (1ll << 28), "gemm: %lld tiles", tiles);
    const unsigned blocks = 8 * (unsigned)((tiles + 7) / 8);
    // (32 x 32 tiles with 16-bit results are faster with their copies looked at: 33 x 768 x 768 13.4 us, 14.0 without)
    const bool whole = K % (KG * FBK) == 0 && (size_t)BM * lda < (1u << 30) && (size_t)BN * K < (1u << 30);
    constexpr int smem = STAGES * KG * (BM + BN) * FBK * 4;
    static_assert(smem <= 65536, "more LDS has to be asked for");
    auto run = [&](auto kernel, auto* to) {
        kernel<<<blocks, 64 * GM * GN * KG, smem, stream>>>(to, a, w, bias, M, N, K, lda, ldo);
        return XR_OK;
    };
    if (out_dtype == XR_BF16) return whole && KG < 4 ? run(k_gemm_f32<bf16_t, false, GM, GN, BM, BN, STAGES, KG, true, RUN>, (bf16_t*)out) : run(k_gemm_f32<bf16_t, false, GM, GN, BM, BN, STAGES, KG, false, RUN>, (bf16_t*)out);
    if (accumulate) return whole ? run(k_gemm_f32<float, true, GM, GN, BM, BN, STAGES, KG, true, RUN>, (float*)out) : run(k_gemm_f32<float, true, GM, GN, BM, BN, STAGES, KG, false, RUN>, (float*)out);
    return whole ? run(k_gemm_f32<float, false, GM, GN, BM, BN, STAGES, KG, true, RUN>, (float*)out) : run(k_gemm_f32<float, false, GM, GN, BM, BN, STAGES, KG, false, RUN>, (float*)out);
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

// NORM: the rows are an RMS norm's input, norm_w its weight: their columns are multiplied by the weight on the way, a wave adds up
// its rows' squares beside its products and scales the sums by 1 / sqrt(mean + eps).  GATED: of the COLS weight rows half are gate rows and
// half up rows (N of each, the up rows behind the gate rows), whose sums meet 32 lanes apart, and act(gate) * up is what is stored.
// (Steps of a few rows on a small model are a chain of launches: with both a layer of the decode step has 6 kernels of 9; a step of
// 3 requests on 2 layers of width 64 has 18 of 23, a replay of 17 such steps takes 2,284 us for 2,408.)
// ACC with `copy`: the sums that are stored also go there, rows of N numbers, for a product that norms them later, when the sums
// themselves may have been added to again.
struct GemvExtra {
    const float* norm_w;
    float inv_width, eps;
    int act;
    float act_param;
    float* copy;
};

template <int MT, int COLS, typename TO, bool ACC, bool NORM = false, bool GATED = false>
__global__ __launch_bounds__(256) void k_gemv_ref(TO* __restrict__ out, const float* __restrict__ a,
                                                   const float* __restrict__ w, const float* __restrict__ bias,
                                                   int M, int N, int K, int lda, int ldo, GemvExtra x) {
    constexpr int OUT = GATED ? COLS / 2 : COLS;        // outputs of a wave
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int n0 = (blockIdx.x * 4 + wave) * OUT;
    if (n0 >= N) return;
    // the c-th weight row, and the output it belongs to
    auto out_of = [&](int c) { return n0 + (GATED ? c % OUT : c); };
    auto row_of = [&](int c) { return out_of(c) + (GATED && c >= OUT ? N : 0); };
    float acc[COLS][MT], sq[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) sq[m] = 0.f;
#pragma unroll
    for (int c = 0; c < COLS; ++c)
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[c][m] = 0.f;
    for (int k = lane * 4; k < K; k += 256) {
        float4 av[MT];
#pragma unroll
        for (int m = 0; m < MT; ++m)
            av[m] = m < M ? *reinterpret_cast<const float4*>(a + (size_t)m * lda + k) : make_float4(0.f, 0.f, 0.f, 0.f);
        if constexpr (NORM) {
            const float4 g = *reinterpret_cast<const float4*>(x.norm_w + k);
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                sq[m] += av[m].x * av[m].x + av[m].y * av[m].y + av[m].z * av[m].z + av[m].w * av[m].w;
                av[m] = make_float4(av[m].x * g.x, av[m].y * g.y, av[m].z * g.z, av[m].w * g.w);
            }
        }
#pragma unroll
        for (int c = 0; c < COLS; ++c) {
            const float4 wv = out_of(c) < N ? *reinterpret_cast<const float4*>(w + (size_t)row_of(c) * K + k) : make_float4(0.f, 0.f, 0.f, 0.f);
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
    float scale[MT];
    if constexpr (NORM) {
#pragma unroll
        for (int m = 0; m < MT; ++m) scale[m] = 1.0f / sqrtf(wave_sum(sq[m]) * x.inv_width + x.eps);
    }
    // 64 sums at a time (a lane ends with one), or all of them where they are fewer
    constexpr int ALL = COLS * MT, GROUP = ALL < 64 ? ALL : 64;
    static_assert(!GATED || (ALL <= 64 && ALL >= 2), "a gate's sum and its up row's are half the sums apart: the tree's first step, 32 lanes");
#pragma unroll
    for (int g0 = 0; g0 < ALL; g0 += GROUP) {
        float v[GROUP];
#pragma unroll
        for (int i = 0; i < GROUP; ++i) v[i] = acc[(g0 + i) / MT][(g0 + i) % MT];
        int mine;
        tree_sums<GROUP>(v, lane, mine);
        const int c = (g0 + mine) / MT, n = out_of(c), m = (g0 + mine) % MT;
        float s = v[0];
        if constexpr (NORM) {
            float f = scale[0];
#pragma unroll
            for (int i = 1; i < MT; ++i) f = m == i ? scale[i] : f;
            s *= f;
        }
        if (bias && n < N) s += bias[row_of(c)];
        if constexpr (GATED) {
            const float up = __shfl_xor(s, 32, 64);
            s = gate_value<false>(x.act, x.act_param, s, up);
        }
        if ((lane & (64 / GROUP - 1)) == 0 && m < M && n < N && !(GATED && c >= OUT)) {
            const size_t at = (size_t)m * ldo + n;
            if (ACC) s += ld<TO>(out, at);
            st<TO>(out, at, s);
            if (ACC && x.copy) x.copy[(size_t)m * N + n] = s;
        }
    }
}

template <int MT, int COLS>
static void launch_gemv_cols(void* out, const float* a, const float* w, const float* bias, int M, int N, int K,
                             int lda, int ldo, int out_dtype, int accumulate, float* copy, hipStream_t stream) {
    const unsigned blocks = (unsigned)((N + 4 * COLS - 1) / (4 * COLS));
    GemvExtra x{};
    x.copy = copy;
    if (out_dtype == XR_BF16) k_gemv_ref<MT, COLS, bf16_t, false><<<blocks, 256, 0, stream>>>((bf16_t*)out, a, w, bias, M, N, K, lda, ldo, x);
    else if (accumulate) k_gemv_ref<MT, COLS, float, true><<<blocks, 256, 0, stream>>>((float*)out, a, w, bias, M, N, K, lda, ldo, x);
    else k_gemv_ref<MT, COLS, float, false><<<blocks, 256, 0, stream>>>((float*)out, a, w, bias, M, N, K, lda, ldo, x);
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
                            int lda, int ldo, int out_dtype, int accumulate, hipStream_t stream, float* copy = nullptr) {
    const int cols = gemv_cols<MT>(N, K);
    if (cols == 8) launch_gemv_cols<MT, 8>(out, a, w, bias, M, N, K, lda, ldo, out_dtype, accumulate, copy, stream);
    else if (cols == 4) launch_gemv_cols<MT, 4>(out, a, w, bias, M, N, K, lda, ldo, out_dtype, accumulate, copy, stream);
    else launch_gemv_cols<MT, 2>(out, a, w, bias, M, N, K, lda, ldo, out_dtype, accumulate, copy, stream);
}

// microseconds of a 32-bit product in tiles of bm x bn made by `waves` waves in `sets`, as f32_tile counts them: `column`
// ns for a column of 32 x 32 results, `ragged` times that where K is no whole stages, `tile` us for a tile's first stage and its sums' way out
static double f32_tile_us(int M, int N, int K, int bm, int bn, int waves, int sets, double column, double ragged, double tile) {
    const double tiles = (double)((M + bm - 1) / bm) * ((N + bn - 1) / bn), most = (double)(((long long)tiles + 255) / 256);
    const double mean = tiles / 256 > 1.0 ? tiles / 256 : 1.0, simd = most * waves / 4.0, ns = K % (sets * FBK) == 0 ? column : column * ragged;
    const double products = (0.722 * most + 0.278 * mean) * ((bm * bn / 1024) * (double)K * ns * 1e-3 + tile) * (simd + 0.501) / simd;
    const double weights = (double)N * K * 4 / 5.0e6;
    return products > weights ? products : weights;
}

// that of tiles 0 to 3
static void f32_tile_times(int M, int N, int K, double (&us)[4]) {
    us[0] = f32_tile_us(M, N, K, 32, 128, 4, 1, 3.84, 1.03, 1.80);
    us[1] = f32_tile_us(M, N, K, 64, 64, 8, 2, 3.58, 1.07, 3.17);
    us[2] = f32_tile_us(M, N, K, 32, 64, 4, 2, 4.07, 1.06, 1.76);
    us[3] = f32_tile_us(M, N, K, 32, 32, 4, 4, 4.49, 1.17, 3.10);
}

// Which tile makes a 32-bit product of more than 16 rows: 0 32 x 128 (one set of waves), 1 64 x 64 (two), 2 32 x 64 (two), 3 32 x 32 (four),
// 4 64 x 64 (two) in runs of 64 columns.
#define XR_F32_TILES 5
static int f32_tile(int M, int N, int K) {
    // The tile that should take the least time: a compute unit's tiles (the fullest one's, and on average) do their products at
    // a rate that grows with its waves (w of them a SIMD: w / (w + 0.5)), less where K is no whole stages (what is copied is
    // then looked at piece by piece), and each pays for its beginning and end.  Fitted to 2,400 timed launches (31 products, 64 to 128,256
    // weight rows, K 64 to 14,336, 17 to 2,048 rows, weights from memory): 0.3% above the best of the four on average.  (Without a
    // tile's own time, fitted to K from 2,048 on, 1.9%: 1024 x 768 x 768 ran in 768 tiles of 32 x 32, 29.2 us, where 64 x 64 ones take 20.5, and
    // 33 x 12288 x 1024 34.2 for 25.0.)  Left out: 64 x 64 with
    // one or four sets, 32 x 64 with four, 32 x 128 with two (0.1 to 0.9% together), 32 x 32 with eight (its registers spill).
    // 401 x 16384 x 2048 343 us -> 234, 401 x 2048 x 8192 187 -> 142, 401 x 3072 x 2048 93 -> 57, 64 x 2048 x 8192 163 -> 60,
    // 2048 x 16384 x 2048 1,302 -> 1,051, 401 x 128256 x 2048 2,010 -> 1,665.
    double tile_us[4];
    f32_tile_times(M, N, K, tile_us);
    // Up to 256 tiles of 64 x 64 at least two sets of waves share the columns: shorter runs, and an error that is smaller by a third
    // where a sum is no more than a few runs (positive numbers, K 64 to 516: 1.07e-7 with two sets, 1.43e-7 with one).  Up to four
    // runs of columns are no work for more sets, and the number of sets then depends on the number of those tiles alone.
    const bool few = (long long)((M + 63) / 64) * ((N + 63) / 64) <= 256;
    const bool few_runs = K <= 4 * RBK * RB_FOLD;
    int best = few ? 1 : 0;
    for (int i = 1; i < 4; ++i)
        if (tile_us[i] < tile_us[best] && !(few_runs && (!few || i == 3))) best = i;
    // Between four runs of columns and eight, the runs of four sets are shorter than 128 columns (192 columns a set at K 768: 128 and 64), and
    // their error is smaller than that of two sets.  They are kept up to 328 tiles of 32 x 32, where they are the fastest or nearly, and where a
    // compute unit would have three of those tiles two sets run 64 x 64 ones in runs of 64 columns (1024 x 768 x 768, us and error against 64 bits:
    // 32 x 32 28.9 and 1.88e-7, so 21.1 and 1.48e-7, in whole runs 20.2 and 2.06e-7).
    if (few && !few_runs && K < 8 * RBK * RB_FOLD) {
        const long long small = (long long)((M + 31) / 32) * ((N + 31) / 32);
        best = small <= 328 ? 3 : small <= 512 ? 2 : small <= 768 ? 4 : 1;
    }
    return best;
}
extern "C" int xr_f32_tile(int M, int N, int K) { return f32_tile(M, N, K); }
// the time that the fastest tile takes by that model, for the choice between these kernels and gemm_f32_parts.hip's
double xr_f32_tiles_us(int M, int N, int K) {
    double tile_us[4], best;
    f32_tile_times(M, N, K, tile_us);
    best = tile_us[0];
    for (int i = 1; i < 4; ++i) best = tile_us[i] < best ? tile_us[i] : best;
    return best;
}

// accumulate != 0: out (float) += product.  variant: 40 + a number of f32_tile's names the tile (tests); any other, the library's choice.
extern "C" int xr_gemm_ref(void* out, const void* a, const void* w, const float* bias, int M, int N, int K,
                           int lda, int ldo, int in_dtype, int out_dtype, int accumulate, int variant, hipStream_t stream) {
    XR_REQUIRE(M >= 0 && N > 0 && K > 0, "gemm: bad sizes M=%d N=%d K=%d", M, N, K);
    XR_REQUIRE(lda >= K && ldo >= N, "gemm: row strides lda=%d ldo=%d are shorter than K=%d N=%d", lda, ldo, K, N);
    XR_REQUIRE(!accumulate || out_dtype == XR_F32, "gemm: accumulation needs a 32-bit output");
    if (M == 0) return XR_OK;
    if (in_dtype == XR_F32 && (out_dtype == XR_F32 || out_dtype == XR_BF16) && K % 4 == 0 && lda % 4 == 0 &&
        ((uintptr_t)a % 16) == 0 && ((uintptr_t)w % 16) == 0) {
        const float* af = (const float*)a;
        const float* wf = (const float*)w;
        if (M > 16) {
            const int tile = variant >= 40 && variant < 40 + XR_F32_TILES ? variant - 40 : f32_tile(M, N, K);
            const int rc = tile == 0   ? launch_gemm_f32<1, 4, 32, 128, 2, 1>(out, af, wf, bias, M, N, K, lda, ldo, out_dtype, accumulate, stream)
                           : tile == 1 ? launch_gemm_f32<2, 2, 64, 64, 2, 2>(out, af, wf, bias, M, N, K, lda, ldo, out_dtype, accumulate, stream)
                           : tile == 2 ? launch_gemm_f32<1, 2, 32, 64, 2, 2>(out, af, wf, bias, M, N, K, lda, ldo, out_dtype, accumulate, stream)
                           : tile == 3 ? launch_gemm_f32<1, 1, 32, 32, 2, 4>(out, af, wf, bias, M, N, K, lda, ldo, out_dtype, accumulate, stream)
                                       : launch_gemm_f32<2, 2, 64, 64, 2, 2, 2>(out, af, wf, bias, M, N, K, lda, ldo, out_dtype, accumulate, stream);
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

// Up to XR_GEMV_EXTRA_ROWS 32-bit rows through a product that norms its rows itself and / or gates its result: out [M, N] is
// norm(a) w^T (+ bias), or with `gated` act(gate) * up of the 2 N weight rows (gate rows, then up rows).  norm_w: the RMS norm's weight [K], or
// null (the rows are taken as they are).  `a` must not be what is written.
#define XR_GEMV_EXTRA_ROWS 4
extern "C" int xr_gemv_extra_rows() { return XR_GEMV_EXTRA_ROWS; }
extern "C" int xr_gemv_extra(float* out, const float* a, const float* w, const float* bias, const float* norm_w, float eps, int gated, int act,
                             float act_param, int M, int N, int K, int lda, int ldo, hipStream_t stream) {
    XR_REQUIRE(M >= 0 && M <= XR_GEMV_EXTRA_ROWS && N > 0 && K > 0, "gemv: bad sizes M=%d (at most %d) N=%d K=%d", M, XR_GEMV_EXTRA_ROWS, N, K);
    XR_REQUIRE(lda >= K && ldo >= N, "gemv: row strides lda=%d ldo=%d are shorter than K=%d N=%d", lda, ldo, K, N);
    XR_REQUIRE(K % 4 == 0 && lda % 4 == 0 && (((uintptr_t)a | (uintptr_t)w | (uintptr_t)norm_w) % 16) == 0, "gemv: operands that are not 16-byte aligned rows of a multiple of 4");
    XR_REQUIRE(norm_w || gated, "gemv: a plain product is xr_gemm_ref's");
    XR_REQUIRE(!gated || (act >= 0 && act < XR_ACT_COUNT), "gemv: unknown activation code %d", act);
    if (M == 0) return XR_OK;
    const GemvExtra x{norm_w, 1.0f / (float)K, eps, act, act_param, nullptr};
    auto run = [&](auto rows) {
        constexpr int MT = decltype(rows)::value;
        // (two weight rows a wave, or two outputs: these are for few rows and small matrices; larger ones by the same lines as plain products)
        const bool wide = gemv_cols<MT>(gated ? 2 * N : N, K) > 2;
#define XV(COLS, NORM, GATED)                                                                                                   \
    {                                                                                                                           \
        constexpr int per = 4 * ((GATED) ? (COLS) / 2 : (COLS));                                                                \
        k_gemv_ref<MT, COLS, float, false, NORM, GATED><<<(unsigned)((N + per - 1) / per), 256, 0, stream>>>(out, a, w, bias, M, N, K, lda, ldo, x); \
    }
        if (gated && norm_w) { if (wide) XV(8, true, true) else XV(2, true, true) }
        else if (gated) { if (wide) XV(8, false, true) else XV(2, false, true) }
        else { if (wide) XV(4, true, false) else XV(2, true, false) }
#undef XV
    };
    if (M == 1) run(std::integral_constant<int, 1>{});
    else run(std::integral_constant<int, 4>{});
    XR_CHECK_LAUNCH("gemv_extra");
    return XR_OK;
}

// Up to XR_GEMV_EXTRA_ROWS 32-bit rows: out [M, N] += a w^T (+ bias), as xr_gemm_ref adds them, and the new rows of `out` also to
// `copy` [M, N], which a later product norms (so that `out` may be added to before it does).
extern "C" int xr_gemv_add_copy(float* out, float* copy, const float* a, const float* w, const float* bias, int M, int N, int K, int lda,
                                int ldo, hipStream_t stream) {
    XR_REQUIRE(M >= 0 && M <= XR_GEMV_EXTRA_ROWS && N > 0 && K > 0, "gemv: bad sizes M=%d (at most %d) N=%d K=%d", M, XR_GEMV_EXTRA_ROWS, N, K);
    XR_REQUIRE(lda >= K && ldo >= N, "gemv: row strides lda=%d ldo=%d are shorter than K=%d N=%d", lda, ldo, K, N);
    XR_REQUIRE(K % 4 == 0 && lda % 4 == 0 && (((uintptr_t)a | (uintptr_t)w) % 16) == 0, "gemv: operands that are not 16-byte aligned rows of a multiple of 4");
    if (M == 0) return XR_OK;
    if (M == 1) launch_gemv_ref<1>(out, a, w, bias, M, N, K, lda, ldo, XR_F32, 1, stream, copy);
    else launch_gemv_ref<4>(out, a, w, bias, M, N, K, lda, ldo, XR_F32, 1, stream, copy);
    XR_CHECK_LAUNCH("gemv_add_copy");
    return XR_OK;
}
