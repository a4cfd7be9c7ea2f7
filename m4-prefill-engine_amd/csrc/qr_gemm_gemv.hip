// qr_gemm_gemv.hip -- quantized projection and fused SwiGLU for a few rows of
// X (M <= 16), one kernel, no K split across workgroups.
//
// A decoded token's projection is bound by streaming the packed weights from
// HBM once; what the split-K kernels of qr_gemm_skinny.hip spend beside that is
// their reduction kernel (~4 - 6 us), and SwiGLU had only the 128-row tiles.
// Here a workgroup of 8 waves owns 16 output columns (SwiGLU: of both
// matrices), and wave w streams its eighth of K straight into registers:
//  * K advances 256 per chunk.  Lane (r, g) = (lane % 16, lane / 16) holds two
//    of column r's eight groups of the chunk whole, so each weight is decoded
//    once, by the whole-group decoders;
//  * MFMA 4 t + e of the chunk's eight (16x16x32, weights as the A operand)
//    takes elements 8 e .. + 7 of its t-th group from every lane; X, the B
//    operand, is read with the same k order (the sum over k is order-free),
//    16 bytes per lane and MFMA, from L2; rows past M read zeros;
//  * the bytes of a chunk are fetched one or two chunks ahead; nothing is staged
//    through LDS and no wave waits for another before the end;
//  * the 8 partial sums of every output meet in LDS in wave order.
#include "qr_decode.h"
#include "qr_kernels.h"

namespace qr {
namespace gemv {

constexpr int kWaves = 8, kThreads = 64 * kWaves;

template <int N>
__device__ __forceinline__ void load_run(__amdgpu_buffer_rsrc_t r, uint32_t off, uint32_t* w) {
#pragma unroll
    for (int i = 0; i + 4 <= N; i += 4) {
        const u4_t v = ld_b128(r, off + 4u * i);
        w[i] = v.x; w[i + 1] = v.y; w[i + 2] = v.z; w[i + 3] = v.w;
    }
    if constexpr (N % 4 == 2) {
        const u2_t v = ld_b64(r, off + 4u * (N - 2));
        w[N - 2] = v.x; w[N - 1] = v.y;
    } else if constexpr (N % 4 == 1) {
        w[N - 1] = ld_b32(r, off + 4u * (N - 1));
    }
}

// The two of a chunk's eight groups that lane group g holds: at(g, t) is the
// t-th; load() fetches both from the column at byte offset `col`, raw() picks
// the words of the t-th for decode_group, and par() is its parity argument.
// In general groups g and g + 4, each by the decoder's own loads; the formats
// of 18 and 20 bytes per group take 2 g and 2 g + 1, one contiguous run of
// 36 or 40 bytes in three loads (MLX, N = 4096, K = 14336: 12.7 -> 11.2 us).
template <int F>
struct Lane {
    using Dec = Decoder<F>;
    static constexpr int kWords = 2 * Dec::kRawWords;
    __device__ static uint32_t at(uint32_t g, int t) { return g + 4u * t; }
    __device__ static void load(__amdgpu_buffer_rsrc_t r, uint32_t col, uint32_t c, uint32_t g, uint32_t* w) {
        Dec::load(r, col, 8u * c + g, w);
        Dec::load(r, col, 8u * c + g + 4u, w + Dec::kRawWords);
    }
    __device__ static void raw(const uint32_t* w, int t, uint32_t* o) {
#pragma unroll
        for (int i = 0; i < Dec::kRawWords; i++) o[i] = w[t * Dec::kRawWords + i];
    }
    __device__ static uint32_t par(uint32_t col, uint32_t c, uint32_t g, int t) { return Dec::parity(col, 8u * c + at(g, t)); }
};
template <int BYTES>
struct RunLane {
    static constexpr int kWords = BYTES / 4;
    __device__ static uint32_t at(uint32_t g, int t) { return 2u * g + t; }
    __device__ static void load(__amdgpu_buffer_rsrc_t r, uint32_t col, uint32_t c, uint32_t g, uint32_t* w) {
        load_run<kWords>(r, col + (4u * c + g) * (uint32_t)BYTES, w);
    }
};
template <> struct Lane<QUANT_Q4_0> : RunLane<36> {  // the second block starts at byte 18
    __device__ static void raw(const uint32_t* w, int t, uint32_t* o) {
#pragma unroll
        for (int i = 0; i < 5; i++) o[i] = w[4 * t + i];
    }
    __device__ static uint32_t par(uint32_t, uint32_t, uint32_t, int t) { return t ? 2u : 0u; }
};
template <> struct Lane<QUANT_MLX_4BIT> : RunLane<40> {
    __device__ static void raw(const uint32_t* w, int t, uint32_t* o) {
#pragma unroll
        for (int i = 0; i < 5; i++) o[i] = w[5 * t + i];
    }
    __device__ static uint32_t par(uint32_t, uint32_t, uint32_t, int) { return 0; }
};
template <> struct Lane<QUANT_MLX_4BIT_G64> : RunLane<36> {  // one 64-element block
    __device__ static void raw(const uint32_t* w, int t, uint32_t* o) {
        o[0] = w[0];
#pragma unroll
        for (int i = 0; i < 4; i++) o[1 + i] = w[1 + 4 * t + i];
    }
    __device__ static uint32_t par(uint32_t, uint32_t, uint32_t, int) { return 0; }
};

// Chunks fetched ahead, and waves per SIMD that the registers are limited to:
// two workgroups per CU, one where the raw blocks are too wide for that.
template <int F, int NT>
constexpr int ahead() { return Decoder<F>::kRawWords <= 5 && Lane<F>::kWords * NT <= 20 ? 2 : 1; }
template <int F, int NT>
constexpr int waves_per_simd() { return Decoder<F>::kRawWords <= (NT == 1 ? 8 : 5) ? 4 : 2; }

}  // namespace gemv

// NC: 16-column tiles per workgroup; PL: weight matrices (2: SwiGLU, gate and up).
template <int F, int NC, int PL>
__global__ void __launch_bounds__(gemv::kThreads, (gemv::waves_per_simd<F, NC * PL>())) gemv_kernel(GemmParams p) {
    using Dec = Decoder<F>;
    using L = gemv::Lane<F>;
    constexpr int NT = NC * PL, A = gemv::ahead<F, NC * PL>(), W = gemv::kWaves, CW = 16 * NC;
    constexpr int RS = 16 + 1;
    __shared__ float red[W * NT * 16 * RS];

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t r16 = lane & 15, g = lane >> 4;
    uint32_t bid = blockIdx.x;
    if (p.ngroups > 1) {  // grouped launch: this workgroup's matrix, output and width
        const uint32_t t0 = (p.N + CW - 1) / CW;
        if (bid >= t0) {
            bid -= t0;
            const uint32_t t1 = (p.Nx[0] + CW - 1) / CW;
            const int gx = (bid < t1 || p.ngroups == 2) ? 0 : 1;
            if (gx == 1) bid -= t1;
            p.W = p.Wx[gx];
            p.Y = p.Yx[gx];
            p.N = p.Nx[gx];
        }
    }
    const uint32_t M = p.M, N = p.N, K = p.K, col_bytes = (uint32_t)p.col_bytes;
    const uint32_t n0 = bid * CW, ncols = min((uint32_t)CW, N - n0);
    const uint32_t nch = K / 256, c0 = nch * (uint32_t)wave / W, c1 = nch * (uint32_t)(wave + 1) / W;

    __amdgpu_buffer_rsrc_t wr[PL];
    wr[0] = make_rsrc(p.W + (size_t)n0 * col_bytes, ncols * col_bytes);
    if constexpr (PL == 2) wr[1] = make_rsrc(p.W2 + (size_t)n0 * col_bytes, ncols * col_bytes);
    const auto xr = make_rsrc(p.X, M * K * 2u);
    uint32_t wo[NC];
#pragma unroll
    for (int i = 0; i < NC; i++) wo[i] = 16u * i + r16 < ncols ? (16u * i + r16) * col_bytes : kOOB;  // past N: zeros
    const uint32_t xo = r16 < M ? r16 * K * 2u : kOOB;

    // weight tile q: columns 16 (q % NC) .. of matrix q / NC
    uint32_t raw[A + 1][NT][L::kWords];
    u4_t xf[2][4];
    auto load_w = [&](uint32_t c, int slot) {
#pragma unroll
        for (int q = 0; q < NT; q++) L::load(wr[q / NC], c < c1 ? wo[q % NC] : kOOB, min(c, nch - 1), g, raw[slot][q]);
    };
    auto load_x = [&](uint32_t c, int t) {
        const uint32_t o = (c < c1 ? xo : kOOB) + (min(c, nch - 1) * 256u + 32u * L::at(g, t)) * 2u;
#pragma unroll
        for (int e = 0; e < 4; e++) xf[t][e] = ld_b128(xr, o + 16u * e);
    };
    f4_t acc[NT];
#pragma unroll
    for (int q = 0; q < NT; q++) acc[q] = f4_t{};
    auto compute = [&](uint32_t c, int slot, int t) {
#pragma unroll
        for (int q = 0; q < NT; q++) {
            uint32_t rg[Dec::kRawWords], o[16];
            L::raw(raw[slot][q], t, rg);
            const uint32_t par = L::par(wo[q % NC], c, g, t);
            decode_half_fast<F>(rg, par, 0, o);
            decode_half_fast<F>(rg, par, 1, o + 8);
            if constexpr (F == QUANT_Q4_K || F == QUANT_Q4_0) {
                if (__any(needs_exact<F>(rg, par))) decode_group<F>(rg, par, o);
            }
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const h8_t a = __builtin_bit_cast(h8_t, u4_t{o[4 * e], o[4 * e + 1], o[4 * e + 2], o[4 * e + 3]});
                acc[q] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, __builtin_bit_cast(h8_t, xf[t][e]), acc[q], 0, 0, 0);
            }
        }
    };

    if (c0 < c1) {
#pragma unroll
        for (int a = 0; a < A; a++) load_w(c0 + a, a);
        load_x(c0, 0);
        load_x(c0, 1);
        for (uint32_t c = c0; c < c1; c += A + 1) {
#pragma unroll
            for (int u = 0; u < A + 1; u++) {  // slot indices static
                if (u && c + u >= c1) break;
                load_w(c + u + A, (u + A) % (A + 1));
#pragma unroll
                for (int t = 0; t < 2; t++) {
                    compute(c + u, u, t);
                    load_x(c + u + 1, t);
                }
            }
        }
    }

    // acc element i of lane (r16, g): column 4 g + i of its tile, row r16
#pragma unroll
    for (int q = 0; q < NT; q++)
#pragma unroll
        for (int i = 0; i < 4; i++) red[((wave * NT + q) * 16 + r16) * RS + 4 * g + i] = acc[q][i];
    __syncthreads();
    for (uint32_t e = tid; e < 16u * CW; e += gemv::kThreads) {
        const uint32_t m = e / CW, nl = e % CW;
        if (m >= M || nl >= ncols) continue;
        float v[PL];
#pragma unroll
        for (int q = 0; q < PL; q++) {
            v[q] = 0.0f;
#pragma unroll
            for (int w = 0; w < W; w++) v[q] += red[((w * NT + q * NC + nl / 16) * 16 + m) * RS + nl % 16];
        }
        float y = v[0];
        if constexpr (PL == 2) y = silu_mul(v[0], v[PL - 1]);
        const uint32_t n = n0 + nl;
        if (p.R) y += (float)p.R[(size_t)m * N + n];
        const size_t o = p.head_D ? ((size_t)(n / p.head_D) * M + m) * p.head_D + n % p.head_D : (size_t)m * N + n;
        p.Y[o] = (_Float16)y;
    }
}

// Column tiles of p, all groups.
static uint32_t column_tiles(const GemmParams& p, uint32_t cw) {
    uint32_t t = (p.N + cw - 1) / cw;
    for (uint32_t g = 1; g < p.ngroups && g < 3; g++) t += (p.Nx[g - 1] + cw - 1) / cw;
    return t;
}

// Two column tiles per workgroup when the workgroups of one would not be
// resident at once (MLX N = 14336, K = 4096, M = 1: 15.5 -> 12.8 us).
uint32_t gemv_tile_columns(const GemmParams& p) { return !p.W2 && column_tiles(p, 16) > 512 ? 32 : 16; }

// ---- the price of this kernel and of the one that would run instead ----
// us: five terms each, fitted (least squares of the relative error) to ~2300 shapes
// per format of 1 .. 16 rows, K 1024 .. 14336, N 256 .. 20000, weights read from
// HBM, launches in a graph; 5 - 7% rms, the tiles' 9 - 12%.
//  few16, few32 (one and two column tiles per workgroup, each over the widths that
//      take it): launch, MB of weights, chunks of the longest wave times workgroups
//      per CU, M K / 1e5 times workgroups per CU (X, which every one of them reads
//      from L2), M K / 1e5;
//  split (the small-M kernel with its K split): launch, MB of weights, K per split / 256
//      times workgroups per CU, partials in 1e6, splits;
//  tiles (the 128-row tiles): launch, MB of weights, K per split / 256 times
//      workgroups per CU, the reduction, partials in 1e6.
struct FewCost {
    float few16[5], few32[5], split[5], tiles[5];
};
static const FewCost& few_cost(int f) {
    static const FewCost q4_0 = {{2.62f, 0.185f, 0.874f, 4.61f, 1.38f}, {3.31f, 0.238f, 0.794f, 6.52f, 3.38f},
                                 {6.04f, 0.173f, 0.417f, 2.74f, 0.298f}, {5.39f, 0.163f, 0.88f, 4.28f, 3.28f}};
    static const FewCost mlx = {{2.6f, 0.164f, 0.944f, 3.49f, 1.54f}, {3.27f, 0.232f, 1.01f, 2.74f, 5.33f},
                                 {5.89f, 0.168f, 0.365f, 2.45f, 0.283f}, {5.4f, 0.123f, 0.861f, 4.32f, 6.09f}};
    static const FewCost q4_k = {{3.03f, 0.154f, 0.928f, 2.85f, 1.67f}, {5.73f, 0.2f, 1.35f, 3.61f, 0},
                                 {6.01f, 0.126f, 0.783f, 2.49f, 0.294f}, {3.63f, 0.175f, 1.38f, 6.49f, 2.77f}};
    static const FewCost ternary = {{2.82f, 0.192f, 0.775f, 2.71f, 0.974f}, {3.68f, 0.237f, 0.736f, 2.56f, 2.06f},
                                 {5.99f, 0.229f, 0.325f, 2.46f, 0.304f}, {4.31f, 0.149f, 0.87f, 3.94f, 5.04f}};
    static const FewCost q8_0 = {{2.62f, 0.136f, 1.34f, 2.03f, 2.63f}, {2.84f, 0.231f, 1.38f, 1.72f, 7.43f},
                                 {}, {4.07f, 0.173f, 1.08f, 5.55f, 4.11f}};
    static const FewCost prism = {{2.81f, 0.219f, 0.939f, 2.73f, 0.836f}, {3.32f, 0.36f, 0.874f, 2.6f, 2.04f},
                                 {}, {4.02f, 0.194f, 0.967f, 4.4f, 3.29f}};
    static const FewCost g64 = {{2.57f, 0.171f, 0.948f, 3.49f, 1.46f}, {3.24f, 0.242f, 1.02f, 3.03f, 4.02f},
                                 {5.76f, 0.155f, 0.38f, 2.68f, 0.297f}, {6.09f, 0.166f, 0.858f, 3.79f, 3.14f}};
    switch (f) {
        case QUANT_MLX_4BIT: return mlx;
        case QUANT_Q4_K: return q4_k;
        case QUANT_TERNARY_1_58: return ternary;
        case QUANT_Q8_0: return q8_0;
        case QUANT_PRISM_Q2_0: return prism;
        case QUANT_MLX_4BIT_G64: return g64;
        default: return q4_0;
    }
}
static float price(const float* w, float a, float b, float c, float d) { return w[0] + w[1] * a + w[2] * b + w[3] * c + w[4] * d; }

// Where this kernel is the fastest.  Every column tile reads all of X from L2, so
// what it loses on is X bytes where the other kernel can split K, and workgroups that
// share a CU unevenly; how well the other one splits depends on K (10752 = 42
// super-blocks splits in two, 8192 in sixteen).  So both are priced, and this one runs where its price
// is lower by 6%, about the fits' error (this kernel / the other, us): MLX M = 7, K = 7168, N = 8720
// 24.5 / 18.0, MLX M = 8, K = 14336, N = 5632 31.4 / 22.4, but Q4_K M = 16, K =
// 10752, N = 1416 14.2 / 45.4, ternary M = 12, K = 13824, N = 3712 15.8 / 37.9.
// Of 15974 shapes 1.92x the other kernels by geometric mean, 39 more than 3% slower
// than them (bounds on M K and tiles in its place: 1.84x, 128).
//  * K up to 1024, below the prices' range: up to 1024 column tiles where the small-M
//    kernel would run (of 6365 shapes 1.62x, 57 more than 3% slower);
//  * SwiGLU, against the 128-row tiles: MLX K = 4096, N = 14336 M = 1 33.2 -> 21.3,
//    M = 16 34.0 -> 33.2; of 800 shapes 23 below 1.2x, two below even, but for VAR_RATE
//    against 16 K splits (K = 8192, N = 512 108 -> 145), EXL3 with short K and many
//    columns (K = 1024, N = 28672 56 -> 65) and Q4_0 past M K = 160 Ki (M = 16, K =
//    14336, N = 5632 60.5 -> 67.9);
//  * VAR_RATE and EXL3 projections: always (M = 16, K = 14336, N = 1536 1.6x);
//  * where the small-M kernel runs as one kernel: one or two rows (MLX 4096 x 4096: M = 1
//    5.5 -> 4.8, M = 2 5.6 -> 5.1, M = 4 5.6 -> 5.7), Q4_K up to 8 (8.2 -> 6.2).
bool gemv_fits(const GemmParams& p) {
    if (p.M > 16 || p.K % 256) return false;
    const int f = p.format;
    const uint32_t tiles = column_tiles(p, 16);
    if (p.W2) {
        const uint32_t ks = gemm_base_ksplit(p);
        return !(f == QUANT_VAR_RATE_AFFINE && ks >= 16) && !(f == QUANT_EXL3 && p.K <= 1024 && tiles > 768) &&
               !(f == QUANT_Q4_0 && ks > 1 && tiles > 256 && (uint64_t)p.M * p.K > 160u << 10);
    }
    if (f == QUANT_VAR_RATE_AFFINE || f == QUANT_EXL3) return true;
    const bool split = p.ngroups <= 1 && skinny_supported(p);
    if (split && skinny_one_kernel(p)) return p.M <= (f == QUANT_Q4_K ? 8u : 2u);
    if (p.K <= 1024) return !split || tiles <= (f == QUANT_Q4_K && p.K < 512 ? 512u : 1024u);
    float n = (float)p.N;
    for (uint32_t g = 1; g < p.ngroups && g < 3; g++) n += (float)p.Nx[g - 1];
    const float mb = n * (float)p.col_bytes * 1e-6f, mk = (float)p.M * (float)p.K;
    const uint32_t cw = gemv_tile_columns(p), ks = split ? skinny_ksplit(p) : gemm_base_ksplit(p);
    auto per_cu = [](uint64_t wgs) { return (float)((wgs + 255) / 256); };
    const FewCost& c = few_cost(f);
    const float wgs = per_cu(column_tiles(p, cw));
    const float few = price(cw == 32 ? c.few32 : c.few16, mb, wgs * (float)((p.K / 256 + 7) / 8), wgs * mk * 1e-5f, mk * 1e-5f);
    const float steps = per_cu((uint64_t)column_tiles(p, split ? 64 : 128) * ks) * (float)p.K / (256.0f * (float)ks);
    const float partials = (float)ks * (float)p.M * n * 1e-6f;
    const float other = split ? price(c.split, mb, steps, partials, (float)ks)
                              : price(c.tiles, mb, steps, ks > 1 ? 1.0f : 0.0f, partials);
    return few < 0.94f * other;
}

template <int F>
static hipError_t launch_gemv_f(const GemmParams& p, hipStream_t st) {
    const uint32_t cw = gemv_tile_columns(p);
    const dim3 grid(column_tiles(p, cw)), block(gemv::kThreads);
    if (p.W2) hipLaunchKernelGGL((gemv_kernel<F, 1, 2>), grid, block, 0, st, p);
    else if (cw == 32) hipLaunchKernelGGL((gemv_kernel<F, 2, 1>), grid, block, 0, st, p);
    else hipLaunchKernelGGL((gemv_kernel<F, 1, 1>), grid, block, 0, st, p);
    return hipGetLastError();
}

hipError_t launch_gemv(const GemmParams& p, hipStream_t st) {
    switch (p.format) {
        case QUANT_Q4_0: return launch_gemv_f<QUANT_Q4_0>(p, st);
        case QUANT_MLX_4BIT: return launch_gemv_f<QUANT_MLX_4BIT>(p, st);
        case QUANT_Q4_K: return launch_gemv_f<QUANT_Q4_K>(p, st);
        case QUANT_TERNARY_1_58: return launch_gemv_f<QUANT_TERNARY_1_58>(p, st);
        case QUANT_VAR_RATE_AFFINE: return launch_gemv_f<QUANT_VAR_RATE_AFFINE>(p, st);
        case QUANT_EXL3: return launch_gemv_f<QUANT_EXL3>(p, st);
        case QUANT_Q8_0: return launch_gemv_f<QUANT_Q8_0>(p, st);
        case QUANT_PRISM_Q2_0: return launch_gemv_f<QUANT_PRISM_Q2_0>(p, st);
        case QUANT_MLX_4BIT_G64: return launch_gemv_f<QUANT_MLX_4BIT_G64>(p, st);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace qr
