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

// Where this kernel is the fastest.  Every column tile reads all of X from L2, so
// what it loses on is X bytes (M K per tile) where the other kernels can split K;
// 3386 shapes of 1 .. 16 rows over all formats, each launch in a graph, us other
// kernel -> this one:
//  * SwiGLU, against the 128-row tiles: MLX K = 4096, N = 14336 M = 1 33.2 -> 21.3,
//    M = 16 34.0 -> 33.2; of 800 shapes 23 below 1.2x, two below even, but for VAR_RATE
//    against 16 K splits (K = 8192, N = 512 108 -> 145), EXL3 with short K and many
//    columns (K = 1024, N = 28672 56 -> 65) and Q4_0 past M K = 160 Ki (M = 16, K =
//    14336, N = 5632 60.5 -> 67.9);
//  * formats without a small-M kernel, and a layer's Q, K and V in one launch: where
//    the tiles split K, up to M K = 128 Ki (ternary M = 16, K = 14336, N = 256 14.4 ->
//    17.7), Q8_0 104 Ki but at 128 to 256 tiles (M = 8, K = 14336, N = 512 19.0 -> 19.8;
//    M = 9, K = 14336, N = 4096 25.0 -> 21.0), and from nine
//    rows past one workgroup per CU Q8_0 48 Ki (M = 16, N = 5632: K = 2048 11.3 -> 9.4, K =
//    4096 14.7 -> 16.1) and PRISM 64 Ki (N = 8192: M = 16, K = 4096 1.04x, M = 11, K =
//    8192 18.8 -> 20.7); VAR_RATE and EXL3 always (M = 16, K = 14336, N = 1536 1.6x);
//  * where the small-M kernel splits K: up to 128 column tiles M K <= 96 Ki (M = 12, K =
//    14336, N = 2048 MLX 14.1 -> 17.7), Q4_K 128 Ki (M = 8 16.8 -> 15.3); past that eight
//    rows (MLX K = 14336, N = 4096, M = 8 19.3 -> 17.2); past one workgroup per CU (256
//    tiles) only what K makes up for the uneven load: MLX and g64 below K = 8192 (g64 M =
//    2, N = 11008: K = 4096 even, K = 8192 19.5 -> 23.0), Q4_0 to M K = 48 Ki; not past
//    1024 tiles, which are not resident at once (N = 28672, M = 1: 19.2 -> 21.8);
//  * where that runs as one kernel: one or two rows (MLX 4096 x 4096: M = 1
//    5.5 -> 4.8, M = 2 5.6 -> 5.1, M = 4 5.6 -> 5.7), Q4_K up to 8 (8.2 -> 6.2).
bool gemv_fits(const GemmParams& p) {
    if (p.M > 16 || p.K % 256) return false;
    const uint32_t tiles = column_tiles(p, 16);
    auto mk_upto = [&](uint32_t ki) { return (uint64_t)p.M * p.K <= (uint64_t)ki << 10; };
    const int f = p.format;
    if (p.W2 || p.ngroups > 1 || !skinny_supported(p)) {
        const uint32_t ks = gemm_base_ksplit(p);
        if (p.W2)
            return !(f == QUANT_VAR_RATE_AFFINE && ks >= 16) && !(f == QUANT_EXL3 && p.K <= 1024 && tiles > 768) &&
                   !(f == QUANT_Q4_0 && ks > 1 && tiles > 256 && !mk_upto(160));
        if (f == QUANT_VAR_RATE_AFFINE || f == QUANT_EXL3) return true;
        if (ks == 1 && (f != QUANT_Q8_0 || tiles <= 1024)) return true;
        if (p.M > 8 && tiles > 256 && ks >= 4 && (f == QUANT_Q8_0 || f == QUANT_PRISM_Q2_0)) return mk_upto(f == QUANT_Q8_0 ? 48 : 64);
        return mk_upto(f == QUANT_Q8_0 && (tiles < 128 || tiles > 256) ? 104 : 128);
    }
    if (skinny_one_kernel(p)) return p.M <= (f == QUANT_Q4_K ? 8u : 2u);
    if (tiles <= 128) return mk_upto(f == QUANT_Q4_K ? 128 : 96);
    if (tiles > 1024 || p.M > 8) return false;
    if (tiles <= 256 || f == QUANT_Q4_K || f == QUANT_TERNARY_1_58) return true;
    return f == QUANT_Q4_0 ? mk_upto(48) : p.K < 8192;
}

// Two column tiles per workgroup when the workgroups of one would not be
// resident at once (MLX N = 14336, K = 4096, M = 1: 15.5 -> 12.8 us).
uint32_t gemv_tile_columns(const GemmParams& p) { return !p.W2 && column_tiles(p, 16) > 512 ? 32 : 16; }

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
