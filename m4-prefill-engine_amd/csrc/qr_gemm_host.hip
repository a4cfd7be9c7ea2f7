// qr_gemm_host.hip -- host side of the tiled projection: format dispatch,
// split-K choice and workspace sizing (kernels in qr_gemm.hip), and the
// split-K reduction kernel shared with the small-M kernel.
#include "qr_device.h"
#include "qr_gemm_shapes.h"

namespace qr {

// Split-K reduction: out[m, n] = epilogue(sum over splits z = 0, 1, ... of
// ws[z][plane][m][n]) with the tiled kernel's epilogue arithmetic (SwiGLU
// silu(g) u in fp32 for DUAL, + fp16 residual, one rounding to fp16,
// [M, N] or head-major [N / head_D, M, head_D]).  The splits are summed in
// split order starting from 0, so the result does not depend on which
// workgroup finished first.  Eight consecutive elements of one row per
// thread (16-byte output stores) when N and head_D are multiples of 8 and Y
// and R are 16-byte aligned; the
// partials are read once, as streaming loads.
constexpr int kRedVec = 8;

template <bool DUAL>
__device__ __forceinline__ void splitk_reduce(const float* __restrict__ ws, uint32_t ks, uint32_t M, uint32_t N,
                                              const _Float16* __restrict__ R, _Float16* __restrict__ Y, uint32_t head_D) {
    const size_t plane = (size_t)M * N;
    const size_t e0 = ((size_t)blockIdx.x * 256 + threadIdx.x) * kRedVec;
    if (e0 >= plane) return;
    const int cnt = plane - e0 < (size_t)kRedVec ? (int)(plane - e0) : kRedVec;
    const bool vec = cnt == kRedVec && (N % kRedVec) == 0 && (head_D % kRedVec) == 0 &&
                     ((reinterpret_cast<uintptr_t>(Y) | reinterpret_cast<uintptr_t>(R)) & 15u) == 0;
    float g[kRedVec], u[kRedVec];
#pragma unroll
    for (int q = 0; q < kRedVec; q++) g[q] = u[q] = 0.0f;
    if (vec) {
        for (uint32_t z = 0; z < ks; z++) {
            const f4_t* src = reinterpret_cast<const f4_t*>(ws + (size_t)z * plane * (DUAL ? 2 : 1) + e0);
            const f4_t a0 = __builtin_nontemporal_load(src), a1 = __builtin_nontemporal_load(src + 1);
            g[0] += a0.x; g[1] += a0.y; g[2] += a0.z; g[3] += a0.w;
            g[4] += a1.x; g[5] += a1.y; g[6] += a1.z; g[7] += a1.w;
            if constexpr (DUAL) {
                const f4_t* sv = reinterpret_cast<const f4_t*>(reinterpret_cast<const float*>(src) + plane);
                const f4_t b0 = __builtin_nontemporal_load(sv), b1 = __builtin_nontemporal_load(sv + 1);
                u[0] += b0.x; u[1] += b0.y; u[2] += b0.z; u[3] += b0.w;
                u[4] += b1.x; u[5] += b1.y; u[6] += b1.z; u[7] += b1.w;
            }
        }
        const uint32_t m = (uint32_t)(e0 / N), n = (uint32_t)(e0 % N);
        float v[kRedVec];
#pragma unroll
        for (int q = 0; q < kRedVec; q++) {
            v[q] = g[q];
            if constexpr (DUAL) v[q] = silu_mul(v[q], u[q]);
        }
        if (R) {
            const u4_t rr = *reinterpret_cast<const u4_t*>(R + e0);
            const uint32_t rw[4] = {rr.x, rr.y, rr.z, rr.w};
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const h2_t hh = as_h2(rw[q]);
                v[2 * q] += (float)hh.x;
                v[2 * q + 1] += (float)hh.y;
            }
        }
        const size_t o = head_D ? ((size_t)(n / head_D) * M + m) * head_D + n % head_D : e0;
        u4_t out;
        out.x = pack_h2(f2h_bits(v[0]), f2h_bits(v[1]));
        out.y = pack_h2(f2h_bits(v[2]), f2h_bits(v[3]));
        out.z = pack_h2(f2h_bits(v[4]), f2h_bits(v[5]));
        out.w = pack_h2(f2h_bits(v[6]), f2h_bits(v[7]));
        *reinterpret_cast<u4_t*>(Y + o) = out;
        return;
    }
    for (uint32_t z = 0; z < ks; z++) {
        const float* src = ws + (size_t)z * plane * (DUAL ? 2 : 1) + e0;
        for (int q = 0; q < cnt; q++) {
            g[q] += src[q];
            if constexpr (DUAL) u[q] += src[plane + q];
        }
    }
    for (int q = 0; q < cnt; q++) {
        const size_t e = e0 + q;
        const uint32_t m = (uint32_t)(e / N), n = (uint32_t)(e % N);
        float v = g[q];
        if constexpr (DUAL) v = silu_mul(v, u[q]);
        if (R) v += (float)R[e];
        const size_t o = head_D ? ((size_t)(n / head_D) * M + m) * head_D + n % head_D : e;
        Y[o] = (_Float16)v;
    }
}

template <bool DUAL>
__global__ void __launch_bounds__(256) splitk_reduce_kernel(const float* __restrict__ ws, uint32_t ks, uint32_t M,
                                                            uint32_t N, const _Float16* __restrict__ R,
                                                            _Float16* __restrict__ Y, uint32_t head_D) {
    splitk_reduce<DUAL>(ws, ks, M, N, R, Y, head_D);
}

// blockIdx.y is the group of a grouped projection (its partials follow the
// previous group's).  A kernel of its own: one matrix's reduction through the
// group tables took 0.2 us longer (small-M projections of 17 .. 64 rows with a K
// split 1.5 - 2.3% slower over 1122 shapes).
struct RedGroups {
    _Float16* Y[3];
    uint32_t N[3];
};
__global__ void __launch_bounds__(256) splitk_reduce_groups_kernel(const float* __restrict__ ws, uint32_t ks, uint32_t M,
                                                                   RedGroups gr, uint32_t head_D) {
    const uint32_t grp = blockIdx.y;
    if (grp > 0) ws += (size_t)ks * M * (gr.N[0] + (grp > 1 ? gr.N[1] : 0u));
    splitk_reduce<false>(ws, ks, M, grp == 0 ? gr.N[0] : (grp == 1 ? gr.N[1] : gr.N[2]), nullptr,
                         grp == 0 ? gr.Y[0] : (grp == 1 ? gr.Y[1] : gr.Y[2]), head_D);
}

static unsigned reduce_blocks(uint32_t M, uint32_t N) {
    const size_t plane = (size_t)M * N;
    return (unsigned)((plane + 256 * kRedVec - 1) / (256 * kRedVec));
}

hipError_t launch_splitk_reduce(const float* ws, uint32_t ks, uint32_t M, uint32_t N, bool dual, const _Float16* R,
                                _Float16* Y, uint32_t head_D, hipStream_t st) {
    const dim3 grid(reduce_blocks(M, N));
    if (dual) hipLaunchKernelGGL(splitk_reduce_kernel<true>, grid, dim3(256), 0, st, ws, ks, M, N, R, Y, head_D);
    else hipLaunchKernelGGL(splitk_reduce_kernel<false>, grid, dim3(256), 0, st, ws, ks, M, N, R, Y, head_D);
    return hipGetLastError();
}

static hipError_t launch_splitk_reduce_groups(const GemmParams& p, hipStream_t st) {
    uint32_t n = p.N;
    for (uint32_t g = 1; g < p.ngroups; g++) n = p.Nx[g - 1] > n ? p.Nx[g - 1] : n;
    hipLaunchKernelGGL(splitk_reduce_groups_kernel, dim3(reduce_blocks(p.M, n), p.ngroups), dim3(256), 0, st, p.ws, p.ksplit,
                       p.M, RedGroups{{p.Y, p.Yx[0], p.Yx[1]}, {p.N, p.Nx[0], p.Nx[1]}}, p.head_D);
    return hipGetLastError();
}

static hipError_t launch_gemm_main(const GemmParams& p, hipStream_t st) {
    switch (p.format) {
        case QUANT_Q4_0: return launch_gemm_format<QUANT_Q4_0>(p, st);
        case QUANT_MLX_4BIT: return launch_gemm_format<QUANT_MLX_4BIT>(p, st);
        case QUANT_Q4_K: return launch_gemm_format<QUANT_Q4_K>(p, st);
        case QUANT_TERNARY_1_58: return launch_gemm_format<QUANT_TERNARY_1_58>(p, st);
        case QUANT_VAR_RATE_AFFINE: return launch_gemm_format<QUANT_VAR_RATE_AFFINE>(p, st);
        case QUANT_EXL3: return launch_gemm_format<QUANT_EXL3>(p, st);
        case QUANT_Q8_0: return launch_gemm_format<QUANT_Q8_0>(p, st);
        case QUANT_PRISM_Q2_0: return launch_gemm_format<QUANT_PRISM_Q2_0>(p, st);
        case QUANT_MLX_4BIT_G64: return launch_gemm_format<QUANT_MLX_4BIT_G64>(p, st);
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_gemm(const GemmParams& p, hipStream_t st) {
    hipError_t e = launch_gemm_main(p, st);
    if (e == hipSuccess && p.ksplit > 1)
        e = p.ngroups > 1 ? launch_splitk_reduce_groups(p, st)
                          : launch_splitk_reduce(p.ws, p.ksplit, p.M, p.N, p.W2 != nullptr, p.R, p.Y, p.head_D, st);
    return e;
}

static uint32_t tiles_of(const GemmParams& p, const RbShape& d) {
    const uint32_t ntm = (p.M + d.bm - 1) / d.bm;
    uint32_t T = ntm * ((p.N + d.bn - 1) / d.bn);
    for (uint32_t g = 1; g < p.ngroups && g < 3; g++) T += ntm * ((p.Nx[g - 1] + d.bn - 1) / d.bn);
    return T;
}

static uint32_t columns_of(const GemmParams& p) {
    uint32_t n = p.N;
    for (uint32_t g = 1; g < p.ngroups && g < 3; g++) n += p.Nx[g - 1];
    return n;
}

// ---- the price of a plan ----
// One workgroup fits a CU, so a grid runs in waves of 256 tiles.  A wave takes
// `fix` us whatever K is (ramp, first loads, epilogue) and, per 4096 of K, `full`
// us when every CU has a tile and `half` when at most half of them have (the
// clock falls as the chip fills; for 64-row tiles the step from `half` to `full`
// starts at an empty chip, else at half).  A K split adds its reduction kernel: r0
// us, r1 per split and rb times the partials' round trip at 4.5 TB/s.
// Least-squares fits to the times of every choice in graphs, weights rotated over
// 300 MB: ~460 shapes per format, M 17 .. 4900, K 1024 .. 14336, N 256 .. 28672
// (relative error 5 - 8% rms: 3 - 4% for the 256-row tiles, 8 - 10% for the 64-row
// ones), less what all choices share (streaming X, W and Y).
// Each format has its own: the decode, the bytes and how they are fetched move the
// tiles against each other (M = 128, K = 4096, N = 14336, 128 x 64 against 64 x 128
// with two K groups: g64 26.9 / 30.9 us, MLX 26.7 / 27.9, ternary 21.9 / 20.9, Q8_0
// 34.8 / 42.7).
struct TileCost {
    float fix, full, half;
};
struct FormatCost {
    TileCost mid, big;          // 128 x 128; 128 x 256 (shape 0, or 3 for Q4_K and ternary)
    TileCost low, low_split;    // 64 x 128 without and with a K split (other kernel instances)
    TileCost kg, low_kg;        // 128 x 64 and 64 x 128 as two K groups
    TileCost wide;              // 256 x 256
    TileCost dual, dual_wide;   // SwiGLU: 128 x 128 and 256 x 128 outputs
    float r0, r1, rb;           // reduction of a projection
    float d0, d1, db;           // reduction of SwiGLU
};
static const FormatCost& format_cost(int f) {
    static const FormatCost q4_0 = {{4.8f, 31.7f, 24.7f}, {7, 59.5f, 43.1f}, {3.2f, 22.7f, 18.5f}, {2.9f, 19.8f, 20},
                                    {5.7f, 14.3f, 11.7f}, {3.4f, 21.3f, 16.8f}, {12.7f, 103.3f, 71.7f},
                                    {4.5f, 55.3f, 45.5f}, {8.2f, 96, 76.5f}, 2.6f, 0.25f, 0.97f, 3.35f, 0.4f, 0.71f};
    static const FormatCost mlx = {{4.8f, 32.5f, 23.9f}, {6.9f, 57.9f, 42.5f}, {2.5f, 21.1f, 18.6f}, {2.5f, 19.4f, 18.7f},
                                   {6, 13, 11.6f}, {4.9f, 15.8f, 12.4f}, {12.1f, 103, 68.1f},
                                   {5.3f, 52.1f, 44.7f}, {7.9f, 96.4f, 71.2f}, 2.8f, 0.25f, 0.94f, 3, 0.27f, 0.71f};
    static const FormatCost q4_k = {{4.5f, 39.8f, 34.6f}, {5.7f, 71.1f, 54.4f}, {3.2f, 29.1f, 29}, {2.7f, 28.8f, 27.9f},
                                    {5.3f, 19.6f, 18.2f}, {4.2f, 23.5f, 22}, {12.3f, 109.9f, 82.8f},
                                    {5, 68.6f, 60}, {8.5f, 105.6f, 85.6f}, 3.85f, 0.15f, 0.55f, 4.1f, 0.31f, 0.73f};
    static const FormatCost ternary = {{5.1f, 29.2f, 24.3f}, {6.7f, 51.6f, 38.4f}, {4, 15.8f, 16.6f}, {2.8f, 15.9f, 15.8f},
                                       {5.5f, 12.8f, 12.2f}, {4.3f, 15.3f, 13.1f}, {12, 89, 67.3f},
                                       {5.4f, 47.9f, 40.6f}, {8.4f, 84.1f, 69.7f}, 3.85f, 0.19f, 0.47f, 3, 0.31f, 0.85f};
    static const FormatCost q8_0 = {{3.2f, 38.4f, 31.4f}, {5.2f, 69.9f, 60.6f}, {1.8f, 29.2f, 27.1f}, {1.8f, 25.6f, 26.4f},
                                    {3.8f, 16.6f, 17.3f}, {1.8f, 29.8f, 27.2f}, {},
                                    {3.1f, 52.1f, 59.3f}, {}, 3.35f, 0.3f, 1.1f, 3.95f, 0.41f, 0.85f};
    static const FormatCost prism = {{4.4f, 32.2f, 26.4f}, {6.7f, 58.9f, 44.6f}, {3.3f, 21.1f, 20}, {2.8f, 21.3f, 19.7f},
                                     {4.5f, 14.9f, 13.5f}, {3.8f, 18.1f, 15.7f}, {},
                                     {4.9f, 47.1f, 44.6f}, {}, 2.9f, 0.27f, 1.2f, 3.35f, 0.41f, 1};
    static const FormatCost g64 = {{5, 31.6f, 24.1f}, {6.7f, 59.4f, 43.2f}, {3, 20.5f, 18.5f}, {2.9f, 18.5f, 17.9f},
                                   {5.2f, 13.4f, 13.2f}, {3.7f, 20, 17}, {12.3f, 102.8f, 68.7f},
                                   {4.4f, 56.5f, 44.6f}, {8.2f, 95.9f, 72.3f}, 3.05f, 0.2f, 0.87f, 3.15f, 0.31f, 1};
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
static float plan_cost(const GemmParams& p, int shape, uint32_t ks) {
    const FormatCost& f = format_cost(p.format);
    const bool low = shape == 4 || shape == 6;
    const TileCost& w = shape == 1 ? f.mid : shape == 0 || shape == 3 ? f.big : shape == 4 ? (ks > 1 ? f.low_split : f.low)
                      : shape == 5 ? f.kg : shape == 6 ? f.low_kg : shape == 7 ? f.wide : shape == 8 ? f.dual_wide : f.dual;
    const uint32_t T = tiles_of(p, rb_dims(shape)) * ks, rem = T % 256;
    const float ramp = low ? (float)rem / 256.0f : rem > 128 ? (float)(rem - 128) / 128.0f : 0.0f;
    float per_k = (float)(T / 256) * w.full;
    if (rem) per_k += w.half + (w.full - w.half) * ramp;
    float c = (float)((T + 255) / 256) * w.fix + per_k * (float)p.K / (4096.0f * (float)ks);
    if (ks > 1) {
        const float mb = (float)ks * (float)p.M * (float)columns_of(p) * (p.W2 ? 16.0f : 8.0f) / 4.5e6f;
        c += p.W2 ? f.d0 + f.d1 * (float)ks + f.db * mb : f.r0 + f.r1 * (float)ks + f.rb * mb;
    }
    return c;
}

// Base choice: the shape of rb_pick, K split (powers of two, whole 256-element
// super-blocks, >= 512 of K per split) while the grid still fits one wave of
// workgroups.
static void base_plan(GemmParams& p) {
    p.shape = rb_pick(p.format, p.M, p.N, p.K, p.W2 != nullptr);
    p.ksplit = 1;
    if (p.shape == 5 || p.shape == 6) return;  // K groups: the tile takes the whole K range
    const uint32_t T = tiles_of(p, rb_dims(p.shape));
    while (T * p.ksplit * 2 <= 256 && p.K % (256 * p.ksplit * 2) == 0 && p.K / (p.ksplit * 2) >= 512) p.ksplit *= 2;
}

uint32_t gemm_base_ksplit(const GemmParams& p0) {
    GemmParams p = p0;
    base_plan(p);
    return p.ksplit;
}

// The base choice, unless another is cheaper by more than its price may be off:
// any shape without a split or, where the base splits, 128- or 64-row tiles with as
// many splits or fewer (so no call needs more split-K partials than the base choice
// would).  2% for tiles of 128 or more rows without a split (SwiGLU's 256-row tiles
// 0: Q4_0 M = 5264, K = 1792, N = 3840 6% faster at an even price), 7% for the others,
// as the fits' errors lie, 12% for fewer splits of more than 2048 of K each (Q4_0, M =
// 128, K = 14336, N = 4096: 8 splits of 128 rows 29.9 us, 4 of 64 33.6).  Over 3368 shapes of 17 rows or more the chosen plans are
// 1.124x as fast as the base ones by geometric mean, 0.5% off the fastest, and 16 are
// more than 3% slower than their base (one table for all formats without a fixed
// cost per wave: 1.107x, 140, Q8_0 by up to 37%).  On 900 shapes outside the fits
// where the choices differ 1.187x, against 1.165x.
void gemm_plan(GemmParams& p) {
    const bool dual = p.W2 != nullptr;
    base_plan(p);
    if (p.format != QUANT_VAR_RATE_AFFINE && p.format != QUANT_EXL3) {  // those have one shape
        const bool groups_ok = p.K % 128 == 0, wide = groups_ok && wide_format(p.format);
        const int cand[6] = {dual ? 2 : 1, dual ? -1 : (big_k_format(p.format) ? 3 : 0), dual ? (wide ? 8 : -1) : (wide ? 7 : -1),
                             dual || !groups_ok ? -1 : 6, dual || !groups_ok || p.M > 128 ? -1 : 5, dual ? -1 : 4};
        const int shape0 = p.shape;
        const uint32_t ks0 = p.ksplit;
        const float base = plan_cost(p, shape0, ks0);
        float best = base;
        auto offer = [&](int s, uint32_t ks, float margin) {
            if (s == shape0 && ks == ks0) return;
            const float c = plan_cost(p, s, ks) + margin * base;
            if (c >= best) return;
            best = c;
            p.shape = s;
            p.ksplit = ks;
        };
        for (int s : cand)
            if (s >= 0) offer(s, 1, s == 4 || s == 5 || s == 6 ? 0.07f : s == 8 ? 0.0f : 0.02f);
        for (int s : {1, 4})
            for (uint32_t ks = 2; !dual && ks <= ks0; ks *= 2)
                offer(s, ks, ks < ks0 && p.K / ks > 2048 ? 0.12f : 0.07f);
    }
    p.group_m = (p.M + rb_dims(p.shape).bm - 1) / rb_dims(p.shape).bm >= 4 ? 4u : 2u;
}

Route choose_route(GemmParams& p) {
    if (gemv_fits(p)) return Route::kFewRows;
    if (p.ngroups <= 1 && skinny_supported(p)) return Route::kSmallM;
    gemm_plan(p);
    return Route::kTiled;
}

TileInfo gemm_tile(const GemmParams& p) {
    const RbShape d = rb_dims(p.shape);
    return {d.bm, d.bn, p.shape == 5 || p.shape == 6 ? 2u : 1u};
}

size_t gemm_workspace_floats(const GemmParams& p) {
    return p.ksplit > 1 ? (size_t)p.ksplit * p.M * columns_of(p) * (p.W2 != nullptr ? 2 : 1) : 0;
}

}  // namespace qr
