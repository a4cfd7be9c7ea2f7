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

// blockIdx.y is the group of a grouped projection (its partials follow the
// previous group's).
struct RedGroups {
    _Float16* Y[3];
    uint32_t N[3];
};

template <bool DUAL>
__global__ void __launch_bounds__(256) splitk_reduce_kernel(const float* __restrict__ ws, uint32_t ks, uint32_t M,
                                                            RedGroups gr, const _Float16* __restrict__ R,
                                                            uint32_t head_D) {
    const uint32_t grp = blockIdx.y;
    if (grp > 0) ws += (size_t)ks * M * (gr.N[0] + (grp > 1 ? gr.N[1] : 0u));
    const uint32_t N = grp == 0 ? gr.N[0] : (grp == 1 ? gr.N[1] : gr.N[2]);
    _Float16* const __restrict__ Y = grp == 0 ? gr.Y[0] : (grp == 1 ? gr.Y[1] : gr.Y[2]);
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

static hipError_t reduce_groups(const float* ws, uint32_t ks, uint32_t M, const RedGroups& gr, uint32_t ngroups, bool dual,
                                const _Float16* R, uint32_t head_D, hipStream_t st) {
    uint32_t n = gr.N[0];
    for (uint32_t g = 1; g < ngroups; g++) n = gr.N[g] > n ? gr.N[g] : n;
    const size_t plane = (size_t)M * n;
    const dim3 grid((unsigned)((plane + 256 * kRedVec - 1) / (256 * kRedVec)), ngroups);
    if (dual) hipLaunchKernelGGL(splitk_reduce_kernel<true>, grid, dim3(256), 0, st, ws, ks, M, gr, R, head_D);
    else hipLaunchKernelGGL(splitk_reduce_kernel<false>, grid, dim3(256), 0, st, ws, ks, M, gr, R, head_D);
    return hipGetLastError();
}

hipError_t launch_splitk_reduce(const float* ws, uint32_t ks, uint32_t M, uint32_t N, bool dual, const _Float16* R,
                                _Float16* Y, uint32_t head_D, hipStream_t st) {
    return reduce_groups(ws, ks, M, RedGroups{{Y, nullptr, nullptr}, {N, 0, 0}}, 1, dual, R, head_D, st);
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
        e = reduce_groups(p.ws, p.ksplit, p.M, RedGroups{{p.Y, p.Yx[0], p.Yx[1]}, {p.N, p.Nx[0], p.Nx[1]}},
                          p.ngroups > 1 ? p.ngroups : 1, p.W2 != nullptr, p.R, p.head_D, st);
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

// One workgroup fits a CU, so a grid runs in waves of 256 tiles.  What a wave
// takes, in us at K = 4096 (it is proportional to K but for ~5 us), per shape:
// `lo` while at most half of the CUs have a tile, rising to `hi` when all have
// (the clock falls as the chip fills).  Measured on MLX and Q4_0 weights (they
// agree to 5%; ternary is ~10% faster at every shape) and on Q4_K, whose decode
// is the heaviest; e.g. MLX at N = 14336: M = 900 128 x 128 tiles 142.7,
// 128 x 256 121.2, 256 x 256 107.4; M = 450 71.4 / 61.6 / 82.4; M = 256
// 37.0 / 52.5 / 81.5.
struct WaveCost {
    float lo, hi;
};
static WaveCost wave_cost(int shape, bool q4k) {
    switch (shape) {
        case 0: return q4k ? WaveCost{68, 77} : WaveCost{51, 72};
        case 3: return q4k ? WaveCost{61, 77} : WaveCost{50, 72};
        case 1: return q4k ? WaveCost{39.5f, 47} : WaveCost{31, 39};
        case 4: return q4k ? WaveCost{33, 34.5f} : WaveCost{25, 28};
        case 5: return q4k ? WaveCost{24, 29} : WaveCost{19, 26};
        case 6: return q4k ? WaveCost{27, 31} : WaveCost{18.5f, 25};
        case 7: return q4k ? WaveCost{97, 130} : WaveCost{81, 122};
        case 8: return q4k ? WaveCost{94, 130} : WaveCost{79, 122};
        default: return q4k ? WaveCost{66, 82} : WaveCost{53, 72};  // 2: SwiGLU 128 x 128
    }
}
static float plan_cost(const GemmParams& p, int shape, uint32_t ks) {
    const WaveCost w = wave_cost(shape, p.format == QUANT_Q4_K);
    const uint32_t T = tiles_of(p, rb_dims(shape)) * ks, rem = T % 256;
    float c = (float)(T / 256) * w.hi;
    if (rem) c += w.lo + (rem > 128 ? (w.hi - w.lo) * (float)(rem - 128) / 128.0f : 0.0f);
    c *= (float)p.K / (4096.0f * (float)ks);
    // the reduction kernel (each split's loads in turn) and the partials' round trip at ~4.5 TB/s
    if (ks > 1) c += 2.5f + 0.35f * (float)ks + (float)ks * (float)p.M * (float)columns_of(p) * (p.W2 ? 16.0f : 8.0f) / 4.5e6f;
    return c;
}

// The base shape with its K split, unless another is cheaper by its tile counts:
// any shape without a split, or, where the base splits, 128- or 64-row tiles with
// as many splits or fewer (so no call needs more split-K partials than the base
// choice would).  MLX, M = 77, K = 8192, N = 2048: 16 splits of 128-row tiles
// 20.8 us, 8 of 64-row tiles 16.4 (launch included); M = 128, K = N = 4096
// 21.1 -> 16.3.
void gemm_plan(GemmParams& p) {
    const bool dual = p.W2 != nullptr;
    p.shape = rb_pick(p.format, p.M, p.N, p.K, dual);
    p.ksplit = 1;
    if (p.shape != 5 && p.shape != 6) {  // K groups: the tile takes the whole K range
        // split K (powers of two, whole 256-element super-blocks, >= 512 of K
        // per split) while the grid still fits one wave
        const uint32_t T = tiles_of(p, rb_dims(p.shape));
        while (T * p.ksplit * 2 <= 256 && p.K % (256 * p.ksplit * 2) == 0 && p.K / (p.ksplit * 2) >= 512) p.ksplit *= 2;
    }
    if (p.format != QUANT_VAR_RATE_AFFINE && p.format != QUANT_EXL3) {  // those have one shape
        const bool heavy = p.format == QUANT_Q4_K || p.format == QUANT_TERNARY_1_58;
        const bool groups_ok = p.K % 128 == 0, wide = groups_ok && wide_format(p.format);
        const int cand[6] = {dual ? 2 : 1, dual ? -1 : (heavy ? 3 : 0), dual ? (wide ? 8 : -1) : (wide ? 7 : -1),
                             dual || !groups_ok ? -1 : 6, dual || !groups_ok || p.M > 128 ? -1 : 5, dual ? -1 : 4};
        const float base = plan_cost(p, p.shape, p.ksplit);
        const float margin = 0.08f * base;  // a near tie keeps the base's split (M = 640, K = 4096, N = 1024 ran even)
        // one kernel without partials on a tie: M = 700, K = 4096, N = 1024 18.7 us, split 19.4
        float best = p.ksplit > 1 ? base : 0.97f * base;
        uint32_t ksplit = p.ksplit;
        for (int s : cand) {
            if (s < 0) continue;
            const float c = plan_cost(p, s, 1);
            if (c < best) {
                best = c;
                p.shape = s;
                ksplit = 1;
            }
        }
        for (int s : {1, 4})
            for (uint32_t ks = 2; !dual && ks <= p.ksplit; ks *= 2) {
                const float c = plan_cost(p, s, ks) + margin;
                if (c < best) {
                    best = c;
                    p.shape = s;
                    ksplit = ks;
                }
            }
        p.ksplit = ksplit;
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
