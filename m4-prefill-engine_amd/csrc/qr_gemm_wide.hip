// qr_gemm_wide.hip -- quantized projection Y = X . W^T on gfx950 MFMA for
// large grids: 256 x 256 output tiles (SwiGLU: 256 x 128 of gate and up),
// weights decoded once per 256 rows into LDS.  Built once per format with
// -DQR_GEMM_FORMAT=F.
//
// What bounds the 128-row tiles of qr_gemm.hip at large M is the decode (3.9 -
// 8.9 VALU ops per MFMA) and the fragment reads; here 4 waves of 128 x 128 wave
// tiles (256 accumulators, one wave per SIMD) halve both:
//  * K advances 32 per step, one quant group of every column.  Thread t decodes
//    column t's group of step i + 2 during step i and writes it to a ring of two
//    LDS slots; every wave reads its 128 rows and 128 columns as fragments, one
//    k-slice ahead.  One barrier per step, placed between the step's two
//    k-slices: every fragment of step i is in registers by then, so its slots
//    can be refilled behind it.
//  * X and the packed weights come by buffer-load-to-LDS copies in inline asm:
//    X as whole 128-byte lines (two steps) two to three steps ahead, the packed
//    bytes of 128 K (72 - 80 bytes a column, coalesced over columns) a round
//    ahead.  The compiler does not know of these copies, so it puts no waits on
//    them; the explicit vmcnt before each barrier counts them exactly (the
//    kernel issues no other vector-memory operation before the epilogue).
//  * Decode, copies and fragment reads are spread over four chunks per k-slice
//    between the MFMAs.
// Measured (MLX g64, M = 8192, K = 4096, N = 14336, SwiGLU and down projection)
// 2762 -> 2365 us, i.e. 1.04 -> 1.22 PF; Q4_K SwiGLU at M = 1000, K = 4096, N = 14336
// 309 -> 241 us.  The matrix pipe is 67% busy at 1.65 GHz (counters, g64), 2.0 - 2.2
// VALU ops and 0.7 LDS ops per MFMA; 47% at 2.0 GHz for Q4_K at M = 1000 (3.1 VALU ops).
#include "qr_decode.h"
#include "qr_gemm_shapes.h"

namespace qr {
namespace wide {

constexpr int kXRing = 3;      // pairs of steps of X held in LDS
constexpr int kWRing = 2;      // steps of decoded weights held in LDS
constexpr int kThreads = 256;  // 2 x 2 waves

template <int TM, int TN>
struct Cfg {
    static constexpr int BM = 64 * TM, BN = 64 * TN;
    static constexpr int XSLOT = BM * 128;                  // bytes of X of two steps
    static constexpr int WSLOT = BN * 64;                   // bytes of the weights of one step
    static constexpr int XCP = XSLOT / 1024 / 8;            // 1 KB copies per wave of half a pair's rows
    static constexpr int ERS = 32 * TN + 16;                // floats per row of the epilogue band
    static constexpr int EPI_BYTES = 4 * 32 * ERS * 4;
    template <int NU> static constexpr int lds_bytes() {    // NU: 16-byte units of a column's round
        constexpr int ring = kXRing * XSLOT + kWRing * WSLOT + BN * NU * 16;
        return ring > EPI_BYTES ? ring : EPI_BYTES;
    }
};

// 64-byte LDS rows hold a row's 32 k values as four 16-byte units; unit u of
// row r sits at u ^ swz(r), chosen so that 16 lanes reading one unit hit distinct
// banks both for 16 consecutive rows and for the rows {0-3, 12-15, 20-27} /
// {4-11, 16-19, 28-31} (M = 8192, N = 4096, K = 14336: 5.2e5 conflict cycles in 2.0e7
// LDS instructions).
__device__ __forceinline__ uint32_t swz(uint32_t r) { return ((r >> 2) & 3u) ^ (r & 2u); }
// 128-byte rows (X of a pair of steps): unit u of row r at u ^ xswz(r).
__device__ __forceinline__ uint32_t xswz(uint32_t r) { return (r ^ (r >> 3)) & 7u; }

// The packed bytes of one column for one round of 4 steps (128 K), as kUnits
// 16-byte units copied to LDS.  off(u) is unit u's byte offset from the round's
// start in the column (72-byte rounds: the last unit is bytes 56..71, so that
// nothing past the round is read, and words 16.. of the units are two on from the
// round's); group() picks the raw words that decode_half_fast takes for group g of
// the round, and returns its parity argument.
constexpr int kRG = 4;
template <int F> struct Round;
template <> struct Round<QUANT_Q4_0> {
    static constexpr int kUnits = 5, kBytes = 72;
    __device__ static uint32_t off(uint32_t u) { return u < 4 ? 16u * u : 56u; }
    __device__ static uint32_t group(const uint32_t* w, int g, uint32_t, uint32_t* raw) {
#pragma unroll
        for (int i = 0; i < 5; i++) {
            const int k = 18 * g / 4 + i;
            raw[i] = w[k < 16 ? k : k + 2];
        }
        return (uint32_t)(18 * g) & 2u;
    }
};
template <> struct Round<QUANT_MLX_4BIT> {
    static constexpr int kUnits = 5, kBytes = 80;
    __device__ static uint32_t off(uint32_t u) { return 16u * u; }
    __device__ static uint32_t group(const uint32_t* w, int g, uint32_t, uint32_t* raw) {
#pragma unroll
        for (int i = 0; i < 5; i++) raw[i] = w[5 * g + i];
        return 0;
    }
};
template <> struct Round<QUANT_MLX_4BIT_G64> {
    static constexpr int kUnits = 5, kBytes = 72;
    __device__ static uint32_t off(uint32_t u) { return u < 4 ? 16u * u : 56u; }
    __device__ static uint32_t group(const uint32_t* w, int g, uint32_t, uint32_t* raw) {
        raw[0] = w[9 * (g >> 1)];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int k = 9 * (g >> 1) + 1 + 4 * (g & 1) + i;
            raw[1 + i] = w[k < 16 ? k : k + 2];
        }
        return 0;
    }
};
template <> struct Round<QUANT_TERNARY_1_58> {
    static constexpr int kUnits = 3, kBytes = 48;
    __device__ static uint32_t off(uint32_t u) { return 16u * u; }
    __device__ static uint32_t group(const uint32_t* w, int g, uint32_t, uint32_t* raw) {
#pragma unroll
        for (int i = 0; i < 3; i++) raw[i] = w[3 * g + i];
        return 0;
    }
};
// Q4_K: half a super-block: its header, then the half's four sub-blocks.
template <> struct Round<QUANT_Q4_K> {
    static constexpr int kUnits = 5, kBytes = 72;
    __device__ static uint32_t off(uint32_t u) { return 16u * u; }
    __device__ static uint32_t group(const uint32_t* w, int g, uint32_t round, uint32_t* raw) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            raw[i] = w[i];
            raw[4 + i] = w[4 + 4 * g + i];
        }
        return 4u * (round & 1u) + (uint32_t)g;
    }
};

}  // namespace wide

template <int F, int TM, int TN, bool DUAL>
__global__ void __launch_bounds__(wide::kThreads, 1) gemm_wide_kernel(GemmParams p) {
    using C = wide::Cfg<TM, TN>;
    using Dec = Decoder<F>;
    constexpr int XR = wide::kXRing, WR = wide::kWRing, XSLOT = C::XSLOT, WSLOT = C::WSLOT, XCP = C::XCP, BM = C::BM;
    constexpr int NJ = DUAL ? TN / 2 : TN;        // 32-column output tiles per wave
    constexpr int BNO = 64 * NJ;                  // output columns of the workgroup
    using RD = wide::Round<F>;
    constexpr int NU = RD::kUnits, NW = 4 * NU;   // 16-byte units and words of a column's round
    constexpr int U = wide::kRG;                  // steps unrolled: one round
    static_assert(C::BN == wide::kThreads, "one column per thread");
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wr = wave >> 1, wc = wave & 1, h = lane >> 5, c32 = lane & 31;

    uint32_t bid = blockIdx.x;
    if (p.ngroups > 1) {
        const uint32_t ntm = (p.M + BM - 1) / BM;
        const uint32_t t0 = ntm * ((p.N + BNO - 1) / BNO);
        if (bid >= t0) {
            bid -= t0;
            const uint32_t t1 = ntm * ((p.Nx[0] + BNO - 1) / BNO);
            const int gx = (bid < t1 || p.ngroups == 2) ? 0 : 1;
            if (gx == 1) bid -= t1;
            p.W = p.Wx[gx];
            p.Y = p.Yx[gx];
            p.N = p.Nx[gx];
        }
    }
    const uint32_t M = p.M, N = p.N, K = p.K;
    const uint32_t nt_m = (M + BM - 1) / BM, nt_n = (N + BNO - 1) / BNO;
    uint32_t tmi, tni;
    tile_of(bid, nt_m, nt_n, p.group_m, tmi, tni);
    const int m0 = tmi * BM, n0 = tni * BNO;
    const uint32_t nsteps = K / 32;
    const uint32_t col_bytes = (uint32_t)p.col_bytes;
    const int mrows = min(BM, (int)M - m0), ncols = min(BNO, (int)N - n0);

    // ---- X copies: a pair of steps is 128 bytes of every row (whole cache
    // lines), copied in two halves of the rows; copy q of this wave fills rows
    // 8 (XCP wave + q) .. + 7 of its half ----
    const u4_t xr = scalar_rsrc(p.X + (size_t)m0 * K, (uint32_t)mrows * K * 2u);
    uint32_t xo[2][XCP];
#pragma unroll
    for (int f = 0; f < 2; f++)
#pragma unroll
        for (int q = 0; q < XCP; q++) {
            const uint32_t r = (uint32_t)(BM / 2 * f) + 8u * (uint32_t)(XCP * wave + q) + (uint32_t)(lane >> 3);
            xo[f][q] = r < (uint32_t)mrows ? (r * K + 8u * (((uint32_t)lane & 7u) ^ wide::xswz(r))) * 2u : kOOB;
        }
    const uint32_t lds0 = (uint32_t)reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) uint8_t*)smem);
    const uint32_t xdst = lds0 + (uint32_t)(XCP * wave) * 1024u;
    auto issue_x = [&](uint32_t pair, int f, uint32_t xoff, int q) {
        const uint32_t soff = 2u * min(pair, nsteps / 2 - 1) * 64u;
        copy_lds(xdst + xoff + (uint32_t)(f * (XSLOT / 2) + q * 1024), xo[f][q], xr, soff);
    };

    // ---- weights: a round's packed bytes are copied to LDS (column after
    // column, NU units each), and thread t decodes column t of the W slots.
    // DUAL: columns 128 w .. + 63 are gate columns 64 w .. + 63, the next 64 the up columns.
    uint8_t* const wring = smem + XR * XSLOT;
    uint8_t* const wraw = wring + WR * WSLOT;
    const uint32_t nrounds = nsteps / wide::kRG;
    const u4_t wrs = scalar_rsrc((DUAL && (wave & 1) ? p.W2 : p.W) + (size_t)n0 * col_bytes, (uint32_t)ncols * col_bytes);
    // copy q of this wave: units 64 (NU wave + q) + lane, i.e. columns 64 wave .. + 63
    uint32_t wo[NU], wodd[F == QUANT_Q4_K ? NU : 1];
#pragma unroll
    for (int q = 0; q < NU; q++) {
        const uint32_t un = 64u * (uint32_t)q + (uint32_t)lane, u = un % NU;
        const uint32_t col = (uint32_t)(DUAL ? 64 * (wave >> 1) : 64 * wave) + un / NU;
        wo[q] = col < (uint32_t)ncols ? col * col_bytes + RD::off(u) : kOOB;
        if constexpr (F == QUANT_Q4_K) wodd[q] = u ? 64u : 0u;
    }
    const uint32_t wrawdst = lds0 + (uint32_t)(XR * XSLOT + WR * WSLOT + NU * wave * 1024);
    auto issue_w = [&](uint32_t rd, int q) {
        const uint32_t r = min(rd, nrounds - 1);
        const uint32_t soff = F == QUANT_Q4_K ? (r >> 1) * 144u : r * (uint32_t)RD::kBytes;
        uint32_t vo = wo[q];
        if constexpr (F == QUANT_Q4_K) vo += (r & 1u) ? wodd[q] : 0u;
        copy_lds(wrawdst + (uint32_t)q * 1024u, vo, wrs, soff);
    };
    uint32_t rw[NW];
    auto read_raw = [&]() {
#pragma unroll
        for (int u = 0; u < NU; u++) {
            const u4_t v = *reinterpret_cast<const u4_t*>(wraw + (tid * NU + u) * 16);
            rw[4 * u] = v.x; rw[4 * u + 1] = v.y; rw[4 * u + 2] = v.z; rw[4 * u + 3] = v.w;
        }
    };
    uint32_t wdst[4];
#pragma unroll
    for (int u = 0; u < 4; u++) wdst[u] = (uint32_t)tid * 64u + 16u * ((uint32_t)u ^ wide::swz((uint32_t)tid));
    // Words 2 q, 2 q + 1 (q = 0 .. 7) of group g of the round in rw.  The whole
    // half is named and the rest dropped by the compiler.
    auto decode_w = [&](uint32_t rd, int g, int q, uint32_t o[16]) {
        uint32_t raw[Dec::kRawWords], t[8];
        const uint32_t par = RD::group(rw, g, rd, raw);
        decode_half_fast<F>(raw, par, q >> 2, t);
        o[2 * q] = t[2 * (q & 3)];
        o[2 * q + 1] = t[2 * (q & 3) + 1];
    };
    // Unit u (words 4 u .. + 3) of a decoded group to the W slot at woff.
    auto write_w = [&](int u, const uint32_t o[16], int woff) {
        *reinterpret_cast<u4_t*>(wring + woff + wdst[u]) = u4_t{o[4 * u], o[4 * u + 1], o[4 * u + 2], o[4 * u + 3]};
    };
    // Groups outside the fast decode's range (Q4_K binade gap, Q4_0 scales with
    // -8 d not finite) are decoded again exactly, over the words just written.
    auto fix_w = [&](uint32_t rd, int g, int woff) {
        if constexpr (F == QUANT_Q4_K || F == QUANT_Q4_0) {
            uint32_t raw[Dec::kRawWords];
            const uint32_t par = RD::group(rw, g, rd, raw);
            const bool slow = needs_exact<F>(raw, par);
            if (__any(slow)) {
                uint32_t ex[16];
                decode_group<F>(raw, par, ex);
                if (slow) {
#pragma unroll
                    for (int u = 0; u < 4; u++) write_w(u, ex, woff);
                }
            }
        }
    };

    // ---- fragments ----
    const uint32_t ar = (uint32_t)(32 * TM * wr + c32), br = (uint32_t)(32 * TN * wc + c32);
    uint32_t ao[4], bo[2];  // slice kk of step parity p: ao[2 p + kk]
#pragma unroll
    for (int q = 0; q < 4; q++) ao[q] = ar * 128u + 16u * ((uint32_t)(2 * q + h) ^ wide::xswz(ar));
#pragma unroll
    for (int kk = 0; kk < 2; kk++) bo[kk] = br * 64u + 16u * ((uint32_t)(2 * kk + h) ^ wide::swz(br));
    h8_t af[2][TM], bf[2][TN];
    // row + 32 flips bit 2 of xswz, i.e. the step parity's half of the row
    auto read_b = [&](int woff, int kk, int j) { bf[kk][j] = *reinterpret_cast<const h8_t*>(wring + woff + bo[kk] + j * 2048); };
    auto read_a = [&](uint32_t xoff, int par, int kk, int i) {
        af[kk][i] = *reinterpret_cast<const h8_t*>(smem + xoff + ao[2 * ((par + i) & 1) + kk] + i * 4096);
    };

    f16v_t acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = f16v_t{};

    // Iteration i = t0 + j of a round, between two barriers: slice 1 of step i,
    // then slice 0 of step i + 1.  The fragments of step i were all read before
    // the barrier that opens it, so its slots are free: the weights of step
    // i + 2 are decoded into W slot i mod 2, and the X pair that ended with step
    // i (odd i) is replaced by the pair three later, half of its rows now and
    // half in the next iteration.  xa, xb, xc: LDS offsets of the X pairs of
    // steps t0, t0 + 2 and t0 + 4.  The packed bytes of a round are read into
    // registers in its first decode (j = 2); the next round's are copied over
    // them from j = 3.
    uint32_t xa = 0, xb = XSLOT, xc = 2u * XSLOT;
    static_assert(TM == 4 && TN == 4 && XCP <= 4, "a chunk is a column tile and a row tile");
    // Slice kk as four chunks: one column tile's MFMAs beside a quarter of the
    // half-group decode, two fragment reads of the next slice and at most two
    // copies (several copies in a row stall the wave at issue while nothing
    // feeds the matrix pipe).
    uint32_t o[16];  // the group being decoded
    auto slice = [&](uint32_t t0, int j, int kk) {
        const uint32_t g = t0 / 2, i = t0 + j, rd = (i + 2) / wide::kRG;
        const uint32_t xoff = j == 0 ? xa : (j == 3 ? xc : xb);
        const int woff = ((j + 1) % WR) * WSLOT, nk = kk ^ 1;
        if (j == 2 && kk == 1) read_raw();
#pragma unroll
        for (int c = 0; c < 4; c++) {
            __builtin_amdgcn_sched_barrier(0);
            if (kk == 1 && c < XCP)
                issue_x(j == 0 ? g + 2 : (j == 3 ? g + 4 : g + 3), j & 1 ? 0 : 1, j == 0 ? xc : (j == 3 ? xb : xa), c);
            if (kk == 0 && j == 3) {
                if (c < NU) issue_w(rd + 1, c);
                if (c + 4 < NU) issue_w(rd + 1, c + 4);
            }
            // fragments of the next slice in the first three chunks
#pragma unroll
            for (int q = 3 * c; q < 3 * c + 3 && q < 8; q++) {
                if (q == 0) read_b(woff, nk, 0);
                else if (q <= 4) read_a(xoff, (j + 1) & 1, nk, q - 1);
                else read_b(woff, nk, q - 4);
            }
#pragma unroll
            for (int r = 0; r < TM; r++)
                acc[r][c] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[kk][r], bf[kk][c], acc[r][c], 0, 0, 0);
            // decode: word pairs 0 | 1 | 2 3 | 4 in slice 1, 5 | 6 7 in slice 0, so
            // that the last LDS write is two chunks old at the barrier
            const int q0 = kk == 1 ? (c == 3 ? 4 : c) : (c == 0 ? 5 : 6);
            const int q1 = kk == 1 ? (c == 2 ? 4 : q0 + 1) : (c == 0 ? 6 : (c == 1 ? 8 : 6));
#pragma unroll
            for (int q = q0; q < q1; q++) {
                decode_w(rd, (j + 2) % 4, q, o);
                // keeps the decode in its chunk (the compiler sinks it behind the MFMAs otherwise)
                asm volatile("" : "+v"(o[2 * q]), "+v"(o[2 * q + 1]));
                if (q & 1) write_w(q >> 1, o, (j % WR) * WSLOT);
            }
#pragma unroll
            for (int q = 0; q < TM; q++) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // DS read
                __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);  // VALU
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        if (kk == 0) fix_w(rd, (j + 2) % 4, (j % WR) * WSLOT);
    };
    auto second = [&](uint32_t t0, int j) {
        slice(t0, j, 0);
        // Copies retire in order.  Before this barrier the X pair of step i + 2,
        // whose second half was issued two or more iterations ago, has to land, and at j = 1 the
        // weight bytes, issued two iterations ago (j = 3) after that one's X.
        // Younger than what has to land are the XCP copies of each of the last
        // two iterations, and at j = 3 and 0 the NU of the weights.  Own LDS
        // reads and writes done.
        if (j == 3 || j == 0) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(2 * XCP + NU) : "memory");
        else asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(2 * XCP) : "memory");
    };

    // ---- prologue: weights of steps 0, 1 decoded, X of steps 0..3 and half of the
    // next pair, the second round's bytes under way, slice 0 of step 0 multiplied ----
#pragma unroll
    for (int q = 0; q < NU; q++) issue_w(0, q);
#pragma unroll
    for (int t = 0; t < 5 * XCP; t++) issue_x(t / XCP / 2, t / XCP & 1, (uint32_t)(t / XCP / 2 * XSLOT), t % XCP);
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(5 * XCP) : "memory");
    read_raw();
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
    for (int q = 0; q < NU; q++) issue_w(1, q);
#pragma unroll
    for (int t = 0; t < 2; t++) {
#pragma unroll
        for (int q = 0; q < 8; q++) decode_w(0, t, q, o);
#pragma unroll
        for (int u = 0; u < 4; u++) write_w(u, o, t * WSLOT);
        fix_w(0, t, t * WSLOT);
    }
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(3 * XCP + NU) : "memory");  // the first X pair
#pragma unroll
    for (int kk = 0; kk < 2; kk++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            read_b(0, kk, i);
            read_a(0, 0, kk, i);
        }
#pragma unroll
    for (int c = 0; c < TN; c++)
#pragma unroll
        for (int r = 0; r < TM; r++)
            acc[r][c] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[0][r], bf[0][c], acc[r][c], 0, 0, 0);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // every wave has read step 0

    for (uint32_t t0 = 0;; t0 += U) {  // whole rounds
#pragma unroll
        for (int j = 0; j < U; j++) {
            slice(t0, j, 1);
            if (j == U - 1 && t0 + U >= nsteps) break;  // slice 1 of the last step
            second(t0, j);
        }
        if (t0 + U >= nsteps) break;
        const uint32_t t = xa;  // two pairs on
        xa = xc;
        xc = xb;
        xb = t;
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");  // copies past the end have landed

    // ---- epilogue, one 32-row band of the wave tile at a time through LDS:
    // accumulator element r of lane l is row 8 (r / 4) + 4 (l / 32) + r % 4,
    // column l % 32 of its 32 x 32 tile; a lane then owns 8 consecutive columns
    // of one row. ----
    const int r0 = m0 + 32 * TM * wr, c0 = n0 + 32 * NJ * wc;
    const bool vec_io = ((reinterpret_cast<uintptr_t>(p.Y) | reinterpret_cast<uintptr_t>(p.R)) & 15u) == 0 &&
                        (N & 7u) == 0 && (p.head_D & 7u) == 0;
    constexpr int ERS = C::ERS;
    float* const E = reinterpret_cast<float*>(smem) + wave * 32 * ERS;
    auto put = [&](int m, int n, float v[8], int cnt) {  // cnt columns of row m from n, one rounding
        if (p.R) {
            const _Float16* r = p.R + (size_t)m * N + n;
#pragma unroll
            for (int q = 0; q < 8; q++)
                if (q < cnt) v[q] += (float)r[q];
        }
#pragma unroll
        for (int q = 0; q < 8; q++) {
            if (q >= cnt) continue;
            const uint32_t nn = (uint32_t)(n + q);
            const size_t o = p.head_D ? ((size_t)(nn / p.head_D) * M + m) * p.head_D + nn % p.head_D : (size_t)m * N + nn;
            p.Y[o] = (_Float16)v[q];
        }
    };
#pragma unroll
    for (int i = 0; i < TM; i++) {
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) E[(8 * (r >> 2) + 4 * h + (r & 3)) * ERS + 32 * j + c32] = acc[i][j][r];
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // own LDS writes done (wave-local region)
        __builtin_amdgcn_wave_barrier();
        constexpr int C8 = 4 * NJ;  // 8-column chunks per row
#pragma unroll 1
        for (int c = lane; c < 32 * C8; c += 64) {
            const int row = c / C8, c8 = c % C8;
            const int m = r0 + i * 32 + row, n = c0 + c8 * 8;
            if (m >= (int)M || n >= (int)N) continue;
            const float* e = E + row * ERS + c8 * 8;
            const f4_t lo = *reinterpret_cast<const f4_t*>(e), hi = *reinterpret_cast<const f4_t*>(e + 4);
            float v[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w}, u[8];
            if constexpr (DUAL) {
                const f4_t ul = *reinterpret_cast<const f4_t*>(e + 32 * NJ), uh = *reinterpret_cast<const f4_t*>(e + 32 * NJ + 4);
                const float uu[8] = {ul.x, ul.y, ul.z, ul.w, uh.x, uh.y, uh.z, uh.w};
#pragma unroll
                for (int q = 0; q < 8; q++) u[q] = uu[q];
            }
            const int cnt = min(8, (int)N - n);
            if constexpr (DUAL) {
#pragma unroll
                for (int q = 0; q < 8; q++) v[q] = silu_mul(v[q], u[q]);
            }
            if (!vec_io) {
                put(m, n, v, cnt);
                continue;
            }
            if (p.R) {
                const u4_t rr = *reinterpret_cast<const u4_t*>(p.R + (size_t)m * N + n);
                const uint32_t rw[4] = {rr.x, rr.y, rr.z, rr.w};
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const h2_t hh = as_h2(rw[q]);
                    v[2 * q] += (float)hh.x;
                    v[2 * q + 1] += (float)hh.y;
                }
            }
            u4_t o;
            o.x = pack_h2(f2h_bits(v[0]), f2h_bits(v[1]));
            o.y = pack_h2(f2h_bits(v[2]), f2h_bits(v[3]));
            o.z = pack_h2(f2h_bits(v[4]), f2h_bits(v[5]));
            o.w = pack_h2(f2h_bits(v[6]), f2h_bits(v[7]));
            const size_t off = p.head_D ? ((size_t)((uint32_t)n / p.head_D) * M + m) * p.head_D + (uint32_t)n % p.head_D
                                        : (size_t)m * N + n;
            *reinterpret_cast<u4_t*>(p.Y + off) = o;
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_wave_barrier();  // band reads done before the next band overwrites
    }
}

template <int F, bool DUAL>
static hipError_t wide_launch(const GemmParams& p, hipStream_t st) {
    using C = wide::Cfg<4, 4>;
    constexpr uint32_t BNO = DUAL ? C::BN / 2 : C::BN;
    auto kern = gemm_wide_kernel<F, 4, 4, DUAL>;
    const uint32_t ntm = (p.M + C::BM - 1) / C::BM;
    uint32_t T = ntm * ((p.N + BNO - 1) / BNO);
    for (uint32_t g = 1; g < p.ngroups && g < 3; g++) T += ntm * ((p.Nx[g - 1] + BNO - 1) / BNO);
    constexpr int lds = C::template lds_bytes<wide::Round<F>::kUnits>();
    if (p.K % 128 || p.ksplit > 1) return hipErrorInvalidValue;  // gemm_plan never asks for these
    static size_t attr[kMaxDevices] = {};
    const hipError_t e = lds_limit_once((const void*)kern, lds, attr);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kern, dim3(T), dim3(wide::kThreads), lds, st, p);
    return hipGetLastError();
}

template <int F>
hipError_t launch_gemm_wide_format(const GemmParams& p, hipStream_t st) {
    return p.W2 ? wide_launch<F, true>(p, st) : wide_launch<F, false>(p, st);
}

#ifndef QR_GEMM_FORMAT
#error "build qr_gemm_wide.hip with -DQR_GEMM_FORMAT=<format id>"
#endif
template hipError_t launch_gemm_wide_format<QR_GEMM_FORMAT>(const GemmParams& p, hipStream_t st);

}  // namespace qr
