// qr_attention.hip -- Q8_0 KV-cache quantization and causal flash attention
// over the Q8_0 cache on gfx950.
//
// Replaces quantize_kv_to_q8_0 (unified_kernels.metal:118-145) and
// flash_attn_mma_64x64_q8_0_impl<D> (brick4_attn_kernels.metal:572-881).
//
//  * The Q8_0 cache is dequantized once per call into an fp16 cache (K' rows,
//    V' transposed), each value the reference's half(q * half(d))
//    (brick4_attn_bench.mm:57-65), so query tiles stage K/V tiles with plain
//    copies instead of decoding them again per query tile.
//  * Each wave owns 32 queries and computes S^T = K . Q^T with
//    v_mfma_f32_32x32x16_f16, so a lane owns ONE query column: the softmax
//    row statistics are lane-local over its 16 accumulator rows plus one
//    exchange with the partner lane (l ^ 32) -- no 32-lane reduction trees.
//  * P stays in registers: the S^T accumulator of a lane already holds the
//    8 keys that lane must supply as the B operand of O^T = V^T . P^T, given
//    the matching key order of the cached V'^T.
//  * fp32 running max / sum / output accumulators (the reference keeps
//    S, P and O in half); the output is rounded to fp16 once.
#include "qr_device.h"
#include "qr_kernels.h"

namespace qr {

// --------------------------------------------------------------------------
// Q8_0 quantization: per 32 values amax in fp32, d = amax / 127 (IEEE
// division), stored as half(d); codes q = round(x * (1/d)) (half away from
// zero) with the UNROUNDED d, clamped to [-128, 127] (unified_kernels.metal:
// 118-145).  One thread per block.
// --------------------------------------------------------------------------
// One block: x[32] -> half(d) bits and 16 code words (two int8 codes each).
__device__ __forceinline__ void quantize_block_q8_0(const float x[32], uint32_t& d16, uint32_t codes[16]) {
    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < 32; i++) amax = fmaxf(amax, fabsf(x[i]));
    const float d = amax / 127.0f;
    const float id = d > 0.0f ? 1.0f / d : 0.0f;
    d16 = f2h_bits(d);
#pragma unroll
    for (int i = 0; i < 16; i++) {
        int q0 = (int)__builtin_roundf(x[2 * i] * id);
        int q1 = (int)__builtin_roundf(x[2 * i + 1] * id);
        q0 = q0 < -128 ? -128 : (q0 > 127 ? 127 : q0);
        q1 = q1 < -128 ? -128 : (q1 > 127 ? 127 : q1);
        codes[i] = (uint32_t)((q0 & 0xff) | ((q1 & 0xff) << 8));
    }
}

__device__ __forceinline__ void load_block_f16(const _Float16* src, float x[32]) {
    const u4_t* s = reinterpret_cast<const u4_t*>(src);
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const u4_t v = s[i];
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int k = 0; k < 4; k++) {
            x[8 * i + 2 * k] = h2f(w[k] & 0xffffu);
            x[8 * i + 2 * k + 1] = h2f(w[k] >> 16);
        }
    }
}

__global__ void __launch_bounds__(256) quantize_q8_0_kernel(const _Float16* src, uint8_t* dst, size_t nblocks) {
    const size_t b = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (b >= nblocks) return;
    float x[32];
    load_block_f16(src + b * 32, x);
    uint32_t d16, codes[16];
    quantize_block_q8_0(x, d16, codes);
    uint16_t* o16 = reinterpret_cast<uint16_t*>(dst + b * 34);  // 34-byte blocks are 2-byte aligned
    o16[0] = (uint16_t)d16;
#pragma unroll
    for (int i = 0; i < 16; i++) o16[1 + i] = (uint16_t)codes[i];
}

hipError_t launch_quantize_q8_0(const _Float16* src, uint8_t* dst, size_t nblocks, hipStream_t st) {
    if (nblocks == 0) return hipSuccess;
    hipLaunchKernelGGL(quantize_q8_0_kernel, dim3((unsigned)((nblocks + 255) / 256)), dim3(256), 0, st, src, dst,
                       nblocks);
    return hipGetLastError();
}

// --------------------------------------------------------------------------
// Flash attention
// --------------------------------------------------------------------------
constexpr int kBKV = 64;      // keys per tile of the cache pass; the fp16 cache pads M to a multiple
// The attention kernel reads a dequantized fp16 working copy of the cache: K'
// [H, Mp, D] (row-major) and V'^T [H, D, Mp] (keys contiguous per dim), Mp = M
// rounded up to whole 64-key tiles, so its LDS tiles are plain 16-byte copies.

// Two Q8_0 codes of bytes 0, 1 (HI = false) or 2, 3 (HI = true) of a code word
// times d: the code plus 128 becomes the binary16 1024 + 128 + q through the
// magic exponent (exact), 1152 is subtracted (exact) and the product rounds
// once -- the reference's half(q * d) (brick4_attn_bench.mm:57-65).
template <bool HI>
__device__ __forceinline__ uint32_t q8_pair(uint32_t codes, h2_t d) {
    const h2_t off = {(_Float16)1152.0f, (_Float16)1152.0f};
    const uint32_t u = codes ^ 0x80808080u;  // two's complement byte -> q + 128
    return as_u32((as_h2(HI ? nib_pair_hi(u) : nib_pair_lo(u)) - off) * d);
}

// In V'^T the keys of every 16 are stored 0-3, 8-11, 4-7, 12-15: the order in
// which a lane holds its P values, so its V^T fragment is one 16-byte read.
//
// Dequantized fp16 cache for the attention kernel, one workgroup per 64-key
// tile of one head.  FROM_Q8: from Q8_0 blocks (half(q * half(d)), the
// reference's dequantizer, brick4_attn_bench.mm:57-65); otherwise from fp16
// K / V through the same quantize-then-dequantize arithmetic as
// quantize_q8_0_kernel + the Q8_0 path (bit-identical values), also writing
// the Q8_0 blocks themselves to Kq / Vq when those are given -- the layer's
// Q8_0 KV cache, produced in the same pass.  Every output goes through LDS so
// it leaves in contiguous runs: K units (one key's block) fill the tile's K'
// rows (one contiguous 64-key run of K'); V units (a key pair's blocks) write
// {V[k][d], V[k+1][d]} words into a tile [d][key] whose rows leave as 128-byte
// runs of V'^T; the Q8_0 blocks of the tile's keys (contiguous in the cache)
// leave as dword runs.  Keys M .. Mp - 1 are zero.
template <bool FROM_Q8>
__device__ __forceinline__ void prep_block(const void* src, size_t blk, uint32_t w[16], uint8_t* q8out) {
    uint32_t d16, codes[8];  // code word c: codes of elements 4c .. 4c + 3
    if constexpr (FROM_Q8) {
        // 34-byte blocks are 2-byte aligned.  From the aligned dword at or
        // below the block, eight dwords plus the next two bytes (block at a
        // dword boundary) or nine dwords (block at 2 mod 4) cover it exactly,
        // so nothing past the block's last byte is read.
        const size_t o = blk * 34;
        const uint8_t* base = static_cast<const uint8_t*>(src) + (o & ~(size_t)3);
        const uint32_t* q = reinterpret_cast<const uint32_t*>(base);
        const bool par = (o & 2u) != 0;
        uint32_t raw[9];
#pragma unroll
        for (int i = 0; i < 8; i++) raw[i] = q[i];
        raw[8] = par ? q[8] : (uint32_t)*reinterpret_cast<const uint16_t*>(base + 32);
        d16 = par ? (raw[0] >> 16) : (raw[0] & 0xffffu);
#pragma unroll
        for (int c = 0; c < 8; c++) codes[c] = par ? raw[c + 1] : __builtin_amdgcn_alignbyte(raw[c + 1], raw[c], 2);
    } else {
        float x[32];
        load_block_f16(static_cast<const _Float16*>(src) + blk * 32, x);
        uint32_t c16[16];
        quantize_block_q8_0(x, d16, c16);
#pragma unroll
        for (int c = 0; c < 8; c++) codes[c] = c16[2 * c] | (c16[2 * c + 1] << 16);
        if (q8out) {  // this block's 34 bytes (2-byte aligned)
            uint16_t* o16 = reinterpret_cast<uint16_t*>(q8out);
            o16[0] = (uint16_t)d16;
#pragma unroll
            for (int i = 0; i < 16; i++) o16[1 + i] = (uint16_t)c16[i];
        }
    }
    const h2_t d = as_h2(d16 | (d16 << 16));
#pragma unroll
    for (int c = 0; c < 8; c++) {
        w[2 * c] = q8_pair<false>(codes[c], d);
        w[2 * c + 1] = q8_pair<true>(codes[c], d);
    }
}

template <int D, bool FROM_Q8>
__global__ void __launch_bounds__(256) kv_prep_kernel(const void* Ksrc, const void* Vsrc, _Float16* Kf, _Float16* Vtf,
                                                      uint8_t* Kq, uint8_t* Vq, uint32_t M, uint32_t Mp) {
    constexpr int NB = D / 32;            // blocks per key
    constexpr int TR = kBKV + 8;          // LDS row (halfs) of the transposed tile
    constexpr int KU = kBKV * NB, VU = (kBKV / 2) * NB;
    __shared__ __attribute__((aligned(16))) _Float16 T[D * TR];
    constexpr int KR = D + 8;  // LDS row (halfs) of the K' tile
    __shared__ __attribute__((aligned(16))) _Float16 KS[kBKV * KR];
    // the tile's Q8_0 blocks (from fp16 input, when the cache is wanted):
    // keys k0 .. k0 + 63 of K, then of V, 34-byte blocks back to back
    constexpr int QB = kBKV * NB * 34;
    __shared__ __attribute__((aligned(16))) uint8_t QS[FROM_Q8 ? 4 : 2 * QB];
    const int tid = threadIdx.x;
    const uint32_t k0 = blockIdx.x * kBKV, hk = blockIdx.y;
    const size_t head_blocks = (size_t)M * NB, head_dst = (size_t)Mp * D;
    for (int u = tid; u < KU + VU; u += 256) {
        if (u < KU) {
            const int key = u % kBKV, db = u / kBKV;
            const uint32_t gk = k0 + key;
            uint32_t w[16] = {};
            if (gk < M)
                prep_block<FROM_Q8>(Ksrc, hk * head_blocks + (size_t)gk * NB + db, w,
                                    (!FROM_Q8 && Kq) ? QS + (key * NB + db) * 34 : nullptr);
            u4_t* dst = reinterpret_cast<u4_t*>(KS + key * KR + db * 32);
#pragma unroll
            for (int c = 0; c < 4; c++) dst[c] = u4_t{w[4 * c], w[4 * c + 1], w[4 * c + 2], w[4 * c + 3]};
        } else {
            const int v = u - KU;
            const int kp = v % (kBKV / 2), db = v / (kBKV / 2);
            uint32_t w[2][16] = {};
#pragma unroll
            for (int e = 0; e < 2; e++) {
                const uint32_t gk = k0 + 2 * kp + e;
                if (gk < M)
                    prep_block<FROM_Q8>(Vsrc, hk * head_blocks + (size_t)gk * NB + db, w[e],
                                        (!FROM_Q8 && Vq) ? QS + QB + ((2 * kp + e) * NB + db) * 34 : nullptr);
            }
            uint32_t* t32 = reinterpret_cast<uint32_t*>(T);
            const int kpos = (kp & ~6) | ((kp & 2) << 1) | ((kp & 4) >> 1);  // keys 4..7 and 8..11 of 16 swapped
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const int dd = db * 32 + 2 * i;
                t32[(dd * TR) / 2 + kpos] = perm(w[1][i], w[0][i], 0x05040100u);
                t32[((dd + 1) * TR) / 2 + kpos] = perm(w[1][i], w[0][i], 0x07060302u);
            }
        }
    }
    __syncthreads();
    // streaming (non-temporal) stores: the working copy is written once and
    // read by the next kernel; measured 11.2 -> 9.9 us (from Q8_0) and 10.5 ->
    // 9.5 us (from fp16) at H = 32, M = 2048, D = 64
    for (int c = tid; c < D * 8; c += 256) {
        const int d = c / 8, kc = c % 8;
        __builtin_nontemporal_store(*reinterpret_cast<const u4_t*>(T + d * TR + kc * 8),
                                    reinterpret_cast<u4_t*>(Vtf + hk * head_dst + (size_t)d * Mp + k0 + kc * 8));
    }
    for (int c = tid; c < kBKV * D / 8; c += 256) {  // the K' tile is one contiguous run
        const int key = c / (D / 8), kc = c % (D / 8);
        __builtin_nontemporal_store(*reinterpret_cast<const u4_t*>(KS + key * KR + kc * 8),
                                    reinterpret_cast<u4_t*>(Kf + hk * head_dst + (size_t)k0 * D + (size_t)c * 8));
    }
    if constexpr (!FROM_Q8) {
        if (Kq) {  // the tile's blocks are one contiguous run of the cache (a multiple of 4 bytes)
            const uint32_t nkeys = min((uint32_t)kBKV, M - k0);
            const size_t first = (hk * head_blocks + (size_t)k0 * NB) * 34;
            if (((reinterpret_cast<uintptr_t>(Kq) | reinterpret_cast<uintptr_t>(Vq)) & 3u) == 0) {
                const int ndw = (int)(nkeys * NB * 34 / 4);
                uint32_t* kd = reinterpret_cast<uint32_t*>(Kq + first);
                uint32_t* vd = reinterpret_cast<uint32_t*>(Vq + first);
                const uint32_t* ks = reinterpret_cast<const uint32_t*>(QS);
                const uint32_t* vs = reinterpret_cast<const uint32_t*>(QS + QB);
                for (int i = tid; i < ndw; i += 256) {
                    kd[i] = ks[i];
                    vd[i] = vs[i];
                }
            } else {  // caches only 2-byte aligned
                const int nh = (int)(nkeys * NB * 17);
                uint16_t* kd = reinterpret_cast<uint16_t*>(Kq + first);
                uint16_t* vd = reinterpret_cast<uint16_t*>(Vq + first);
                const uint16_t* ks = reinterpret_cast<const uint16_t*>(QS);
                const uint16_t* vs = reinterpret_cast<const uint16_t*>(QS + QB);
                for (int i = tid; i < nh; i += 256) {
                    kd[i] = ks[i];
                    vd[i] = vs[i];
                }
            }
        }
    }
}

// --------------------------------------------------------------------------
// Causal attention over the fp16 cache.  A workgroup is 4 waves (one per SIMD;
// two workgroups per CU, whose softmax and matrix phases overlap because no
// barrier ties them): 4 / NK blocks of 32 queries times NK key groups, group kg
// taking the kg-th share of every tile's 32-key units, the partial states
// merged through LDS at the end of a query tile.  Per 32 x 32 unit a wave issues
// D / 16 MFMAs for S^T = K . Q^T, a softmax of ~90 VALU ops, 16 of them
// exponentials (16 cycles each), and D / 16 MFMAs for O^T += V^T . P^T, and reads
// 128 D bytes of LDS.  Counters: D = 128, M = 8100 5.6 VALU ops per MFMA (90 per unit),
// the matrix pipe 50% busy at 1.8 GHz; D = 64, M = 2048 12.9 (103 per unit, masks and
// merges included), 18% busy, waves waiting 37% of their cycles.
//
// Key tiles of 32 KB (K rows, then V^T rows) are double-buffered in LDS, copied
// there by buffer loads in inline asm one tile ahead; the only barrier is one
// per tile, behind the wave's own vmcnt(0).  Units above a wave's diagonal are
// skipped.  Softmax in log2 units with the scale folded into one fma; the
// reference point moves lazily (only past 2^8, checked once per two units), the
// halves of a row combined only then; fp32 state; P rounded to fp16 once, for
// the MFMA and for the row sums alike.
//
// Before, one 8-wave workgroup per CU (4 waves at D = 128, one per SIMD) ran an
// in-wave software pipeline of the two phases; at one wave per SIMD the compiler
// moved the accumulators between register files (11.7 VALU ops per MFMA at D = 128, M =
// 2048) and nothing covered its waits.  us with the cache pass, before ->
// now: D = 128, H = 32, Hkv = 8, M = 8100 984 -> 578; M = 1000 49.4 -> 27.5;
// D = 64, H = 32, M = 2048 42.7 -> 39.9, M = 8192 433 -> 370, M = 500 19.5 -> 12.5.
// --------------------------------------------------------------------------
constexpr int tile_keys(int D) { return D == 64 ? 128 : 64; }  // 32 KB of K and V^T per tile at either width
constexpr int kTileBytes = 32768;
constexpr int kLmBytes = 2048;  // row sums and maxima of the merge
// Reference point of a row that has seen no score above -infinity: finite, so
// that such scores weigh exp2(-inf - kNoScore) = 0 in every key group (from
// -infinity it would be exp2(NaN), and one key group whose first keys all score
// -infinity would make the whole row NaN).
constexpr float kNoScore = -3.402823466e38f;

__device__ __forceinline__ float max3(float a, float b, float c) { return fmaxf(fmaxf(a, b), c); }

template <int D, int NK>  // NK: key groups; 4 / NK blocks of 32 queries per workgroup
__global__ void __launch_bounds__(256, 2) flash_attn_kernel(AttnParams p, int paired) {
    constexpr int KT = tile_keys(D), UPT = KT / 32, UW = UPT / NK, NQ = 4 / NK, BQ = 32 * NQ;
    constexpr int DT = D / 32, KK = D / 16;
    constexpr int KB = KT * D * 2;             // bytes of a K tile
    constexpr int KU = D / 8, VU = KT / 8;     // 16-byte units per K row, per V^T row
    constexpr int CPW = kTileBytes / 2 / 1024 / 4;  // copies per wave of K, and of V^T
    constexpr int NB = UW < 2 ? 1 : 2;         // units per softmax batch
    static_assert(KB == kTileBytes / 2 && D * KT * 2 == kTileBytes / 2, "tile bytes");
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int qb_ = wave % NQ, kg = wave / NQ;  // query block and key group
    const int g = lane >> 5, j = lane & 31;
    const int M = (int)p.M, Mp = (int)p.Mp;
    const int qtiles = (M + BQ - 1) / BQ;
    const int pr = (int)blockIdx.x / (int)p.H, h = (int)blockIdx.x % (int)p.H;
    // paired: a light and a heavy query tile; else one, the heavy half of them
    // first, descending, then the light half, ascending (workgroups half a
    // grid apart, which share a CU when the grid fills it twice, then add up alike)
    const int nh = (qtiles + 1) / 2;
    const int qz = pr < nh ? qtiles - 1 - pr : pr - nh;
    const int qa = paired ? pr : qz;
    auto tiles_for = [&](int qt) { return (min((qt + 1) * BQ, M) - 1) / KT + 1; };
    const int Tl = qa == qz ? 0 : tiles_for(qa);
    const int S = Tl + tiles_for(qz);
    auto tile_of = [&](int s) { return s < Tl ? s : s - Tl; };

    const size_t head_elems = (size_t)M * D;
    const int hk = p.Hkv ? h / ((int)p.H / (int)p.Hkv) : h;
    const uint32_t cbytes = (uint32_t)((size_t)Mp * D * 2);
    const u4_t kr = scalar_rsrc(p.Kf + (size_t)hk * Mp * D, cbytes);
    const u4_t vr = scalar_rsrc(p.Vtf + (size_t)hk * Mp * D, cbytes);
    const auto qr_ = make_rsrc(p.Q + (size_t)h * head_elems, (uint32_t)(head_elems * 2));

    // ---- tile copies.  K rows (keys) hold KU 16-byte units, V^T rows (dims) VU;
    // unit u of row r sits at u ^ swz, which depends on r mod 32 only and puts
    // the 16 rows of a fragment-read pass on distinct banks ----
    auto swz = [](int units, uint32_t r) -> uint32_t {
        r &= 31u;
        return units == 16 ? (r & 15u) : ((r ^ (r >> 3)) & 7u);
    };
    uint32_t ko[CPW], vo[CPW], vk[CPW];
#pragma unroll
    for (int q = 0; q < CPW; q++) {
        const uint32_t un = 64u * (uint32_t)(CPW * wave + q) + (uint32_t)lane;
        const uint32_t kr_ = un / KU, ku = (un % KU) ^ swz(KU, kr_);
        ko[q] = (kr_ * D + 8u * ku) * 2u;
        const uint32_t vr_ = un / VU, vu = (un % VU) ^ swz(VU, vr_);
        vk[q] = 8u * vu;
        vo[q] = (vr_ * (uint32_t)Mp + 8u * vu) * 2u;
    }
    const uint32_t lds0 = (uint32_t)reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) uint8_t*)smem);
    auto issue = [&](int s) {
        const uint32_t k0 = (uint32_t)(tile_of(s) * KT);
        const uint32_t dst = lds0 + (uint32_t)(s & 1) * kTileBytes + (uint32_t)(CPW * wave) * 1024u;
        const bool part = k0 + KT > (uint32_t)Mp;  // a V^T chunk past Mp would be the next dim's first keys
#pragma unroll
        for (int q = 0; q < CPW; q++) {
            copy_lds(dst + q * 1024u, ko[q] + k0 * D * 2u, kr, 0);  // rows past Mp: past the head's cache
            copy_lds(dst + KB + q * 1024u, part && k0 + vk[q] >= (uint32_t)Mp ? kOOB : vo[q], vr, k0 * 2u);
        }
    };

    float c = p.scale * 1.4426950408889634f;  // log2 units
    const bool neg = c < 0.0f;
    if (neg) c = -c;

    // fragment offsets in a tile: K row 32 u + j, unit 2 kk + g; V^T row 32 t + j,
    // unit 4 u + 2 t2 + g, for this wave's units u = kg UW + b
    uint32_t kof[KK], vof[UW * 2];
#pragma unroll
    for (int kk = 0; kk < KK; kk++) kof[kk] = (uint32_t)j * (KU * 16u) + 16u * ((uint32_t)(2 * kk + g) ^ swz(KU, (uint32_t)j));
#pragma unroll
    for (int x = 0; x < UW * 2; x++)
        vof[x] = (uint32_t)j * (VU * 16u) + 16u * ((uint32_t)(4 * kg * UW + 2 * x + g) ^ swz(VU, (uint32_t)j));

    h8_t qf[KK];
    f16v_t o[DT];
    float m_run, l_run;  // l_run: this lane's half of the row sum of P
    int qw = 0;
    auto start = [&](int qt) {
        qw = qt * BQ + qb_ * 32;
        const int my_q = qw + j;
#pragma unroll
        for (int kk = 0; kk < KK; kk++) {
            const uint32_t off = my_q < M ? ((uint32_t)my_q * D + kk * 16 + 8 * g) * 2u : kOOB;
            qf[kk] = __builtin_bit_cast(h8_t, ld_b128(qr_, off));
            if (neg) qf[kk] = -qf[kk];
        }
        m_run = kNoScore;
        l_run = 0.0f;
#pragma unroll
        for (int t = 0; t < DT; t++) o[t] = f16v_t{};
    };
    auto store = [&]() {
        const float l = l_run + __shfl_xor(l_run, 32);
        const float inv = 1.0f / l;
        const int my_q = qw + j;
        if (my_q >= M) return;
#pragma unroll
        for (int t = 0; t < DT; t++)
#pragma unroll
            for (int r4 = 0; r4 < 4; r4++) {
                const int d0 = t * 32 + 8 * r4 + 4 * g;
                const f2_t a = {o[t][4 * r4] * inv, o[t][4 * r4 + 1] * inv};
                const f2_t b = {o[t][4 * r4 + 2] * inv, o[t][4 * r4 + 3] * inv};
                const size_t idx = p.o_token_major ? ((size_t)my_q * p.H + h) * D + d0
                                                   : (size_t)h * head_elems + (size_t)my_q * D + d0;
                *reinterpret_cast<u2_t*>(p.O + idx) =
                    u2_t{as_u32(__builtin_convertvector(a, h2_t)), as_u32(__builtin_convertvector(b, h2_t))};
            }
    };

    // ---- this wave's units b0 .. b0 + NB - 1 of the tile in `buf` (first key
    // key0), the first `live` of them at or below its last query ----
    const h2_t one2 = {(_Float16)1.0f, (_Float16)1.0f};
    auto batch = [&](const uint8_t* buf, int b0, int key0, int live) {
        f16v_t s[NB];
#pragma unroll
        for (int b = 0; b < NB; b++) {
            if (b >= live) break;
            const uint8_t* kb = buf + (kg * UW + b0 + b) * 32 * (KU * 16);
            s[b] = f16v_t{};
#pragma unroll
            for (int kk = 0; kk < KK; kk++)
                s[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(*reinterpret_cast<const h8_t*>(kb + kof[kk]), qf[kk], s[b], 0, 0, 0);
        }
#pragma unroll
        for (int b = 0; b < NB; b++) {
            if (b >= live) break;
            const int k0 = key0 + 32 * b;
            if (k0 + 31 > qw || k0 + 31 >= M) {  // the diagonal, or the end of the keys
                const int my_q = qw + j;
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int key = k0 + 8 * (r >> 2) + 4 * g + (r & 3);
                    s[b][r] = (key <= my_q && key < M) ? s[b][r] : -INFINITY;
                }
            }
        }
        // Row maximum of each lane's half decides whether the reference point
        // must move (by more than 2^8); only then are the halves combined.
        float mx[4];
#pragma unroll
        for (int q = 0; q < 4; q++) mx[q] = fmaxf(max3(s[0][4 * q], s[0][4 * q + 1], s[0][4 * q + 2]), s[0][4 * q + 3]);
        if (NB > 1 && live > 1) {
#pragma unroll
            for (int q = 0; q < 4; q++)
                mx[q] = max3(max3(mx[q], s[NB - 1][4 * q], s[NB - 1][4 * q + 1]), s[NB - 1][4 * q + 2], s[NB - 1][4 * q + 3]);
        }
        const float m_cand = fmaxf(max3(mx[0], mx[1], mx[2]), mx[3]) * c;
        if (__any(m_cand > m_run + 8.0f)) {
            const float m_new = fmaxf(m_run, fmaxf(m_cand, __shfl_xor(m_cand, 32)));
            const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
            m_run = m_new;
#pragma unroll
            for (int t = 0; t < DT; t++)
#pragma unroll
                for (int r = 0; r < 16; r++) o[t][r] *= alpha;
            l_run *= alpha;
        }
        // raised wave priority over the exponentials and their MFMAs: the SIMD's
        // other wave, in its S phase, yields (M = 8100, D = 128 2% faster)
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int b = 0; b < NB; b++) {
            if (b >= live) break;
            uint32_t pk[8];
#pragma unroll
            for (int r = 0; r < 16; r += 2) {
                const f2_t e = {__builtin_amdgcn_exp2f(__builtin_fmaf(s[b][r], c, -m_run)),
                                __builtin_amdgcn_exp2f(__builtin_fmaf(s[b][r + 1], c, -m_run))};
                const h2_t pp = __builtin_convertvector(e, h2_t);
                pk[r >> 1] = as_u32(pp);
                l_run = __builtin_amdgcn_fdot2(pp, one2, l_run, false);  // row sum of the rounded P
            }
            const uint8_t* vb = buf + KB;
#pragma unroll
            for (int t2 = 0; t2 < 2; t2++) {
                const h8_t pf = __builtin_bit_cast(h8_t, u4_t{pk[4 * t2], pk[4 * t2 + 1], pk[4 * t2 + 2], pk[4 * t2 + 3]});
#pragma unroll
                for (int t = 0; t < DT; t++) {
                    const h8_t va = *reinterpret_cast<const h8_t*>(vb + t * 32 * (VU * 16) + vof[2 * (b0 + b) + t2]);
                    o[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(va, pf, o[t], 0, 0, 0);
                }
            }
        }
        __builtin_amdgcn_s_setprio(0);
    };

    // ---- merge of the key groups' partial states through the tile buffer that
    // every wave has finished reading (after a barrier): group 0 takes the others in order ----
    auto merge = [&](uint8_t* buf) {
        float* const lm = reinterpret_cast<float*>(smem + 2 * kTileBytes);
        const int slot = (kg - 1) * NQ + qb_;
        if (kg > 0) {
            float* x = reinterpret_cast<float*>(buf) + slot * (DT * 16 * 64);
#pragma unroll
            for (int t = 0; t < DT; t++)
#pragma unroll
                for (int r = 0; r < 16; r += 4)
                    *reinterpret_cast<f4_t*>(x + ((t * 4 + r / 4) * 64 + lane) * 4) = f4_t{o[t][r], o[t][r + 1], o[t][r + 2], o[t][r + 3]};
            *reinterpret_cast<f2_t*>(lm + (slot * 64 + lane) * 2) = f2_t{l_run, m_run};
        }
        __syncthreads();
        if (kg == 0) {
#pragma unroll 1
            for (int k = 1; k < NK; k++) {
                const int sl = (k - 1) * NQ + qb_;
                const float* x = reinterpret_cast<const float*>(buf) + sl * (DT * 16 * 64);
                const f2_t q = *reinterpret_cast<const f2_t*>(lm + (sl * 64 + lane) * 2);
                const float m = fmaxf(q.y, m_run);
                const float fa = __builtin_amdgcn_exp2f(q.y - m), fb = __builtin_amdgcn_exp2f(m_run - m);
#pragma unroll
                for (int t = 0; t < DT; t++)
#pragma unroll
                    for (int r = 0; r < 16; r += 4) {
                        const f4_t v = *reinterpret_cast<const f4_t*>(x + ((t * 4 + r / 4) * 64 + lane) * 4);
                        o[t][r] = o[t][r] * fb + v.x * fa;
                        o[t][r + 1] = o[t][r + 1] * fb + v.y * fa;
                        o[t][r + 2] = o[t][r + 2] * fb + v.z * fa;
                        o[t][r + 3] = o[t][r + 3] * fb + v.w * fa;
                    }
                l_run = l_run * fb + q.x * fa;
                m_run = m;
            }
        }
    };

    // ---- one stream of tiles: the light query tile's, then the heavy one's ----
    start(Tl > 0 ? qa : qz);
    issue(0);
    for (int s = 0; s < S; s++) {
        if (s == Tl && s > 0) start(qz);
        // own copies of step s have landed, every wave is past step s - 1
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (s + 1 < S) issue(s + 1);
        uint8_t* const buf = smem + (s & 1) * kTileBytes;
        const int key_t = tile_of(s) * KT;
#pragma unroll
        for (int b = 0; b < UW; b += NB) {
            const int key0 = key_t + 32 * (kg * UW + b);
            const int live = key0 > qw + 31 ? 0 : (NB > 1 && key0 + 32 <= qw + 31 ? NB : 1);
            if (live > 0) batch(buf, b, key0, live);
        }
        if (s == Tl - 1 || s == S - 1) {
            if constexpr (NK > 1) {
                asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
                merge(buf);
            }
            if (kg == 0) store();
        }
    }
}

template <int D, int NK>
static hipError_t launch_attn(const AttnParams& p, int paired, hipStream_t st) {
    constexpr uint32_t bq = 128 / NK;
    constexpr size_t lds = 2 * kTileBytes + kLmBytes;
    const uint32_t qtiles = (p.M + bq - 1) / bq;
    static size_t attr[kMaxDevices] = {};  // more than the default 64 KB of LDS
    const hipError_t e = lds_limit_once((const void*)flash_attn_kernel<D, NK>, lds, attr);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((flash_attn_kernel<D, NK>), dim3((paired ? (qtiles + 1) / 2 : qtiles) * p.H), dim3(256), lds, st, p, paired);
    return hipGetLastError();
}

hipError_t launch_flash_attn_q8_0(const AttnParams& p, hipStream_t st) {
    // the kernels read the dequantized fp16 cache (launch_kv_prep)
    if (p.Kf == nullptr || p.Vtf == nullptr || p.Mp < p.M || p.Mp % kBKV) return hipErrorInvalidValue;
    if (p.D != 64 && p.D != 128) return hipErrorInvalidValue;
    auto qtiles = [&](uint32_t nk) { return (p.M + 128 / nk - 1) / (128 / nk); };
    // One pair of query tiles per workgroup while that fills every CU twice
    // (512 workgroups), with as few key groups as do; else one query tile each,
    // on two key groups if that is more than one workgroup per CU, else (D = 64)
    // on four.  us at H = 32, with the cache pass: D = 64, M = 4096 pairs on one
    // / two key groups 101 / 116; M = 2048 46 / 40; M = 1024 two key groups,
    // pairs / single tiles 22.3 / 20.3; M = 512 single tiles, two / four key
    // groups 13.5 / 12.5; D = 128, M = 1000 two key groups, pairs / single 29.8 / 27.6.
    uint32_t nk = 1;
    while (nk < 2 && (qtiles(nk) + 1) / 2 * p.H < 512) nk *= 2;
    const int paired = (qtiles(nk) + 1) / 2 * p.H >= 512;
    if (!paired && p.D == 64 && qtiles(2) * p.H <= 256) nk = 4;
    switch (p.D + nk) {
        case 65: return launch_attn<64, 1>(p, paired, st);
        case 66: return launch_attn<64, 2>(p, paired, st);
        case 68: return launch_attn<64, 4>(p, paired, st);
        case 129: return launch_attn<128, 1>(p, paired, st);
        default: return launch_attn<128, 2>(p, paired, st);
    }
}

uint32_t kv_padded_len(uint32_t M) { return (M + kBKV - 1) / kBKV * kBKV; }

hipError_t launch_kv_prep(const void* K, const void* V, bool from_q8, _Float16* Kf, _Float16* Vtf, uint32_t Hkv,
                          uint32_t M, uint32_t D, hipStream_t st, uint8_t* Kq, uint8_t* Vq) {
    const uint32_t Mp = kv_padded_len(M);
    dim3 grid(Mp / kBKV, Hkv);
    if (from_q8) Kq = Vq = nullptr;  // the blocks are the input
    switch (D * 2 + (from_q8 ? 1 : 0)) {
        case 128: hipLaunchKernelGGL((kv_prep_kernel<64, false>), grid, dim3(256), 0, st, K, V, Kf, Vtf, Kq, Vq, M, Mp); break;
        case 129: hipLaunchKernelGGL((kv_prep_kernel<64, true>), grid, dim3(256), 0, st, K, V, Kf, Vtf, Kq, Vq, M, Mp); break;
        case 256: hipLaunchKernelGGL((kv_prep_kernel<128, false>), grid, dim3(256), 0, st, K, V, Kf, Vtf, Kq, Vq, M, Mp); break;
        case 257: hipLaunchKernelGGL((kv_prep_kernel<128, true>), grid, dim3(256), 0, st, K, V, Kf, Vtf, Kq, Vq, M, Mp); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace qr
