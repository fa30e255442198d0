/*
 * qmm_gemm.hip -- the stock path's matrix products (gfx950), y[M,N] = x[M,K] . dequant(W)[N,K]^T:
 * below, many rows of one 16-bit dtype of x, scales, biases and y; at the end of the file, the
 * fp32 form of every other call.
 *
 * The codes enter the MFMAs as exact small integers and everything else stays in fp32: per
 * quantisation group P = sum x (MAGIC + q), y += s * P + b * X - MAGIC * s * X with X = sum x.
 * bf16 4-bit codes carry MAGIC = 16 (8 VALU operations make the 8 operands of a word); fp16 codes
 * take one packed subtraction more and carry none; 8-bit bf16 codes are converted.
 *
 *  - Precision.  The GEMV corrects each lane's 32 or 16 k at once, in 64 chains; here one
 *    accumulator holds up to four groups' s P before the X terms meet them.  The error of the
 *    sums before the output's rounding, as a share of the result's norm, K = 1024 to 17408,
 *    activations of either sign / of one sign (GEMV in brackets): 4-bit bf16 1.8e-7 to 3.2e-7 /
 *    1.9e-6 to 3.0e-6 (7.4e-7 to 8.3e-7 / 3.9e-6 to 4.1e-6; with a MAGIC of 128 here 1.4e-6 to
 *    1.7e-6 / 1.3e-5 to 2.0e-5); 4-bit fp16 1.0e-7 to 3.2e-7 / 6.7e-7 to 1.9e-6 (1.4e-5 /
 *    6.4e-5); 8-bit 0.9e-7 to 3.4e-7 / 0.6e-6 to 2.8e-6 (0.4e-7 to 1.4e-7 / 1.0e-7 to 2.8e-7).
 *    The output's own rounding is 1.7e-3 in bf16 and 2.1e-4 in fp16.
 *
 *  - s * P is one fp32 FMA an accumulator element and group: 64 issue cycles a 32 x 32 tile
 *    against 128 matrix cycles at group 64, so the vector and the matrix pipes run side by
 *    side.  A group of 128 is taken as two of 64 (the partial sums of a whole tile row would
 *    not fit in registers).
 *  - the X terms are a product over groups, so they go through the matrix cores too: X is
 *    split exactly into three bf16 values (24 bits), and 4 groups x (Xh, Xm, Xl, 0) are the
 *    16 k slots of one MFMA against b, and of a second against -MAGIC s (or, for fp16, the
 *    second part of b, split exactly into two bf16 values): one or two MFMAs per 16.
 *
 *    X itself is one more product, ones . x, shared out over the column strips: summed on the
 *    vector pipe as x is staged instead, a 128 x 128 step alone took 1.07 us against 0.83.
 *
 * A workgroup computes 32 RT MW rows x 32 CT NW columns in KW slices of K; a wave holds RT x CT
 * tiles of one slice.  x is staged in LDS 64 k a step, in two buffers, permuted into the order
 * of the nibbles and XOR-swizzled by row so that neither writes nor reads conflict; codes are
 * staged by whole 128-byte lines of their rows (4 or 2 steps), with the line's scales and
 * biases.  Read straight into the operand registers instead, 32 bytes a row and step, the lines
 * of 128 columns and their scales outlived the 32 KB L1 and each was fetched several times:
 * 2048 x 17408, K 5120 took 556 us against 535, 16 x 5120 25.7 against 20.9.  All loads run a
 * step (x) or a line (codes) ahead, and are clamped rather than predicated: with a branch
 * around them the compiler waited for each at once (636 against 556 us).  KW > 1 slices are
 * summed through LDS at the end, in slice order.
 *
 * The next step is staged after all but the last two row tiles' LDS reads, which its writes
 * would otherwise hold up (2048 x 17408, K 5120: 527 us after the first, 513).
 *
 * Measured on MI355X against the GEMV's launches it replaces (us a pass): 512 x 5120, K 5120,
 * 4-bit bf16 1537 -> 59.9; 2048 x 17408, K 5120 12548 -> 527 (693 TFLOP/s); an MLP of 333 rows,
 * 8-bit fp16 6566 -> 423.  A wave's step of 128 x 32 has 704 matrix cycles, of which 512 are the
 * product, 128 the x sums (31 of 32 columns of ones . x are the same) and 64 the X products, and
 * about 150 vector instructions, up to six of which issue behind an MFMA of their own wave, but
 * another wave's only one (measured: an FMA every 32 cycles beside a wave of MFMAs), so two waves a
 * SIMD hardly fill each other's gaps.  Where a grid leaves one workgroup a CU (512 x 5120: 240)
 * there is one wave a SIMD, and LDS reads, vector work and MFMAs add up.
 */
#include "qmm_device.h"
#include "qmm_params.h"

namespace {

typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

template <bool F16>
__device__ __forceinline__ f32x16_t mfma32(u32x4_t a, u32x4_t b, f32x16_t c) {
    if constexpr (F16)
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a),
                                                      __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                       __builtin_bit_cast(bf16x8_t, b), c, 0, 0,
                                                       0);
}

/* 8 nibbles of a word -> bf16 (MAGIC + q) pairs (q_i, q_{i+4}) with MAGIC = 16: each code right
 * below the leading one.  One operation more than nibble_operand's 128 + q: there the sums are
 * 128 sum x too large until the X terms meet them, which in a long-lived accumulator costs
 * precision (see the head comment).  TURNED words have been turned left by 3 bits as they were
 * staged, which takes the operation out of the step's chain: 512 x 5120, K 5120 59.7 us against
 * 61.4; with four row tiles a wave the registers of it spill (2048 x 17408 540 us against 531,
 * with the 128 of before 525). */
constexpr int kMagic = 16;
template <bool TURNED>
__device__ __forceinline__ u32x4_t nibble_operand16(uint32_t p, uint32_t mask, uint32_t magic) {
    u32x4_t v;
    v[0] = ((TURNED ? p : p << 3) & mask) | magic;
    v[1] = ((p >> (TURNED ? 4 : 1)) & mask) | magic;
    v[2] = ((p >> (TURNED ? 8 : 5)) & mask) | magic;
    v[3] = ((TURNED ? __builtin_amdgcn_alignbit(p, p, 12) : p >> 9) & mask) | magic;
    return v;
}

/* (1024 + q) pairs -> q pairs, exact. */
__device__ __forceinline__ uint32_t less_1024(uint32_t v) {
    const f16x2_t m = {(_Float16)1024.0f, (_Float16)1024.0f};
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(f16x2_t, v) - m);
}

/* fp32 -> the output's dtype, to nearest even (one instruction in either dtype). */
template <bool F16>
__device__ __forceinline__ uint16_t round_out(float f) {
    if constexpr (F16) return __builtin_bit_cast(uint16_t, (_Float16)f);
    else return __builtin_bit_cast(uint16_t, (__bf16)f);
}

/* The operand of one word of 4-bit codes, or of two words of 8-bit codes. */
template <int BITS, bool F16, bool TURNED>
__device__ __forceinline__ u32x4_t code_operand(const uint32_t* w, uint32_t mask,
                                                uint32_t magic) {
    u32x4_t v;
    if constexpr (BITS == 4) {
        if constexpr (F16) v = nibble_operand<true>(w[0], mask, magic);
        else v = nibble_operand16<TURNED>(w[0], mask, magic);
    } else if constexpr (F16) {
        v[0] = __builtin_amdgcn_perm(0x64646464u, w[0], 0x04010400u);
        v[1] = __builtin_amdgcn_perm(0x64646464u, w[0], 0x04030402u);
        v[2] = __builtin_amdgcn_perm(0x64646464u, w[1], 0x04010400u);
        v[3] = __builtin_amdgcn_perm(0x64646464u, w[1], 0x04030402u);
    } else {
        return byte_operand<false>(w[0], w[1]);
    }
    if constexpr (F16)
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = less_1024(v[e]);
    return v;
}

template <int BITS, int GS, bool F16, int RT, int CT, int MW, int NW, int KW>
__device__ __forceinline__ void qmm_gemm(const QmmGemmParams& p) {
    static_assert(GS == 32 || GS == 64, "sub-groups of a step");
    constexpr int BM = 32 * RT * MW, BN = 32 * CT * NW;
    constexpr int NP = 64 / GS;         // groups a step of 64 k holds
    constexpr int JP = 4 / NP;          // MFMAs a group
    constexpr int SS = 4 / NP;          // steps of the four groups of an X product
    constexpr int NWD = BITS;           // code words a lane takes per column and step
    constexpr int LS = 16 / BITS;       // steps of a 128-byte line of codes
    constexpr int LG = LS * NP;         // groups of a line
    constexpr int ST = 64 * MW * NW;    // threads of a slice
    constexpr int XI = BM * 8 / ST;     // 16-byte chunks of x each of them stages a step
    constexpr int WI = BN * 8 / ST;     // 16-byte chunks of codes, a line
    constexpr int SI = 2 * BN > ST ? 2 * BN / ST : 1;  // columns' scales or biases, a line
    constexpr bool kTwo = F16 || BITS == 4;  // a second X product
    constexpr bool kTurned = BITS == 4 && !F16 && RT < 4;  // see nibble_operand16
    static_assert(XI * ST == BM * 8 && WI * ST == BN * 8, "whole chunks");
    static_assert(SI * ST == 2 * BN || SI == 1, "whole rows of scales");
    /* bytes of a step's x, of four groups' X, of a line of codes and of its scales + biases */
    constexpr int kA = BM * 128, kX = BM * 32, kW = BN * 128, kS = BN * LG * 4;
    constexpr int SR = LG == 2 ? 4 : 2;  // lines of scales kept: an X product may need two
    constexpr int kSlice = 2 * (kA + kX + kW) + SR * kS;
    constexpr int kRed = (KW - 1) * MW * NW * RT * CT * 4096;
    __shared__ __attribute__((aligned(16))) uint8_t lds[KW * kSlice > kRed ? KW * kSlice : kRed];

    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kw = wave / (MW * NW), wn = wave % NW, wm = wave / NW % MW, tl = tid - kw * ST;
    const int M = p.M, N = p.N, K = p.K, gpr = p.gpr;
    /* XCD x takes one contiguous run of tiles (rows fastest), so that the row tiles of a
     * column strip share its codes in one L2 */
    const int G = gridDim.x;
    int id = blockIdx.x;
    if (p.xcd8) {
        const int x = id & 7, base = G >> 3, rem = G & 7;
        id = x * base + min(x, rem) + (id >> 3);
    }
    const int nt = id / p.tiles_m, m0 = (id - nt * p.tiles_m) * BM, n0 = nt * BN;

    /* the slice's steps, from a fourth one: every slice walks `per` (the barriers are
     * shared), the last ones may own fewer; loads past K read its last step or line again
     * and are not used */
    const int steps = (K + 63) >> 6;
    const int per = ((steps + KW - 1) / KW + 3) & ~3;
    const int first = kw * per, mine = min(per, steps - first);
    const int walk = KW == 1 ? steps : per;
    uint8_t* abuf = lds + kw * kSlice;
    uint8_t* xbuf = abuf + 2 * kA;
    uint8_t* wbuf = xbuf + 2 * kX;
    uint8_t* sbuf = wbuf + 2 * kW;
    const int c8 = tl & 7;

    /* x: chunk c of row r of the tile, rows past M read the last one */
    const uint8_t* xg = (const uint8_t*)p.x + (size_t)m0 * K * 2;
    uint32_t xoff[XI];
    int xr[XI];
#pragma unroll
    for (int i = 0; i < XI; ++i) {
        xr[i] = (tl + i * ST) >> 3;
        xoff[i] = (uint32_t)min(xr[i], M - 1 - m0) * (uint32_t)K * 2u + (uint32_t)c8 * 16u;
    }
    u32x4_t xv[XI];
    auto load_x = [&](int st) {
        const uint32_t k0 = (uint32_t)min(first + st, steps - 1) * 64u;
        const uint8_t* src = xg + (size_t)k0 * 2;
        /* the half step a K of odd 32s ends in: chunks past it read the half before */
        const uint32_t back = (GS == 32 && k0 + (uint32_t)c8 * 8u >= (uint32_t)K) ? 64u : 0u;
#pragma unroll
        for (int i = 0; i < XI; ++i) xv[i] = *(const u32x4_t*)(src + (xoff[i] - back));
    };
    auto stage_x = [&](int st) {
        const bool in = GS == 64 || (first + st) * 64 + c8 * 8 < K;
        uint8_t* ab = abuf + (st & 1) * kA;
#pragma unroll
        for (int i = 0; i < XI; ++i) {
            if constexpr (GS == 32)
#pragma unroll
                for (int e = 0; e < 4; ++e) xv[i][e] = in ? xv[i][e] : 0u;
            *(u32x4_t*)(ab + xr[i] * 128 + ((c8 ^ (xr[i] & 7)) * 16)) =
                BITS == 4 ? nibble_permute(xv[i]) : xv[i];
        }
    };

    /* a line of codes: chunk c of column r (the last one past N); chunks past K repeat its
     * last one */
    const uint32_t RB = (uint32_t)K * BITS / 8u;
    const uint8_t* wg = (const uint8_t*)p.w + (size_t)n0 * RB;
    uint32_t wrow[WI];
#pragma unroll
    for (int i = 0; i < WI; ++i) wrow[i] = (uint32_t)min((tl + i * ST) >> 3, N - 1 - n0) * RB;
    u32x4_t wv[WI];
    /* scales (items below BN) and biases of a line's groups */
    uint32_t srow[SI];
#pragma unroll
    for (int i = 0; i < SI; ++i)
        srow[i] = (uint32_t)min((tl + i * ST) % BN, N - 1 - n0) * (uint32_t)gpr;
    const uint16_t* sg[SI];
#pragma unroll
    for (int i = 0; i < SI; ++i)
        sg[i] = (const uint16_t*)(tl + i * ST < BN ? p.scales : p.biases) + (size_t)n0 * gpr;
    uint32_t sv[SI][(LG + 1) / 2];
    auto load_w = [&](int line) {
        const uint32_t off = min((uint32_t)line * 128u + (uint32_t)c8 * 16u, RB - 16u);
#pragma unroll
        for (int i = 0; i < WI; ++i) wv[i] = *(const u32x4_t*)(wg + (wrow[i] + off));
        if (p.svec) {  // whole lines' groups, aligned: one load
            const uint32_t g = min((uint32_t)line * LG, (uint32_t)(gpr - LG));
#pragma unroll
            for (int i = 0; i < SI; ++i) {
                const uint16_t* src = sg[i] + (srow[i] + g);
                if constexpr (LG == 8) {
                    const u32x4_t v = *(const u32x4_t*)src;
#pragma unroll
                    for (int e = 0; e < 4; ++e) sv[i][e] = v[e];
                } else if constexpr (LG == 4) {
                    const u32x2_t v = *(const u32x2_t*)src;
                    sv[i][0] = v[0];
                    sv[i][1] = v[1];
                } else {
                    sv[i][0] = *(const uint32_t*)src;
                }
            }
        } else {
#pragma unroll
            for (int i = 0; i < SI; ++i)
#pragma unroll
                for (int e = 0; e < LG; e += 2) {
                    const uint32_t g = (uint32_t)(line * LG + e) >> p.gshift;
                    const uint32_t g1 = (uint32_t)(line * LG + e + 1) >> p.gshift;
                    const uint32_t a = sg[i][srow[i] + min(g, (uint32_t)(gpr - 1))];
                    const uint32_t b = sg[i][srow[i] + min(g1, (uint32_t)(gpr - 1))];
                    sv[i][e / 2] = a | (b << 16);
                }
        }
    };
    auto stage_w = [&](int line) {
        uint8_t* wb = wbuf + (line & 1) * kW;
#pragma unroll
        for (int i = 0; i < WI; ++i) {
            const int r = (tl + i * ST) >> 3;
            if constexpr (kTurned)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    wv[i][e] = __builtin_amdgcn_alignbit(wv[i][e], wv[i][e], 29);
            *(u32x4_t*)(wb + r * 128 + ((c8 ^ (r & 7)) * 16)) = wv[i];
        }
        uint32_t* sb = (uint32_t*)(sbuf + (line & (SR - 1)) * kS);
#pragma unroll
        for (int i = 0; i < SI; ++i)
#pragma unroll
            for (int e = 0; e < LG / 2; ++e)
                if (SI * ST == 2 * BN || tl < 2 * BN) sb[(tl + i * ST) * (LG / 2) + e] = sv[i][e];
    };

    f32x16_t acc[RT][CT];
#pragma unroll
    for (int t = 0; t < CT; ++t)
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[r][t][e] = 0.0f;
    uint32_t magic = F16 ? 0x64006400u : 0x41804180u;
    uint32_t nmask = F16 ? 0x000F000Fu : 0x00780078u;
    __asm__ volatile("" : "+v"(magic));  // opaque: keep in a VGPR (see nibble_operand)
    __asm__ volatile("" : "+s"(nmask));  // opaque: keep in an SGPR

    const int line0 = first / LS;
    /* X of one row tile's groups in step st (the strips share the row tiles): ones . x puts row
     * l32's sum in every element of its lanes */
    auto x_sums = [&](const uint8_t* ab, int st) {
        const int xrow = (wm * RT + wn % RT) * 32 + l32;
        const uint8_t* row = ab + xrow * 128;
        uint8_t* xb = xbuf + ((st / SS) & 1) * kX + xrow * 32;
        const u32x4_t ones = F16 ? u32x4_t{0x3c003c00u, 0x3c003c00u, 0x3c003c00u, 0x3c003c00u}
                                 : u32x4_t{0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u};
#pragma unroll
        for (int q = 0; q < NP; ++q) {
            f32x16_t P = {};
#pragma unroll
            for (int j = 0; j < JP; ++j) {
                const int c = (8 / NP) * q + JP * h + j;
                P = mfma32<F16>(ones, *(const u32x4_t*)(row + ((c ^ (l32 & 7)) * 16)), P);
            }
            const float X = P[0];
            /* an infinite X has no low parts (inf - inf) and stays an infinity */
            const bool inf = __builtin_fabsf(X) == __builtin_inff();
            const uint32_t hi = __float_as_uint(X) & 0xffff0000u;
            const float r1 = inf ? 0.0f : X - __uint_as_float(hi);
            const uint32_t mid = __float_as_uint(r1) & 0xffff0000u;
            const uint32_t lo = __float_as_uint(r1 - __uint_as_float(mid));
            const int g = (NP == 1) ? (st & 3) : ((st & 1) * 2 + q);
            *(u32x2_t*)(xb + g * 8) = u32x2_t{mid | (hi >> 16), lo >> 16};  // (halves agree)
        }
    };
    /* the X products of the (up to) four groups that end with step st's */
    auto x_products = [&](int st) {
        const uint8_t* xb = xbuf + ((st / SS) & 1) * kX;
        u32x4_t b1[CT], b2[CT];
#pragma unroll
        for (int t = 0; t < CT; ++t) {
            const int col = (wn * CT + t) * 32 + l32;
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                /* the lane half's groups 2h and 2h + 1 of the four; none past K */
                const int g = st / SS * 4 + 2 * h + e;
                const uint16_t* sl =
                    (const uint16_t*)(sbuf + ((line0 + g / LG) & (SR - 1)) * kS) + col * LG +
                    g % LG;
                const bool in = (first * NP + g) * GS < K;
                const uint32_t cs = in ? sl[0] : 0u, cb = in ? sl[BN * LG] : 0u;
                uint32_t v1, v2;  // the bf16 factors, in the low half
                if constexpr (F16) {
                    /* the low part of a short b would be 0, and NaN against an infinite X: two
                     * halves, so that b X has the sign of both (or is NaN for b = 0, as the
                     * GEMV's is) and s P of the other sign makes NaN, not its own infinity */
                    const float b = elem_to_f32<true>(cb);
                    const uint32_t top = __float_as_uint(b) & 0xffff0000u;
                    const bool whole = __uint_as_float(top) == b;
                    const float hi = whole ? 0.5f * b : __uint_as_float(top);
                    v1 = __float_as_uint(hi) >> 16;
                    v2 = __float_as_uint(whole ? hi : b - hi) >> 16;
                } else {
                    v1 = cb;
                    v2 = __float_as_uint(-(float)kMagic * elem_to_f32<false>(cs)) >> 16;
                }
                /* an infinite b meets X's high part alone: the low ones may be 0 */
                const bool finite = (v1 & 0x7f80u) != 0x7f80u;
                const uint32_t l1 = finite ? v1 : 0u, l2 = !F16 || finite ? v2 : 0u;
                b1[t][2 * e] = v1 | (l1 << 16);
                b1[t][2 * e + 1] = l1;
                b2[t][2 * e] = v2 | (l2 << 16);
                b2[t][2 * e + 1] = l2;
            }
        }
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            const u32x4_t X =
                *(const u32x4_t*)(xb + ((wm * RT + r) * 32 + l32) * 32 + h * 16);
#pragma unroll
            for (int t = 0; t < CT; ++t) {
                acc[r][t] = mfma32<false>(X, b1[t], acc[r][t]);
                if constexpr (kTwo) acc[r][t] = mfma32<false>(X, b2[t], acc[r][t]);
            }
        }
    };

    load_x(0);
    load_w(line0);
    stage_x(0);
    stage_w(line0);
    load_x(1);

    for (int l = 0; l * LS < walk; ++l) {
        const int line = line0 + l;
#pragma unroll
        for (int ls = 0; ls < LS; ++ls) {
            const int st = l * LS + ls;
            if (st >= walk) break;
            __syncthreads();  // step st is staged, step st - 1 has been read
            if (st > 0 && (st & (SS - 1)) == 0 && st <= mine) x_products(st - 1);
            if (KW > 1 && st >= mine) continue;
            /* the next step: past the end clamped addresses are read, and what nothing reads is
             * staged.  Placed after the LDS reads of a row tile, which it would hold up */
            auto stage_next = [&]() {
                stage_x(st + 1);
                load_x(st + 2);
                if (ls == LS - 1) stage_w(line + 1);
                if (ls == 0) load_w(line + 1);
            };
            const uint8_t* wb = wbuf + (line & 1) * kW;
            const uint16_t* sb = (const uint16_t*)(sbuf + (line & (SR - 1)) * kS);
            u32x4_t B[CT][4];
            float s[CT][NP];
#pragma unroll
            for (int t = 0; t < CT; ++t) {
                const int col = (wn * CT + t) * 32 + l32;
                const uint8_t* row = wb + col * 128;
                uint32_t w[NWD];
                constexpr int W = NWD / NP;  // words of a group
#pragma unroll
                for (int q = 0; q < NP; ++q) {
                    /* the lane's words of group q: byte ls * 8 BITS + q * 8 W + h * 4 W */
                    if constexpr (W == 2) {
                        const u32x2_t v = *(const u32x2_t*)(
                            row + (((ls * 2 + q) ^ (col & 7)) * 16 + h * 8));
                        w[q * W] = v[0];
                        w[q * W + 1] = v[1];
                    } else {
#pragma unroll
                        for (int j = 0; j < W / 4; ++j) {
                            const int c = ls * (BITS / 2) + q * (W / 2) + h * (W / 4) + j;
                            const u32x4_t v = *(const u32x4_t*)(row + ((c ^ (col & 7)) * 16));
#pragma unroll
                            for (int e = 0; e < 4; ++e) w[q * W + j * 4 + e] = v[e];
                        }
                    }
                    s[t][q] = elem_to_f32<F16>(sb[col * LG + ls * NP + q]);
                    if (GS == 32 && (first + st) * 64 + q * GS >= K) s[t][q] = 0.0f;
                }
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    B[t][j] = code_operand<BITS, F16, kTurned>(w + j * NWD / 4, nmask, magic);
            }
            const uint8_t* ab = abuf + (st & 1) * kA;
            x_sums(ab, st);
#pragma unroll
            for (int r = 0; r < RT; ++r) {
                const uint8_t* row = ab + ((wm * RT + r) * 32 + l32) * 128;
                u32x4_t A[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int c = (8 / NP) * (j / JP) + JP * h + j % JP;
                    A[j] = *(const u32x4_t*)(row + ((c ^ (l32 & 7)) * 16));
                }
#pragma unroll
                for (int t = 0; t < CT; ++t)
#pragma unroll
                    for (int q = 0; q < NP; ++q) {
                        f32x16_t P = {};
#pragma unroll
                        for (int j = 0; j < JP; ++j)
                            P = mfma32<F16>(A[q * JP + j], B[t][q * JP + j], P);
#pragma unroll
                        for (int e = 0; e < 16; ++e)
                            acc[r][t][e] = __builtin_fmaf(s[t][q], P[e], acc[r][t][e]);
                    }
                if (r == (RT > 2 ? RT - 2 : 0)) stage_next();
            }
        }
    }
    /* the last set's slots past the slice's last step: the sums of two sets before are still
     * there (or nothing yet), and an infinity among them would make NaN of the factor 0 */
    const int over = mine > 0 ? mine & (SS - 1) : 0;
    if (over) {
        uint8_t* xb = xbuf + ((mine / SS) & 1) * kX + ((wm * RT + wn % RT) * 32 + l32) * 32;
        for (int g = over * NP; g < 4; ++g) *(u32x2_t*)(xb + g * 8) = u32x2_t{0u, 0u};
    }
    __syncthreads();
    if (over || mine == walk) x_products(mine - 1);

    if constexpr (KW > 1) {  // the other slices' sums to slice 0
        __syncthreads();
        f32x4_t* red = (f32x4_t*)lds;
        constexpr int kV = RT * CT * 4;  // 16-byte values of a lane
        if (kw > 0) {
            f32x4_t* o = red + (size_t)((kw - 1) * MW * NW + wm * NW + wn) * kV * 64 + lane;
#pragma unroll
            for (int i = 0; i < kV; ++i) {
                const f32x16_t& a = acc[i / 4 / CT][i / 4 % CT];
                o[i * 64] = f32x4_t{a[i % 4 * 4], a[i % 4 * 4 + 1], a[i % 4 * 4 + 2],
                                    a[i % 4 * 4 + 3]};
            }
        }
        __syncthreads();
        if (kw > 0) return;
#pragma unroll
        for (int k2 = 0; k2 < KW - 1; ++k2) {
            const f32x4_t* o = red + (size_t)(k2 * MW * NW + wm * NW + wn) * kV * 64 + lane;
#pragma unroll
            for (int i = 0; i < kV; ++i) {
                const f32x4_t v = o[i * 64];
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[i / 4 / CT][i / 4 % CT][i % 4 * 4 + e] += v[e];
            }
        }
    }

    const uint16_t* lb = (const uint16_t*)p.lbias;
    uint16_t* y = (uint16_t*)p.y;
#pragma unroll
    for (int t = 0; t < CT; ++t) {
        const int n = n0 + (wn * CT + t) * 32 + l32;
        if (n >= N) continue;
        const float add = lb ? elem_to_f32<F16>(lb[n]) : 0.0f;
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int m = m0 + (wm * RT + r) * 32 + (e & 3) + 8 * (e >> 2) + 4 * h;
                if (m < M) y[(size_t)m * N + n] = round_out<F16>(acc[r][t][e] + add);
            }
    }
}

}  // namespace

#define DFQ_GEMM_KERNEL(BITS, GS, F16, NAME, TILE, RT, CT, MW, NW, KW)                     \
    extern "C" __global__ void __launch_bounds__(64 * MW * NW * KW, 2)                            \
        dfq_gemm_b##BITS##_g##GS##_##NAME##_##TILE(QmmGemmParams p) {                        \
        qmm_gemm<BITS, GS, F16, RT, CT, MW, NW, KW>(p);                                      \
    }
/* rows x columns of a workgroup's tile, and slices of K (kGemmTiles in qmm_runtime.cpp) */
#define DFQ_GEMM_FORMAT(BITS, GS, F16, NAME)                       \
    DFQ_GEMM_KERNEL(BITS, GS, F16, NAME, 96x128, 3, 1, 1, 4, 1)    \
    DFQ_GEMM_KERNEL(BITS, GS, F16, NAME, 64x128, 2, 1, 1, 4, 1)    \
    DFQ_GEMM_KERNEL(BITS, GS, F16, NAME, 64x128_k2, 2, 1, 1, 4, 2) \
    DFQ_GEMM_KERNEL(BITS, GS, F16, NAME, 32x128_k2, 1, 1, 1, 4, 2) \
    DFQ_GEMM_KERNEL(BITS, GS, F16, NAME, 32x64_k4, 1, 1, 1, 2, 4)
#define DFQ_GEMM_FORMAT64(BITS, F16, NAME)                        \
    DFQ_GEMM_KERNEL(BITS, 64, F16, NAME, 128x128, 4, 1, 1, 4, 1) \
    DFQ_GEMM_FORMAT(BITS, 64, F16, NAME)

DFQ_GEMM_FORMAT(4, 32, false, bf16)
DFQ_GEMM_FORMAT64(4, false, bf16)
DFQ_GEMM_FORMAT(8, 32, false, bf16)
DFQ_GEMM_FORMAT64(8, false, bf16)
DFQ_GEMM_FORMAT(4, 32, true, f16)
DFQ_GEMM_FORMAT64(4, true, f16)
DFQ_GEMM_FORMAT(8, 32, true, f16)
DFQ_GEMM_FORMAT64(8, true, f16)

/* ---------------------------------------------------------------------------------- */
/* The stock path in fp32: promoted dtypes, fp32 arrays, 2-bit codes, other groups      */
/* ---------------------------------------------------------------------------------- */

namespace {

constexpr int kF32Waves = 16;

/* Eight codes as floats, in k order. */
template <int BITS>
__device__ __forceinline__ void codes8(const uint32_t* w, float (&q)[8]) {
    if constexpr (BITS == 8) {
#pragma unroll
        for (int t = 0; t < 8; ++t) q[t] = (float)((w[t >> 2] >> (8 * (t & 3))) & 0xffu);
    } else if constexpr (BITS == 4) {
        const uint32_t lo = w[0] & 0x0f0f0f0fu, hi = (w[0] >> 4) & 0x0f0f0f0fu;
#pragma unroll
        for (int t = 0; t < 8; ++t) q[t] = (float)(((t & 1 ? hi : lo) >> (8 * (t >> 1))) & 0xffu);
    } else {  // the low 16 bits
#pragma unroll
        for (int t = 0; t < 8; ++t) q[t] = (float)((w[0] >> (2 * t)) & 3u);
    }
}

/* Element i of an array of dtype dt as loaded, and its value: apart, so that the loads of a step
 * are in flight together (a conversion in the branch on dt would wait for its own). */
__device__ __forceinline__ uint32_t load_bits(const void* ptr, int dt, size_t i) {
    if (dt == 2) return ((const uint32_t*)ptr)[i];
    return ((const uint16_t*)ptr)[i];
}
__device__ __forceinline__ float bits_to_f32(uint32_t v, int dt) {
    return dt == 2 ? __uint_as_float(v) : dt == 1 ? elem_to_f32<true>(v) : elem_to_f32<false>(v);
}

/* y = x . dequant(W)^T with every weight, product and sum in fp32: w = s q + b is formed in
 * fp32 as the per-element kernel forms it, and the products run on the fp32 matrix
 * instruction (16 x 16 x 4), which needs x and w unsplit.
 *
 * A workgroup computes 16 columns x 16 RT rows; its 16 waves take the steps of 4 KL k round
 * robin.  Lane 16 j + n holds column n's KL consecutive codes at KL j of the step (one group,
 * so one scale and bias), lane 16 j + m row m's x at the same k, so that product t of a step
 * takes element t of either and no operand is moved between lanes.  A wave keeps four sums
 * (t mod 4): 64 chains in a workgroup, as the per-element kernel's lanes, which keeps the
 * rounding error where it was.  The waves' sums meet in LDS and are added as a tree.
 *
 * With one row tile the loads of two of a wave's steps are issued together (more tiles would
 * spill): 16 x 16, K 17408, all fp32 58.7 -> 48.7 us.
 *
 * Measured on MI355X, fp32 x over bf16 scales, 6 x 4096, K 4096, 4-bit: 172 us a pass by the
 * per-element kernel, 12.5 here, 10 to 11 of them the kernel; both are 1.6e-7 from the 64-bit
 * result.  Bound by latency, a wave has two steps, and by the 16 rows of a tile that 6 fill (3.4 us
 * of matrix time). */
template <int BITS, int KL, int XDT, int RT>
__device__ __forceinline__ void qmm_f32(const QmmGenericParams& p) {
    __shared__ f32x4_t part[kF32Waves * RT * 64];
    constexpr int CB = KL * BITS / 8;  // bytes of a lane's codes
    constexpr int XB = XDT == 2 ? 4 : 2;
    constexpr int U = RT == 1 ? 2 : 1;  // steps whose loads are issued together
    const int tid = threadIdx.x, lane = tid & 63, n16 = lane & 15, j = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int M = p.M, N = p.N, K = p.K;
    const int n0 = blockIdx.x * 16, m0 = blockIdx.y * 16 * RT;
    const int n = min(n0 + n16, N - 1);  // columns past N and rows past M repeat the last
    const int gpr = K / p.gs;
    const uint8_t* wr = (const uint8_t*)p.w + (size_t)n * ((size_t)K * BITS / 8);
    const uint8_t* xr[RT];
#pragma unroll
    for (int r = 0; r < RT; ++r)
        xr[r] = (const uint8_t*)p.x + (size_t)min(m0 + r * 16 + n16, M - 1) * K * XB;

    f32x4_t acc[RT][4];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int a = 0; a < 4; ++a) acc[r][a] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    const int steps = (K - 1) / (4 * KL) + 1;
    constexpr int XW = XDT == 2 ? KL / 4 : KL / 8;  // 16-byte loads of a lane's x of one row
    constexpr int WD = CB < 4 ? 1 : CB / 4;         // words of its codes
    struct Step {
        uint32_t w[WD];
        u32x4_t x[U > 1 ? XW : 1];  // the one row tile's (more of them would spill)
        uint32_t s, b;  // as loaded
        int kc;
        bool in;
    };
    auto load_x = [&](int r, int i, int kc) {
        return *(const u32x4_t*)(xr[r] + (size_t)kc * XB + i * 16);
    };
    auto load = [&](int st) {
        Step v;
        /* (unsigned: the last step of a K near 2^31 ends past it.  K is a multiple of KL) lanes
         * past K read its last codes */
        const uint32_t k = (uint32_t)st * (4 * KL) + (uint32_t)(j * KL);
        const bool in = k < (uint32_t)K;
        const int kc = in ? (int)k : K - KL;
        const uint8_t* ws = wr + (size_t)kc * BITS / 8;
        if constexpr (CB == 2) {
            v.w[0] = *(const uint16_t*)ws;
        } else if constexpr (CB == 4) {
            v.w[0] = *(const uint32_t*)ws;
        } else if constexpr (CB == 8) {
            const u32x2_t c = *(const u32x2_t*)ws;
            v.w[0] = c[0];
            v.w[1] = c[1];
        } else {
#pragma unroll
            for (int i = 0; i < CB / 16; ++i) {
                const u32x4_t c = *(const u32x4_t*)(ws + i * 16);
#pragma unroll
                for (int e = 0; e < 4; ++e) v.w[i * 4 + e] = c[e];
            }
        }
        const size_t g = (size_t)n * gpr + kc / p.gs;
        v.s = load_bits(p.scales, p.sdt, g);
        v.b = load_bits(p.biases, p.sdt, g);
        v.kc = kc;
        v.in = in;
        if constexpr (U > 1)
#pragma unroll
            for (int i = 0; i < XW; ++i) v.x[i] = load_x(0, i, kc);
        return v;
    };
    auto add = [&](const Step& v) {
        const float s = v.in ? bits_to_f32(v.s, p.sdt) : 0.0f;
        const float b = v.in ? bits_to_f32(v.b, p.sdt) : 0.0f;
#pragma unroll
        for (int c = 0; c < KL / 8; ++c) {
            float q[8];
            uint32_t wc[2];
            if constexpr (BITS == 8) {
                wc[0] = v.w[2 * c];
                wc[1] = v.w[2 * c + 1];
            } else if constexpr (BITS == 4) {
                wc[0] = v.w[c];
            } else {
                wc[0] = v.w[c / 2] >> (16 * (c & 1));
            }
            codes8<BITS>(wc, q);
#pragma unroll
            for (int t = 0; t < 8; ++t) q[t] = __builtin_fmaf(q[t], s, b);
#pragma unroll
            for (int r = 0; r < RT; ++r) {
                constexpr int XC = XDT == 2 ? 2 : 1;  // 16-byte pieces of 8 elements
                u32x4_t xv[XC];
#pragma unroll
                for (int i = 0; i < XC; ++i)
                    xv[i] = U > 1 ? v.x[(U > 1) * (XC * c + i)] : load_x(r, XC * c + i, v.kc);
                float x[8];
#pragma unroll
                for (int t = 0; t < 8; ++t) {
                    if constexpr (XDT == 2) {
                        x[t] = __uint_as_float(xv[t / 4][t & 3]);
                    } else {
                        const uint32_t e = xv[0][t / 2];
                        x[t] = elem_to_f32<XDT == 1>(t & 1 ? e >> 16 : e & 0xffffu);
                    }
                }
                if (!v.in)  // lanes past K add nothing, whatever their row holds
#pragma unroll
                    for (int t = 0; t < 8; ++t) x[t] = 0.0f;
#pragma unroll
                for (int t = 0; t < 8; ++t)
                    acc[r][t & 3] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[t], q[t],
                                                                         acc[r][t & 3], 0, 0, 0);
            }
        }
    };
    int st = wave;
    if constexpr (U > 1)
        for (; st + (U - 1) * kF32Waves < steps; st += U * kF32Waves) {
            Step v[U];
#pragma unroll
            for (int u = 0; u < U; ++u) v[u] = load(st + u * kF32Waves);
#pragma unroll
            for (int u = 0; u < U; ++u) add(v[u]);
        }
    for (; st < steps; st += kF32Waves) add(load(st));
#pragma unroll
    for (int r = 0; r < RT; ++r)
        part[(wave * RT + r) * 64 + lane] = (acc[r][0] + acc[r][1]) + (acc[r][2] + acc[r][3]);
    __syncthreads();
    const float* ps = (const float*)part;
    for (int o = tid; o < RT * 256; o += kF32Waves * 64) {
        float v[kF32Waves];
#pragma unroll
        for (int i = 0; i < kF32Waves; ++i) v[i] = ps[i * RT * 256 + o];
#pragma unroll
        for (int d = 1; d < kF32Waves; d *= 2)
#pragma unroll
            for (int i = 0; i < kF32Waves; i += 2 * d) v[i] += v[i + d];
        /* element e of lane l: column l % 16, row 4 (l / 16) + e */
        const int l = (o & 255) >> 2, on = n0 + (l & 15);
        const int om = m0 + (o >> 8) * 16 + (l >> 4) * 4 + (o & 3);
        if (on < N && om < M) {
            float y = v[0];
            if (p.lbias) y += load_any(p.lbias, p.sdt, on);
            store_any(p.y, p.ydt, (size_t)om * N + on, y);
        }
    }
}

}  // namespace

#define DFQ_F32_KERNEL(BITS, KL, XDT, NAME, RT)                                             \
    extern "C" __global__ void __launch_bounds__(kF32Waves * 64)                             \
        dfq_f32_b##BITS##_k##KL##_##NAME##_r##RT(QmmGenericParams p) {                       \
        qmm_f32<BITS, KL, XDT, RT>(p);                                                       \
    }
#define DFQ_F32_ROWS(BITS, KL, XDT, NAME)  \
    DFQ_F32_KERNEL(BITS, KL, XDT, NAME, 1) \
    DFQ_F32_KERNEL(BITS, KL, XDT, NAME, 2) \
    DFQ_F32_KERNEL(BITS, KL, XDT, NAME, 4)
#define DFQ_F32_FORMAT(BITS, KL)       \
    DFQ_F32_ROWS(BITS, KL, 0, bf16)    \
    DFQ_F32_ROWS(BITS, KL, 1, f16)     \
    DFQ_F32_ROWS(BITS, KL, 2, f32)

DFQ_F32_FORMAT(2, 8)
DFQ_F32_FORMAT(2, 32)
DFQ_F32_FORMAT(4, 8)
DFQ_F32_FORMAT(4, 32)
DFQ_F32_FORMAT(8, 8)
DFQ_F32_FORMAT(8, 32)
