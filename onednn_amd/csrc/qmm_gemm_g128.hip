// Tiled GEMM over 4-bit weights whose scales change every 128 k (or less often),
// for many rows: hip:gfx950:decode_w4 (f16 / bf16 activations, f32 sums) and
// hip:gfx950:mfma_w4a8 (s8 activations, s32 sums inside a group of 128 k). The
// arithmetic is that of qmm_gemm_w4f.hip / qmm_gemm_w4a8.hip, operation for
// operation but for one: bf16 takes the offset off the group's sum in one fma, where
// qmm_gemm_w4f.hip rounds the product first. What differs is the shape of the work.
//
// Both problems are bound by instruction issue: next to its MFMAs a wave has to
// expand the nibbles of its columns and to fold a finished group into f32
// accumulators, and the vector ALU shares its issue slots with the matrix
// cores. So the wave tile is as tall as 256 registers allow with two waves per SIMD:
// 128 rows for s8, 96 for f16 / bf16, whose expanded weights take twice the
// registers; or 64, where the taller one leaves more of the last round empty. Three
// forms stand one step over: s8 with 128 rows spills 4 registers (20 bytes of scratch
// a lane, from the second pass over the groups that huge row scales need; without it
// 247 registers), bf16 with 96 rows 1 (s4 weights 4).
//   * four waves side by side own 16 FM rows x 256 columns, a wave all the rows
//     of its 64 columns: a nibble is expanded once for up to 128 rows, where the
//     other kernels expand it once for 64 (the 64-row form has none of this gain: its
//     comes from the next point and from two workgroups on a CU);
//   * the group is the unit of the loop: a 16 x 16 fragment of the result runs
//     its MFMAs over the whole group (4 of 16 x 16 x 32 f16, 2 of 16 x 16 x 64
//     i8) in four registers and is folded into the f32 accumulators at once, so
//     the group's sums never need a second accumulator tile;
//   * f16 weights: two of a dword's four nibble pairs are taken where they lie
//     (0x6400 | w << 4 is 1024 + 16 w, and one packed fma makes that w - z), 9
//     instructions for 8 weights instead of 11;
//   * s8 x 4 bit: a group's s32 sum starts at 0x4B400000, the bits of the float
//     1.5 * 2^23, so it IS the float 1.5 * 2^23 + sum (|sum| = |16 s w'| <= 2^21
//     in a group of 128) and the conversion, the subtraction of the bias and the
//     product with the row scale are one fma: fma(f, ss, -1.5 * 2^23 * ss). The
//     bias times a 16-bit scale is exact, so the one rounding is that of
//     (float)sum * ss. Two vector instructions per result and group, not three.
//     Where the product with the bias overflows (an infinite scale, a bf16 one of
//     2^100 and more), the sums are formed again with (f - 1.5 * 2^23) * ss;
//   * the row and column scales of the next group are fetched by the threads
//     of the workgroup, one of each, and go through LDS as f32: no pre-pass.
// Source rows come through LDS (double-buffered per group, direct loads), a
// wave's packed weights through a private piece of LDS that is refilled as soon
// as its nibbles are in registers. One barrier per group.
//
// Measured on 4096 x 14336 weights, launches back to back, the kernels named above /
// this one: s8 x s4, 1000 rows 121 / 87 us, 2176 rows 230 / 163 us, 4096 rows 407 / 284
// us (1.69 POP/s); f16 x u4, 1000 rows (64-row tiles) 230 / 158 us, 2048 rows 402 / 259
// us (0.93 PFLOP/s); bf16 x u4, 1000 rows 256 / 178 us. The second pass of the s8 form
// costs 3 % where it is not taken (2176 rows 155 us without). With parts switched off
// (1000 rows, s8, without that pass, 88 us): no MFMAs 66, no fold 64, neither 43 us
// (prologue, expanding, LDS reads, epilogue), no loads inside the loop 88: the parts
// add up, whether the fold stands behind a row block's MFMAs or between them. f16 x u4
// (1000 rows, 156 us; 2048 rows, 252 us): no MFMAs 126; 185, no fold 140; 230, neither 112;
// 164, these two and the expanding of nibbles off 58; 100.
#include <algorithm>
#include <type_traits>

#include "qmm_device.hpp"
#include "qmm_hip.h"
#include "qmm_plan.hpp"

namespace qmm {
#if defined(QMM_G128_PART)
namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));

constexpr int WAVES = 4, FN = 4, WN = 16 * FN, BN = WAVES * WN;
constexpr int B_WAVE = FN * 1024; // a wave's packed weights of one group
constexpr int STG_PITCH = WN + 4; // floats per staged row of results

template <int KIND, int FM>
struct geo {
    static constexpr int BM = 16 * FM;
    static constexpr int ROW = KIND == G_S8 ? 128 : 256; // bytes of a row's group
    static constexpr int A_BYTES = BM * ROW;
    static constexpr int B_OFF = 2 * A_BYTES;
    static constexpr int X_OFF = B_OFF + WAVES * B_WAVE;
    // per-group scales as f32 (s8): {ss, -1.5 * 2^23 * ss} per row, sw per column
    static constexpr int X_BYTES = KIND == G_S8 ? BM * 8 + BN * 4 : 0;
    static constexpr int LOOP = X_OFF + 2 * X_BYTES;
    static constexpr int PF = FM == 8 || FM == 6 ? FM / 2 : FM; // row blocks staged at a time
    static_assert(FM % PF == 0, "");
    static constexpr int EPI = WAVES * 16 * PF * STG_PITCH * 4;
    static constexpr int LDS = LOOP > EPI ? LOOP : EPI;
};

QMM_D void dma16(uint32_t lds_addr, uint32_t voff, const uint8_t *sbase) {
    asm volatile("s_mov_b32 m0, %0\n\t"
                 "s_nop 0\n\t"
                 "global_load_lds_dwordx4 %1, %2" ::"s"(lds_addr),
                 "v"(voff), "s"(sbase)
                 : "memory", "m0");
}
QMM_D const uint8_t *uniform_ptr(const uint8_t *q) {
    const uint64_t v = (uint64_t)q;
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return (const uint8_t *)(((uint64_t)hi << 32) | lo);
}
constexpr int WAIT_VM0 = (7 << 4) | (15 << 8); // vmcnt(0) alone
constexpr int WAIT_LGKM0 = 15 | (7 << 4) | (3 << 14); // lgkmcnt(0) alone

template <int KIND>
QMM_D v4f mma(const v4u &a, const v4u &b, const v4f &c) {
    if constexpr (KIND == G_S8)
        return __builtin_bit_cast(v4f,
                __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(v4i, a),
                        __builtin_bit_cast(v4i, b), __builtin_bit_cast(v4i, c), 0,
                        0, 0));
    else if constexpr (KIND == G_F16)
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, a),
                __builtin_bit_cast(v8h, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                __builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, b), c, 0, 0,
                0);
}

QMM_D float half_bits(uint32_t raw, bool f16) { // a 16-bit scale's value
    const float h = (float)__builtin_bit_cast(_Float16, (uint16_t)raw);
    const float b = u2f(raw << 16);
    return f16 ? h : b;
}

// The fragment a result comes from, by kind. s8: the weights are the MFMA's
// first operand, so a lane holds ONE row (lane % 16) and four neighbouring
// columns (4 (lane / 16) + register): a row scale is one value per lane. f16 /
// bf16: the activations are, so a lane holds ONE column (lane % 16) and four
// rows: scale and zero point are one value per lane.
template <int KIND, int FM, bool WSIGNED>
__global__ void __launch_bounds__(WAVES * 64, 2)
gemm_g128_kernel(const g128_params_t p) {
    using G = geo<KIND, FM>;
    constexpr int BM = G::BM;
    constexpr bool S8 = KIND == G_S8, F16 = KIND == G_F16;
    constexpr int STEPS = S8 ? 2 : 4; // MFMAs of a fragment and group
    typedef __attribute__((address_space(3))) uint8_t lds_u8;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, c = lane >> 4;

    // XCD-aware tile order: consecutive logical tiles run on one XCD
    const int ntiles = p.tiles_m * p.tiles_n;
    int lt = blockIdx.x;
    if (ntiles >= 64) {
        const int per = (ntiles + 7) / 8;
        const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
        lt = xcd * per + slot;
        if (slot >= per || lt >= ntiles) return;
    }
    constexpr int GROUP_M = 8;
    const int gid = lt / (GROUP_M * p.tiles_n);
    const int first_m = gid * GROUP_M;
    const int gsz = min(p.tiles_m - first_m, GROUP_M);
    const int tile_m = first_m + (lt % (GROUP_M * p.tiles_n)) % gsz;
    const int tile_n = (lt % (GROUP_M * p.tiles_n)) / gsz;
    const int m0 = tile_m * BM, n0 = tile_n * BN, n_w = n0 + wave * WN;

    const uint32_t lds_base = __builtin_amdgcn_readfirstlane(
            (uint32_t)(uintptr_t)(lds_u8 *)lds);
    const int NG = p.ng;

    // ---- direct loads: 1 KiB an instruction. Source rows: 16-byte chunk q of a
    // row lies at chunk q ^ swz(row), so that the 16 rows of a fragment read
    // hit every bank group once; rows past M repeat the last one.
    constexpr int CPR = G::ROW / 16; // chunks per row
    constexpr int RPI = 64 / CPR; // rows per instruction
    constexpr int A_LD = BM / RPI / WAVES;
    static_assert(A_LD * RPI * WAVES == BM, "");
    auto swz = [](int row) { return S8 ? (row >> 1) & 7 : row & 15; };
    uint32_t a_vo[A_LD];
#pragma unroll
    for (int j = 0; j < A_LD; j++) {
        const int row = (wave * A_LD + j) * RPI + lane / CPR;
        a_vo[j] = (uint32_t)(min(m0 + row, p.M - 1) - m0) * (uint32_t)p.lda
                + (uint32_t)(((lane % CPR) ^ swz(row)) * 16);
    }
    const uint8_t *sa = uniform_ptr(p.A + (int64_t)m0 * p.lda);
    const uint32_t lds_a = lds_base + wave * A_LD * 1024;
    // Packed weights: 1 KiB per 16 columns and group (f16, bf16: four column
    // blocks; s8: two blocks of 32 columns of two 1 KiB tiles each); blocks past
    // the last one repeat it and are never stored.
    const uint8_t *sb[FN];
#pragma unroll
    for (int j = 0; j < FN; j++) {
        if constexpr (S8)
            sb[j] = uniform_ptr(p.B
                    + ((int64_t)min(n_w / 32 + (j >> 1), p.nb - 1) * NG * 2
                              + (j & 1))
                            * 1024);
        else
            sb[j] = uniform_ptr(
                    p.B + (int64_t)min(n_w / 16 + j, p.nb - 1) * NG * 1024);
    }
    constexpr int B_STEP = S8 ? 2048 : 1024;
    const uint32_t lds_b = lds_base + G::B_OFF + wave * B_WAVE;
    auto fetch_a = [&](int g) {
        const uint8_t *s = sa + (int64_t)g * G::ROW;
        const uint32_t d = lds_a + (g & 1) * G::A_BYTES;
#pragma unroll
        for (int j = 0; j < A_LD; j++)
            dma16(d + j * 1024, a_vo[j], s);
    };
    auto fetch_b = [&](int g) {
#pragma unroll
        for (int j = 0; j < FN; j++)
            dma16(lds_b + j * 1024, lane * 16, sb[j] + (int64_t)g * B_STEP);
    };

    // ---- scales and zero points, requested a group ahead in storage types
    const uint16_t *x_row = nullptr, *x_col[FN];
    uint32_t raw_row = 0, raw_col[FN];
    uint32_t raw_zp[FN];
    if constexpr (S8) { // thread t: row t of the tile, column t of the tile
        x_row = (const uint16_t *)p.ss + (int64_t)min(m0 + min(tid, BM - 1), p.M - 1) * p.ss_sm;
        x_col[0] = (const uint16_t *)p.scales + (int64_t)min(n0 + tid, p.N - 1) * p.sw_sn;
    } else {
#pragma unroll
        for (int j = 0; j < FN; j++) {
            const int n = min(n_w + 16 * j + r, p.N - 1);
            x_col[j] = (const uint16_t *)p.scales + (p.scale_per_n ? n : 0);
        }
    }
    // (an absent zero-point buffer: the weights stand in, the value is not used)
    const uint8_t *const zps = p.zps ? (const uint8_t *)p.zps : p.B;
    auto zp_index = [&](int g, int j) {
        const int64_t gz = p.gz_shift < 0 ? 0 : g >> p.gz_shift;
        const int n = min(n_w + 16 * j + r, p.N - 1);
        return !p.zps ? (int64_t)0 : p.zp_per_n ? gz * p.N + n : gz;
    };
    auto fetch_x = [&](int g0) {
        const int g = min(g0, NG - 1); // (past the end: the last group, not used)
        if constexpr (S8) {
            raw_row = x_row[g * p.ss_sk];
            raw_col[0] = x_col[0][g * p.sw_sk];
        } else {
            const int64_t gs = p.gs_shift < 0 ? 0 : g >> p.gs_shift;
#pragma unroll
            for (int j = 0; j < FN; j++) {
                raw_col[j] = x_col[j][p.scale_per_n ? gs * p.N : gs];
                const int64_t zi = zp_index(g, j);
                raw_zp[j] = zps[p.zp4 ? zi >> 1 : zi];
            }
        }
    };
    constexpr float BIAS = 12582912.f; // 1.5 * 2^23, bits 0x4B400000
    int huge = 0; // s8: a row scale whose product with BIAS is no number
    auto stage_x = [&](int g) { // s8: the fetched scales of group g to LDS
        if constexpr (S8) {
            float *x = (float *)(lds + G::X_OFF + (g & 1) * G::X_BYTES);
            const float s = half_bits(raw_row, p.ss_f16);
            if (tid < BM) *(float2 *)(x + 2 * tid) = make_float2(s, -BIAS * s);
            huge |= !(__builtin_fabsf(s) < 0x1p100f);
            x[2 * BM + tid] = half_bits(raw_col[0], p.sw_f16) * 0.0625f;
        }
    };

    float res[FM][FN][4]; // (scalars: as vectors they must lie in aligned tuples)
    const v4f p0 = S8 ? v4f {BIAS, BIAS, BIAS, BIAS} : v4f {0.f, 0.f, 0.f, 0.f};

    auto sum_groups = [&](auto any_scale) {
    constexpr bool ANY_SCALE = decltype(any_scale)::value;
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++)
#pragma unroll
            for (int e = 0; e < 4; e++) res[i][j][e] = 0.f;

    fetch_x(0);
    fetch_a(0);
    fetch_b(0);
    stage_x(0);
#pragma unroll 1
    for (int g = 0; g < NG; g++) {
        // this wave's loads of group g have landed; behind the barrier so have
        // the others', and everyone is done with the other stage
        __builtin_amdgcn_s_waitcnt(WAIT_VM0);
        __syncthreads();
        float sc[FN], off[FN];
        uint32_t k_lo[FN], k_hi[FN];
        if constexpr (!S8) {
#pragma unroll
            for (int j = 0; j < FN; j++) {
                sc[j] = half_bits(raw_col[j], p.sw_f16);
                const int odd = p.zp4 ? (int)(zp_index(g, j) & 1) : 0;
                const int zbits = p.zp4 ? 4 : 8;
                const uint32_t zraw = (raw_zp[j] >> (4 * odd)) & ((1u << zbits) - 1u);
                const int zsx = (int)(zraw << (32 - zbits)) >> (32 - zbits);
                const float z = p.zps ? (float)(p.zp_signed ? zsx : (int)zraw) : 0.f;
                const float soff = WSIGNED ? 8.f : 0.f;
                off[j] = 128.f + soff + z; // bf16: leaves through the row sums
                const uint32_t l = __builtin_bit_cast(
                        uint16_t, (_Float16)(-(1024.f + soff + z)));
                const uint32_t h = __builtin_bit_cast(
                        uint16_t, (_Float16)(-(64.f + soff + z)));
                k_lo[j] = l | (l << 16);
                k_hi[j] = h | (h << 16);
            }
        }
        if (g + 1 < NG) fetch_a(g + 1);
        fetch_x(g + 1);

        // ---- the group's weights as MFMA operands
        v4u w[FN][STEPS];
        const uint8_t *bw = lds + G::B_OFF + wave * B_WAVE;
#pragma unroll
        for (int j = 0; j < FN; j++) {
            // s8: lane (r, c) takes the packed lane r + 16 (j % 2) + 32 (c % 2) of
            // tile c / 2 of the group: its k are 64 (c / 2) + 32 step + 16 (c % 2)
            const v4u d4 = *(const v4u *)(S8 ? bw + (j >> 1) * 2048 + (c >> 1) * 1024
                            + (r + 16 * (j & 1) + 32 * (c & 1)) * 16
                                             : bw + j * 1024 + lane * 16);
#pragma unroll
            for (int s = 0; s < STEPS; s++) {
                if constexpr (S8) {
                    const uint32_t d0 = d4[2 * s], d1 = d4[2 * s + 1];
                    w[j][s] = v4u {(d0 << 4) & 0xF0F0F0F0u, d0 & 0xF0F0F0F0u,
                            (d1 << 4) & 0xF0F0F0F0u, d1 & 0xF0F0F0F0u};
                } else {
                    const uint32_t d = WSIGNED ? d4[s] ^ 0x88888888u : d4[s];
                    if constexpr (F16) {
                        const uint32_t e = d >> 8;
                        const v2h lo = __builtin_bit_cast(v2h, k_lo[j]);
                        const v2h hi = __builtin_bit_cast(v2h, k_hi[j]);
                        const v2h q = {(_Float16)0.0625f, (_Float16)0.0625f};
                        auto f = [&](uint32_t x, bool up) {
                            const v2h v = __builtin_bit_cast(v2h, x | 0x64006400u);
                            return __builtin_bit_cast(uint32_t,
                                    up ? __builtin_elementwise_fma(v, q, hi)
                                       : v + lo);
                        };
                        w[j][s] = v4u {f(d & 0x000F000Fu, false),
                                f(d & 0x00F000F0u, true),
                                f(e & 0x000F000Fu, false),
                                f(e & 0x00F000F0u, true)};
                    } else {
                        w[j][s] = v4u {(d & 0x000F000Fu) | 0x43004300u,
                                ((d >> 4) & 0x000F000Fu) | 0x43004300u,
                                ((d >> 8) & 0x000F000Fu) | 0x43004300u,
                                ((d >> 12) & 0x000F000Fu) | 0x43004300u};
                    }
                }
            }
        }
        // the packed bytes are in registers: the next group's may overwrite them
        __builtin_amdgcn_s_waitcnt(WAIT_LGKM0);
        if (g + 1 < NG) fetch_b(g + 1);

        const uint8_t *As = lds + (g & 1) * G::A_BYTES + r * G::ROW;
        const float *x = (const float *)(lds + G::X_OFF + (g & 1) * G::X_BYTES);
        v4f sw[FN];
        if constexpr (S8) {
#pragma unroll
            for (int j = 0; j < FN; j++)
                sw[j] = *(const v4f *)(x + 2 * BM + wave * WN + 16 * j + 4 * c);
        }
        const v4u ones = {0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u};
        // A source fragment is read again, for the next row block, as soon as the
        // MFMAs of its step have been issued
        v4u a[STEPS];
        auto read_a = [&](int i, int s) {
            // (swz(16 i + r) == swz(r): 16 rows are whole swizzle periods)
            const int q = S8 ? 4 * (c >> 1) + 2 * s + (c & 1) : 4 * s + c;
            return *(const v4u *)(As + i * 16 * G::ROW + (q ^ swz(r)) * 16);
        };
#pragma unroll
        for (int s = 0; s < STEPS; s++) a[s] = read_a(0, s);
        // A row block's fragments are computed in units of UJ column blocks. The
        // MFMAs of a unit go out between the instructions that fold the unit
        // before it, in exactly this order: the empty asm statements pin the
        // arithmetic (which the compiler would otherwise sink behind the last
        // unit, all group sums live), the scheduling barriers the order.
        constexpr int UJ = S8 ? FN : FN / 2, NU = FN / UJ; // units per row block
        constexpr int NM = STEPS * UJ, RPM = 4 * UJ / NM; // results per MFMA
        static_assert(RPM * NM == 4 * UJ, "");
        v4f P[2][UJ], S[2];
        float2 ss[2];
        auto read_ss = [&](int i) { return *(const float2 *)(x + 2 * (16 * i + r)); };
        if constexpr (S8) ss[0] = read_ss(0);
#pragma unroll
        for (int u = -1; u < FM * NU; u++) {
            const int i = u / NU, j0 = u % NU * UJ; // folded (u >= 0)
            const int in = (u + 1) / NU, jn = (u + 1) % NU * UJ; // multiplied
            const bool more = u + 1 < FM * NU;
            if (S8 && more && u >= 0) ss[in & 1] = read_ss(in);
#pragma unroll
            for (int t = 0; t < NM; t++) {
                const int s = t / UJ, j = t % UJ;
                if (more) {
                    v4f &d = P[(u + 1) & 1][j];
                    const v4f c0 = s == 0 ? p0 : d;
                    d = S8 ? mma<KIND>(w[jn + j][s], a[s], c0)
                           : mma<KIND>(a[s], w[jn + j][s], c0);
                    asm volatile("" : "+v"(d));
                    if (j == UJ - 1) {
                        if (KIND == G_BF16 && jn == 0) {
                            v4f &q = S[in & 1];
                            const v4f q0 = s == 0 ? p0 : q;
                            q = mma<KIND>(a[s], ones, q0);
                            asm volatile("" : "+v"(q));
                        }
                        if (jn + UJ == FN && in + 1 < FM) a[s] = read_a(in + 1, s);
                    }
                }
                if (u >= 0) {
#pragma unroll
                    for (int q = t * RPM; q < (t + 1) * RPM; q++) {
                        const int jf = q / 4, e = q % 4;
                        const float v = P[u & 1][jf][e];
                        float &o = res[i][j0 + jf][e];
                        if constexpr (S8 && ANY_SCALE)
                            o = __builtin_fmaf((v - BIAS) * ss[i & 1].x, sw[jf][e], o);
                        else if constexpr (S8)
                            o = __builtin_fmaf(
                                    __builtin_fmaf(v, ss[i & 1].x, ss[i & 1].y),
                                    sw[jf][e], o);
                        else
                            o = __builtin_fmaf(sc[j0 + jf],
                                    F16 ? v
                                        : __builtin_fmaf(
                                                  -off[j0 + jf], S[i & 1][e], v),
                                    o);
                        asm volatile("" : "+v"(o));
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        stage_x(g + 1);
    }
    };
    sum_groups(std::false_type {});
    // LDS is reused behind this barrier, by the sums once more or the epilogue
    if constexpr (S8) {
        if (__syncthreads_or(huge)) {
            sum_groups(std::true_type {});
            __syncthreads();
        }
    } else {
        __syncthreads();
    }

    // ---- epilogue: up to 64 rows at a time through a wave-private LDS tile, so that a
    // lane gets four neighbouring columns of a row and 16 lanes a whole row piece
    constexpr int PF = G::PF;
    float *const stg = (float *)lds + wave * 16 * PF * STG_PITCH;
    const int ecol = (lane & 15) * 4, en = n_w + ecol;
    const int envalid = min(4, p.N - en);
    ep_cols_t cols;
    epilogue_cols_load(p.ep, cols, 0, en, envalid > 0 ? envalid : 0);
    // the row interpreter reads the parameter block where it lies (the kernel
    // argument segment): its run-time indexing must not drag `p` into memory
    const epilogue_t &epk
            = ((const g128_params_t *)__builtin_amdgcn_kernarg_segment_ptr())->ep;
    const bool has_ss = p.ep.src_scale.ptr != nullptr;
    const bool fast = S8 && p.ep.fast != EP_FAST_NONE && !p.ep.fast_ext;
    const bool bare = !fast && !has_ss && !cols.has_ws && !cols.has_bias
            && !cols.has_ds && !cols.has_zp && p.ep.npo == 0;
    const float ss0 = has_ss ? ep_load(p.ep.src_scale, 0, 0, 0) : 1.f;
    // (half of a tall tile at a time: while the row loop below, which holds the post-op
    // interpreter, runs, at most 64 accumulator registers are live)
    auto stage = [&](auto h_tag) { // (h a constant: the results stay in registers)
        constexpr int h = decltype(h_tag)::value;
        if constexpr (PF * h < FM) {
#pragma unroll
            for (int i2 = 0; i2 < PF; i2++)
#pragma unroll
                for (int j = 0; j < FN; j++) {
                    if constexpr (S8) {
                        *(v4f *)&stg[(16 * i2 + r) * STG_PITCH + 16 * j + 4 * c]
                                = v4f {res[PF * h + i2][j][0], res[PF * h + i2][j][1],
                                        res[PF * h + i2][j][2], res[PF * h + i2][j][3]};
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; e++)
                            stg[(16 * i2 + 4 * c + e) * STG_PITCH + 16 * j + r]
                                    = res[PF * h + i2][j][e];
                    }
                }
        }
    };
#pragma unroll 1
    for (int h = 0; h < FM / PF; h++) {
        if (h == 0) stage(std::integral_constant<int, 0> {});
        else stage(std::integral_constant<int, 1> {});
        // (wave-private: ordered by the compiler's waits, no barrier)
#pragma unroll 1
        for (int it = 0; it < 4 * PF; it++) {
            const int row = it * 4 + c;
            const v4f t = *(const v4f *)&stg[row * STG_PITCH + ecol];
            const int m = m0 + 16 * PF * h + row;
            if (m < p.M && en < p.N) {
                float v[4] = {t.x, t.y, t.z, t.w};
                if (bare)
                    epilogue_store4(p.ep, v, (int64_t)m * p.ep.dst.sm + en * p.ep.dst.sn,
                            envalid);
                else if (fast)
                    epilogue_fast4(p.ep, v, has_ss, ss0, cols.has_ws, cols.ws, 0,
                            m, en, envalid);
                else
                    epilogue_rows4(epk, cols, v, has_ss, ss0, 0, m, en, envalid);
            }
        }
    }
}

template <int KIND, int FM, bool WSIGNED>
void launch_one(const g128_params_t &p, hipStream_t stream) {
    using G = geo<KIND, FM>;
    static_assert(2 * G::LDS <= 160 * 1024, "two workgroups per CU");
    g128_params_t q = p;
    q.tiles_m = (p.M + G::BM - 1) / G::BM;
    q.tiles_n = (p.N + BN - 1) / BN;
    const int ntiles = q.tiles_m * q.tiles_n;
    const int grid = ntiles >= 64 ? (ntiles + 7) / 8 * 8 : ntiles;
    auto kern = gemm_g128_kernel<KIND, FM, WSIGNED>;
    ensure_dynamic_lds((const void *)kern, G::LDS);
    hipLaunchKernelGGL(kern, dim3(grid), dim3(WAVES * 64), G::LDS, stream, q);
}

template <int KIND, bool WSIGNED>
void launch_rows(const g128_params_t &p, int rows, hipStream_t stream) {
    if (rows == 64) launch_one<KIND, 4, WSIGNED>(p, stream);
    else launch_one<KIND, KIND == G_S8 ? 8 : 6, WSIGNED>(p, stream);
}

} // namespace

#if QMM_G128_PART == 0
void launch_gemm_g128_s8(const g128_params_t &p, int rows, hipStream_t stream) {
    launch_rows<G_S8, false>(p, rows, stream);
}
#elif QMM_G128_PART == 1
void launch_gemm_g128_f16(const g128_params_t &p, int rows, hipStream_t stream) {
    if (p.wei_signed) launch_rows<G_F16, true>(p, rows, stream);
    else launch_rows<G_F16, false>(p, rows, stream);
}
#else
void launch_gemm_g128_bf16(const g128_params_t &p, int rows, hipStream_t stream) {
    if (p.wei_signed) launch_rows<G_BF16, true>(p, rows, stream);
    else launch_rows<G_BF16, false>(p, rows, stream);
}
#endif
#else
// us per group of 128 k for so many tiles, one / two workgroups on a CU (a CU that
// has n takes n / 2 pairs and n % 2 single ones, one after the other)
static double group_us(int64_t tiles, double one, double two) {
    const int64_t n = (tiles + 255) / 256;
    return (double)(n / 2) * two + (double)(n % 2) * one;
}
// us of the kernels of qmm_gemv_w4.hip (up to 16 rows) and qmm_gemm_w4f.hip for few
// rows. Up to 16 rows: per 1000 columns what launching their workgroups takes, or
// reading their weights; 17 to 32 rows: rounds of 32 x 128 tiles, one on a CU.
static double few_rows_us(int M, int N, int groups) {
    if (M > 16) return (double)(((int64_t)N + 32767) / 32768) * (5.5 + 0.68 * groups);
    const double launch = M <= 4 ? 0.31 : M <= 8 ? 0.43 : 0.93;
    const double read = M <= 4 ? 0.012 : M <= 8 ? 0.017 : 0.0178;
    return 1e-3 * N * std::max(launch, read * groups);
}

// Rows of the tile for an M x N x K problem, 0: the other kernels are as fast.
// us per group of 128 k, one / two workgroups on a CU, prologue and epilogue of a
// 4096-k problem shared out over its groups:
//   s8:   64 rows 1.10 / 1.45, 128 rows 1.75 / 2.45
//   f16:  64 rows 1.75 / 2.35,  96 rows 2.2  / 2.7 (bf16 a tenth more on each)
// Over 530 problems (100 ... 4096 rows, 4096 ... 28672 columns, 1024 and 4096 k) the
// tile chosen with these is 0.9 % (s8), 0.2 % (f16), 0.5 % (bf16) behind the better one
// on average, 15 % (s8, 257 rows x 28672 columns), 3 % and 5 % at most. Costs from the
// slope over K alone (s8 0.84 / 1.28 and 1.27 / 2.26) choose worse (s8: 4.6 %).
// The gates: the kernel of qmm_gemm_w4f.hip takes 1.85 us for a 64 x 256 block and
// runs one on a CU (4096 x 14336 weights: 256 rows, 224 blocks, 62 against 63 us;
// 512 rows, 448 blocks, 117 against 82 us); that of qmm_gemm_w4a8.hip was faster by
// up to 5 % at 64 ... 128 blocks and slower from 224 on (200 rows 49.4 against
// 42.2 us; 128 rows 40.9 against 40.9 us; 65 rows x 4096 columns 38.0 against 39.9).
// f16 / bf16 with at most 32 rows pass the gate where there are more than 65536
// columns, and are then a question of time against time: most of a 64-row tile is
// padding, but the other kernels pay by the column. bf16, other kernels / this one:
// 4096 x 128256 weights, 1 row 49 / 84, 8 rows 74 / 85, 16 rows 119 / 87, 32 rows
// 109 / 91; 4096 x 65792, 1 row 26 / 82, 16 rows 73 / 84, 32 rows 79 / 86, 33 rows
// 121 / 87; 1024 x 128256, 1 row 39 / 25 us. (s8: up to 64
// rows have kernels of their own, which the launch takes before it asks here.)
int gemm_g128_rows(int M, int N, int K, int kind) {
    const bool s8 = kind == G_S8;
    const int64_t tn = ((int64_t)N + 255) / 256;
    const int tall = s8 ? 128 : 96;
    const int64_t t64 = ((int64_t)M + 63) / 64 * tn;
    const int64_t tt = ((int64_t)M + tall - 1) / tall * tn;
    if (t64 <= (s8 ? 192 : 256) || (s8 && M <= 64)) return 0;
    const double c64 = s8 ? group_us(t64, 1.10, 1.45) : group_us(t64, 1.75, 2.35);
    const double ct = s8 ? group_us(tt, 1.75, 2.45) : group_us(tt, 2.2, 2.7);
    if (!s8 && M <= 32) {
        const int groups = K / 128;
        const double us
                = 5.0 + groups * std::min(c64, ct) * (kind == G_BF16 ? 1.1 : 1.0);
        if (few_rows_us(M, N, groups) <= us) return 0;
    }
    return c64 < ct ? 64 : tall;
}
// what that tile takes (5 us of start and end aside the groups)
double gemm_g128_us(int M, int N, int K, int kind) {
    const bool s8 = kind == G_S8;
    const int64_t tn = ((int64_t)N + 255) / 256;
    const int tall = s8 ? 128 : 96;
    const int64_t t64 = ((int64_t)M + 63) / 64 * tn, tt = ((int64_t)M + tall - 1) / tall * tn;
    const double us = s8 ? std::min(group_us(t64, 1.10, 1.45), group_us(tt, 1.75, 2.45))
                         : std::min(group_us(t64, 1.75, 2.35), group_us(tt, 2.2, 2.7));
    return 5.0 + K / 128 * us * (kind == G_BF16 ? 1.1 : 1.0);
}
#endif
} // namespace qmm

#if !defined(QMM_G128_PART)
extern "C" int qmm_gemm_g128_rows(int src_dt, int64_t M, int64_t N, int64_t K) {
    using namespace qmm;
    if (M < 1 || N < 1 || K < 1 || M > INT32_MAX || N > INT32_MAX || K > INT32_MAX)
        return 0;
    if (src_dt != dt_s8 && src_dt != dt_f16 && src_dt != dt_bf16) return 0;
    return gemm_g128_rows((int)M, (int)N, (int)K,
            src_dt == dt_s8 ? G_S8 : src_dt == dt_f16 ? G_F16 : G_BF16);
}
#endif
