// hip:gfx950:decode_w4 between the decode step and the long prompts: 16-bit activations
// [M,K] x 4- or 8-bit weights of QMM_LAYOUT_MFMA_W4 / _W8 (arithmetic of qmm_gemv_w4.hip:
// src/cpu/matmul/ref_matmul.cpp:140-173 with fpmath_mode apply_to_int), where tiles that
// walk all of K leave most of the chip idle. A workgroup owns 16 RB x 16 CB results; its
// eight waves cut K between them, a 128-k tile each in turn, and each holds all the
// results: no wave waits for another before the sum at the end.
//   * Activations of a tile are requested one tile ahead, four lanes to 64 bytes of a row, and
//     change to operand order in a piece of LDS of the wave's own: no barrier. (Requested in
//     operand order, lane l from row l % 16, 8 waves of a CU get 11.5 bytes a cycle from L2,
//     with quads of lanes 32 ... 40; 164 x 6528 x 3552 25.2 against 19.4 us.) Fragments of
//     weights are the layout's own, requested with scales and zero points two tiles ahead.
//   * f16: the offset and zero point leave the weights in one packed operation (integers
//     below 2048, exact; odd pairs of nibbles stay in place as 1024 + 16 w, so that a dword
//     takes one shift), and the products need no row sums. 8-bit weights are put together
//     from both nibbles first, one product per step instead of two. bf16 takes the row
//     sums from products with ones, as the decode kernel does.
//   * FOLD: a scale per K group, folded into a second set of sums behind every tile; else
//     one scale per column, applied at the end.
// Bound: a tile of 32 x 64 results costs a CU 1.3 us per 128 k of its eight waves: 480 cycles a
// SIMD of products, 1400 of vector instructions, 2400 of requests through L1 (12 KB a wave).
// 48 x 64 needs the fewest bytes per product and all 256 registers; 64 x 64, and 48 x 64 in
// bf16, spill (204 x 12928 x 2176 25.0 us in 32 x 64, 51.5 in 48 x 64). One workgroup is
// resident per CU; 32 x 32 results in 128 registers for two spill as well (8.3 -> 16.2 us).
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "qmm_device.hpp"
#include "qmm_kcut.hpp"
#include "qmm_plan.hpp"

// Instantiated per activation type and weights width (QMM_W4K_PART = 0..3: bit 0 f16
// activations, bit 1 8-bit weights); the unit without the macro holds the launcher.
namespace qmm {
constexpr int WK_WAVES = 8;

// Workgroup w runs on XCD w % 8; an XCD takes a run of neighbouring items, the row blocks
// of a column block one after another, so that weights are read into one L2 and no XCD
// gets more than its share.
struct w4k_map_t {
    int nrb, total, share;
};
__host__ __device__ inline w4k_map_t w4k_map(int M, int nb16, int rb, int cb) {
    const int nrb = (M + 16 * rb - 1) / (16 * rb), ncb = (nb16 + cb - 1) / cb;
    return {nrb, nrb * ncb, (nrb * ncb + 7) / 8};
}

// (f16 and one scale per column: the tiles' sums need no scale of their own)
inline bool w4k_fold(const gemv_params_t &p) {
    return !p.act_f16 || p.gs_shift >= 0 || p.gz_shift >= 0;
}
// 48 x 64 results: without spills, or all but
constexpr bool w4k_tall(bool f16, bool w8, bool fold) { return f16 && !(w8 && fold); }

#if defined(QMM_W4K_PART)
namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));

template <bool F16>
QMM_D v4f mfma16(const v4u &a, const v4u &b, const v4f &c) {
    if constexpr (F16)
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, a),
                __builtin_bit_cast(v8h, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, a),
                __builtin_bit_cast(v8bf, b), c, 0, 0, 0);
}

QMM_D uint32_t pk_sub(uint32_t x, uint32_t y) {
    return __builtin_bit_cast(
            uint32_t, __builtin_bit_cast(v2h, x) - __builtin_bit_cast(v2h, y));
}

QMM_D uint32_t pk_sixteenth(uint32_t x, uint32_t y) { // x / 16 - y, rounded once
    const v2h sixteenth = {(_Float16)0.0625f, (_Float16)0.0625f};
    return __builtin_bit_cast(uint32_t,
            __builtin_elementwise_fma(
                    __builtin_bit_cast(v2h, x), sixteenth, -__builtin_bit_cast(v2h, y)));
}

// bytes of a wave: its activations of a tile, later its results in rows of BN + 4 floats
constexpr int w4k_wave_lds(int rb, int cb) {
    const int results = 16 * rb * (16 * cb + 4) * 4;
    return results > rb * 4096 ? results : rb * 4096;
}

// flags_m / shifts: as gemv_w4_fast_kernel (qmm_gemv_w4.hip)
template <bool F16, bool W8, bool WSIGNED, int RB, int CB, bool FOLD>
__global__ void __launch_bounds__(WK_WAVES * 64)
gemm_w4k_kernel(const gemv_params_t p, const int shifts, const int flags_m) {
    constexpr int NP = W8 ? 2 : 1, TILE_BYTES = 1024 * NP;
    constexpr bool W8F = W8 && F16; // both nibbles in one f16 value
    extern __shared__ __attribute__((aligned(16))) uint8_t lds_raw[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane >> 4, r = lane & 15;
    const int M = p.M, N = p.N, tiles = p.kg128, nb16 = p.nb16;
    const w4k_map_t map = w4k_map(M, nb16, RB, CB);
    const int item = (blockIdx.x & 7) * map.share + (blockIdx.x >> 3);
    if (item >= map.total) return;
    const int m0 = item % map.nrb * (16 * RB), nb0 = item / map.nrb * CB;

    const int gs_shift = (int8_t)(shifts & 0xff), gz_shift = (int8_t)(shifts >> 8);
    const bool scale_per_n = flags_m & 1, zp_per_n = flags_m & 2;
    const bool zp4 = flags_m & 4, zp_signed = flags_m & 8, sc_f16 = flags_m & 16;
    const bool has_zp = flags_m & 64;
    constexpr float OFFSET = F16 ? 1024.f : 128.f;
    constexpr uint32_t ONE2 = 0x3F803F80u; // (bf16 only)
    const v4u ones = {ONE2, ONE2, ONE2, ONE2};
    constexpr uint32_t sflip = WSIGNED ? 0x88888888u : 0u;
    constexpr float soff = WSIGNED ? (W8 ? 128.f : 8.f) : 0.f;
    // (mask in a scalar, exponent in a vector register: one v_and_or_b32)
    uint32_t MAGIC = F16 ? 0x64006400u : 0x43004300u;
    asm volatile("" : "+v"(MAGIC));
    constexpr uint32_t MAGIC_HI = 0x45004500u; // bf16, high nibbles: 2048 + 16 h
    uint32_t NIB = 0x000F000Fu, NIBH = 0x00F000F0u;
    asm volatile("" : "+s"(NIB), "+s"(NIBH));

    // column blocks past the last one repeat it, rows past M the last one: never stored
    const uint8_t *Bt[CB];
    uint32_t scol[CB], zcol[CB];
#pragma unroll
    for (int cb = 0; cb < CB; cb++) {
        Bt[cb] = p.B + (int64_t)min(nb0 + cb, nb16 - 1) * tiles * TILE_BYTES;
        const int nn = min((nb0 + cb) * 16 + r, N - 1);
        scol[cb] = scale_per_n ? nn : 0;
        zcol[cb] = has_zp && zp_per_n ? nn : 0;
    }
    // Activations are requested four lanes to 64 bytes of a row (lane l: row l / 4, piece
    // l % 4) and change to operand order in a piece of LDS of the wave's own, where unit u of
    // 16 bytes of row r lies at u ^ g(r): neither 16 lanes that write (four units of four
    // rows) nor 16 that read (one unit of 16 rows) meet in a bank. g(r) = 4 (r % 4) + r / 4.
    uint32_t aoff[RB]; // bytes (the caller checks that they fit)
#pragma unroll
    for (int rb = 0; rb < RB; rb++)
        aoff[rb] = ((uint32_t)min(m0 + 16 * rb + (lane >> 2), M - 1) * (uint32_t)p.lda
                           + 8 * (lane & 3))
                * 2;
    uint8_t *const stage = lds_raw + wave * w4k_wave_lds(RB, CB);
    const uint32_t wr_at = (lane >> 2) * 256 + ((((lane >> 2) & 3) << 6) | ((lane >> 4) ^ (lane & 3)) << 4);
    const uint32_t rd_at = r * 256 + (((r & 3) << 6) | ((r >> 2) ^ c) << 4);
    // (no branch on any of these in the loop: one would wait for every load before it)
    const int gs_sh = gs_shift < 0 ? 31 : gs_shift, gz_sh = gz_shift < 0 ? 31 : gz_shift;
    // from one group's scales / zero points to the next: a row of N, or one for all columns
    const uint32_t sN = scale_per_n ? N : 1, zN = !has_zp ? 0 : zp_per_n ? N : 1;
    const uint8_t *const pZP = has_zp ? (const uint8_t *)p.zps : p.B;
    const uint32_t zhalf = zp4 ? 1 : 0;
    const uint32_t zmask = !has_zp ? 0u : zp4 ? 15u : 255u;
    const uint32_t zsign = zp_signed ? (zp4 ? 8u : 128u) : 0u;
    const uint8_t *const pA = (const uint8_t *)p.A;

    // uniform base + 32-bit offset of the lane; made anew in front of each request, else the
    // compiler widens the offset once and adds 64 bits per request
    auto at = [](const uint8_t *base, uint32_t off) {
        asm volatile("" : "+v"(off));
        return base + off;
    };
    // the wave's tiles: wave, wave + 8, ..
    const int cnt = tiles > wave ? (tiles - 1 - wave) / WK_WAVES + 1 : 0;
    auto tile_of = [&](int i) { return wave + WK_WAVES * min(i, cnt - 1); };

    // scale and zero point of tile t's group, as they are stored
    auto load_q = [&](int t, int cb, uint16_t &sc, uint8_t &zp) {
        sc = *(const uint16_t *)at(
                (const uint8_t *)p.scales + (int64_t)(t >> gs_sh) * sN * 2, scol[cb] * 2);
        zp = *at(pZP, ((t >> gz_sh) * zN + zcol[cb]) >> zhalf);
    };
    v4u a[4][RB], wt[2][CB][NP];
    constexpr int NQ = FOLD ? 2 : 1; // (one group: loaded once)
    uint16_t scp[NQ][CB];
    uint8_t zpp[NQ][CB];
    auto load_w = [&](int i, auto slot) {
        constexpr int sl = decltype(slot)::value;
        const int t = tile_of(i);
#pragma unroll
        for (int cb = 0; cb < CB; cb++) {
#pragma unroll
            for (int pl = 0; pl < NP; pl++)
                wt[sl][cb][pl] = *(const v4u *)(at(Bt[cb] + (int64_t)t * TILE_BYTES, lane * 16)
                        + pl * 1024);
            if constexpr (FOLD) load_q(t, cb, scp[sl][cb], zpp[sl][cb]);
        }
    };
    auto load_a = [&](int i) {
        const uint8_t *const tile = pA + (int64_t)tile_of(i) * 256;
#pragma unroll
        for (int rb = 0; rb < RB; rb++) {
            const uint8_t *const row = at(tile, aoff[rb]);
#pragma unroll
            for (int s = 0; s < 4; s++) a[s][rb] = *(const v4u *)(row + s * 64);
        }
    };

    v4f out[RB][CB];
#pragma unroll
    for (int rb = 0; rb < RB; rb++)
#pragma unroll
        for (int cb = 0; cb < CB; cb++) out[rb][cb] = v4f {0.f, 0.f, 0.f, 0.f};
    float sc_end[CB];
#pragma unroll
    for (int cb = 0; cb < CB; cb++) sc_end[cb] = 0.f;

    auto step = [&](int i, auto slot) {
        constexpr int sl = decltype(slot)::value;
        float sc[CB], off[CB];
        uint32_t sub[CB], sub16[CB]; // f16 pairs: offset + zero point, 1024 / 16 + zero point
#pragma unroll
        for (int cb = 0; cb < CB; cb++) {
            constexpr int q = FOLD ? sl : 0;
            sc[cb] = sc_f16 ? (float)__builtin_bit_cast(_Float16, scp[q][cb])
                            : u2f((uint32_t)scp[q][cb] << 16);
            const uint32_t odd = ((tile_of(i) >> gz_sh) * zN + zcol[cb]) & zhalf;
            const uint32_t z = ((uint32_t)zpp[q][cb] >> (4 * odd)) & zmask;
            const float zp = (float)((int)(z ^ zsign) - (int)zsign);
            // (bf16, both planes in one sum: 17 * offset)
            off[cb] = (W8 && !F16 ? 17.f * OFFSET : OFFSET) + soff + zp;
            const uint32_t h = __builtin_bit_cast(uint16_t, (_Float16)off[cb]);
            sub[cb] = h | (h << 16);
            sub16[cb] = pk_sub(sub[cb], 0x63806380u); // (1024 - 64 = 960)
        }
        // (wave-private and in order: behind the reads of the tile before)
#pragma unroll
        for (int s = 0; s < 4; s++)
#pragma unroll
            for (int rb = 0; rb < RB; rb++)
                *(v4u *)(stage + rb * 4096 + (wr_at ^ (s << 6))) = a[s][rb];
        __builtin_amdgcn_sched_barrier(0x6);
        load_a(i + 1);
        __builtin_amdgcn_sched_barrier(0x6);
        v4u ops[2][RB];
        auto read_a = [&](int s) {
#pragma unroll
            for (int rb = 0; rb < RB; rb++)
                ops[s & 1][rb] = *(const v4u *)(stage + rb * 4096 + (rd_at ^ (s << 6)));
        };
        read_a(0);
        v4f P[RB][CB], S[RB];
        if constexpr (FOLD) {
#pragma unroll
            for (int rb = 0; rb < RB; rb++) {
                S[rb] = v4f {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int cb = 0; cb < CB; cb++) P[rb][cb] = v4f {0.f, 0.f, 0.f, 0.f};
            }
        }
#pragma unroll
        for (int s = 0; s < 4; s++) {
            if (s < 3) read_a(s + 1);
            const v4u *const op = ops[s & 1];
            if constexpr (!F16) {
#pragma unroll
                for (int rb = 0; rb < RB; rb++) S[rb] = mfma16<F16>(op[rb], ones, S[rb]);
            }
#pragma unroll
            for (int cb = 0; cb < CB; cb++) {
                const uint32_t d = wt[sl][cb][0][s] ^ sflip;
                v4u b, bl;
                if constexpr (W8F) {
                    const uint32_t dl = wt[sl][cb][NP - 1][s];
                    b[0] = (dl & NIB) | MAGIC | ((d << 4) & NIBH);
                    b[1] = ((dl >> 4) & NIB) | MAGIC | (d & NIBH);
                    b[2] = ((dl >> 8) & NIB) | MAGIC | ((d >> 4) & NIBH);
                    b[3] = ((dl >> 12) & NIB) | MAGIC | ((d >> 8) & NIBH);
                } else if constexpr (W8) {
                    const uint32_t dl = wt[sl][cb][NP - 1][s];
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        b[e] = ((d >> (4 * e)) & NIB) | MAGIC_HI;
                        bl[e] = ((dl >> (4 * e)) & NIB) | MAGIC;
                    }
                } else if constexpr (F16) {
                    // the odd pairs stay where they are: 1024 + 16 w, over 16
                    const uint32_t d8 = d >> 8;
                    b[0] = (d & NIB) | MAGIC;
                    b[1] = (d & NIBH) | MAGIC;
                    b[2] = (d8 & NIB) | MAGIC;
                    b[3] = (d8 & NIBH) | MAGIC;
                } else {
#pragma unroll
                    for (int e = 0; e < 4; e++) b[e] = ((d >> (4 * e)) & NIB) | MAGIC;
                }
                if constexpr (F16) {
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        b[e] = W8 || e % 2 == 0 ? pk_sub(b[e], sub[cb])
                                                : pk_sixteenth(b[e], sub16[cb]);
                }
#pragma unroll
                for (int rb = 0; rb < RB; rb++) {
                    v4f &acc = FOLD ? P[rb][cb] : out[rb][cb];
                    acc = mfma16<F16>(op[rb], b, acc);
                    if constexpr (W8 && !F16) acc = mfma16<F16>(op[rb], bl, acc);
                }
            }
            __builtin_amdgcn_sched_barrier(0x6); // (one step's operands ahead, not all)
        }
        load_w(i + 2, slot);
        __builtin_amdgcn_sched_barrier(0x6);
#pragma unroll
        for (int cb = 0; cb < CB; cb++) {
            if constexpr (FOLD) {
#pragma unroll
                for (int rb = 0; rb < RB; rb++)
#pragma unroll
                    for (int j = 0; j < 4; j++)
                        out[rb][cb][j] = __builtin_fmaf(sc[cb],
                                F16 ? P[rb][cb][j] : P[rb][cb][j] - off[cb] * S[rb][j],
                                out[rb][cb][j]);
            } else {
                sc_end[cb] = sc[cb];
            }
        }
    };
    if constexpr (!FOLD) {
#pragma unroll
        for (int cb = 0; cb < CB; cb++) load_q(0, cb, scp[0][cb], zpp[0][cb]);
    }
    const std::integral_constant<int, 0> even;
    const std::integral_constant<int, 1> odd;
    if (cnt > 0) {
        // (in the order of their first use: results return in the order of the requests)
        load_w(0, even);
        __builtin_amdgcn_sched_barrier(0);
        load_a(0);
        __builtin_amdgcn_sched_barrier(0);
        load_w(1, odd);
        __builtin_amdgcn_sched_barrier(0);
        int i = 0;
        for (; i + 2 <= cnt; i += 2) {
            step(i, even);
            step(i + 1, odd);
        }
        if (i < cnt) step(i, even);
    }

    // The waves' sums meet in LDS, in the waves' order; four columns of a row per thread.
    // MFMA output: register j of lane (r, c) is row 4 c + j, column r.
    constexpr int BM = 16 * RB, BN = 16 * CB, PITCH = BN + 4, W_LDS = w4k_wave_lds(RB, CB);
    constexpr int QUADS = BN / 4, RPP = WK_WAVES * 64 / QUADS; // rows per pass
    constexpr int PASSES = (BM + RPP - 1) / RPP;
    const int cg = tid % QUADS * 4, tr = tid / QUADS, n = nb0 * 16 + cg;
    const int nvalid = min(4, N - n);
    ep_cols_t cols; // requested before the waves meet
    epilogue_cols_load(p.ep, cols, 0, n, nvalid);
    const bool has_ss = p.ep.src_scale.ptr != nullptr;
    const float ss = has_ss ? ep_load(p.ep.src_scale, 0, 0, 0) : 1.f; // (one for all rows)
    float *const red = (float *)(lds_raw + wave * W_LDS);
#pragma unroll
    for (int rb = 0; rb < RB; rb++)
#pragma unroll
        for (int cb = 0; cb < CB; cb++)
#pragma unroll
            for (int j = 0; j < 4; j++)
                red[(16 * rb + 4 * c + j) * PITCH + 16 * cb + r]
                        = FOLD ? out[rb][cb][j] : sc_end[cb] * out[rb][cb][j];
    __syncthreads();
    const epilogue_t &epk
            = ((const gemv_params_t *)__builtin_amdgcn_kernarg_segment_ptr())->ep;
#pragma unroll
    for (int q = 0; q < PASSES; q++) {
        const int row = q * RPP + tr, m = m0 + row;
        if (row >= BM || m >= M || nvalid <= 0) continue;
        v4f v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < WK_WAVES; w++)
            v += *(const v4f *)(lds_raw + w * W_LDS + (row * PITCH + cg) * 4);
        float d[4] = {v[0], v[1], v[2], v[3]};
        epilogue_rows4(epk, cols, d, has_ss, ss, 0, m, n, nvalid);
    }
}

} // namespace

#define QMM_W4K_NAME2(n) launch_gemm_w4k_part##n
#define QMM_W4K_NAME(n) QMM_W4K_NAME2(n)
void QMM_W4K_NAME(QMM_W4K_PART)(const gemv_params_t &p, int rb, int cb, int shifts,
        int flags_m, hipStream_t stream) {
    constexpr bool F = (QMM_W4K_PART & 1) != 0, W = (QMM_W4K_PART & 2) != 0;
    const w4k_map_t map = w4k_map(p.M, p.nb16, rb, cb);
    auto go = [&](auto kern) {
        const int lds = WK_WAVES * w4k_wave_lds(rb, cb);
        if (lds > 65536) ensure_dynamic_lds((const void *)kern, lds);
        hipLaunchKernelGGL(kern, dim3((unsigned)(8 * map.share)), dim3(WK_WAVES * 64), lds,
                stream, p, shifts, flags_m);
    };
    const bool fold = w4k_fold(p);
    auto by_shape = [&](auto sgn, auto fld) {
        constexpr bool S = decltype(sgn)::value, D = decltype(fld)::value;
        if constexpr (w4k_tall(F, W, D)) {
            if (rb == 3) {
                go(gemm_w4k_kernel<F, W, S, 3, 4, D>);
                return;
            }
        }
        if (cb == 4) go(gemm_w4k_kernel<F, W, S, 2, 4, D>);
        else go(gemm_w4k_kernel<F, W, S, 2, 2, D>);
    };
    auto by_fold = [&](auto sgn) {
        if constexpr (F) {
            if (!fold) {
                by_shape(sgn, std::false_type {});
                return;
            }
        }
        by_shape(sgn, std::true_type {});
    };
    if (p.wei_signed) by_fold(std::true_type {});
    else by_fold(std::false_type {});
}

#else // the launcher

void launch_gemm_w4k_part0(const gemv_params_t &, int, int, int, int, hipStream_t);
void launch_gemm_w4k_part1(const gemv_params_t &, int, int, int, int, hipStream_t);
void launch_gemm_w4k_part2(const gemv_params_t &, int, int, int, int, hipStream_t);
void launch_gemm_w4k_part3(const gemv_params_t &, int, int, int, int, hipStream_t);

double gemm_w4f_us(const gemv_params_t &p);
double gemm_g128_us(int M, int N, int K, int kind);
int gemm_g128_rows(int M, int N, int K, int kind);

// Row and column blocks of a workgroup as 16 * rb + cb, 0: another kernel is faster. Before /
// now (us): f16 x u4 164 x 6528 x 3552 54 / 19, 64 x 4096 x 4096 20.2 / 8.3, 563 x 2048 x
// 1248 22.7 / 11.5, 269 x 9856 x 5168 82 / 53; bf16 x u4 204 x 12928 x 2176 111 / 25, 711 x
// 9088 x 3520 131 / 102; f16 x u8 148 x 12800 x 1424 83 / 19, 64 x 4096 x 14336 51 / 28; the
// other kernels stay ahead from 450 rows and 8 million weights on (727 x 4480 x 4064 64 / 65,
// bf16 684 x 9472 x 14016 252 / 381, 1324 x 13824 x 2544 192 / 220). Over 260 shapes of 17 ... 2048 rows 1.75 times as fast in
// the mean, the choice within 0.5 % of the faster kernel in the mean and 20 % at most; over 1900 further ones 8 % at
// most slower than the others (bf16 948 x 6912 x 3328 104 / 113). A round
// of workgroups (one on a CU, 32 on an XCD) costs a start, an end and the waves' K; a begun
// round costs most of a whole one. us at K = 1024 (f16 x u4, one round 32 x 32 / 32 x 64 /
// 48 x 64 results): 4.6 / 5.8 / 7.5, and 1.1 / 1.5 / 2.2 per further 1024 k.
// 9 ... 16 rows: past 256 blocks of 16 columns the decode kernel has more than one
// workgroup on a CU and stages no rows; 29 problems there 1.15 ... 2.2 times as fast here
// (u8 16 x 1280 x 4160 13.1 / 6.1, 14 x 8704 x 11712 45 / 28; u4 f16 15 x 3456 x 5408 11.7 / 7.8,
// bf16 12 x 2432 x 12432 17.5 / 9.3); with fewer it may be ahead (u4 14 x 7808 x 3440 9.9 / 11.5).
// Over 65536 columns and more, few k under 4-bit weights are the tall tiles' (qmm_gemm_g128.hip:
// bf16 10 x 128 x 95648 10.3 / 21.6, 15 x 512 x 78560 18.0 / 21.9, f16 12 x 512 x 69472 16.7 / 19.9).
int gemm_w4k_shape(const gemv_params_t &p) {
    if (p.M <= 8 || (p.M <= 16 && p.N <= 4096) || p.K % 128 != 0
            || (int64_t)p.M * p.lda * 2 >= (int64_t)1 << 32
            || (int64_t)p.kg128 * p.N >= (int64_t)1 << 31)
        return 0;
    const int kind = p.act_f16 ? G_F16 : G_BF16;
    const double other = !p.w8 && gemm_g128_rows(p.M, p.N, p.K, kind)
            ? gemm_g128_us(p.M, p.N, p.K, kind)
            : p.M <= 16 ? 1e30
                        : gemm_w4f_us(p);
    const bool tall = w4k_tall(p.act_f16, p.w8, w4k_fold(p));
    // {once, per round, per round and 1024 k}
    static const double f16[3][3] = {{1.1, 2.4, 1.09}, {0.4, 3.9, 1.54}, {-0.6, 5.9, 2.19}};
    static const double bf16[3][3] = {{2.0, 1.6, 1.29}, {1.2, 3.0, 1.76}, {0, 0, 0}};
    static const double w8[3][3] = {{2.3, 2.2, 1.25}, {1.0, 4.4, 2.06}, {0.8, 5.9, 2.37}};
    const double(*const c)[3] = p.w8 ? w8 : p.act_f16 ? f16 : bf16;
    static const int shapes[3][2] = {{2, 2}, {2, 4}, {3, 4}};
    double best = other / 1.1; // (clearly, or not)
    int pick = 0;
    const double rows = many_rows(p.M, p.K, 0.25);
    for (int i = 0; i < (tall ? 3 : 2); i++) {
        const double rounds = w4k_map(p.M, p.nb16, shapes[i][0], shapes[i][1]).share / 32.0;
        const double us = (p.w8 && !p.act_f16 ? 1.2 : 1.0)
                * (c[i][0]
                        + std::max(1.0, 0.8 * std::ceil(rounds) + 0.2 * rounds)
                                * (c[i][1] + c[i][2] * p.K / 1024) * rows);
        if (us < best) {
            best = us;
            pick = 16 * shapes[i][0] + shapes[i][1];
        }
    }
    return pick;
}

void launch_gemm_w4k(const gemv_params_t &p, int rb, int cb, int shifts, int flags_m,
        hipStream_t stream) {
    switch ((p.act_f16 ? 1 : 0) | (p.w8 ? 2 : 0)) {
        case 0: launch_gemm_w4k_part0(p, rb, cb, shifts, flags_m, stream); break;
        case 1: launch_gemm_w4k_part1(p, rb, cb, shifts, flags_m, stream); break;
        case 2: launch_gemm_w4k_part2(p, rb, cb, shifts, flags_m, stream); break;
        default: launch_gemm_w4k_part3(p, rb, cb, shifts, flags_m, stream); break;
    }
}
#endif

} // namespace qmm

#if !defined(QMM_W4K_PART)
extern "C" int qmm_gemm_w4k_shape(
        int src_dt, int weights_bits, int per_column, int64_t M, int64_t N, int64_t K) {
    using namespace qmm;
    const int64_t top = 1 << 24;
    if ((src_dt != dt_f16 && src_dt != dt_bf16) || (weights_bits != 4 && weights_bits != 8) || M < 1
            || N < 1 || K < 1 || M > top || N > top || K > top)
        return 0;
    gemv_params_t p = {};
    p.M = (int32_t)M;
    p.N = (int32_t)N;
    p.K = (int32_t)K;
    p.lda = K;
    p.kg128 = (int32_t)((K + 127) / 128);
    p.nb16 = (int32_t)((N + 15) / 16);
    p.act_f16 = src_dt == dt_f16;
    p.w8 = weights_bits == 8;
    p.gs_shift = p.gz_shift = per_column ? -1 : 0;
    return gemm_w4k_shape(p);
}
#endif
