// hip:gfx950:mfma_b8 from one row to some hundred: s8 / u8 x s8 and f8_e4m3 with K
// a multiple of 128 and no weights zero points, where tiles that walk all of K leave most of
// the chip idle (arithmetic of qmm_gemm_b8.hip: src/cpu/matmul/ref_matmul_int8.cpp:165-259).
// A workgroup owns 16 RB x 16 CB results; its eight waves cut K between them, 128 k each in
// turn, and each holds all the results: no wave waits for another before the sum at the end.
//   * Products are of 16 x 16 x 64 (s8) or 16 x 16 x 128 (fp8). The order of k inside a tile is
//     free as long as both operands agree: lane (c, r) takes the 16 bytes that
//     QMM_LAYOUT_MFMA_B8 holds for column r, fragment 2 i + c / 2, half c % 2, as operand i;
//     for fp8 operands 0 and 1 are one.
//   * Rows are requested eight lanes to 128 bytes and change to operand order in a piece of
//     LDS of the wave's own: no barrier. Weights are requested two tiles ahead.
// Bound: HBM and a start and an end of 4 us where the weights are read once (64 x 4096 x 14336
// 20.0 us, 2.9 TB/s, with 224 of 256 CUs; 16.4 with the weights in the memory-side cache), else the requests through L1: 64 x 64 results need 16
// KB per 128 k of a wave, 32 x 64 12, which is why the largest tile wins as soon as it fills
// the chip (413 x 12672 x 3584, fp8, in 16 x 64 / 32 x 64 / 64 x 64: 76 / 55 / 49 us).
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "qmm_device.hpp"
#include "qmm_kcut.hpp"
#include "qmm_hip.h"
#include "qmm_plan.hpp"

namespace qmm {
namespace {
constexpr int WK_WAVES = 8;

typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef unsigned v8u __attribute__((ext_vector_type(8)));

// Workgroup w runs on XCD w % 8; an XCD takes a run of neighbouring items, the row blocks
// of a column block one after another, so that weights are read into one L2.
struct b8k_map_t {
    int nrb, total, share;
};
__host__ __device__ inline b8k_map_t b8k_map(int M, int nb16, int rb, int cb) {
    const int nrb = (M + 16 * rb - 1) / (16 * rb), ncb = (nb16 + cb - 1) / cb;
    return {nrb, nrb * ncb, (nrb * ncb + 7) / 8};
}

// bytes of a wave: rows of a tile, later its results in rows of BN + 4 floats
constexpr int b8k_wave_lds(int rb, int cb) {
    const int results = 16 * rb * (16 * cb + 4) * 4, stage = rb * 2048;
    return results > stage ? results : stage;
}

// tiles of rows requested ahead: as many as the registers allow
constexpr int B8K_DW = 2;
constexpr int b8k_da(int rb) { return rb <= 2 ? 2 : 1; }

template <bool F8, int RB, int CB, bool NT>
__global__ void __launch_bounds__(WK_WAVES * 64, RB * CB <= 4 ? 4 : 2)
gemm_b8k_kernel(const gemm_params_t p) {
    typedef typename std::conditional<F8, v4f, v4i>::type acc_t;
    constexpr int DW = B8K_DW, DA = b8k_da(RB);
    extern __shared__ __attribute__((aligned(16))) uint8_t lds_raw[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane >> 4, r = lane & 15;
    const int M = p.M, N = p.N, tiles = p.K / 128, nb16 = (N + 15) / 16;
    const b8k_map_t map = b8k_map(M, nb16, RB, CB);
    const int item = (blockIdx.x & 7) * map.share + (blockIdx.x >> 3);
    if (item >= map.total) return;
    const int m0 = item % map.nrb * (16 * RB), nb0 = item / map.nrb * CB;

    // column blocks past the last one repeat it, rows past M the last one: never stored
    const uint8_t *Bt[CB];
#pragma unroll
    for (int cb = 0; cb < CB; cb++) {
        const int b = min(nb0 + cb, nb16 - 1);
        Bt[cb] = p.B + (int64_t)(b >> 1) * p.kb32 * 1024 + (b & 1) * 256;
    }
    const uint32_t boff = (c >> 1) * 1024 + (c & 1) * 512 + r * 16;
    // 16-byte unit u of row r lies at u ^ (r / 2) of the row's 128 bytes: neither 16 lanes
    // that write (two rows) nor 16 that read (one unit of 16 rows) meet in a bank
    uint32_t aoff[RB][2]; // bytes (the caller checks that they fit)
#pragma unroll
    for (int rb = 0; rb < RB; rb++)
#pragma unroll
        for (int h = 0; h < 2; h++)
            aoff[rb][h] = (uint32_t)min(m0 + 16 * rb + 8 * h + (lane >> 3), M - 1)
                            * (uint32_t)p.lda
                    + 16 * (lane & 7);
    uint8_t *const stage = lds_raw + wave * b8k_wave_lds(RB, CB);
    const uint32_t wr_at = (lane >> 3) * 128 + (((lane & 7) ^ (lane >> 4)) << 4);
    const uint32_t rd_at = r * 128 + ((c ^ (r >> 1)) << 4);
    const uint32_t flip = p.a_is_u8 && !p.a_preflipped ? 0x80808080u : 0u;

    // uniform base + 32-bit offset of the lane; made anew in front of each request, else the
    // compiler widens the offset once and adds 64 bits per request
    auto at = [](const void *base, uint32_t off) {
        asm volatile("" : "+v"(off));
        return (const uint8_t *)base + off;
    };
    // the wave's tiles: wave, wave + 8, ..
    const int cnt = tiles > wave ? (tiles - 1 - wave) / WK_WAVES + 1 : 0;
    auto tile_of = [&](int i) { return wave + WK_WAVES * min(i, cnt - 1); };
    // requests past the wave's last tile are made, all lanes for the same bytes (a branch
    // around them would wait for every load before it)
    auto lanes = [&](int i) { return i < cnt ? ~0u : 0u; };

    v4u a[DA][RB][2], wt[DW][CB][2];
    auto load_w = [&](int i, auto slot) {
        constexpr int sl = decltype(slot)::value;
        const int t = tile_of(i);
#pragma unroll
        for (int cb = 0; cb < CB; cb++) {
            const uint8_t *const q = at(Bt[cb] + (int64_t)t * 4096, boff & lanes(i));
#pragma unroll
            for (int h = 0; h < 2; h++)
                if constexpr (NT)
                    wt[sl][cb][h] = __builtin_nontemporal_load((const v4u *)(q + h * 2048));
                else
                    wt[sl][cb][h] = *(const v4u *)(q + h * 2048);
        }
    };
    auto load_a = [&](int i, auto slot) {
        constexpr int sl = decltype(slot)::value;
        const int t = tile_of(i);
#pragma unroll
        for (int rb = 0; rb < RB; rb++)
#pragma unroll
            for (int h = 0; h < 2; h++)
                a[sl][rb][h] = *(const v4u *)at(p.A + (int64_t)t * 128, aoff[rb][h] & lanes(i));
    };

    acc_t out[RB][CB];
#pragma unroll
    for (int rb = 0; rb < RB; rb++)
#pragma unroll
        for (int cb = 0; cb < CB; cb++) out[rb][cb] = acc_t {0, 0, 0, 0};

    auto step = [&](int i, auto j_tag) {
        constexpr int j = decltype(j_tag)::value;
        constexpr std::integral_constant<int, j % DW> ws;
        constexpr std::integral_constant<int, j % DA> as;
        // (wave-private and in order: behind the reads of the tile before)
#pragma unroll
        for (int rb = 0; rb < RB; rb++)
#pragma unroll
            for (int h = 0; h < 2; h++)
                *(v4u *)(stage + rb * 2048 + h * 1024 + (wr_at ^ (h << 6)))
                        = F8 ? a[as][rb][h] : a[as][rb][h] ^ flip;
        __builtin_amdgcn_sched_barrier(0x6);
        load_a(i + DA, as);
        __builtin_amdgcn_sched_barrier(0x6);
        v4u ops[RB][2];
#pragma unroll
        for (int rb = 0; rb < RB; rb++)
#pragma unroll
            for (int h = 0; h < 2; h++)
                ops[rb][h] = *(const v4u *)(stage + rb * 2048 + (rd_at ^ (h << 6)));
#pragma unroll
        for (int cb = 0; cb < CB; cb++) {
            const v4u *const w = wt[ws][cb];
            if constexpr (F8) {
                const v8u b = __builtin_shufflevector(w[0], w[1], 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
                for (int rb = 0; rb < RB; rb++) {
                    const v8u o = __builtin_shufflevector(
                            ops[rb][0], ops[rb][1], 0, 1, 2, 3, 4, 5, 6, 7);
                    out[rb][cb] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
                            __builtin_bit_cast(v8i, o), __builtin_bit_cast(v8i, b), out[rb][cb],
                            0, 0, 0, 0, 0, 0);
                }
            } else {
#pragma unroll
                for (int h = 0; h < 2; h++)
#pragma unroll
                    for (int rb = 0; rb < RB; rb++)
                        out[rb][cb] = __builtin_amdgcn_mfma_i32_16x16x64_i8(
                                __builtin_bit_cast(v4i, ops[rb][h]),
                                __builtin_bit_cast(v4i, w[h]), out[rb][cb], 0, 0, 0);
            }
        }
        __builtin_amdgcn_sched_barrier(0x6);
        load_w(i + DW, ws);
        __builtin_amdgcn_sched_barrier(0x6);
    };
    if (cnt > 0) {
        // (in the order of their first use: results return in the order of the requests)
        auto first = [&](auto j_tag) {
            constexpr int j = decltype(j_tag)::value;
            load_w(j, j_tag);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (j < DA) load_a(j, j_tag);
            __builtin_amdgcn_sched_barrier(0);
        };
        first(std::integral_constant<int, 0> {});
        first(std::integral_constant<int, 1> {});
        int i = 0;
        for (; i + 2 <= cnt; i += 2) {
            step(i, std::integral_constant<int, 0> {});
            step(i + 1, std::integral_constant<int, 1> {});
        }
        if (i < cnt) step(i, std::integral_constant<int, 0> {});
    }

    // The waves' sums meet in LDS, in the waves' order; four columns of a row per thread.
    // MFMA output: register j of lane (c, r) is row 4 c + j, column r.
    constexpr int BM = 16 * RB, BN = 16 * CB, PITCH = BN + 4, W_LDS = b8k_wave_lds(RB, CB);
    constexpr int QUADS = BN / 4, RPP = WK_WAVES * 64 / QUADS; // rows per pass
    constexpr int PASSES = (BM + RPP - 1) / RPP;
    const int cg = tid % QUADS * 4, tr = tid / QUADS, n = nb0 * 16 + cg;
    const int nvalid = min(4, N - n);
    ep_cols_t cols; // requested before the waves meet
    epilogue_cols_load(p.ep, cols, 0, n, nvalid);
    const bool has_ss = p.ep.src_scale.ptr != nullptr;
    float ss[PASSES];
#pragma unroll
    for (int q = 0; q < PASSES; q++)
        ss[q] = has_ss ? ep_load(p.ep.src_scale, 0, min(m0 + q * RPP + tr, M - 1), 0) : 1.f;
    int comp = p.a_is_u8 ? 128 : 0;
    if (p.src_zp) comp -= load_int(p.src_zp_dt, p.src_zp, 0);
    v4u cs = {0, 0, 0, 0};
    if (!F8 && comp != 0 && p.colsum) {
#pragma unroll
        for (int e = 0; e < 4; e++)
            if (e < nvalid) cs[e] = (uint32_t)comp * (uint32_t)p.colsum[n + e];
    }
    uint32_t *const red = (uint32_t *)stage;
#pragma unroll
    for (int rb = 0; rb < RB; rb++)
#pragma unroll
        for (int cb = 0; cb < CB; cb++) {
            const v4u v = __builtin_bit_cast(v4u, out[rb][cb]);
#pragma unroll
            for (int j = 0; j < 4; j++)
                red[(16 * rb + 4 * c + j) * PITCH + 16 * cb + r] = v[j];
        }
    __syncthreads();
    const epilogue_t &epk
            = ((const gemm_params_t *)__builtin_amdgcn_kernarg_segment_ptr())->ep;
#pragma unroll
    for (int q = 0; q < PASSES; q++) {
        const int row = q * RPP + tr, m = m0 + row;
        if (row >= BM || m >= M || nvalid <= 0) continue;
        float d[4];
        v4u s = cs;
        v4f f = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < WK_WAVES; w++) {
            const v4u x = *(const v4u *)(lds_raw + w * W_LDS + (row * PITCH + cg) * 4);
            if constexpr (F8) f += __builtin_bit_cast(v4f, x);
            else s += x; // s32 arithmetic that wraps as the reference's int accumulation
        }
#pragma unroll
        for (int e = 0; e < 4; e++) d[e] = F8 ? f[e] : (float)(int32_t)s[e];
        epilogue_rows4(epk, cols, d, has_ss, ss[q], 0, m, n, nvalid);
    }
}

} // namespace

int gemm_b8_tile(const gemm_params_t &p, bool f8, bool post_ops);
bool gemm_b8x_two_per_cu(const gemm_params_t &p, bool f8);

// us of the kernels that gemm_b8_tile chooses between (4900 problems of 128 ... 16384 k, 33 ...
// 2500 rows and 16 ... 131072 columns, weights in and out of the caches, 5 ... 12 % rms): {rows,
// columns and workgroups of a round, once, per round, per round and 1024 k, a begun round's share;
// what workgroups alone on their CUs save once and per 1024 k; columns off a multiple of
// `align`, per round; per MB of results}. The last three are the kernels of 256 rows, which take half as
// long over few k where columns are aligned (s8 2398 x 128 x 1152 9.8 us, 2423 x 128 x 1264 16.3).
static double b8_other_us(const gemm_params_t &p, bool f8, bool post_ops) {
    static const struct {
        int rows, cols, slots;
        double once, start, k1024, begun, alone, alone_k1024;
        int align;
        double tail, mb;
    } kernels[] = {
            {32, 32, 512, 2.12, 3.84, 2.12, 0.31, 0, 1.02, 1, 0, 0},
            {32, 32, 512, 1.86, 3.48, 2.18, 0.29, 0, 1.17, 1, 0, 0},
            {64, 64, 256, 3.7, 4.0, 3.1, 0.5, 0, 0, 1, 0, 0},
            {64, 64, 256, 2.8, 3.5, 3.5, 0.5, 0, 0, 1, 0, 0},
            {128, 128, 256, 16.1, 1.46, 4.72, 0.62, 0, -0.77, 1, 0, 0},
            {128, 128, 256, 13.6, 2.0, 5.1, 0.5, 0, 0, 1, 0, 0},
            {256, 256, 256, 31.0, -8.6, 12.3, 0.3, 11.6, 2.5, 128, 6.7, 0.89},
            {256, 128, 512, -3.8, 12.4, 12.6, 0.31, 0, 5.4, 64, 5.2, 0.13},
            {256, 256, 256, 10.8, 11.9, 12.1, 0.6, 4.3, 0, 64, 0, 0.13},
    };
    gemm_params_t q = p;
    const int64_t tiles256 = (((int64_t)p.M + 255) / 256) * (((int64_t)p.N + 255) / 256);
    double flip = 0;
    if (p.a_is_u8 && p.K > 256 && p.K % 64 == 0 && tiles256 >= 192
            && !gemm_b8x_two_per_cu(p, f8)) { // (rewritten as s8 by a pre-pass)
        q.a_preflipped = 1;
        flip = 3 + (double)p.M * p.K / 2e6;
    }
    const int tile = gemm_b8_tile(q, f8, post_ops);
    const auto &t = kernels[tile == 32 ? !f8 : tile == 64 ? 2 + !f8 : tile == 128 ? 4 + !f8
                    : f8                                                          ? 6
                    : gemm_b8x_two_per_cu(q, f8)                                  ? 7
                                                                                  : 8];
    const int64_t wgs = (((int64_t)p.M + t.rows - 1) / t.rows) * ((p.N + t.cols - 1) / t.cols);
    const double k = p.K / 1024.0, x = (double)wgs / t.slots;
    const double rounds = std::max(1.0, t.begun * std::ceil(x) + (1 - t.begun) * x);
    // (three rows of tiles and more find their weights in L2: 2055 x 8832 x 1024 59 us)
    const double alone_k1024 = t.alone_k1024 + (t.rows == 256 && t.cols == 128 && p.M > 512 ? 0.5 : 0.0);
    const double mb = (double)p.M * p.N * (p.ep.dst.dt == dt_f32 || p.ep.dst.dt == dt_s32 ? 4e-6 : 2e-6);
    return t.once + flip + t.mb * mb
            + rounds * (t.start + t.k1024 * k + (p.N % t.align ? t.tail : 0.0))
            - (wgs <= 256 ? t.alone + alone_k1024 * k : 0.0);
}

// Row and column blocks of a workgroup as 16 * rb + cb, 0: another kernel is faster. Before /
// now (us, weights in the memory-side cache): s8 64 x 4096 x 14336 21.3 / 16.4, 16 x 12288 x 2048 14.8 /
// 10.3, 195 x 6912 x 3296 27.6 / 16.0, 256 x 4096 x 4096 19.0 / 12.5, u8 256 x 1024 x 1024 5.5 / 4.7; fp8
// 413 x 12672 x 3584 73 / 46, 350 x 8704 x 1472 30 / 14.7; weights from HBM 24.1 / 20.0, 15.7 / 15.3, 28.7 /
// 18.4, 19.7 / 14.9, 6.4 / 5.9; 84 / 54, 30 / 17.5. The tiles that walk all of K stay ahead
// from some hundred rows on (fp8 967 x 8576 x 4064 66 / 83, s8 894 x 2944 x 12624 61 / 108), over few k
// and many aligned columns from 33 rows on (fp8 65 x 640 x 62464 21 / 50, 1102 x 640 x 4608 20.6 / 45,
// 40 x 384 x 56928 21 / 27; s8 74 x 6016 x 49408 84 / 121) and for u8 rows where these are rewritten once
// for many tiles (1934 x 14336 x 4112 184 / 284); and
// where the streaming kernel requests all of its K at once: up to 4 rows of 4096 k (from HBM, 1 x
// 4096 x 4832 8.2 / 8.5, 1 x 4096 x 14336 14.2 / 15.1; 3072 k and less, or very wide weights, are the same or
// faster here: 2 x 2944 x 4192 7.6 / 7.6, 2 x 3200 x 65072 42 / 36, 1 x 12032 x 9248 27.6 / 24.5) and up to 32
// of 2048 (25 x 1536 x 21808 12.6 / 13.6, 20 x 1664 x 85952 40 / 44). Over 640 problems
// of 1 ... 2500 rows 1.25 times as fast in the mean; over 5300 further ones 1.17 times, and up to 17 %
// slower than the kernels before (fp8 82 x 15232 x 35968 164 / 191; u8 165 x 128 x 10208 12.0 / 13.4). A round of workgroups costs a start, an end and the waves' K; a CU holds one,
// or (up to 16 x 64 or 32 x 32 results) two. The caller checks that there is one matrix and no
// weights zero point.
int gemm_b8k_shape(const gemm_params_t &p, bool f8, bool post_ops) {
    if (p.K % 128 != 0 || (int64_t)p.M * p.lda >= (int64_t)1 << 32) return 0;
    // K that the streaming kernel requests all at once: up to 4096 with 4 rows, 2048 with 32
    if (p.M <= 4 && p.K > 3072 && p.K <= 4096 && p.N > 4096 && p.N <= 16384) return 0;
    if (p.M > 16 && p.M <= 32 && p.K > 1408 && p.K <= 2048 && p.N > 16384) return 0;
    // {.., once, per round, per round and 1024 k, a begun round's share, the second on a CU}
    static const struct {
        int rb, cb;
        double once, start, k1024, begun, second;
    } shapes[] = {{1, 2, 3.83, 0.95, 0.54, 1.0, 0.85}, {1, 4, 3.13, 1.86, 0.97, 1.0, 0.65},
            {2, 2, 3.44, 1.45, 0.71, 0.97, 1.0}, {2, 4, 1.35, 3.94, 1.16, 0.91, 0},
            {4, 2, 0.97, 3.75, 1.13, 0.92, 0}, {4, 4, -0.27, 6.84, 1.57, 0.92, 0},
            // (one row of workgroups, few k: the rounds overlap; 56 x 384 x 126800 in 32 x 32 73 us, so 60)
            {4, 4, 2.2, 4.6, 1.57, 0.92, 0}};
    double best = 1e30;
    int pick = 0;
    const bool short_k = p.M <= 64 && p.K <= 1024 && !f8;
    const double rows = many_rows(p.M, p.K, f8 ? 0.25 : 0.1);
    for (const auto &s : shapes) {
        if (s.rb * s.cb == 16 && (s.once > 0) != short_k) continue;
        // workgroups on a CU (32 on an XCD)
        const double wgs = b8k_map(p.M, (p.N + 15) / 16, s.rb, s.cb).share / 32.0;
        // (17 ... 32 rows bound by HBM: 32 x 32 results twice on a CU, 23 x 3584 x 124496 99.5 / 86)
        if (s.rb == 2 && s.cb == 4 && p.M <= 32 && wgs > 2) continue;
        double rounds = s.begun * std::ceil(wgs) + (1 - s.begun) * wgs;
        if (s.second > 0) { // pairs
            const double full = std::floor(wgs / 2), rest = wgs - 2 * full;
            rounds = full * (1 + s.second)
                    + (rest <= 0          ? 0.0
                                    : rest <= 1 ? 1.0
                                                : 1 + s.second * (s.begun + (1 - s.begun) * (rest - 1)));
        }
        const double us = s.once + std::max(1.0, rounds) * (s.start + s.k1024 * p.K / 1024) * rows;
        if (us < best) {
            best = us;
            pick = 16 * s.rb + s.cb;
        }
    }
    if (p.M <= 32 || (p.M <= 64 && (!f8 || gemm_b8_tile(p, f8, post_ops) == 32))) return pick;
    // (64 x 64 fp8 results of few k take longer than priced: 104 x 6352 x 128 8.4 / 9.0)
    if (f8 && p.K <= 512 && pick == 0x44) best += 1.6;
    // (clearly, or not; very tall problems are off what was measured: s8 16384 x 1024 x 128
    // 13.7 / 16.9, 16384 x 4096 x 64 28.7 / 22.5; fp8 up to 64 rows in tiles is priced too high)
    const double margin = p.M > 2500 ? 1.3 : p.M > 64 ? 1.05 : 1.25;
    return best < b8_other_us(p, f8, post_ops) / margin ? pick : 0;
}

void launch_gemm_b8k(const gemm_params_t &p, bool f8, int shape, hipStream_t stream) {
    const int rb = shape / 16, cb = shape % 16;
    const b8k_map_t map = b8k_map(p.M, (p.N + 15) / 16, rb, cb);
    auto go = [&](auto kern) {
        const int lds = WK_WAVES * b8k_wave_lds(rb, cb);
        if (lds > 65536) ensure_dynamic_lds((const void *)kern, lds);
        hipLaunchKernelGGL(kern, dim3((unsigned)(8 * map.share)), dim3(WK_WAVES * 64), lds,
                stream, p);
    };
    auto by_shape = [&](auto f, auto n) {
        constexpr bool F = decltype(f)::value, NT = decltype(n)::value;
        switch (shape) {
            case 0x12: go(gemm_b8k_kernel<F, 1, 2, NT>); break;
            case 0x14: go(gemm_b8k_kernel<F, 1, 4, NT>); break;
            case 0x22: go(gemm_b8k_kernel<F, 2, 2, NT>); break;
            case 0x24: go(gemm_b8k_kernel<F, 2, 4, NT>); break;
            case 0x42: go(gemm_b8k_kernel<F, 4, 2, NT>); break;
            default: go(gemm_b8k_kernel<F, 4, 4, NT>); break;
        }
    };
    // Weights that are read once go past the caches from 128 MB on, where not even two of them fit
    // the 256 MB memory-side cache. us, through / past the caches, weights from HBM: 64 x 8192 x 28672
    // 59.5 / 57.2, 64 x 4096 x 14336 20.0 / 19.5, 4 x 2048 x 13000 9.8 / 9.8; weights in that cache: 44.6 /
    // 54.4, 16.4 / 17.6, 8.1 / 9.1. Over 640 problems from HBM 0 % are won below 30 MB, 2 to 3 % from 40 to
    // 100, 4 from 100 to 200 and 7 from there; what is in the cache loses 8 ... 14 %.
    const bool nt = map.nrb == 1 && (int64_t)p.K * p.N >= (int64_t)128 << 20;
    auto by_nt = [&](auto f) {
        if (nt) by_shape(f, std::true_type {});
        else by_shape(f, std::false_type {});
    };
    if (f8) by_nt(std::true_type {});
    else by_nt(std::false_type {});
}

} // namespace qmm

extern "C" int qmm_gemm_b8k_shape(
        int src_dt, int64_t M, int64_t N, int64_t K, int post_ops) {
    using namespace qmm;
    const int64_t top = 1 << 24;
    const bool f8 = src_dt == dt_f8_e4m3;
    if ((!f8 && src_dt != dt_s8 && src_dt != dt_u8) || M < 1 || N < 1 || K < 128 || K % 128 != 0
            || M > top || N > top || K > top)
        return 0;
    gemm_params_t p = {};
    p.M = (int32_t)M;
    p.N = (int32_t)N;
    p.K = (int32_t)K;
    p.lda = K;
    p.batch = 1;
    p.kb32 = (int32_t)(K / 32);
    p.a_is_u8 = src_dt == dt_u8;
    return gemm_b8k_shape(p, f8, post_ops);
}
