// hip:gfx950:mfma_w4a8 from one row to some hundred: s8 activations [M,K] x s4 weights of
// QMM_LAYOUT_MFMA_W4K64, 16-bit scales per row / column and 128 k, no zero points (the
// arithmetic of qmm_gemm_w4a8.hip: an s32 sum per group, times the row's and the column's
// scale, added in f32). A workgroup owns 16 RB x 16 CB results; its eight waves cut K
// between them, a group each in turn, and each holds all the results: no wave waits for
// another before the sum at the end, and there is no pre-pass over the scales.
//   * Products are of 16 x 16 x 64. The order of k inside a group is free as long as both
//     operands agree: lane (c, r) takes the 16 bytes that the packed layout holds for
//     column r, tile c / 2 of the group, half c % 2, and with them the k 64 (c / 2) +
//     16 (c % 2) + 32 i ... + 15 as operand i. One 16-byte load per 16 columns and group.
//   * Rows are requested eight lanes to the 128 bytes of a group (DA groups ahead), row
//     scales one lane a row, and both change to operand order in a piece of LDS of the
//     wave's own: no barrier. Weights and their scales are requested DW groups ahead.
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

// Workgroup w runs on XCD w % 8; an XCD takes a run of neighbouring items, the row blocks
// of a column block one after another, so that weights are read into one L2.
struct w4a8k_map_t {
    int nrb, total, share;
};
__host__ __device__ inline w4a8k_map_t w4a8k_map(int M, int nb16, int rb, int cb) {
    const int nrb = (M + 16 * rb - 1) / (16 * rb), ncb = (nb16 + cb - 1) / cb;
    return {nrb, nrb * ncb, (nrb * ncb + 7) / 8};
}

// bytes of a wave: rows and row scales of a group, later its results in rows of BN + 4 floats
constexpr int w4a8k_wave_lds(int rb, int cb) {
    const int results = 16 * rb * (16 * cb + 4) * 4, stage = rb * (2048 + 64);
    return results > stage ? results : stage;
}

// groups of rows requested ahead: as many as the registers allow
constexpr int W4A8K_DW = 2;
constexpr int w4a8k_da(int rb) { return rb <= 2 ? 2 : 1; }

template <int RB, int CB>
__global__ void __launch_bounds__(WK_WAVES * 64, RB * CB <= 4 ? 4 : 2)
gemm_w4a8k_kernel(const g128_params_t p) {
    constexpr int DW = W4A8K_DW, DA = w4a8k_da(RB);
    extern __shared__ __attribute__((aligned(16))) uint8_t lds_raw[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane >> 4, r = lane & 15;
    const int M = p.M, N = p.N, groups = p.ng, nb16 = (N + 15) / 16;
    const w4a8k_map_t map = w4a8k_map(M, nb16, RB, CB);
    const int item = (blockIdx.x & 7) * map.share + (blockIdx.x >> 3);
    if (item >= map.total) return;
    const int m0 = item % map.nrb * (16 * RB), nb0 = item / map.nrb * CB;

    // column blocks past the last one repeat it, rows past M the last one: never stored
    const uint8_t *Bt[CB];
    uint32_t scol[CB];
#pragma unroll
    for (int cb = 0; cb < CB; cb++) {
        const int b = min(nb0 + cb, nb16 - 1);
        Bt[cb] = p.B + (int64_t)(b >> 1) * groups * 2048 + (b & 1) * 256;
        scol[cb] = (uint32_t)(min((nb0 + cb) * 16 + r, N - 1) * p.sw_sn) * 2;
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
    const uint32_t soff = (uint32_t)(min(m0 + min(lane, 16 * RB - 1), M - 1) * p.ss_sm) * 2;
    uint8_t *const stage = lds_raw + wave * w4a8k_wave_lds(RB, CB);
    float *const stage_s = (float *)(stage + RB * 2048);
    const uint32_t wr_at = (lane >> 3) * 128 + (((lane & 7) ^ (lane >> 4)) << 4);
    const uint32_t rd_at = r * 128 + (((4 * (c >> 1) + (c & 1)) ^ (r >> 1)) << 4);

    // uniform base + 32-bit offset of the lane; made anew in front of each request, else the
    // compiler widens the offset once and adds 64 bits per request
    auto at = [](const void *base, uint32_t off) {
        asm volatile("" : "+v"(off));
        return (const uint8_t *)base + off;
    };
    // the wave's groups: wave, wave + 8, ..
    const int cnt = groups > wave ? (groups - 1 - wave) / WK_WAVES + 1 : 0;
    auto group_of = [&](int i) { return wave + WK_WAVES * min(i, cnt - 1); };

    v4u a[DA][RB][2], wt[DW][CB];
    uint16_t ssr[DA], swr[DW][CB];
    auto load_w = [&](int i, auto slot) {
        constexpr int sl = decltype(slot)::value;
        const int t = group_of(i);
#pragma unroll
        for (int cb = 0; cb < CB; cb++) {
            wt[sl][cb] = *(const v4u *)at(Bt[cb] + (int64_t)t * 2048, boff);
            swr[sl][cb] = *(const uint16_t *)at(
                    (const uint8_t *)p.scales + (int64_t)t * p.sw_sk * 2, scol[cb]);
        }
    };
    auto load_a = [&](int i, auto slot) {
        constexpr int sl = decltype(slot)::value;
        const int t = group_of(i);
#pragma unroll
        for (int rb = 0; rb < RB; rb++)
#pragma unroll
            for (int h = 0; h < 2; h++)
                a[sl][rb][h] = *(const v4u *)at(p.A + (int64_t)t * 128, aoff[rb][h]);
        ssr[sl] = *(const uint16_t *)at(
                (const uint8_t *)p.ss + (int64_t)t * p.ss_sk * 2, soff);
    };
    auto scale = [](bool f16, uint16_t s) {
        return f16 ? (float)__builtin_bit_cast(_Float16, s) : u2f((uint32_t)s << 16);
    };

    v4f out[RB][CB];
#pragma unroll
    for (int rb = 0; rb < RB; rb++)
#pragma unroll
        for (int cb = 0; cb < CB; cb++) out[rb][cb] = v4f {0.f, 0.f, 0.f, 0.f};

    auto step = [&](int i, auto j_tag) {
        constexpr int j = decltype(j_tag)::value;
        constexpr std::integral_constant<int, j % DW> ws;
        constexpr std::integral_constant<int, j % DA> as;
        // (wave-private and in order: behind the reads of the group before)
#pragma unroll
        for (int rb = 0; rb < RB; rb++)
#pragma unroll
            for (int h = 0; h < 2; h++)
                *(v4u *)(stage + rb * 2048 + h * 1024 + (wr_at ^ (h << 6)))
                        = a[as][rb][h];
        if (lane < 16 * RB) stage_s[lane] = scale(p.ss_f16, ssr[as]);
        __builtin_amdgcn_sched_barrier(0x6);
        load_a(i + DA, as);
        __builtin_amdgcn_sched_barrier(0x6);
        v4i ops[RB][2];
        v4f ss[RB];
#pragma unroll
        for (int rb = 0; rb < RB; rb++) {
#pragma unroll
            for (int h = 0; h < 2; h++)
                ops[rb][h] = *(const v4i *)(stage + rb * 2048 + (rd_at ^ (h << 5)));
            ss[rb] = *(const v4f *)(stage_s + 16 * rb + 4 * c);
        }
#pragma unroll
        for (int cb = 0; cb < CB; cb++) {
            const v4u w = wt[ws][cb];
            // nibbles as bytes 16 w: the factor leaves with the column's scale
            v4i b[2];
#pragma unroll
            for (int h = 0; h < 2; h++)
                b[h] = v4i {(int)((w[2 * h] << 4) & 0xF0F0F0F0u), (int)(w[2 * h] & 0xF0F0F0F0u),
                        (int)((w[2 * h + 1] << 4) & 0xF0F0F0F0u),
                        (int)(w[2 * h + 1] & 0xF0F0F0F0u)};
            const float sw = scale(p.sw_f16, swr[ws][cb]) * 0.0625f;
            v4i P[RB];
#pragma unroll
            for (int rb = 0; rb < RB; rb++)
                P[rb] = __builtin_amdgcn_mfma_i32_16x16x64_i8(
                        ops[rb][0], b[0], v4i {0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
            for (int rb = 0; rb < RB; rb++)
                P[rb] = __builtin_amdgcn_mfma_i32_16x16x64_i8(ops[rb][1], b[1], P[rb], 0, 0, 0);
#pragma unroll
            for (int rb = 0; rb < RB; rb++)
#pragma unroll
                for (int e = 0; e < 4; e++)
                    out[rb][cb][e] = __builtin_fmaf(
                            (float)P[rb][e] * ss[rb][e], sw, out[rb][cb][e]);
            if constexpr (RB > 2) __builtin_amdgcn_sched_barrier(0x6); // (a column's operands at a time)
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
    constexpr int BM = 16 * RB, BN = 16 * CB, PITCH = BN + 4, W_LDS = w4a8k_wave_lds(RB, CB);
    constexpr int QUADS = BN / 4, RPP = WK_WAVES * 64 / QUADS; // rows per pass
    constexpr int PASSES = (BM + RPP - 1) / RPP;
    const int cg = tid % QUADS * 4, tr = tid / QUADS, n = nb0 * 16 + cg;
    const int nvalid = min(4, N - n);
    ep_cols_t cols; // requested before the waves meet
    epilogue_cols_load(p.ep, cols, 0, n, nvalid);
    const bool has_ss = p.ep.src_scale.ptr != nullptr;
    const float ss = has_ss ? ep_load(p.ep.src_scale, 0, 0, 0) : 1.f;
    const bool fast = p.ep.fast != EP_FAST_NONE && !p.ep.fast_ext;
    float *const red = (float *)stage;
#pragma unroll
    for (int rb = 0; rb < RB; rb++)
#pragma unroll
        for (int cb = 0; cb < CB; cb++)
#pragma unroll
            for (int j = 0; j < 4; j++)
                red[(16 * rb + 4 * c + j) * PITCH + 16 * cb + r] = out[rb][cb][j];
    __syncthreads();
    const epilogue_t &epk
            = ((const g128_params_t *)__builtin_amdgcn_kernarg_segment_ptr())->ep;
#pragma unroll
    for (int q = 0; q < PASSES; q++) {
        const int row = q * RPP + tr, m = m0 + row;
        if (row >= BM || m >= M || nvalid <= 0) continue;
        v4f v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < WK_WAVES; w++)
            v += *(const v4f *)(lds_raw + w * W_LDS + (row * PITCH + cg) * 4);
        float d[4] = {v[0], v[1], v[2], v[3]};
        if (fast)
            epilogue_fast4(p.ep, d, has_ss, ss, cols.has_ws, cols.ws, 0, m, n, nvalid);
        else
            epilogue_rows4(epk, cols, d, has_ss, ss, 0, m, n, nvalid);
    }
}

} // namespace

int gemm_g128_rows(int M, int N, int K, int kind);
double gemm_g128_us(int M, int N, int K, int kind);

// us of the tiled kernel of qmm_gemm_w4a8.hip and its pre-pass, from 65 rows to where
// gemm_g128_rows takes over (194 problems, within 8 %): two of its workgroups on a CU
static double w4a8_tiled_us(int M, int N, int K) {
    const int64_t big = (int64_t)((M + 127) / 128) * ((N + 127) / 128);
    const int64_t mid = (int64_t)((M + 63) / 64) * ((N + 127) / 128);
    const int64_t tiles = big >= 256 ? big : mid;
    const double one = 5.6 + 6.85 * K / 1024;
    return 3.9 - 0.34 * K / 1024 + one * (tiles <= 256 ? 1.0 : 1.24 * (double)((tiles + 511) / 512));
}

// Row and column blocks of a workgroup as 16 * rb + cb, 0: another kernel is faster. The other
// kernels / this one (us), weights from HBM: 1 x 4096 x 14336 10.5 / 10.3, 64 x 4096 x 14336
// 23.6 / 19.7, 8 x 4096 x 4096 17.2 / 6.7, 1 x 13312 x 1312 11.5 / 10.3; in the caches: 9.3 /
// 8.5, 22.8 / 16.3, 16.1 / 5.7, 10.4 / 8.7, 128 x 12288 x 2048 85 / 12.9, 435 x 5376 x 3888
// 43 / 31, 1941 x 1024 x 1072 18.8 / 18.0; the tall tiles of qmm_gemm_g128.hip stay ahead from some 200 rows and 15 million
// weights on (256 x 4096 x 14336 37 / 50, 1000 x 4096 x 4096 37 / 58, 1267 x 14336 x 2768 109 / 129). Up to 64 rows no
// problem but the one below was faster without. Over 1785 problems of 1 ... 4096 rows, HBM and
// caches, the choice is 1.74 times as fast as the other kernels in the mean and up to 5 % slower
// (17 ... 32 rows of few k over some 20000 columns up to 12 %: 17 x 640 x 22400 7.8 / 8.7). A round of workgroups costs a start, an end and the waves' K; a CU holds one, or (16
// rows) two, which take about twice as long as one.
int gemm_w4a8k_shape(const g128_params_t &p) {
    // 32-bit offsets of rows, row scales and column scales
    if ((int64_t)p.M * p.lda >= (int64_t)1 << 32 || (int64_t)p.M * p.ss_sm >= (int64_t)1 << 31
            || (int64_t)p.N * p.sw_sn >= (int64_t)1 << 31)
        return 0;
    const int K = p.ng * 128;
    // (the single-token kernel reads past the caches: 1 x 4096 x 128256 49 / 54, 4 x 4096 x
    // 65536 28.7 / 31 us)
    if (p.M <= 4 && (int64_t)K * p.N >= (int64_t)128 << 20) return 0;
    double best = 1e30;
    if (p.M > 64)
        best = (gemm_g128_rows(p.M, p.N, K, G_S8) ? gemm_g128_us(p.M, p.N, K, G_S8)
                                                  : w4a8_tiled_us(p.M, p.N, K))
                / 1.05; // (clearly, or not)
    // {once, per round, per round and 1024 k, a begun round's share of a whole one}
    static const struct {
        int rb, cb;
        double once, start, k1024, begun;
    } shapes[] = {{1, 2, 2.79, 0.98, 0.44, 0.79}, {1, 4, 3.17, 1.17, 0.68, 0.95},
            {2, 4, 1.49, 3.14, 1.03, 0.99}, {3, 4, 1.03, 4.14, 1.33, 0.94}};
    int pick = 0;
    const double rows = many_rows(p.M, K, 0.25);
    for (const auto &s : shapes) {
        // workgroups on a CU (32 on an XCD)
        const double wgs = w4a8k_map(p.M, (p.N + 15) / 16, s.rb, s.cb).share / 32.0;
        double rounds;
        if (s.rb == 1) { // pairs
            const double pair = s.cb == 2 ? 2.02 : 1.9, full = std::floor(wgs / 2);
            const double rest = wgs - 2 * full;
            rounds = full * pair
                    + (rest <= 0      ? 0.0
                              : rest <= 1 ? 1.0
                                          : 1 + (pair - 1) * (s.begun + (1 - s.begun) * (rest - 1)));
        } else {
            rounds = s.begun * std::ceil(wgs) + (1 - s.begun) * wgs;
        }
        const double us
                = s.once + std::max(1.0, rounds) * (s.start + s.k1024 * K / 1024) * rows;
        if (us < best) {
            best = us;
            pick = 16 * s.rb + s.cb;
        }
    }
    return pick;
}

void launch_gemm_w4a8k(const g128_params_t &p, int shape, hipStream_t stream) {
    const int rb = shape / 16, cb = shape % 16;
    const w4a8k_map_t map = w4a8k_map(p.M, (p.N + 15) / 16, rb, cb);
    auto go = [&](auto kern) {
        const int lds = WK_WAVES * w4a8k_wave_lds(rb, cb);
        if (lds > 65536) ensure_dynamic_lds((const void *)kern, lds);
        hipLaunchKernelGGL(kern, dim3((unsigned)(8 * map.share)), dim3(WK_WAVES * 64), lds,
                stream, p);
    };
    // (loads past the caches gain nothing from HBM and lose where weights are in the memory-side
    // cache, us, so / past them: 1 x 4096 x 28672 15.6 / 15.9 and 12.6 / 13.9, 16 x 2048 x 128256
    // 39.0 / 43.8 and 27.2 / 39.4)
    switch (shape) {
        case 0x12: go(gemm_w4a8k_kernel<1, 2>); break;
        case 0x14: go(gemm_w4a8k_kernel<1, 4>); break;
        case 0x24: go(gemm_w4a8k_kernel<2, 4>); break;
        default: go(gemm_w4a8k_kernel<3, 4>); break;
    }
}

} // namespace qmm

extern "C" int qmm_gemm_w4a8k_shape(int64_t M, int64_t N, int64_t K) {
    using namespace qmm;
    const int64_t top = 1 << 24;
    if (M < 1 || N < 1 || K < 128 || K % 128 != 0 || M > top || N > top || K > top) return 0;
    g128_params_t p = {};
    p.M = (int32_t)M;
    p.N = (int32_t)N;
    p.ng = (int32_t)(K / 128);
    p.lda = K;
    p.ss_sm = p.ng;
    p.sw_sn = 1;
    return gemm_w4a8k_shape(p);
}
