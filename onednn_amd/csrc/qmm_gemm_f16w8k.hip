// hip:gfx950:mfma_f16w8 where 256 x 256 tiles are few: f16 activations x 8-bit weights of
// QMM_LAYOUT_MFMA_B8, one scale and zero point per column or in all, K a multiple of 128
// (arithmetic of qmm_gemm_f16w8.hip). A workgroup owns 16 RB x 64 results; its eight waves cut K
// between them, 128 k each in turn, and each holds all the results, as in qmm_gemm_b8k.hip.
//   * A lane's 16 weight bytes (column r, k 64 h + 16 c ...) are two operands of 16 x 16 x 32: k
//     8 e ... + 7 of them, e = 0, 1; the rows' operand is the 16 bytes of the same k.
//   * Rows are requested four lanes to 64 bytes and change to operand order in a piece of LDS
//     of the wave's own, where unit u of 16 bytes of row r lies at u ^ (4 (r % 4) + r / 4):
//     neither 16 lanes that write nor 16 that read meet in a bank.
// Bound: trips to memory where K is short, else the vector ALU and requests through L1 (64 x 64
// results and 128 k of the eight waves 2.7 us: 320 instructions to convert, 24 KB a wave). 250
// registers, one workgroup on a CU.
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

typedef float v4f __attribute__((ext_vector_type(4)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));

// Workgroup w runs on XCD w % 8; an XCD takes a run of neighbouring items, the row blocks
// of a column block one after another, so that weights are read into one L2.
struct f16w8k_map_t {
    int nrb, total, share;
};
__host__ __device__ inline f16w8k_map_t f16w8k_map(int M, int nb16, int rb, int cb) {
    const int nrb = (M + 16 * rb - 1) / (16 * rb), ncb = (nb16 + cb - 1) / cb;
    return {nrb, nrb * ncb, (nrb * ncb + 7) / 8};
}

// bytes of a wave: rows of a tile, later its results in rows of BN + 4 floats
constexpr int f16w8k_wave_lds(int rb, int cb) {
    const int results = 16 * rb * (16 * cb + 4) * 4, stage = rb * 4096;
    return results > stage ? results : stage;
}

template <int RB, int CB>
__global__ void __launch_bounds__(WK_WAVES * 64, 2)
gemm_f16w8k_kernel(const gemm_params_t p) {
    constexpr int DW = 2; // weights tiles requested ahead
    extern __shared__ __attribute__((aligned(16))) uint8_t lds_raw[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane >> 4, r = lane & 15;
    const int M = p.M, N = p.N, tiles = p.K / 128, nb16 = (N + 15) / 16;
    const f16w8k_map_t map = f16w8k_map(M, nb16, RB, CB);
    const int item = (blockIdx.x & 7) * map.share + (blockIdx.x >> 3);
    if (item >= map.total) return;
    const int m0 = item % map.nrb * (16 * RB), nb0 = item / map.nrb * CB;

    // column blocks past the last one repeat it, rows past M the last one: never stored
    const uint8_t *Bt[CB];
    v2h zc[CB]; // 1152 - w_off + zero point: an f16 number
#pragma unroll
    for (int cb = 0; cb < CB; cb++) {
        const int b = min(nb0 + cb, nb16 - 1);
        Bt[cb] = p.B + (int64_t)(b >> 1) * p.kb32 * 1024 + (b & 1) * 256;
        const int n = min((nb0 + cb) * 16 + r, N - 1);
        const int z = p.wei_zp ? load_int(p.wei_zp_dt, p.wei_zp, (int64_t)n * p.wei_zp_sn) : 0;
        const _Float16 f = (_Float16)(float)(1152 - p.w_off + z);
        zc[cb] = v2h {f, f};
    }
    const uint32_t boff = (c >> 1) * 1024 + (c & 1) * 512 + r * 16;
    uint32_t aoff[RB]; // bytes (the caller checks that they fit)
#pragma unroll
    for (int rb = 0; rb < RB; rb++)
        aoff[rb] = (uint32_t)min(m0 + 16 * rb + (lane >> 2), M - 1) * (uint32_t)p.lda
                + 16 * (lane & 3);
    uint8_t *const stage = lds_raw + wave * f16w8k_wave_lds(RB, CB);
    const uint32_t wr_at = (lane >> 2) * 256
            + ((((lane >> 2) & 3) << 6) | ((lane >> 4) ^ (lane & 3)) << 4);
    const uint32_t rd_at = r * 256 + (((2 * c) ^ (((r & 3) << 2) | (r >> 2))) << 4);

    // uniform base + 32-bit offset of the lane; made anew in front of each request, else the
    // compiler widens the offset once and adds 64 bits per request
    auto at = [](const void *base, uint32_t off) {
        asm volatile("" : "+v"(off));
        return (const uint8_t *)base + off;
    };
    // the wave's tiles: wave, wave + 8, ..
    const int cnt = tiles > wave ? (tiles - 1 - wave) / WK_WAVES + 1 : 0;
    auto tile_of = [&](int i) { return wave + WK_WAVES * min(i, cnt - 1); };

    v4u a[4][RB], wt[DW][CB][2];
    auto load_w = [&](int i, auto slot) {
        constexpr int sl = decltype(slot)::value;
        const int t = tile_of(i);
#pragma unroll
        for (int cb = 0; cb < CB; cb++) {
            const uint8_t *const q = at(Bt[cb] + (int64_t)t * 4096, boff);
#pragma unroll
            for (int h = 0; h < 2; h++) wt[sl][cb][h] = *(const v4u *)(q + h * 2048);
        }
    };
    auto load_a = [&](int i) {
        const uint8_t *const tile = p.A + (int64_t)tile_of(i) * 256;
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

    auto step = [&](int i, auto slot) {
        constexpr int sl = decltype(slot)::value;
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
        auto read_a = [&](int s) { // (s = 2 h + e)
#pragma unroll
            for (int rb = 0; rb < RB; rb++)
                ops[s & 1][rb] = *(const v4u *)(stage + rb * 4096
                        + (rd_at ^ ((8 * (s >> 1) + (s & 1)) << 4)));
        };
        read_a(0);
#pragma unroll
        for (int s = 0; s < 4; s++) {
            if (s < 3) read_a(s + 1);
#pragma unroll
            for (int cb = 0; cb < CB; cb++) {
                v4u b;
#pragma unroll
                for (int k = 0; k < 2; k++) {
                    // the byte as an unsigned one behind 0x64: the f16 number 1024 + u
                    const uint32_t x = wt[sl][cb][s >> 1][2 * (s & 1) + k] ^ 0x80808080u;
                    const uint32_t lo = __builtin_amdgcn_perm(0x64646464u, x, 0x04010400u);
                    const uint32_t hi = __builtin_amdgcn_perm(0x64646464u, x, 0x04030402u);
                    b[2 * k] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(v2h, lo) - zc[cb]);
                    b[2 * k + 1]
                            = __builtin_bit_cast(uint32_t, __builtin_bit_cast(v2h, hi) - zc[cb]);
                }
#pragma unroll
                for (int rb = 0; rb < RB; rb++)
                    out[rb][cb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                            __builtin_bit_cast(v8h, ops[s & 1][rb]), __builtin_bit_cast(v8h, b),
                            out[rb][cb], 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0x6); // (one step's operands ahead, not all)
        }
        load_w(i + DW, slot);
        __builtin_amdgcn_sched_barrier(0x6);
    };
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
    // MFMA output: register j of lane (c, r) is row 4 c + j, column r.
    constexpr int BM = 16 * RB, BN = 16 * CB, PITCH = BN + 4, W_LDS = f16w8k_wave_lds(RB, CB);
    constexpr int QUADS = BN / 4, RPP = WK_WAVES * 64 / QUADS; // rows per pass
    constexpr int PASSES = (BM + RPP - 1) / RPP;
    const int cg = tid % QUADS * 4, tr = tid / QUADS, n = nb0 * 16 + cg;
    const int nvalid = min(4, N - n);
    ep_cols_t cols; // requested before the waves meet
    epilogue_cols_load(p.ep, cols, 0, n, nvalid);
    const bool has_ss = p.ep.src_scale.ptr != nullptr;
    const float ss = has_ss ? ep_load(p.ep.src_scale, 0, 0, 0) : 1.f; // (one for all rows)
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
            = ((const gemm_params_t *)__builtin_amdgcn_kernarg_segment_ptr())->ep;
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

int gemm_f16w8_splits(int64_t M, int64_t N, int64_t K);

// us of the 256 x 256 kernel with as many K slices as it would take (1500 problems of 256 ...
// 3000 rows). What it takes besides its K is the store of its results: whole quads of 128
// columns 15 us, 4 more with a post-op, and up to 0.4 per row past a multiple of 64; columns that end inside 128 26 us
// more, with a post-op 67 (786 x 256 x 896 31 us, 778 x 752 x 640 52, with a swish 832 x 256 x
// 512 28, 875 x 656 x 896 108). Slices store f32 sums and leave the post-ops to a second kernel.
static double f16w8_tiled_us(const gemm_params_t &p) {
    const int splits = gemm_f16w8_splits(p.M, p.N, p.K);
    const int64_t tiles = (int64_t)((p.M + 255) / 256) * ((p.N + 255) / 256) * splits;
    const double rounds = (double)((tiles + 255) / 256), k = p.K / 1024.0 / splits;
    const bool ends = p.N % 128 != 0, post = p.ep.npo > 0;
    if (splits > 1)
        return 22.4 + rounds * (19.7 * k - 4 + (ends ? 10.3 : 0)) + 1.8e-6 * splits * p.M * p.N;
    const double tail = ends ? (post ? 67 : 26) : (post ? 0.4 : 0.15) * (p.M % 64);
    return 1 + rounds * (14.5 + (post ? 4 : 0) + 18 * k) + tail;
}

// Row and column blocks of a workgroup as 16 * rb + cb, 0: 256 x 256 tiles are faster. Before /
// now (us): 263 x 1280 x 3040 43.4 / 12.6, 350 x 2688 x 2384 44.6 / 14, 424 x 2816 x 5344 63 / 40,
// 468 x 10496 x 1792 51 / 31, 872 x 8192 x 2208 79 / 55, 303 x 5632 x 12304 102 / 90; there from
// some 500 rows and 20 million weights on (614 x 1664 x 10400 56 / 70, 1922 x 2304 x 2864 63 / 82, 4096 x 1024 x 1024 36 / 42),
// earlier where columns come in whole multiples of 128 (331 x 256 x 8960 22 / 24, 1103 x 5504 x 2560 65 / 73), and
// with long rows (1473 x 14464 x 1344 106 / 124, 2102 x 9216 x 816 75 / 81; but 885 x 12160 x 1472 90 / 69).
// Over 1750 problems of 256 ... 3000 rows 1.7 times as fast in the mean and up to 6 % slower than before
// (2141 x 3456 x 1152 57 / 61). One workgroup on a CU (32 on an XCD); a begun round costs most of a whole one.
int gemm_f16w8k_shape(const gemm_params_t &p) {
    if (p.K % 128 != 0 || (int64_t)p.M * p.lda >= (int64_t)1 << 32) return 0;
    static const struct {
        int rb, cb;
        double once, start, k1024, begun;
    } shapes[] = {{2, 4, 2.48, 4.28, 1.9, 0.69}, {3, 4, 1.45, 5.95, 2.29, 0.76},
            {4, 4, 0.72, 7.07, 2.69, 0.68}};
    double best = f16w8_tiled_us(p) / 1.1; // (clearly, or not)
    int pick = 0;
    const double rows = many_rows(p.M, p.K, 0.25);
    for (const auto &s : shapes) {
        const double wgs = f16w8k_map(p.M, (p.N + 15) / 16, s.rb, s.cb).share / 32.0;
        const double rounds = std::max(1.0, s.begun * std::ceil(wgs) + (1 - s.begun) * wgs);
        const double us = s.once + rounds * (s.start + s.k1024 * p.K / 1024) * rows;
        if (us < best) {
            best = us;
            pick = 16 * s.rb + s.cb;
        }
    }
    return pick;
}

void launch_gemm_f16w8k(const gemm_params_t &p, int shape, hipStream_t stream) {
    const int rb = shape / 16, cb = shape % 16;
    const f16w8k_map_t map = f16w8k_map(p.M, (p.N + 15) / 16, rb, cb);
    auto go = [&](auto kern) {
        const int lds = WK_WAVES * f16w8k_wave_lds(rb, cb);
        if (lds > 65536) ensure_dynamic_lds((const void *)kern, lds);
        hipLaunchKernelGGL(kern, dim3((unsigned)(8 * map.share)), dim3(WK_WAVES * 64), lds,
                stream, p);
    };
    switch (shape) {
        case 0x24: go(gemm_f16w8k_kernel<2, 4>); break;
        case 0x44: go(gemm_f16w8k_kernel<4, 4>); break;
        default: go(gemm_f16w8k_kernel<3, 4>); break;
    }
}

} // namespace qmm

extern "C" int qmm_gemm_f16w8k_shape(int64_t M, int64_t N, int64_t K) {
    using namespace qmm;
    const int64_t top = 1 << 24;
    if (M < 1 || N < 1 || K < 256 || K % 128 != 0 || M > top || N > top || K > top) return 0;
    gemm_params_t p = {};
    p.M = (int32_t)M;
    p.N = (int32_t)N;
    p.K = (int32_t)K;
    p.lda = 2 * K;
    return gemm_f16w8k_shape(p);
}
