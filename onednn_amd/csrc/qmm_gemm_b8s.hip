// hip:gfx950:mfma_b8, many small matrices with a short K (attention scores: batches of s8 x s8
// with K 64 or 128 and, most often, an f32 mask added): a launch writes its results and does
// little else, so what counts is requests in flight and whole lines in L2. A wave owns 32 x 64
// results and never waits for another one: operands straight into registers (16 x 16 x 64
// products; a lane's 16 bytes of QMM_LAYOUT_MFMA_B8 are an operand, as in qmm_gemm_b8k.hip),
// the mask requested with them, results turned to rows in a piece of LDS of its own, stored
// as 16 lanes to 256 bytes of a row. An XCD takes a run of neighbouring items, columns first:
// where rows start off a line, both writers of that line share an L2. Bound: the trip to
// memory and back for few tokens, else writes that end inside lines (16 x 1361 x 1361 2.5 TB/s).
// Source scales looked up per row cost 0.7 us, one matrix after the other (a shared mask then
// comes from the memory side for each) 10 % at 2047 rows.
#include <algorithm>
#include <type_traits>

#include "qmm_device.hpp"
#include "qmm_hip.h"
#include "qmm_plan.hpp"

namespace qmm {
namespace {
constexpr int BS_WAVES = 4, BS_RB = 2, BS_CB = 4; // a workgroup: 64 rows x 128 columns
constexpr int BS_PITCH = 16 * BS_CB + 4;

typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v4f_any __attribute__((ext_vector_type(4), aligned(4)));

struct b8s_map_t {
    int tm, tn;
    int64_t total, share;
};
__host__ __device__ inline b8s_map_t b8s_map(int M, int N, int batch) {
    const int tm = (M + 63) / 64, tn = (N + 127) / 128;
    const int64_t total = (int64_t)batch * tm * tn;
    return {tm, tn, total, (total + 7) / 8};
}

// KC: K / 64. ADD: nothing but scales and an f32 operand added, dense along n
template <int KC, bool ADD>
__global__ void __launch_bounds__(BS_WAVES * 64, 3)
gemm_b8s_kernel(const gemm_params_t p) {
    __shared__ __attribute__((aligned(16))) float lds[BS_WAVES][16 * BS_RB * BS_PITCH];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane >> 4, r = lane & 15;
    const b8s_map_t map = b8s_map(p.M, p.N, p.batch);
    const int item = (int)((blockIdx.x & 7) * map.share + (blockIdx.x >> 3));
    if (item >= map.total) return;
    // 256 rows of every matrix, then the next 256: what one mask for all has of them stays in L2
    const int group = 4 * map.tn * p.batch, g = item / group, gm = min(4, map.tm - 4 * g);
    const int b = item % group / (gm * map.tn), t = item % group % (gm * map.tn);
    const int m0 = (4 * g + t / map.tn) * 64 + (wave >> 1) * 32;
    const int n0 = t % map.tn * 128 + (wave & 1) * 64;
    if (m0 >= p.M || n0 >= p.N) return; // (no barrier in this kernel)

    // rows past M and columns past N repeat the last ones: never stored
    const uint8_t *const A = p.A + b * p.a_sb, *const B = p.B + b * p.b_sb;
    const int nb16 = (p.N + 15) / 16;
    v4i a[BS_RB][KC], w[BS_CB][KC];
#pragma unroll
    for (int rb = 0; rb < BS_RB; rb++)
#pragma unroll
        for (int i = 0; i < KC; i++)
            a[rb][i] = *(const v4i *)(A + (int64_t)min(m0 + 16 * rb + r, p.M - 1) * p.lda
                    + 64 * i + 16 * c);
#pragma unroll
    for (int cb = 0; cb < BS_CB; cb++) {
        const int nb = min(n0 / 16 + cb, nb16 - 1);
        const uint8_t *const q = B + (int64_t)(nb >> 1) * p.kb32 * 1024 + (nb & 1) * 256
                + (c >> 1) * 1024 + (c & 1) * 512 + r * 16;
#pragma unroll
        for (int i = 0; i < KC; i++) w[cb][i] = *(const v4i *)(q + i * 2048);
    }
    // a lane's results: columns n ... n + 3 of rows m0 + c + 4 q
    constexpr int ROWS = 4 * BS_RB;
    const int cg = r * 4, n = n0 + cg, nvalid = min(4, p.N - n);
    v4f add[ROWS];
    if constexpr (ADD) {
        const float *const q0 = (const float *)p.ep.po[0].t.ptr + b * p.ep.po[0].t.sb;
#pragma unroll
        for (int q = 0; q < ROWS; q++) {
            const float *const y = q0 + (int64_t)min(m0 + c + 4 * q, p.M - 1) * p.ep.po[0].t.sm;
            if (nvalid == 4) {
                add[q] = *(const v4f_any *)(y + n);
            } else {
#pragma unroll
                for (int i = 0; i < 4; i++) add[q][i] = y[min(n + i, p.N - 1)];
            }
        }
    }
    ep_cols_t cols;
    epilogue_cols_load(p.ep, cols, b, n, nvalid);
    const bool has_ss = p.ep.src_scale.ptr != nullptr;
    // (one trip to memory for all rows where they share a scale)
    const bool ss_rows = has_ss && p.ep.src_scale.sm != 0;
    const float ss0 = has_ss ? ep_load(p.ep.src_scale, b, min(m0 + c, p.M - 1), 0) : 1.f;

    float *const stage = lds[wave];
#pragma unroll
    for (int rb = 0; rb < BS_RB; rb++)
#pragma unroll
        for (int cb = 0; cb < BS_CB; cb++) {
            v4i acc = {0, 0, 0, 0};
#pragma unroll
            for (int i = 0; i < KC; i++)
                acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[rb][i], w[cb][i], acc, 0, 0, 0);
            // register j of lane (c, r) is row 4 c + j, column r
#pragma unroll
            for (int j = 0; j < 4; j++)
                stage[(16 * rb + 4 * c + j) * BS_PITCH + 16 * cb + r] = (float)acc[j];
        }
    const epilogue_t &epk
            = ((const gemm_params_t *)__builtin_amdgcn_kernarg_segment_ptr())->ep;
    if (nvalid <= 0) return;
#pragma unroll
    for (int q = 0; q < ROWS; q++) {
        const int row = c + 4 * q, m = m0 + row;
        if (m >= p.M) continue;
        const v4f v = *(const v4f *)(stage + row * BS_PITCH + cg);
        const float ss = ss_rows ? ep_load(p.ep.src_scale, b, m, 0) : ss0;
        float d[4] = {v[0], v[1], v[2], v[3]};
        if constexpr (ADD) {
            // (an absent scale is the factor 1: the same bits)
#pragma unroll
            for (int i = 0; i < 4; i++) d[i] = d[i] * ss * cols.ws[i] + add[q][i];
            epilogue_store4(p.ep, d, b * p.ep.dst.sb + m * p.ep.dst.sm + n, nvalid);
        } else {
            epilogue_rows4(epk, cols, d, has_ss, ss, b, m, n, nvalid);
        }
    }
}

} // namespace

int gemm_b8_tile(const gemm_params_t &p, bool f8, bool post_ops);
static bool adds_f32(const gemm_params_t &p) {
    return p.ep.fast == EP_FAST_ADD && !p.ep.fast_ext;
}

// Several matrices, s8 x s8 without zero points (the caller checks), f32 rows that start off the
// 16-byte boundaries, which the kernels with tiles store and add at a fraction of their rate.
// us, those / this one, with a mask: 16 x 1361 x 1361 x 64 70 / 47, 8 x 2047 x 2047 x 128 73 / 59,
// 20 x 922 x 922 x 128 50 / 34, 32 x 309 x 309 x 64 19.9 / 10.3, 4 x 439 x 439 x 128 18.2 / 9.9.
// Rows on such boundaries stay there: 32 x 2048 x 2048 x 128 117 / 184, 32 x 1024 42 / 48; so do
// the problems of 64 x 64 tiles (8 x 201 x 201 x 128 5.9 / 7.8, 4 x 131 x 131 x 64 5.6 / 9.6).
bool gemm_b8s_takes(const gemm_params_t &p) {
    return p.batch > 1 && (p.K == 64 || p.K == 128) && p.M > 128 && p.N > 128
            && p.ep.dst.dt == dt_f32 && p.ep.dst.sn == 1 && p.ep.dst.sm % 4 != 0
            && (adds_f32(p) || p.ep.npo == 0)
            && b8s_map(p.M, p.N, p.batch).total < (int64_t)1 << 26
            && gemm_b8_tile(p, false, p.ep.npo > 0) > 64;
}

void launch_gemm_b8s(const gemm_params_t &p, hipStream_t stream) {
    const b8s_map_t map = b8s_map(p.M, p.N, p.batch);
    auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3((unsigned)(8 * map.share)), dim3(BS_WAVES * 64), 0, stream, p);
    };
    const bool add = adds_f32(p);
    if (p.K == 64) add ? go(gemm_b8s_kernel<1, true>) : go(gemm_b8s_kernel<1, false>);
    else add ? go(gemm_b8s_kernel<2, true>) : go(gemm_b8s_kernel<2, false>);
}

} // namespace qmm

extern "C" int qmm_gemm_b8s_takes(
        int64_t batch, int64_t M, int64_t N, int64_t K, int64_t dst_pitch, int add) {
    using namespace qmm;
    const int64_t top = 1 << 24;
    if (batch < 1 || M < 1 || N < 1 || K < 16 || K % 16 || dst_pitch < N || batch > top || M > top || N > top || K > top)
        return 0;
    gemm_params_t p = {};
    p.M = (int32_t)M;
    p.N = (int32_t)N;
    p.K = (int32_t)K;
    p.lda = K;
    p.batch = (int32_t)batch;
    p.kb32 = (int32_t)((K + 31) / 32);
    p.ep.dst.dt = dt_f32;
    p.ep.dst.sm = dst_pitch;
    p.ep.dst.sn = 1;
    p.ep.npo = add ? 1 : 0;
    p.ep.fast = add ? EP_FAST_ADD : EP_FAST_PLAIN;
    return gemm_b8s_takes(p);
}
