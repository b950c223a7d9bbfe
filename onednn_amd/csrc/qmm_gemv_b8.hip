// hip:gfx950:mfma_b8, few source rows (the decode step of a W8A8 linear layer, one
// token or a small batch of them) or few results: a launch is one read of the weights,
// or one per 32 rows, the later ones from L2, so the kernel is organised
// around memory parallelism instead of tiles. A workgroup owns 32 columns (one
// block of QMM_LAYOUT_MFMA_B8, whose 1 KiB fragments already are the MFMA
// operand per lane) and at most 32 rows; its 8 waves cut K between them and each
// streams its fragments straight into registers, 16 requested at a time together with the
// matching source bytes, and multiplies them with v_mfma_i32_32x32x32_i8 (the
// first M rows of the 32 x 32 result are the source rows; the others repeat the
// last row and are dropped: MR = 4 keeps only registers 0..3 of lanes 0..31,
// MR = 32 everything), or with the 64-k fp8 MFMA. The waves' s32 sums are added
// through LDS -- integer addition, so the result does not depend on the cut (f32 sums:
// always in the waves' order) -- and the epilogue runs on four columns per thread:
//   (float)(P + comp * colsum[n] - z_w'[n] * (rowsum[m] + K * comp)),
// source scale, weights scale, bias, post-ops, dst quantization
// (src/cpu/matmul/ref_matmul_int8.cpp:165-259). The row sums that a weights
// zero point needs come from dot products of the source fragments with ones.
// Bound: at M = 1 HBM (4096 x 14336 13.3 us, 4.5 TB/s); with 64 rows of that the waves'
// chain of request, wait, multiply (22.6; 24.9 with one result per thread and trip to
// memory at the end); for small problems launch, one or two trips to memory and the
// sum (256 x 1024 x 1024 6.3 us, 9.1 ... 10.3 in 64 x 64 tiles).
#include <type_traits>

#include "qmm_device.hpp"
#include "qmm_plan.hpp"

namespace qmm {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));

constexpr int GB8_WAVES = 8;
constexpr int GB8_CH = 16; // fragments in flight per wave

// MR = 32: the source bytes of a chunk go through a wave-private piece of LDS --
// requested as whole 256-byte row pieces (16 lanes a row, 4 rows an
// instruction) instead of one 16-byte piece per lane out of 32 different rows
// -- and come back in operand order. The same bytes hold the wave's results
// for the sum across waves afterwards.
constexpr int GB8_CH32 = 8; // fragments per chunk with 32 rows
constexpr int GB8_APITCH = GB8_CH32 * 32 + 16; // bytes of a staged row
constexpr int gb8_wave_lds(int mr) { // >= mr x 32 s32 of results + row sums
    return mr == 32 ? 32 * GB8_APITCH : (4 * 32 + 4) * 4;
}
static_assert(gb8_wave_lds(32) >= 32 * 32 * 4 + 32 * 4, "");

// (by value: of a vector's element in place the builtin takes the first one's bits)
template <typename T>
QMM_D int bits(T v) {
    return __builtin_bit_cast(int, v);
}

// Column block and first row of a workgroup, more than 32 rows. Workgroup w runs on XCD
// w % 8. A column block's row blocks go to one XCD, one after another: close in time and
// on one L2 (counted there: 256 x 4096 x 4096 fetches 27.9 MB, 8.4 of them the rows once per
// XCD, so its 16.8 MB of weights 1.1 times; 32 rows 18.3 MB in all). With many of them (an XCD has 32 CUs) the columns past the last whole group
// of 8 would leave XCDs idle: there every XCD takes an eighth of their blocks (s8, us, one
// XCD a column / so: 43008 x 4096 x 32 191 / 46.3, 16384 x 4096 x 64 68.2 / 25.4, 2000 x
// 4096 x 288 22.5 / 18.0; with few row blocks the other way, 226 x 8192 x 2055 25.0 / 29.4).
// False: nothing left for it.
struct gb8_map_t {
    int nrb, whole, share; // row blocks; columns of whole groups; rest of an XCD, or 0
};
__host__ __device__ inline gb8_map_t gb8_map(int M, int nb32) {
    const int nrb = (M + 31) / 32;
    return {nrb, nb32 / 8 * 8, nrb >= 32 ? (nrb * (nb32 % 8) + 7) / 8 : 0};
}
__host__ __device__ inline int gb8_grid(int M, int nb32) {
    const gb8_map_t g = gb8_map(M, nb32);
    return g.share ? g.nrb * g.whole + 8 * g.share : g.nrb * ((nb32 + 7) / 8 * 8);
}
__host__ __device__ inline bool gb8_block(int M, int nb32, int w, int &nb, int &m0) {
    const gb8_map_t g = gb8_map(M, nb32);
    nb = w / (8 * g.nrb) * 8 + w % 8;
    m0 = w / 8 % g.nrb * 32;
    if (g.share && nb >= g.whole) {
        w -= g.nrb * g.whole;
        const int item = w % 8 * g.share + w / 8;
        nb = g.whole + item / g.nrb;
        m0 = item % g.nrb * 32;
    }
    return nb < nb32;
}

// What a thread adds up and stores: four neighbouring columns of one row, so that a
// block of 32 columns is one pass of the workgroup and everything the epilogue reads
// per row and column is requested before the waves meet. red: the waves' results,
// [rows][32] s32 and `mr` row sums each, `pitch` bytes apart. epk: the epilogue where
// the kernel's arguments lie (its post-op list is indexed at run time).
struct gb8_tail_t {
    ep_cols_t cols;
    int cs[4], zw[4], comp, nvalid;
    float ss;
};
QMM_D void gb8_tail_load(const gemm_params_t &p, bool need_rs, int m, int n, gb8_tail_t &t) {
    t.nvalid = m < p.M ? min(4, p.N - n) : 0;
    t.comp = p.a_is_u8 ? 128 : 0;
    if (p.src_zp) t.comp -= load_int(p.src_zp_dt, p.src_zp, 0);
    epilogue_cols_load(p.ep, t.cols, 0, n, t.nvalid);
#pragma unroll
    for (int i = 0; i < 4; i++) {
        t.cs[i] = t.zw[i] = 0;
        if (i < t.nvalid) {
            if (t.comp != 0 && p.colsum) t.cs[i] = t.comp * p.colsum[n + i];
            if (need_rs)
                t.zw[i] = (p.wei_zp ? load_int(p.wei_zp_dt, p.wei_zp,
                                   (int64_t)(n + i) * p.wei_zp_sn)
                                    : 0)
                        - p.w_off;
        }
    }
    t.ss = t.nvalid > 0 && p.ep.src_scale.ptr ? ep_load(p.ep.src_scale, 0, m, 0) : 1.f;
}
template <bool F8>
QMM_D void gb8_tail_store(const gemm_params_t &p, const epilogue_t &epk,
        const gb8_tail_t &t, const uint8_t *red,
        int pitch, int mr, int r, int m, int n) {
    if (t.nvalid <= 0) return;
    float d[4] = {0.f, 0.f, 0.f, 0.f};
    v4u v = {0, 0, 0, 0};
    uint32_t rs = 0;
#pragma unroll
    for (int w = 0; w < GB8_WAVES; w++) {
        const v4u x = *(const v4u *)(red + w * pitch + (r * 32 + (n & 31)) * 4);
        if constexpr (F8) {
#pragma unroll
            for (int i = 0; i < 4; i++) d[i] += u2f(x[i]);
        } else {
            v += x;
            rs += ((const uint32_t *)(red + w * pitch))[mr * 32 + r];
        }
    }
#pragma unroll
    for (int i = 0; i < 4 && !F8; i++) // s32 arithmetic that wraps as the reference's int accumulation
        d[i] = (float)(int32_t)(v[i] + (uint32_t)t.cs[i]
                - (uint32_t)t.zw[i] * (rs + (uint32_t)p.K * (uint32_t)t.comp));
    epilogue_rows4(epk, t.cols, d, p.ep.src_scale.ptr != nullptr, t.ss, 0, m, n, t.nvalid);
}

// F8: f8_e4m3 on both sides, f32 sums (two fragments to an MFMA of 64 k)
// QUADS: the end takes four columns per thread; else, for at most 16 rows, a thread per
// result: a long post-op is one chain of them and not four (16 x 4096 x 4096 8.3 / 8.8,
// 1 x 1024 x 4096 with a swish 6.0 / 6.7 us; 32 x 4096 x 4096 9.9 / 9.4 the other way).
// Kernels of their own: either end behind a branch cost the few rows 0.4 us.
template <int MR, bool F8, bool QUADS>
__global__ void __launch_bounds__(GB8_WAVES * 64)
gemv_b8_kernel(const gemm_params_t p) {
    typedef typename std::conditional<F8, v16f, v16i>::type acc_t;
    static_assert(MR == 4 || MR == 32, "");
    constexpr int CH = MR == 32 ? GB8_CH32 : GB8_CH;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds_raw[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    constexpr int WAVE_LDS = gb8_wave_lds(MR);
    // a wave's results [MR][32] and row sums [MR], s32
    auto red = [&](int w, int r, int c) -> int & {
        return ((int *)(lds_raw + w * WAVE_LDS))[r * 32 + c];
    };
    auto red_rs = [&](int w, int r) -> int & {
        return ((int *)(lds_raw + w * WAVE_LDS))[MR * 32 + r];
    };
    int nb = blockIdx.x, m0 = 0;
    if (QUADS && p.M > 32 && !gb8_block(p.M, p.nb32, blockIdx.x, nb, m0)) return;
    const int rows = p.M - m0;
    const uint8_t *const A = p.A + (int64_t)m0 * p.lda;
    // the wave's fragments (32 k each): an even cut of the K / 32 that hold data
    const int nfrag = (p.K + 31) / 32;
    int per = (nfrag + GB8_WAVES - 1) / GB8_WAVES;
    if (F8) per = (per + 1) & ~1; // (K is a multiple of 64)
    const int f0 = min(wave * per, nfrag), f1 = min(f0 + per, nfrag);
    const v4u *bsrc = (const v4u *)(p.B + (int64_t)nb * p.kb32 * 1024) + lane;
    // A operand: lane l is row l % 32, bytes 16 (l / 32) .. + 15 of the fragment
    const int row = min(lane & 31, rows - 1);
    const uint8_t *arow = A + (int64_t)row * p.lda;
    const uint32_t flip = p.a_is_u8 && !p.a_preflipped ? 0x80808080u : 0u;
    const bool need_rs = p.wei_zp != nullptr || p.w_off != 0;
    uint8_t *const stage = lds_raw + wave * WAVE_LDS;

    acc_t acc;
    int rsum = 0;
#pragma unroll
    for (int r = 0; r < 16; r++) acc[r] = 0;
    for (int fb = f0; fb < f1; fb += CH) {
        v4u bq[CH];
        uint4 av[CH];
        // every request of the chunk before the first use; fragments past the
        // wave's end repeat its last one and are skipped below
        if constexpr (MR == 32) {
            // piece l % 16 of rows l / 16 + 4 i (K is a multiple of 16: a piece
            // is inside the row or past it)
            static_assert(CH == 8, "a block of 32 rows is 8 row quadruples");
            const int k = fb * 32 + (lane & 15) * 16;
#pragma unroll
            for (int i = 0; i < CH; i++) {
                const int r = min(4 * i + (lane >> 4), rows - 1);
                av[i] = *(const uint4 *)(A + (int64_t)r * p.lda + min(k, p.K - 16));
            }
#pragma unroll
            for (int j = 0; j < CH; j++)
                bq[j] = __builtin_nontemporal_load(bsrc + (int64_t)min(fb + j, f1 - 1) * 64);
#pragma unroll
            for (int i = 0; i < CH; i++)
                *(uint4 *)(stage + (4 * i + (lane >> 4)) * GB8_APITCH + (lane & 15) * 16)
                        = k >= p.K ? make_uint4(flip, flip, flip, flip) // zero after the flip
                                   : av[i];
#pragma unroll
            for (int j = 0; j < CH; j++)
                av[j] = *(const uint4 *)(stage + (lane & 31) * GB8_APITCH + j * 32
                        + (lane >> 5) * 16);
        } else {
#pragma unroll
            for (int j = 0; j < CH; j++) {
                const int f = min(fb + j, f1 - 1);
                bq[j] = __builtin_nontemporal_load(bsrc + (int64_t)f * 64);
                // K is a multiple of 16: a half fragment is inside the row or past it
                const int k = f * 32 + (lane >> 5) * 16;
                av[j] = *(const uint4 *)(arow + min(k, p.K - 16));
                if (k >= p.K) av[j] = make_uint4(flip, flip, flip, flip); // zero after the flip
            }
        }
#pragma unroll
        for (int j = 0; j < CH; j += F8 ? 2 : 1) {
            if (fb + j < f1) {
                if constexpr (F8) {
                    const uint4 a0 = av[j], a1 = av[j + 1];
                    const v8i a = {(int)a0.x, (int)a0.y, (int)a0.z, (int)a0.w,
                            (int)a1.x, (int)a1.y, (int)a1.z, (int)a1.w};
                    const v8i b = {(int)bq[j].x, (int)bq[j].y, (int)bq[j].z,
                            (int)bq[j].w, (int)bq[j + 1].x, (int)bq[j + 1].y,
                            (int)bq[j + 1].z, (int)bq[j + 1].w};
                    acc = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(
                            a, b, acc, 0, 0, 0, 0, 0, 0);
                } else {
                    const v4i b = {(int)bq[j].x, (int)bq[j].y, (int)bq[j].z,
                            (int)bq[j].w};
                    const v4i a = {(int)(av[j].x ^ flip), (int)(av[j].y ^ flip),
                            (int)(av[j].z ^ flip), (int)(av[j].w ^ flip)};
                    if (need_rs) {
#pragma unroll
                        for (int q = 0; q < 4; q++)
                            rsum = __builtin_amdgcn_sdot4(a[q], 0x01010101, rsum, false);
                    }
                    acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, acc, 0, 0, 0);
                }
            }
        }
    }
    // accumulator register r of lane l is row 8 (r / 4) + 4 (l / 32) + r % 4,
    // column l % 32; the two k halves of row r's sum sit in lanes r and r + 32
    if constexpr (MR == 4) {
        if (lane < 32) {
#pragma unroll
            for (int r = 0; r < 4; r++) red(wave, r, lane) = bits(acc[r]);
        }
    } else {
#pragma unroll
        for (int r = 0; r < 16; r++)
            red(wave, 8 * (r / 4) + 4 * (lane >> 5) + r % 4, lane & 31) = bits(acc[r]);
    }
    const int tot = rsum + __shfl_xor(rsum, 32);
    if (lane < MR) red_rs(wave, lane) = tot;
    const int tid = threadIdx.x;
    if constexpr (!QUADS) {
        __syncthreads();
        const int r = tid >> 5, n = nb * 32 + (tid & 31);
        if (r >= rows || r >= MR || n >= p.N) return;
        float d = 0.f;
        uint32_t v = 0, rs = 0;
#pragma unroll
        for (int w = 0; w < GB8_WAVES; w++) {
            const int x = red(w, r, tid & 31);
            if constexpr (F8) {
                d += u2f((uint32_t)x);
            } else {
                v += (uint32_t)x;
                rs += (uint32_t)red_rs(w, r);
            }
        }
        if constexpr (!F8) {
            int comp = p.a_is_u8 ? 128 : 0;
            if (p.src_zp) comp -= load_int(p.src_zp_dt, p.src_zp, 0);
            const int cs = comp != 0 && p.colsum ? comp * p.colsum[n] : 0;
            const int zw = need_rs
                    ? (p.wei_zp ? load_int(p.wei_zp_dt, p.wei_zp, (int64_t)n * p.wei_zp_sn)
                                : 0)
                            - p.w_off
                    : 0;
            // s32 arithmetic that wraps as the reference's int accumulation
            v += (uint32_t)cs - (uint32_t)zw * (rs + (uint32_t)p.K * (uint32_t)comp);
            d = (float)(int32_t)v;
        }
        epilogue_apply_store(p.ep, d, 0, m0 + r, n);
    } else {
        const int tr = tid >> 3, tn = nb * 32 + (tid & 7) * 4;
        gb8_tail_t tail;
        if (tr < MR) gb8_tail_load(p, need_rs, m0 + tr, tn, tail);
        __syncthreads();
        const epilogue_t &epk
                = ((const gemm_params_t *)__builtin_amdgcn_kernarg_segment_ptr())->ep;
        if (tr < MR)
            gb8_tail_store<F8>(p, epk, tail, lds_raw, WAVE_LDS, MR, tr, m0 + tr, tn);
    }
}

// 33 ... 64 rows over many columns: both blocks of 32 rows against the same weights.
// A chunk is CH fragments of k: its source bytes, 128-byte row pieces, go through the
// wave's piece of LDS, and the next chunk is requested before the products.
__global__ void __launch_bounds__(GB8_WAVES * 64, 4)
gemv_b8_rows64_kernel(const gemm_params_t p) {
    constexpr int MR = 64, CH = 4, PITCH = CH * 32 + 16, W_LDS = MR * PITCH;
    constexpr int NI = MR / 8; // row pieces of a lane
    extern __shared__ __attribute__((aligned(16))) uint8_t lds_raw[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    uint8_t *const stage = lds_raw + wave * W_LDS;
    const int nb = blockIdx.x;
    const int nfrag = (p.K + 31) / 32;
    const int per = (nfrag + GB8_WAVES - 1) / GB8_WAVES;
    const int f0 = min(wave * per, nfrag), f1 = min(f0 + per, nfrag);
    const int last = f0 + (f1 - 1 - f0) / CH * CH; // the wave's last chunk
    const uint32_t flip = p.a_is_u8 && !p.a_preflipped ? 0x80808080u : 0u;
    const bool need_rs = p.wei_zp != nullptr || p.w_off != 0;
    const v4u *bsrc = (const v4u *)(p.B + (int64_t)nb * p.kb32 * 1024) + lane;
    v16i acc[2];
    int rsum[2] = {0, 0};
#pragma unroll
    for (int rb = 0; rb < 2; rb++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[rb][r] = 0;
    const int pr = lane >> 3, pk = (lane & 7) * 16;
    v4u as[NI], bq[2][CH];
    // (requests past the wave's end repeat its last chunk or fragment; K is a multiple
    // of 16: a piece is inside the row or past it)
    auto request = [&](int fb, auto slot) {
        constexpr int s = decltype(slot)::value;
        fb = min(fb, last);
        const uint8_t *ak = p.A + min(fb * 32 + pk, p.K - 16);
#pragma unroll
        for (int i = 0; i < NI; i++)
            as[i] = *(const v4u *)(ak + (int64_t)min(8 * i + pr, p.M - 1) * p.lda);
#pragma unroll
        for (int j = 0; j < CH; j++)
            bq[s][j] = __builtin_nontemporal_load(bsrc + (int64_t)min(fb + j, f1 - 1) * 64);
    };
    auto stage_rows = [&](int fb) {
        const bool past = fb * 32 + pk >= p.K;
#pragma unroll
        for (int i = 0; i < NI; i++) // (past K: zero after the flip)
            *(v4u *)(stage + (8 * i + pr) * PITCH + pk)
                    = past ? v4u {flip, flip, flip, flip} : as[i];
    };
    auto multiply = [&](int fb, auto slot) {
        constexpr int s = decltype(slot)::value;
#pragma unroll
        for (int j = 0; j < CH; j++) {
            if (fb + j >= f1) continue;
#pragma unroll
            for (int rb = 0; rb < 2; rb++) {
                const v4u v = *(const v4u *)(stage + (32 * rb + (lane & 31)) * PITCH
                        + j * 32 + (lane >> 5) * 16);
                const v4i a = __builtin_bit_cast(v4i, v ^ flip);
                if (need_rs) {
#pragma unroll
                    for (int q = 0; q < 4; q++)
                        rsum[rb] = __builtin_amdgcn_sdot4(a[q], 0x01010101, rsum[rb], false);
                }
                acc[rb] = __builtin_amdgcn_mfma_i32_32x32x32_i8(
                        a, __builtin_bit_cast(v4i, bq[s][j]), acc[rb], 0, 0, 0);
            }
        }
    };
    if (f0 < f1) {
        const std::integral_constant<int, 0> even;
        const std::integral_constant<int, 1> odd;
        request(f0, even);
        for (int fb = f0;; fb += 2 * CH) {
            stage_rows(fb);
            request(fb + CH, odd);
            multiply(fb, even);
            if (fb + CH >= f1) break;
            stage_rows(fb + CH);
            request(fb + 2 * CH, even);
            multiply(fb + CH, odd);
            if (fb + 2 * CH >= f1) break;
        }
    }
    // the waves' results [64][32] and row sums
    static_assert(W_LDS >= 64 * 32 * 4 + 64 * 4, "");
    const int tid = threadIdx.x, tr = tid >> 3, tn = nb * 32 + (tid & 7) * 4;
    gb8_tail_t tail;
    gb8_tail_load(p, need_rs, tr, tn, tail);
    int *const red = (int *)stage;
#pragma unroll
    for (int rb = 0; rb < 2; rb++) {
#pragma unroll
        for (int r = 0; r < 16; r++)
            red[(32 * rb + 8 * (r / 4) + 4 * (lane >> 5) + r % 4) * 32 + (lane & 31)]
                    = acc[rb][r];
        const int tot = rsum[rb] + __shfl_xor(rsum[rb], 32);
        if (lane < 32) red[MR * 32 + 32 * rb + lane] = tot;
    }
    __syncthreads();
    const epilogue_t &epk
            = ((const gemm_params_t *)__builtin_amdgcn_kernarg_segment_ptr())->ep;
    gb8_tail_store<false>(p, epk, tail, lds_raw, W_LDS, MR, tr, tr, tn);
}

} // namespace

// One read of the weights (or, with more rows, one per 32 rows, from L2): up to how many
// rows and columns this is the faster kernel. Per workgroup of 32 x 32 results the
// operands are read once, 64 K bytes; the tiled kernels read less but leave CUs idle,
// walk K in one chain and post-process in a longer one. us, tiled / here, s8 x s8:
// 256 x 1024 x 1024 10.3 / 6.3 (256 workgroups), 128 x 4096 x 1024 18.0 / 7.9, 256 x
// 4096 x 4096 28.7 / 19.4, 96 x 14336 x 8192 97.8 / 54.7, 512 x 14336 x 2048 85.5 /
// 63.1, 1000 x 4096 x 1024 35.7 / 21.8 (all at most 1024), 320 x 4096 x 4096 36.2 /
// 24.0 (1280), 70 x 4096 x 14336 31.6 / 27.4 (1344), 384 x 4096 x 4096 27.6 / 29.6
// (1536), 128 x 4096 x 14336 27.8 / 33.6 (1792). With fewer than 2048 k the 256-row
// kernels come level earlier: 1024 x 1024 x 1024 12.5 / 13.3 (1024), 256 x 1024 x 4096
// 12.4 / 11.7 (1024), 70 x 1024 x 16384 17.5 / 18.1 (1536), 300 x 1024 x 3072 23.5 / 11.6 (960).
// f8_e4m3 (tiled / here): 256 x 1024 x 1024 12.8 / 7.1, 512 x 4096 x 4096 43.5 / 35.5
// (2048), 1024 x 2048 x 2048 31.9 / 27.7 (2048), 919 x 1152 x 1664 22.8 / 23.9 (1508),
// 2048 x 1024 x 1024 23.0 / 26.7 (2048), 700 x 14336 x 2048 85.0 / 94.6 (1408), 100 x 4096 x
// 16384 37.7 / 36.8 (2048), 100 x 6144 x 16384 46.0 / 55.9, 200 x 6144 x 8192 45.5 / 46.3 (1792).
//
// Against 64 x 64 tiles (fewer than 64 tiles of 128 x 128 and not the 256-row kernels),
// which keep every CU at one workgroup and take 10.4 / 11.8 / 13.0 / 19.7 / 32 us at K =
// 1024 / 1536 / 2048 / 4096 / 8192: up to 512 workgroups here always (7.7 at 256 x 1024 x
// 2048); up to 768 past K = 1024 (256 x 2816, with a swish 11.4 / 11.6 / 11.9 / 16.5 / 26.1);
// above that with no post-op to walk and between (226 x 3552 11.6 / 12.1 / 12.8 / 18.3 / 31,
// with a swish 12.9 / 13.5 / 14.3 / 19.1 / 31.8; 128 x 8000 36.6 at 8192).
// f8_e4m3, 33 ... 64 rows (tiles / here): 33 x 4096 x 16384 31.1 / 22.9 (1024), 64 x 14336 x
// 16384 97.8 / 73.7, 64 x 8192 x 24576 69.1 / 62.2 (1536), 33 x 14336 x 24576 97.8 / 114,
// 33 x 4096 x 32768 34.6 / 41.5 (2048), 64 x 8192 x 65536 118.7 / 166.9.
bool gemv_b8_takes(int64_t M, int64_t N, int64_t K, bool f8, bool tile256, bool post_ops) {
    const int64_t wgs = (M + 31) / 32 * ((N + 31) / 32);
    if (M <= (f8 ? 32 : 64)) return true;
    if (M <= 64) return wgs <= (K > 8192 ? 1024 : 1536);
    if (!tile256 && (M + 127) / 128 * ((N + 127) / 128) < 64) {
        if (wgs <= 512) return true;
        if (wgs <= 768) return K > 1024;
        return !f8 && !post_ops && K >= 2048 && K < 8192;
    }
    if (f8) return wgs <= (K >= 8192 ? 1024 : K > 4096 ? 1536 : K >= 2048 ? 2048 : 1344);
    return wgs <= (K >= 2048 ? 1344 : tile256 ? 960 : 1024);
}

// one batch; integer operands, or f8_e4m3 with K a multiple of 64 (the caller checks)
void launch_gemv_b8(const gemm_params_t &p, bool f8, hipStream_t stream) {
    if (p.M <= 0 || p.N <= 0) return;
    auto go = [&](auto kern, int64_t blocks, int lds) {
        if (lds > 65536) ensure_dynamic_lds((const void *)kern, lds);
        hipLaunchKernelGGL(
                kern, dim3((unsigned)blocks), dim3(GB8_WAVES * 64), lds, stream, p);
    };
    constexpr int lds4 = GB8_WAVES * gb8_wave_lds(4), lds32 = GB8_WAVES * gb8_wave_lds(32);
    const int64_t grid32 = p.M > 32 ? gb8_grid((int)p.M, p.nb32) : p.nb32;
    if (p.M <= 4)
        f8 ? go(gemv_b8_kernel<4, true, false>, p.nb32, lds4)
           : go(gemv_b8_kernel<4, false, false>, p.nb32, lds4);
    else if (p.M <= 16)
        f8 ? go(gemv_b8_kernel<32, true, false>, p.nb32, lds32)
           : go(gemv_b8_kernel<32, false, false>, p.nb32, lds32);
    // 33 ... 64 rows as two blocks of 32 where these are at most one workgroup to a CU
    // (64 rows, us, two blocks / one of 64: 4096 x 4096 8.6 / 11.6, 14336 x 4096 20.8 /
    // 28.5, 1024 x 6144 7.5 / 6.5, 8192 x 8192 23.7 / 21.7, 4096 x 14336 23.1 / 22.6)
    else if (f8 || p.M <= 32 || p.M > 64 || p.nb32 <= 128)
        f8 ? go(gemv_b8_kernel<32, true, true>, grid32, lds32)
           : go(gemv_b8_kernel<32, false, true>, grid32, lds32);
    else
        go(gemv_b8_rows64_kernel, p.nb32, GB8_WAVES * 64 * (4 * 32 + 16));
}

} // namespace qmm

extern "C" int64_t qmm_gemv_b8_block(int64_t M, int64_t N, int64_t workgroup) {
    int nb = 0, m0 = 0;
    if (M <= 32 || M > 1 << 20 || N < 1 || N > 1 << 20 || workgroup < 0
            || workgroup >= qmm::gb8_grid((int)M, (int)((N + 31) / 32))
            || !qmm::gb8_block((int)M, (int)((N + 31) / 32), (int)workgroup, nb, m0))
        return -1;
    return (int64_t)m0 << 32 | nb;
}
