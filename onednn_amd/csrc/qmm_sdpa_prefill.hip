// Scaled dot-product attention over many queries, K and V in the queries' 16-bit
// type (or written in it first), head sizes 64 and 128, causal or not, no explicit
// mask (the rest: qmm_sdpa.hip, which also describes the arithmetic).
//
// A workgroup owns 128 queries of a head; its eight waves are two groups of four,
// a wave 32 queries, and the groups take the keys' tiles of 64 in turn, each with
// statistics and accumulators of its own, merged at the end through LDS. That
// keeps two waves on every SIMD to the end of a long causal walk, and the two are
// held half a step apart by the barriers: one multiplies (the scores of a tile and
// the values of the tile before) while the other forms its probabilities, so that
// the matrix cores and the vector ALU work at the same time.
//   * S^T = K x Q^T and O^T += V^T x P^T on 32 x 32 x 16 MFMAs: a lane holds 16 of
//     32 keys' scores of ONE query, its statistics need one lane exchange, and the
//     probabilities packed to 16 bits are the second operand of the other product
//     (k index 8 h + i <-> key 4 h + i for i < 4, 8 + 4 h + i - 4 otherwise, h the
//     half of the wave);
//   * K and V tiles come by direct global -> LDS loads, two buffers each, requested in
//     the vector slot before the one they are needed in; the fragments of a matrix
//     slot are read four products ahead;
//   * the accumulators are rescaled whenever a maximum grew, so that the largest
//     probability is exactly 1. Letting it lag (up to 2^8) from 2048 keys on gained
//     2 ... 4 % at 4096 ... 16384 keys and cost precision: where one late key outweighs
//     the rest, its rounded weight no longer is what the sum has of it.
// Bound: the power limit (1.5 GHz in a long run, matrix cores busy 57 % of its
// cycles) and, below that, the vector ALU: a wave alone issues one instruction in
// about 5 cycles, and the probabilities of a slot are about 190 of them next to
// 1024 cycles of MFMAs; a workgroup's start takes 3.9 us, its end 1.4.
// Measured (us; the kernel of qmm_sdpa.hip / this one, launches back to back): causal,
// f16, 32 heads x 2048 tokens of 128 84.5 / 49.3, x 1000 46.6 / 24.8, 16 x 320 17.3 /
// 11.1, 4 x 100 10.4 / 8.7; bf16, 8 x 3500 of 128 135.8 / 52.7, 32 x 666 of 64 20.5 /
// 13.2, 32 x 155 of 64 8.4 / 7.0; f16, 40 over 4 K / V heads x 4096 of 64 154.8 / 144.
// Not kept: workgroups that stay and walk several query tiles with the next one's
// loads under way (49.6), the loads spread between the products (the same), products
// and probabilities interleaved in one stream (57.7: the compiler keeps to neither
// order), both waves of a SIMD in step (56).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "qmm_plan.hpp"
#include "qmm_sdpa.hpp"

namespace qmm {
namespace {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef short v8s __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) uint8_t lds_u8;

template <bool BF>
QMM_D v16f mma32(const v8h &a, const v8h &b, const v16f &c) {
    if constexpr (BF)
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                __builtin_bit_cast(v8b, a), __builtin_bit_cast(v8b, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}
template <bool BF>
QMM_D uint32_t cvt_pair(float a, float b) {
    if constexpr (BF) {
        typedef __bf16 b2 __attribute__((ext_vector_type(2)));
        return __builtin_bit_cast(uint32_t, b2 {(__bf16)a, (__bf16)b});
    } else
        return __builtin_bit_cast(uint32_t, h2 {(_Float16)a, (_Float16)b});
}

QMM_D void dma16(uint32_t lds_addr, uint32_t voff, const uint8_t *sbase) {
    asm volatile("s_mov_b32 m0, %0\n\t"
                 "s_nop 0\n\t"
                 "global_load_lds_dwordx4 %1, %2" ::"s"(lds_addr),
                 "v"(voff), "s"(sbase)
                 : "m0");
}
QMM_D const uint8_t *uniform_ptr(const uint8_t *q) {
    const uint64_t v = (uint64_t)q;
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return (const uint8_t *)(((uint64_t)hi << 32) | lo);
}
// a barrier that waits for nothing but the waves; nothing is moved across it
QMM_D void phase_barrier() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}
template <int N>
QMM_D void wait_loads() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

constexpr int QW = 4, KT = 64; // waves of a group, 32 queries each; keys of a tile

template <int DC, bool BF>
__global__ void __launch_bounds__(512, 2)
sdpa_prefill_kernel(const sdpa_params_t p) {
    constexpr int D = 32 * DC, ROW = D * 2; // bytes of a row
    constexpr int KG = 8 / QW; // groups of waves that share the keys
    constexpr int KB = KT / 32; // blocks of 32 keys
    constexpr int CH = D / 8; // 16-byte chunks of a row
    constexpr int TILE = KT * ROW;
    constexpr int GROUP = 4 * TILE; // K twice, V twice
    constexpr int NL = TILE / 1024 / QW; // loads of a wave and tile
    constexpr int RPL = 1024 / ROW; // rows of a load
    constexpr int QUADS = 4 * DC, OWN = QUADS / KG; // see the end
    typedef __attribute__((address_space(3))) v8h lds_v8h;
    typedef __attribute__((address_space(3))) v4s lds_v4s;
    typedef __attribute__((address_space(3))) float lds_f;
    typedef __attribute__((address_space(3))) v4f lds_v4f;
    typedef uint32_t v4u __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) v4u lds_v4u;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = wave / QW, qw = wave % QW;
    const int c = lane & 31, h = lane >> 5;

    const uint32_t lds_base = __builtin_amdgcn_readfirstlane(
            (uint32_t)(uintptr_t)(lds_u8 *)lds);
    const uint32_t gbase = lds_base + g * GROUP;
    const uint32_t k_row = (uint32_t)p.k.row * 2, v_row = (uint32_t)p.v.row * 2;

    // ---- direct loads of 1 KiB. LDS row i holds tile row i, its 16-byte chunk x at
    // x ^ k_swz(i) or x ^ v_swz(i): the 16 lanes of a K fragment that are read at a
    // time (16 rows, one chunk) and the 32 of a transposing V read (4 rows, 4 chunks)
    // then lie in different 16 bytes of the 256 that LDS delivers. A wave's loads are
    // 4 RPL rows apart, which neither sees, so they share one address
    auto k_swz = [](int i) { return D == 128 ? i & 15 : (i >> 1) & 7; };
    auto v_swz = [](int i) { return D == 128 ? 4 * (i & 3) : 4 * ((i >> 1) & 1); };
    const int l_row = qw * RPL + lane / CH, l_ch = lane % CH;
    const uint32_t k_ch = (l_ch ^ k_swz(l_row)) * 16, v_ch = (l_ch ^ v_swz(l_row)) * 16;
    const uint32_t k_vo = l_row * k_row + k_ch, v_vo = l_row * v_row + v_ch;
    auto load = [&](const uint8_t *base, uint32_t row_bytes, uint32_t vo, uint32_t ch,
                        uint32_t dst, int kt) {
        const int key0 = kt * KT;
        dst += qw * 1024;
        if (key0 + KT <= p.S) {
            const uint8_t *sb = base + (uint64_t)key0 * row_bytes;
#pragma unroll
            for (int j = 0; j < NL; j++)
                dma16(dst + j * (QW * 1024), vo,
                        sb + (uint64_t)(j * QW * RPL) * row_bytes);
        } else {
#pragma unroll
            for (int j = 0; j < NL; j++)
                dma16(dst + j * (QW * 1024),
                        (uint32_t)min(key0 + j * QW * RPL + l_row, p.S - 1) * row_bytes
                                + ch,
                        base);
        }
    };

    // LDS addresses of the fragments, up to immediate offsets
    uint32_t ka[2 * DC], va[DC];
#pragma unroll
    for (int dc = 0; dc < 2 * DC; dc++)
        ka[dc] = gbase + c * ROW + (((2 * dc + h) ^ k_swz(c)) * 16);
    {
        const int j = lane & 15, s = (lane >> 4) & 1;
        const int row = 4 * h + (j >> 2);
#pragma unroll
        for (int db = 0; db < DC; db++)
            va[db] = gbase + 2 * TILE + row * ROW
                    + (((4 * db + 2 * s + ((j & 3) >> 1)) ^ v_swz(row)) * 16)
                    + (j & 1) * 8;
    }

    const int b1 = blockIdx.x % p.B1, b0 = blockIdx.x / p.B1;
    const int kb0 = b0 / p.kv_div0, kb1 = b1 / p.kv_div1;
    // heads first, the longest walks of a causal mask first: as workgroups end, the
    // next ones in that order take their CUs, the shortest last
    const int q_wg = (int)(gridDim.y - 1 - blockIdx.y) * (32 * QW);
    const int q_wave = q_wg + qw * 32;
    const uint8_t *Kp = uniform_ptr((const uint8_t *)((const uint16_t *)p.K
            + kb0 * p.k.b0 + kb1 * p.k.b1));
    const uint8_t *Vp = uniform_ptr((const uint8_t *)((const uint16_t *)p.V
            + kb0 * p.v.b0 + kb1 * p.v.b1));
    int n_keys = p.S;
    if (p.causal) n_keys = min(n_keys, min(q_wg + 32 * QW, p.Qn));
    const int n_tiles = (n_keys + KT - 1) / KT, steps = (n_tiles + KG - 1) / KG;
    auto load_k = [&](int t) {
        const int kt = t * KG + g;
        if (kt < n_tiles) load(Kp, k_row, k_vo, k_ch, gbase + (t & 1) * TILE, kt);
    };
    auto load_v = [&](int t) {
        const int kt = t * KG + g;
        if (kt < n_tiles) load(Vp, v_row, v_vo, v_ch, gbase + (2 + (t & 1)) * TILE, kt);
    };
    load_k(0);
    load_v(0);
    load_k(1);

    v8h qf[2 * DC];
    {
        const int q = min(q_wave + c, p.Qn - 1);
        const uint16_t *Qr = p.Q + b0 * p.q.b0 + b1 * p.q.b1 + q * p.q.row + h * 8;
#pragma unroll
        for (int dc = 0; dc < 2 * DC; dc++) qf[dc] = *(const v8h *)(Qr + dc * 16);
    }
    float sc = 1.f;
    if (p.scale) {
        sc = load_float(p.scale_dt, p.scale, 0);
        if (p.invert_scale) sc = 1.f / sc;
    }
    const float sc2 = sc * 1.44269504088896340736f;

    // whether the wave has anything to do with tile kt
    auto wanted = [&](int kt) {
        return kt < n_tiles && !(p.causal && kt * KT > q_wave + 31);
    };
    v16f oacc[DC], st[KB];
#pragma unroll
    for (int d = 0; d < DC; d++)
#pragma unroll
        for (int i = 0; i < 16; i++) oacc[d][i] = 0.f;
    v8h pb[2 * KB];
    float m_run = -INFINITY, l_run = 0.f;
    bool have_p = false, half = false;

    // ---- one slot of matrix work: the scores of tile t, then the values of t - 1
    auto scores = [&](auto par_tag) {
        constexpr int par = decltype(par_tag)::value;
#pragma unroll
        for (int kb = 0; kb < KB; kb++)
#pragma unroll
            for (int i = 0; i < 16; i++) st[kb][i] = 0.f;
#pragma unroll
        for (int dc = 0; dc < 2 * DC; dc++)
#pragma unroll
            for (int kb = 0; kb < KB; kb++) {
                const v8h a = *(const lds_v8h *)(uintptr_t)(ka[dc] + par * TILE
                        + kb * 32 * ROW);
                st[kb] = mma32<BF>(a, qf[dc], st[kb]);
            }
    };
    // one slot of matrix work: the scores of the tile after the one whose
    // values are due (past the wave's last tile they are formed and not used),
    // fragments read AHEAD products ahead
    auto matrix = [&](auto par_tag) {
        constexpr int par = decltype(par_tag)::value;
        constexpr int NS = 2 * DC * KB, N = NS + 2 * KB * DC;
        constexpr int AHEAD = 4;
        if (!have_p) return;
        auto fragment = [&](int i) {
            if (i < NS)
                return *(const lds_v8h *)(uintptr_t)(ka[i / KB] + par * TILE
                        + i % KB * 32 * ROW);
            const uint32_t at = va[(i - NS) % DC] + (1 - par) * TILE
                    + (i - NS) / DC * 16 * ROW;
            const v4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    (lds_v4s *)(uintptr_t)at);
            const v4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    (lds_v4s *)(uintptr_t)(at + 8 * ROW));
            return __builtin_bit_cast(v8h,
                    v8s {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]});
        };
        v8h f[AHEAD];
#pragma unroll
        for (int i = 0; i < AHEAD; i++) f[i] = fragment(i);
#pragma unroll
        for (int kb = 0; kb < KB; kb++)
#pragma unroll
            for (int i = 0; i < 16; i++) st[kb][i] = 0.f;
        __builtin_amdgcn_sched_barrier(0);
        auto product = [&](int i) {
            if (i < NS)
                st[i % KB] = mma32<BF>(f[i % AHEAD], qf[i / KB], st[i % KB]);
            else
                oacc[(i - NS) % DC] = mma32<BF>(
                        f[i % AHEAD], pb[(i - NS) / DC], oacc[(i - NS) % DC]);
            if (i + AHEAD < N) f[i % AHEAD] = fragment(i + AHEAD);
            __builtin_amdgcn_sched_barrier(0);
        };
#pragma unroll
        for (int i = 0; i < N - 2 * DC; i++) product(i);
        if (half) return;
#pragma unroll
        for (int i = N - 2 * DC; i < N; i++) product(i);
    };

    // ---- one slot of vector work: the probabilities of tile t
    auto softmax = [&](int t) {
        const int key0 = (t * KG + g) * KT;
        load_v(t + 1);
        load_k(t + 2);
        have_p = wanted(t * KG + g);
        // the tile's last 32 keys, hidden from every query of the wave, stay out of the
        // products: probability 0 times a value that is not finite would be NaN
        half = p.causal && key0 + 32 > q_wave + 31;
        if (have_p) {
            const bool edge = key0 + KT > p.S
                    || (p.causal && key0 + KT - 1 > q_wave) || !(sc2 > 0.f);
            float mul = sc2;
            if (edge) {
                // scaled scores, hidden keys at -inf
                mul = 1.f;
                const int q = q_wave + c;
                const int last = (p.causal ? min(q, p.S - 1) : p.S - 1) - key0 - 4 * h;
#pragma unroll
                for (int kb = 0; kb < KB; kb++)
#pragma unroll
                    for (int i = 0; i < 16; i++) {
                        const int key = 32 * kb + 8 * (i >> 2) + (i & 3);
                        st[kb][i] = key > last ? -INFINITY : st[kb][i] * sc2;
                    }
            }
            float mx = st[0][0];
#pragma unroll
            for (int kb = 0; kb < KB; kb++)
#pragma unroll
                for (int i = 0; i < 16; i++) mx = fmaxf(mx, st[kb][i]);
            {
                const unsigned u = f2u(mx);
                const v2u x = __builtin_amdgcn_permlane32_swap(u, u, false, false);
                mx = fmaxf(u2f(x.x), u2f(x.y)) * mul;
            }
            if (__builtin_amdgcn_ballot_w64(mx > m_run)) {
                const float m_new = fmaxf(m_run, mx);
                const float alpha = m_new == -INFINITY
                        ? 1.f
                        : __builtin_amdgcn_exp2f(m_run - m_new);
                m_run = m_new;
                l_run *= alpha;
#pragma unroll
                for (int d = 0; d < DC; d++) oacc[d] *= alpha;
            }
            const float m_neg = m_run == -INFINITY ? 0.f : -m_run;
            float ls = 0.f;
#pragma unroll
            for (int kb = 0; kb < KB; kb++)
#pragma unroll
                for (int i = 0; i < 16; i += 8) {
                    uint32_t w[4];
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        const float e0 = __builtin_amdgcn_exp2f(__builtin_fmaf(
                                st[kb][i + 2 * k], mul, m_neg));
                        const float e1 = __builtin_amdgcn_exp2f(__builtin_fmaf(
                                st[kb][i + 2 * k + 1], mul, m_neg));
                        ls += e0;
                        ls += e1;
                        w[k] = cvt_pair<BF>(e0, e1);
                    }
                    pb[2 * kb + i / 8] = __builtin_bit_cast(
                            v8h, v4u {w[0], w[1], w[2], w[3]});
                }
            l_run += ls;
        }
        // tile t of V and t + 1 of K have landed: all but this slot's loads
        if ((t + 2) * KG + g < n_tiles)
            wait_loads<2 * NL>();
        else if ((t + 1) * KG + g < n_tiles)
            wait_loads<NL>();
        else
            wait_loads<0>();
        if (key0 < p.S && key0 + KT > p.S) {
            // keys past the end: zero, so that probability 0 x V stays 0
#pragma unroll
            for (int j = 0; j < NL; j++)
                if (key0 + j * QW * RPL + l_row >= p.S)
                    *(lds_v4u *)(uintptr_t)(gbase + (2 + (t & 1)) * TILE
                            + (j * QW + qw) * 1024 + lane * 16)
                            = v4u {0, 0, 0, 0};
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        }
    };

    // K's first tile and the queries (consumed here, so that no wait for them
    // stands between the products)
#pragma unroll
    for (int dc = 0; dc < 2 * DC; dc++) asm volatile("" : "+v"(qf[dc]));
    wait_loads<0>();
    phase_barrier();
    // the two waves of a SIMD half a step apart: one multiplies while the other
    // forms its probabilities
    if (wave >= 4) phase_barrier();
    const std::integral_constant<int, 0> even;
    const std::integral_constant<int, 1> odd;
    if (wanted(g)) scores(even);
    for (int t = 0;; t += 2) {
        phase_barrier();
        softmax(t);
        phase_barrier();
        matrix(odd);
        if (t + 1 >= steps) break;
        phase_barrier();
        softmax(t + 1);
        phase_barrier();
        matrix(even);
        if (t + 2 >= steps) break;
    }
    if (wave < 4) phase_barrier();
    phase_barrier(); // every tile has been read

    // ---- merge the groups' states, in the LDS that V's tiles had: per wave the
    // accumulators that other groups finish, a quad [lane][4] each, then maxima
    // and sums
    {
        const unsigned u = f2u(l_run);
        const v2u x = __builtin_amdgcn_permlane32_swap(u, u, false, false);
        l_run = u2f(x.x) + u2f(x.y);
    }
    auto quad_at = [&](int w, int slot) { // slot: the quad's place among the sent
        return lds_base + (w / QW) * GROUP + 2 * TILE
                + ((w % QW) * (QUADS - OWN) + slot) * 1024;
    };
    const uint32_t ml = lds_base + KG * GROUP; // [wave][32 queries], twice
    if (h == 0) {
        *(lds_f *)(uintptr_t)(ml + (wave * 32 + c) * 4) = m_run;
        *(lds_f *)(uintptr_t)(ml + 1024 + (wave * 32 + c) * 4) = l_run;
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    phase_barrier();
    float m_all = -INFINITY, l_all = 0.f, mg[KG];
#pragma unroll
    for (int i = 0; i < KG; i++) {
        mg[i] = *(lds_f *)(uintptr_t)(ml + ((i * QW + qw) * 32 + c) * 4);
        m_all = fmaxf(m_all, mg[i]);
    }
    const float m_use = m_all == -INFINITY ? 0.f : m_all;
#pragma unroll
    for (int i = 0; i < KG; i++)
        l_all += __builtin_amdgcn_exp2f(mg[i] - m_use)
                * *(lds_f *)(uintptr_t)(ml + 1024 + ((i * QW + qw) * 32 + c) * 4);
    const float mine = __builtin_amdgcn_exp2f(m_run - m_use);
#pragma unroll
    for (int d = 0; d < DC; d++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int quad = 4 * d + j, owner = quad / OWN;
            if (owner != g)
                *(lds_v4f *)(uintptr_t)(quad_at(wave, quad - (owner > g ? OWN : 0))
                        + lane * 16)
                        = v4f {oacc[d][4 * j] * mine, oacc[d][4 * j + 1] * mine,
                                oacc[d][4 * j + 2] * mine, oacc[d][4 * j + 3] * mine};
        }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    phase_barrier();
    const int q = q_wave + c;
    uint16_t *Or = p.dst + b0 * p.o.b0 + b1 * p.o.b1 + (int64_t)q * p.o.row;
    const float inv = 1.f / l_all;
    auto finish = [&](int d, int j) {
        const int quad = 4 * d + j;
        v4f o = v4f {oacc[d][4 * j] * mine, oacc[d][4 * j + 1] * mine,
                oacc[d][4 * j + 2] * mine, oacc[d][4 * j + 3] * mine};
#pragma unroll
        for (int i = 1; i < KG; i++) {
            const int og = (g + i) % KG;
            o += *(lds_v4f *)(uintptr_t)(quad_at(og * QW + qw,
                                                 quad - (g > og ? OWN : 0))
                    + lane * 16);
        }
        return make_uint2(cvt_pair<BF>(o[0] * inv, o[1] * inv),
                cvt_pair<BF>(o[2] * inv, o[3] * inv));
    };
#pragma unroll
    for (int d = 0; d < DC; d++)
#pragma unroll
        for (int j = 0; j < 4; j += 2) {
            if ((4 * d + j) / OWN != g) continue;
            const uint2 x = finish(d, j), y = finish(d, j + 1);
            // lane half 0: columns 8 j .. + 7 of the block, half 1: the next eight
            const v2u s0 = __builtin_amdgcn_permlane32_swap(x.x, y.x, false, false);
            const v2u s1 = __builtin_amdgcn_permlane32_swap(x.y, y.y, false, false);
            typedef uint32_t v4ua __attribute__((ext_vector_type(4), aligned(8)));
            if (q < p.Qn)
                *(v4ua *)(Or + d * 32 + j * 8 + h * 8)
                        = v4ua {s0.x, s1.x, s0.y, s1.y};
        }
}

// An 8-bit cache for the kernel above: K and V as dense [head][key][D] arrays of the
// queries' type, with the values (and the arithmetic) of the kernels that dequantize
// while they stage. Bound: HBM; one pass here instead of one per 128 queries there.
template <bool BF>
__global__ void __launch_bounds__(256)
sdpa_dequant_kernel(const sdpa_params_t p, int D, int kv1, uint16_t *K, uint16_t *V) {
    const int per_row = D / 8;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (int64_t)p.S * per_row) return;
    const int key = (int)(i / per_row), ch = (int)(i % per_row);
    const int kb0 = blockIdx.y / kv1, kb1 = blockIdx.y % kv1;
    const bool v = blockIdx.z != 0;
    const sdpa_strides_t &st = v ? p.v : p.k;
    const uint2 w = *(const uint2 *)((const uint8_t *)(v ? p.V : p.K) + kb0 * st.b0
            + kb1 * st.b1 + (int64_t)key * st.row + ch * 8);
    const int64_t qi = kb0 * p.qz_b0 + kb1 * p.qz_b1 + key;
    const void *sp = v ? p.v_scale : p.k_scale, *zp = v ? p.v_zp : p.k_zp;
    const float s = sp ? ld_scale(v ? p.vs_dt : p.ks_dt, sp, qi) : 1.f;
    const float z = zp ? ld_zp(v ? p.vz_dt : p.kz_dt, zp, qi) : 0.f;
    const bool sgn = p.kv_dt == dt_s8;
    const uint32_t flip = sgn ? 0x80808080u : 0u;
    const float zb = z + (sgn ? 128.f : 0.f);
    const uint32_t b[2] = {w.x ^ flip, w.y ^ flip};
    uint4 o;
    if (p.fastq) {
        o = dequant8_f16(b[0], b[1], twice(s), twice(1024.f + zb));
    } else {
        float f[8];
#pragma unroll
        for (int j = 0; j < 8; j++)
            f[j] = s * ((float)((b[j >> 2] >> (8 * (j & 3))) & 0xff) - zb);
        o = make_uint4(cvt_pair<BF>(f[0], f[1]), cvt_pair<BF>(f[2], f[3]),
                cvt_pair<BF>(f[4], f[5]), cvt_pair<BF>(f[6], f[7]));
    }
    *(uint4 *)((v ? V : K) + ((int64_t)blockIdx.y * p.S * D + i * 8)) = o;
}

} // namespace

// Keys from which the kernel beats that of qmm_sdpa.hip. Its workgroups of eight waves
// take longer to start and to merge, two fit a CU at head size 64 and one at 128, and
// what they gain is the shorter walk: alone on a CU one wins from 97 keys on (causal 33;
// 8 heads x 512, us, there / here: 64 keys of 128 7.9 / 8.2, 128 10.3 / 9.2, 700 32.7 /
// 17.0), with n of them to a CU only from a longer walk on, since the other kernel's
// small workgroups then hide each other's latency. Head size 64: 512 workgroups x 320
// keys 16.2 / 17.2, x 512 22.4 / 21.0; 768 x 640 35.4 / 35.6; 1024 x 512 38.2 / 40.7,
// x 1024 64.9 / 63.2; 2048 x 1024 119.7 / 124.0, x 2048 226.4 / 218.8; causal, 256 heads
// x 256 13.7 / 16.8, 512 x 512 50.7 / 72.1, 64 x 2048 70.8 / 67.3, 128 x 2048 127.1 /
// 134.9, x 4096 470 / 462. Head size 128: 512 x 256 22.5 / 23.5, x 400 30.4 / 30.3;
// 1024 x 512 61.0 / 61.9, x 640 72.6 / 70.4; 2048 x 700 149.9 / 157.1, x 1024 206 / 199;
// causal, 256 heads x 512 46.7 / 61.5, 128 x 700 40.0 / 47.0, 64 x 1400 65.3 / 57.8,
// 256 x 2048 461 / 461, 128 x 4096 802 / 724. bf16 alike.
//
// An 8-bit cache is dequantized into the scratchpad first, from 257 queries on: a second
// launch and the scratchpad's order cost 8 us, dequantizing while staging, which the
// other kernel does once per 128 queries, more the more keys there are (us, there / here,
// s8, f16). Head size 64: 8 heads x 300 queries x 64 keys 7.0 / 13.9, x 256 14.6 / 15.3,
// x 300 17.6 / 16.8; causal, 128 heads x 400 24.3 / 25.2, x 600 38.2 / 33.7, 256 x 600
// 48.2 / 57.9, x 900 92.0 / 102, x 2048 319 / 297, 64 x 4096 queries x 384 67.9 / 74.2,
// x 512 85.0 / 84.3. Head size 128: 32 over 8 heads x 300 x 64 10.1 / 17.7, x 150 17.1 /
// 19.2, x 200 21.4 / 19.7, x 4096 343 / 67; 64 x 4096 x 128 72.8 / 76.0, x 256 116 / 93.9.
static bool walk_is_long(const sdpa_params_t &p, int D, bool dequant) {
    const int64_t n = ((int64_t)p.B0 * p.B1 * ((p.Qn + 127) / 128) + 255) / 256;
    const double S = p.causal ? std::min(p.S, p.Qn) : p.S;
    // the mean over the workgroups
    const double walk = p.causal ? S * (1 - S / (2.0 * p.Qn)) + 64 : S;
    if (dequant) {
        if (D == 128) return walk > 160;
        return n <= 1 ? S > 280 : walk > std::min(p.causal ? 800.0 : 500.0, 70.0 * n + 150);
    }
    if (n <= 1) return S > (p.causal ? 32 : 96);
    if (D == 64) return walk > (n == 2 ? (p.causal ? 264 : 420) : std::min(1800.0, 275.0 * n - 250));
    return walk > (n == 2 ? 315 : n == 3 ? 570 : std::min(1000.0, 120.0 * n + 100));
}

// byte offsets inside a head have 32 bits here; at most 256 MiB of scratchpad
bool sdpa_prefill_takes(const sdpa_params_t &p, int D) {
    if ((D != 64 && D != 128) || p.mask_dt != dt_undef || p.Qn <= 16) return false;
    if (p.kv_dt == (p.bf ? dt_bf16 : dt_f16))
        return (int64_t)p.S * p.k.row * 2 < (int64_t)1 << 31
                && (int64_t)p.S * p.v.row * 2 < (int64_t)1 << 31 && walk_is_long(p, D, false);
    const int64_t heads = (int64_t)(p.B0 / p.kv_div0) * (p.B1 / p.kv_div1);
    return p.Qn > 256 && heads <= 65535 && heads * p.S * D * 4 <= (int64_t)256 << 20
            && walk_is_long(p, D, true);
}

size_t sdpa_prefill_scratch(const sdpa_params_t &p, int D) {
    if (!sdpa_prefill_takes(p, D) || p.kv_dt == (p.bf ? dt_bf16 : dt_f16)) return 0;
    return (size_t)(p.B0 / p.kv_div0) * (p.B1 / p.kv_div1) * p.S * D * 4;
}

bool sdpa_prefill_launch(
        const sdpa_params_t &p0, int D, void *scratch, void *hip_stream) {
    sdpa_params_t p = p0;
    const dim3 grid((unsigned)(p.B0 * p.B1), (unsigned)((p.Qn + 32 * QW - 1) / (32 * QW)));
    if (grid.y > 65535) return false;
    if (p.kv_dt != (p.bf ? dt_bf16 : dt_f16)) {
        if (!scratch) return false;
        const int kv0 = p.B0 / p.kv_div0, kv1 = p.B1 / p.kv_div1;
        uint16_t *const K = (uint16_t *)scratch, *const V = K + (int64_t)kv0 * kv1 * p.S * D;
        const dim3 dq((unsigned)(((int64_t)p.S * (D / 8) + 255) / 256), (unsigned)(kv0 * kv1), 2);
        if (p.bf)
            hipLaunchKernelGGL(sdpa_dequant_kernel<true>, dq, dim3(256), 0,
                    (hipStream_t)hip_stream, p, D, kv1, K, V);
        else
            hipLaunchKernelGGL(sdpa_dequant_kernel<false>, dq, dim3(256), 0,
                    (hipStream_t)hip_stream, p, D, kv1, K, V);
        p.K = K;
        p.V = V;
        p.k.row = p.v.row = D;
        p.k.b1 = p.v.b1 = (int64_t)p.S * D;
        p.k.b0 = p.v.b0 = (int64_t)kv1 * p.S * D;
    }
    const int lds = 8 / QW * 4 * KT * D * 2 + 2048;
    auto go = [&](auto kern) {
        ensure_dynamic_lds((const void *)kern, lds);
        hipLaunchKernelGGL(kern, grid, dim3(512), lds, (hipStream_t)hip_stream, p);
    };
    if (D == 128)
        p.bf ? go(sdpa_prefill_kernel<4, true>)
             : go(sdpa_prefill_kernel<4, false>);
    else
        p.bf ? go(sdpa_prefill_kernel<2, true>)
             : go(sdpa_prefill_kernel<2, false>);
    return true;
}

} // namespace qmm

extern "C" int qmm_sdpa_pipelined(int head_size, int causal, int64_t heads, int64_t kv_heads,
        int64_t queries, int64_t keys, int cache_8bit) {
    const int64_t top = 1 << 30;
    if (heads < 1 || kv_heads < 1 || heads > top || heads % kv_heads || queries < 1
            || queries > top || keys < 1 || keys > top)
        return 0;
    qmm::sdpa_params_t p = {};
    p.B0 = p.kv_div0 = 1;
    p.B1 = (int32_t)heads;
    p.kv_div1 = (int32_t)(heads / kv_heads);
    p.Qn = (int32_t)queries;
    p.S = (int32_t)keys;
    p.causal = causal;
    p.mask_dt = qmm::dt_undef;
    p.kv_dt = cache_8bit ? qmm::dt_s8 : qmm::dt_f16;
    p.k.row = p.v.row = head_size;
    return qmm::sdpa_prefill_takes(p, head_size);
}
