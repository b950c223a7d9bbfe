// What the attention kernels share: the launch parameters, the 16-bit MFMA and
// conversion by type, lane exchanges, and the 8-bit cache's dequantization.
#ifndef QMM_SDPA_HPP
#define QMM_SDPA_HPP

#include <hip/hip_runtime.h>

#include "qmm_device.hpp"
#include "qmm_hip.h"

namespace qmm {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));

typedef short v4s __attribute__((ext_vector_type(4)));
typedef __bf16 v8b __attribute__((ext_vector_type(8)));

// BF: the 16-bit type of Q, K, V and dst is bf16 (else f16). Operands travel
// as raw 16-byte vectors; only the MFMA and the conversions know the type.
template <bool BF>
QMM_D v4f mma16(const v8h &a, const v8h &b, const v4f &c) {
    if constexpr (BF)
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                __builtin_bit_cast(v8b, a), __builtin_bit_cast(v8b, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}
template <bool BF>
QMM_D _Float16 cvt16(float v) { // the bits of v in the 16-bit type, carried as _Float16
    if constexpr (BF)
        return __builtin_bit_cast(_Float16, (__bf16)v); // v_cvt_pk_bf16_f32
    else
        return (_Float16)v;
}

struct sdpa_strides_t {
    int64_t b0, b1, row; // two outer dims, then the row dim (elements)
};

struct sdpa_params_t {
    const uint16_t *Q;
    const void *K, *V;
    uint16_t *dst;
    const void *mask; // nullptr: none
    const void *scale; // nullptr: 1
    const void *k_scale, *k_zp, *v_scale, *v_zp; // per (kv batch, key)
    sdpa_strides_t q, k, v, o, m;
    int64_t m_col; // mask stride over keys (0 or 1)
    int32_t B0, B1; // outer dims of Q / dst
    int32_t kv_div0, kv_div1; // q batch index / div = kv batch index
    int64_t qz_b0, qz_b1; // scale / zero-point index = kb0 * qz_b0 + kb1 * qz_b1 + key
    int32_t Qn, S;
    int32_t scale_dt, mask_dt, invert_scale, causal;
    int32_t kv_dt; // the queries' type, or dt_s8 / dt_u8
    int32_t ks_dt, kz_dt, vs_dt, vz_dt;
    int32_t pair_halves; // the grid fits the chip at once: see the kernel
    // few queries (decode): the keys are cut into nsplit ranges of tps tiles
    int32_t nsplit, tps;
    int32_t fastq, bf; // f16 scales and 8-bit zero points: f16 dequantisation
    int32_t pack; // few queries: heads of one K / V head that share a workgroup
    int32_t packs; // B1 / pack
    float *part; // [head][split], part_pitch each: [query][D + 2]: O (unnormalised), m, l
};

// Lanes that differ only in their 16-lane row hold parts of one query. The two
// exchange steps (row r <-> r ^ 1, half <-> other half) as vector-ALU lane
// swaps: v_permlane16_swap returns (rows 0 0 2 2, rows 1 1 3 3) of its two
// inputs' rows, v_permlane32_swap (lower lower, upper upper) halves; with both
// inputs the same value the two results are the partners of a butterfly.
typedef unsigned v2u __attribute__((ext_vector_type(2)));
QMM_D float rows_max(float v) {
    unsigned u = f2u(v);
    const v2u a = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    u = f2u(fmaxf(u2f(a.x), u2f(a.y)));
    const v2u b = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return fmaxf(u2f(b.x), u2f(b.y));
}
QMM_D float rows_sum(float v) {
    unsigned u = f2u(v);
    const v2u a = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    u = f2u(u2f(a.x) + u2f(a.y));
    const v2u b = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return u2f(b.x) + u2f(b.y);
}

// the mask is f32 or one of the 16-bit types
QMM_D float ld_mask(int dt, const void *p, int64_t i) {
    if (dt == dt_f32) return ((const float *)p)[i];
    const uint16_t h = ((const uint16_t *)p)[i];
    return dt == dt_bf16 ? __uint_as_float((uint32_t)h << 16)
                         : (float)__builtin_bit_cast(_Float16, h);
}

// the cache's scales are f16 or f32, its zero points s8, u8 or s32
QMM_D float ld_scale(int dt, const void *p, int64_t i) {
    return dt == dt_f16 ? (float)((const _Float16 *)p)[i] : ((const float *)p)[i];
}
QMM_D float ld_zp(int dt, const void *p, int64_t i) {
    return dt == dt_s8  ? (float)((const int8_t *)p)[i]
            : dt == dt_u8 ? (float)((const uint8_t *)p)[i]
                          : (float)((const int32_t *)p)[i];
}

// Eight cache bytes -> eight f16 values scale * (x - zero_point), in f16
// arithmetic: byte b behind the exponent pattern 0x64 is the f16 number
// 1024 + b, (1024 + b) - (1024 + z) is exact (integers up to 2048 are f16
// numbers), and an f16 scale times that small integer has at most 20
// significant bits, so rounding the f16 product is the same single rounding as
// f16(f32 product): the values of the reference's dequantizing reorder, at 1.5
// instructions per element. `raw`: bytes with the sign bit already flipped for
// s8; sc: the scale twice; off: 1024 + zero point (+ 128 for s8), twice: an integer
// within [896, 1407], so that off and every difference (at most 383 away from 0) are
// f16 numbers.
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
QMM_D h2 twice(float v) {
    return h2 {(_Float16)v, (_Float16)v};
}
QMM_D uint4 dequant8_f16(uint32_t w0, uint32_t w1, const h2 &sc, const h2 &off) {
    const uint32_t w[2] = {w0, w1};
    uint32_t o[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const uint32_t m = __builtin_amdgcn_perm(
                0x64646464u, w[j >> 1], (j & 1) ? 0x04030402u : 0x04010400u);
        const h2 v = (__builtin_bit_cast(h2, m) - off) * sc;
        o[j] = __builtin_bit_cast(uint32_t, v);
    }
    return make_uint4(o[0], o[1], o[2], o[3]);
}

// many queries without an explicit mask (qmm_sdpa_prefill.hip); scratch: what
// sdpa_prefill_scratch asks for, an 8-bit cache in the queries' type
bool sdpa_prefill_takes(const sdpa_params_t &p, int D);
size_t sdpa_prefill_scratch(const sdpa_params_t &p, int D);
bool sdpa_prefill_launch(const sdpa_params_t &p, int D, void *scratch, void *hip_stream);

} // namespace qmm

#endif
