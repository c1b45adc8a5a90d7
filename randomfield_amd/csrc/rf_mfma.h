// rf_mfma.h -- shared by the matrix-core spectral sums (rf_mfma.hip,
// rf_lat.hip): operand types, the FP16/BF16 hi/lo split and the store of a
// wave's accumulator tiles.
#pragma once
#include "rf_internal.h"

namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef __bf16 b8 __attribute__((ext_vector_type(8)));
typedef float f16x __attribute__((ext_vector_type(16)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

template <typename V> struct Elem;
template <> struct Elem<h8> { typedef _Float16 T; };
template <> struct Elem<b8> { typedef __bf16 T; };

__device__ inline f16x mfma(const h8& a, const h8& b, const f16x& c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}
__device__ inline f16x mfma(const b8& a, const b8& b, const f16x& c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// (c, s) -> hi and lo halves at positions 2q, 2q+1 of the basis fragments.
// FP16: one packed conversion for hi, the residuals v - hi by mixed-precision
// FMAs reading the f16 halves in place (v_fma_mix_f32), one packed conversion
// for lo.  BF16: plain conversions.
template <typename V>
__device__ inline void split_pair(float c, float s, int q, V* bh, V* bl) {
    typedef typename Elem<V>::T T;
    const T ch = (T)c, sh = (T)s;
    (*bh)[2 * q] = ch;
    (*bh)[2 * q + 1] = sh;
    (*bl)[2 * q] = (T)(c - (float)ch);
    (*bl)[2 * q + 1] = (T)(s - (float)sh);
}
template <>
__device__ inline void split_pair<h8>(float c, float s, int q, h8* bh, h8* bl) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    const h2 hi = {(_Float16)c, (_Float16)s};        // v_cvt_pk_f16_f32 (RNE)
    const unsigned hb = __builtin_bit_cast(unsigned, hi);
    float lc, ls;
    asm("v_fma_mix_f32 %0, -%1, 1.0, %2 op_sel:[0,0,0] op_sel_hi:[1,0,0]" : "=v"(lc) : "v"(hb), "v"(c));
    asm("v_fma_mix_f32 %0, -%1, 1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(ls) : "v"(hb), "v"(s));
    (*bh)[2 * q] = hi.x;
    (*bh)[2 * q + 1] = hi.y;
    (*bl)[2 * q] = (_Float16)lc;
    (*bl)[2 * q + 1] = (_Float16)ls;
}

// The MT 32x32 accumulator tiles of a wave (point pt, M-tiles from mt0, lane
// half h) to the field.
template <int MT>
__device__ __forceinline__ void store_tiles(const rf_sum_args& a, const f16x* acc, float outScale, int64_t pt, int mt0,
                                            int h) {
    // D layout of a 32x32 tile: lane column n, rows 8*(r/4) + 4*h + r%4.
    // The marginal map and the output type are uniform: one store loop each,
    // so the common cases carry no exp evaluation or dtype select per value.
    auto store = [&](auto map, auto* out) {
#pragma unroll
        for (int m = 0; m < MT; m++) {
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int real = (mt0 + m) * 32 + 8 * (r >> 2) + 4 * h + (r & 3);
                if (real < a.Nmc) out[(int64_t)real * a.N + pt] = map(acc[m][r] * outScale);
            }
        }
    };
    const float sc = (float)a.epi.scale, sh = (float)a.epi.shift;
    auto none = [](float u) { return u; };
    auto gauss = [=](float u) { return fmaf(u, sc, sh); };
    auto logn = [=](float u) { return expf(fmaf(u, sc, sh)); };
    auto none64 = [](float u) { return (double)u; };
    auto gauss64 = [=](float u) { return (double)fmaf(u, sc, sh); };
    auto logn64 = [=](float u) { return (double)expf(fmaf(u, sc, sh)); };
    float* o32 = static_cast<float*>(a.out);
    double* o64 = static_cast<double*>(a.out);
    if (a.outDtype == RF_DTYPE_F64) {
        if (a.epi.margi == RF_FOM_NONE) store(none64, o64);
        else if (a.epi.margi == RF_FOM_LOGNORMAL) store(logn64, o64);
        else store(gauss64, o64);
    } else {
        if (a.epi.margi == RF_FOM_NONE) store(none, o32);
        else if (a.epi.margi == RF_FOM_LOGNORMAL) store(logn, o32);
        else store(gauss, o32);
    }
}

// The field of tile b of a grouped launch.
__device__ inline int group_find(const rf_group_req* __restrict__ reqs, int nReq, int64_t b) {
    int lo = 0, hi = nReq - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (reqs[mid].tile0 <= b) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

}  // namespace
