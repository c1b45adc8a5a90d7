// rf_grid_dev.h -- device helpers shared by the grid-form kernels (rf_grid.hip,
// rf_strip.hip): operand addressing, the FP16 hi/lo split, the fused blend's
// targets, the drawn coefficients and the placement of tiles.
#pragma once
#include "rf_internal.h"
#include "rf_philox.h"

namespace {

// element offsets of column n in B and in D (two-level when nLo > 0)
__device__ __forceinline__ int64_t col_b(const rf_gemm_desc& g, int n) {
    return g.nLo ? (int64_t)(n / g.nLo) * g.bSnHi + (int64_t)(n % g.nLo) * g.bSn : (int64_t)n * g.bSn;
}
__device__ __forceinline__ int64_t col_d(const rf_gemm_desc& g, int n) {
    return g.nLo ? (int64_t)(n / g.nLo) * g.dSnHi + (int64_t)(n % g.nLo) * g.dSn : (int64_t)n * g.dSn;
}

typedef float f32x16 __attribute__((ext_vector_type(16)));

typedef float f2v __attribute__((ext_vector_type(2)));
typedef const f2v __attribute__((address_space(1))) gf2;      // global-memory views
typedef f2v __attribute__((address_space(1))) gf2o;
typedef float __attribute__((address_space(1))) gfo;
typedef double __attribute__((address_space(1))) gdo;
typedef float f4v __attribute__((ext_vector_type(4)));
typedef const f4v __attribute__((address_space(1))) gf4;
typedef _Float16 hv8 __attribute__((ext_vector_type(8)));
typedef _Float16 hv4 __attribute__((ext_vector_type(4)));

// Fused blend: the group-grid column offset of plane column n, or -1 where
// another field also covers it.
__device__ __forceinline__ int64_t grp_col(const rf_gemm_desc& g, int n) {
    const int x = n % g.grpNx, y = n / g.grpNx;
    return (x >= g.grpXlo && x < g.grpXhi && y >= g.grpYlo && y < g.grpYhi)
               ? g.grpCol0 + x + g.grpG0 * (int64_t)y : (int64_t)-1;
}
// Fused blend: plane column n inside a first-axis overlap band sits in the
// band array of its side (*side 0 low, 1 high) at element offset (return) +
// m * (*rowStride) for row m; -1 outside the bands.
// (selects, not early returns: the blend's lookup of the same bands was
// miscompiled in an if-return form)
__device__ __forceinline__ int64_t band_col(const rf_gemm_desc& g, int n, int batch, int* side, int* rowStride) {
    const int x = n % g.grpNx, y = n / g.grpNx;
    const int wLo = g.grpXlo, wHi = g.grpNx - g.grpXhi;
    const bool lo = g.bandLo != nullptr && x < g.grpXlo;
    const bool hi = !lo && g.bandHi != nullptr && x >= g.grpXhi;
    const int64_t offLo = (int64_t)batch * g.bandLoStrideB + (int64_t)y * wLo + x;
    const int64_t offHi = (int64_t)batch * g.bandHiStrideB + (int64_t)y * wHi + (x - g.grpXhi);
    *side = hi ? 1 : 0;
    *rowStride = lo ? g.grpNy * wLo : hi ? g.grpNy * wHi : 0;
    return lo ? offLo : hi ? offHi : (int64_t)-1;
}

// v -> FP16 hi (round to nearest) and lo = v - hi: packed conversions for
// hi and lo, the residuals by mixed-precision FMAs reading the f16 halves in
// place (v_fma_mix_f32), two instructions per value.
__device__ inline void split4(const float* v, hv4* hi, hv4* lo) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
#pragma unroll
    for (int i = 0; i < 4; i += 2) {
        const h2 h = {(_Float16)v[i], (_Float16)v[i + 1]};       // v_cvt_pk_f16_f32
        const unsigned hb = __builtin_bit_cast(unsigned, h);
        float l0, l1;
        asm("v_fma_mix_f32 %0, -%1, 1.0, %2 op_sel:[0,0,0] op_sel_hi:[1,0,0]" : "=v"(l0) : "v"(hb), "v"(v[i]));
        asm("v_fma_mix_f32 %0, -%1, 1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(l1) : "v"(hb), "v"(v[i + 1]));
        (*hi)[i] = h.x;
        (*hi)[i + 1] = h.y;
        (*lo)[i] = (_Float16)l0;
        (*lo)[i + 1] = (_Float16)l1;
    }
}

// cos and sin of 2 pi U for U in [0, 1): FP32 sincospi of the FP32 part Uh
// and the first-order term of the remainder U - Uh (|U - Uh| <= 2^-25), a few
// FP32 ulps from the FP64 values -- the coefficients are FP32.
__device__ __forceinline__ void cis_rev(double U, float* c, float* s) {
    const float uh = (float)U;
    const float ul = (float)(U - (double)uh);
    float sh, ch;
    sincospif(2.0f * uh, &sh, &ch);
    const float d = 6.28318530717958648f * ul;
    *s = fmaf(d, ch, sh);
    *c = fmaf(-d, sh, ch);
}

// The folded coefficient of row (r, j3, q, j2) and column (h, j1) with its
// phase drawn from element drawBase + src of the stream (seed, tag 2): the
// one formula of the coefficient fold and of the first contraction that forms
// its coefficients itself.
__device__ __forceinline__ float2 fold_coef_draw(const rf_fold_desc& f, unsigned r, unsigned j3, unsigned q,
                                                 unsigned j2, unsigned j1, unsigned h, uint64_t seed,
                                                 int64_t drawBase) {
#pragma clang fp contract(off)
    unsigned b = 0;
    if (f.fold) b = f.nDim == 3 ? (q == 0 ? (h ? 3u : 0u) : (h ? 1u : 2u)) : h;
    const int64_t jb = (int64_t)b * f.kNu + ((int64_t)j3 * f.nk2 + j2) * f.nk1 + j1;   // b kNu + j
    const int64_t src = (int64_t)r * f.kNr + jb;
    const double a = f.amp[(int64_t)r * f.ampStrideR + jb] * f.ampMult;
    float cs, sn;
    cis_rev(rf_uniform(seed, 2u, (uint64_t)(drawBase + src)), &cs, &sn);
    return make_float2((float)(a * (double)cs), (float)(h ? -(a * (double)sn) : a * (double)sn));
}

// Placement.  Workgroups go round-robin to the 8 XCDs, each with its own L2;
// block b runs logical tile (b % 8) * P + b / 8, so every XCD walks a contiguous
// range of P tiles and what neighbours share (streamed lines between table
// groups, amplitudes, cache lines at strip edges) is re-read from its L2.
constexpr int kXcd = 8;

__device__ inline int64_t xcd_tile(int64_t b, int64_t nTiles) {
    const int64_t per = (nTiles + kXcd - 1) / kXcd;
    return (b % kXcd) * per + b / kXcd;
}

// Grouped form: the GEMMs of several fields in one launch; GEMM q owns
// logical tiles tile0 .. tile0 + tiles(q) - 1.
__device__ inline int gemm_find(const rf_gemm_desc* __restrict__ gs, int nG, int64_t b) {
    int lo = 0, hi = nG - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (gs[mid].tile0 <= b) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

}  // namespace
