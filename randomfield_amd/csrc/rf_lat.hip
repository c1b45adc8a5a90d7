// rf_lat.hip -- the Shinozuka sum on scattered points through the product form
// of its lattice.
//
// The lattice of a sign block is a tensor product (spectra_RF.f90:87-133), so
// with a = k1_j1 x1, b = k2_j2 x2, c = k3_j3 x3
//   cos(a + s2 b + s3 c) = ca cb cc - s2 s3 ca sb sc - s2 sa sb cc - s3 sa cb sc
//   sin(a + s2 b + s3 c) = sa cb cc + s2 ca sb cc + s3 ca cb sc - s2 s3 sa sb sc
// and the four blocks (two in 2-D) of a lattice point (j1, j2, j3) share the
// eight (four) products of per-axis sines and cosines:
//   u[r][i] = sum_j sum_e  P[r][j][e] Phi[j][e][i],
// P the sums over the blocks of +-A cos(phi), +-A sin(phi), formed in FP64.  The
// contraction is the one of rf_mfma.hip -- FP16 or BF16 hi/lo operands, three
// v_mfma_f32_32x32x16 products per K-step, FP32 accumulation -- but a basis
// value costs two mixed-precision FMAs (hi and lo half of a product) instead of
// an FP64 k.x, a fraction, a hardware sine or cosine and the split: ~20 instead
// of ~67 VALU cycles per 64 (point, wavevector) pairs.  The per-axis factors are formed in FP64 reduction
// and accurate FP32 sines, so the basis is good to ~2 FP32 ulps (the hardware
// sines are not).
//
// K-step (16 entries), 3-D: lane half h takes j1 = 2 t + h and its 8 products
// e = 4 f1 + 2 f2 + f3 (f = 0 cosine, 1 sine); 2-D: j1 = 4 t + 2 h + u,
// e = 4 u + 2 f1 + f2.  Steps run t fastest, then j2, then j3.
#include <type_traits>

#include "rf_mfma.h"
#include "rf_per_device.h"
#include "rf_philox.h"

namespace {

// cos and sin of 2 pi t, |t| any: FP64 reduction, FP32 sincospi of the FP32
// part and the first-order term of the remainder.
__device__ __forceinline__ float2 cis_turns(double t) {
    const double f = t - rint(t);
    const float fh = (float)f;
    const float d = 6.28318530717958648f * (float)(f - (double)fh);
    float s, c;
    sincospif(2.0f * fh, &s, &c);
    return make_float2(fmaf(-d, s, c), fmaf(d, c, s));
}

// Basis values x0 y, x1 y as a packed pair of hi halves and their residuals.
// FP16: four mixed-precision FMAs, hi = f16(x y), lo = f16(x y - hi) with the
// product unrounded (separate multiplications and conversions: six).
template <typename V>
__device__ __forceinline__ void prod_pair(float x0, float x1, float y, unsigned* hi, unsigned* lo);
template <>
__device__ __forceinline__ void prod_pair<h8>(float x0, float x1, float y, unsigned* hi, unsigned* lo) {
    unsigned a, b;
    asm("v_fma_mixlo_f16 %0, %1, %2, 0" : "=v"(a) : "v"(x0), "v"(y));
    asm("v_fma_mixhi_f16 %0, %1, %2, 0" : "+v"(a) : "v"(x1), "v"(y));
    asm("v_fma_mixlo_f16 %0, %1, %2, -%3 op_sel:[0,0,0] op_sel_hi:[0,0,1]" : "=v"(b) : "v"(x0), "v"(y), "v"(a));
    asm("v_fma_mixhi_f16 %0, %1, %2, -%3 op_sel:[0,0,1] op_sel_hi:[0,0,1]" : "+v"(b) : "v"(x1), "v"(y), "v"(a));
    *hi = a;
    *lo = b;
}
template <>
__device__ __forceinline__ void prod_pair<b8>(float x0, float x1, float y, unsigned* hi, unsigned* lo) {
    typedef __bf16 b2 __attribute__((ext_vector_type(2)));
    const float v0 = x0 * y, v1 = x1 * y;
    const b2 h = {(__bf16)v0, (__bf16)v1};
    const b2 l = {(__bf16)(v0 - (float)h.x), (__bf16)(v1 - (float)h.y)};
    *hi = __builtin_bit_cast(unsigned, h);
    *lo = __builtin_bit_cast(unsigned, l);
}

// K-steps per stage and K-group (8 KB of panels)
constexpr int lat_steps(int MT) { return MT == 1 ? 4 : 2; }
constexpr int lat_units(int KG) { return 512 * KG; }   // 16-byte units of a stage
// The accumulators of 64 K-steps, of 16 where a group has up to 128, are added to the
// running sums: a serial FP32 accumulation over all ~1,400 steps of a 10-correlation-
// length lattice is off by 5e-6, so by 4e-7 (general form 1.9e-6).  On short groups 64
// are nearly one sum: FP16 errors of 33,000 points in 2-D boxes of 7 and 10 correlation
// lengths (28 and 56 steps) were 2.8e-7 and 3.8e-7, in a 3-D box of 3 (75) 4.0e-7, more
// than the general form's 2.7e-7, 3.6e-7 and 3.8e-7; so 1.9e-7, 2.0e-7 and 2.1e-7.  (16
// everywhere: 1.5-3 % of the time.)
constexpr int lat_flush(int64_t nG) { return nG <= 128 ? 16 : 64; }
// BF16 halves carry eight bits each, and the dropped product of the low halves is
// a third of the form's error variance.  Products of sines and cosines lie less
// near 1, where a rounding weighs least, than the general form's single sines do:
// without it errors are 5-8 % above that form's (3-D box of 6 correlation lengths, 32
// realizations: 4.25e-6 against 3.94e-6).  So the first kLatLowPart-th of the K-steps --
// the slow axis' long waves, most of the field -- takes it too: 3.66e-6 for 5-8 % of
// the time (on every step 3.38e-6 for up to 20 %).  Where the K-steps are split over
// groups of waves every other stage does (3.84e-6 for 3-9 %): two loops spill there
// (39 %), and a choice per step does in both shapes.
constexpr int kLatLowPart = 3;

// One block: points pt0 .. pt0 + 32 W - 1 (clipped to a.i1), M-tiles mt0 ..
// mt0 + MT - 1.  W waves side by side take 32 points each; KG such groups take
// 1/KG of the K-steps each, their sums added in group order at the end.  Two
// shapes, chosen by the field's N alone so that a field's result does not
// depend on what else is launched with it:
//   W = 8, KG = 1 (two blocks per CU): the fewest panel bytes per point, and
//     the stages of one block fill the barriers of the other; 48 served
//     requests of up to 300,000 points 10.4 ms, all in the other shape 12.6 ms
//     (a sine and cosine per term: 13.2 ms);
//   W = 4, KG = 4, N <= kLatSmallN: a field of 20,000 points has 157 blocks, and
//     without the split each SIMD has one wave, which waits on its own LDS
//     reads and MFMA chain: 229 us, 153 us split (before: 644 us).
// tab: per-point tables of axis 1 (P1 rows) and axis 2 (n2 rows), [row][point]
// (cos, sin); axis 3 is formed when j3 advances.  panA, panB: the stage being
// read and the next, copied through registers one stage ahead; one barrier per
// stage.  The LDS reads of a step (its panels, the table value of the basis
// after next) are issued before the VALU work on the next step's basis, the
// MFMAs follow it.
template <typename V, int D, int MT, int W, int KG>
__device__ __forceinline__ void lat_block(const rf_sum_args& a, const rf_lat_dev& L, int mtTotal,
                                          const u32x4* __restrict__ panels, float outScale, int64_t pt0, int mt0,
                                          u32x4* panA, u32x4* panB, float2* tab) {
    constexpr int kPts = 32 * W, kThreads = 64 * W * KG;
    constexpr int S = lat_steps(MT), kCopy = lat_units(KG) / kThreads, kGroupUnits = S * MT * 128;
    static_assert(kGroupUnits * KG == lat_units(KG) && kCopy * kThreads == lat_units(KG), "stage size");
    constexpr int J = D == 3 ? 1 : 2;                   // axis-1 points of a lane per step
    const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, n = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), pw = wave % W, kg = wave / W;
    const int pl = pw * 32 + n;                         // this lane's point in the block
    const int64_t pt = pt0 + pl;
    const int64_t stepUnits = (int64_t)mtTotal * 128;
    const int64_t nG = L.nSteps / KG;               // K-steps of a group, a multiple of 4
    const int64_t nStages = nG / S;
    const int flush = lat_flush(nG) / S;                // stages

    u32x4 pre[kCopy];
    const u32x4* src[kCopy];                            // this thread's units of the stage to fetch
#pragma unroll
    for (int i = 0; i < kCopy; i++) {
        const int e = tid + i * kThreads, eg = e % kGroupUnits;
        src[i] = panels + (e / kGroupUnits * nG + eg / (MT * 128)) * stepUnits + mt0 * 128 + eg % (MT * 128);
    }
    auto fetch = [&]() {                                // stage by stage
#pragma unroll
        for (int i = 0; i < kCopy; i++) {
            pre[i] = *src[i];
            src[i] += S * stepUnits;
        }
    };
    auto stash = [&](u32x4* dst) {
#pragma unroll
        for (int i = 0; i < kCopy; i++) dst[tid + i * kThreads] = pre[i];
    };
    fetch();
    float2* T1 = tab;
    float2* T2 = tab + L.P1 * kPts;
    double x3 = 0.0;
    {
        // kThreads / kPts threads per point share its rows
        constexpr int kRows = kThreads / kPts;
        const int p = tid % kPts;
        const int64_t i = pt0 + p < a.i1 ? pt0 + p : a.i1 - 1;
        const double t1 = a.x[i * D] / a.corrL[0] * L.kd[0];
        const double t2 = a.x[i * D + 1] / a.corrL[1] * L.kd[1];
        for (int j = tid / kPts; j < L.P1 + L.n2; j += kRows) {
            const int j2 = j - L.P1;
            tab[j * kPts + p] = j < L.n1 || j2 >= 0 ? cis_turns(j2 < 0 ? t1 * (double)j : t2 * (double)j2)
                                                    : make_float2(0.f, 0.f);
        }
        if (D == 3) {
            const int64_t ic = pt < a.i1 ? pt : a.i1 - 1;
            x3 = a.x[ic * D + (D - 1)] / a.corrL[D - 1] * L.kd[D - 1];
        }
    }
    stash(panA);
    __syncthreads();

    // (t, j2, j3): the step whose table value q holds; p: its axis-2/3 products
    int t, j2, j3;
    {
        const int64_t s0 = kg * nG, row = s0 / L.TS;
        t = (int)(s0 - row * L.TS);
        j3 = (int)(row / L.n2);
        j2 = (int)(row - (int64_t)j3 * L.n2);
    }
    float2 c3 = D == 3 ? cis_turns(x3 * (double)j3) : make_float2(1.f, 0.f);
    float p[4];
    float2 q[J];
    const float2* T1l = T1 + J * h * kPts + pl;
    auto products = [&]() {
        const float2 y = T2[j2 * kPts + pl];
        if (D == 3) {
            p[0] = y.x * c3.x;
            p[1] = y.x * c3.y;
            p[2] = y.y * c3.x;
            p[3] = y.y * c3.y;
        } else {
            p[0] = y.x;
            p[1] = y.y;
        }
    };
    auto load_q = [&]() {
#pragma unroll
        for (int u = 0; u < J; u++) q[u] = T1l[(2 * J * t + u) * kPts];
    };
    products();
    load_q();
    // fragments of the step at (t, j2, j3)
    auto form = [&](V* vh, V* vl) {
        u32x4 wh, wl;
        unsigned hh, ll;
        if (D == 3) {
            prod_pair<V>(p[0], p[1], q[0].x, &hh, &ll); wh[0] = hh; wl[0] = ll;
            prod_pair<V>(p[2], p[3], q[0].x, &hh, &ll); wh[1] = hh; wl[1] = ll;
            prod_pair<V>(p[0], p[1], q[0].y, &hh, &ll); wh[2] = hh; wl[2] = ll;
            prod_pair<V>(p[2], p[3], q[0].y, &hh, &ll); wh[3] = hh; wl[3] = ll;
        } else {
#pragma unroll
            for (int u = 0; u < J; u++) {
                prod_pair<V>(p[0], p[1], q[u].x, &hh, &ll); wh[2 * u] = hh; wl[2 * u] = ll;
                prod_pair<V>(p[0], p[1], q[u].y, &hh, &ll); wh[2 * u + 1] = hh; wl[2 * u + 1] = ll;
            }
        }
        *vh = __builtin_bit_cast(V, wh);
        *vl = __builtin_bit_cast(V, wl);
    };
    auto advance = [&]() {
        if (++t == L.TS) {                              // uniform
            t = 0;
            if (++j2 == L.n2) {
                j2 = 0;
                j3++;
                if (D == 3) c3 = cis_turns(x3 * (double)j3);
            }
            products();
        }
        load_q();
    };
    V bh, bl;
    form(&bh, &bl);
    advance();

    f16x acc[MT], tot[MT];
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
            acc[m][r] = 0.0f;
            tot[m][r] = 0.0f;
        }
    int left = flush;
    // one stage; lowToo: with the product of the low halves
    auto stage = [&](int64_t u, const u32x4* cur, u32x4* nxt, auto lowToo) {
        if (u + 1 < nStages) fetch();
#pragma unroll
        for (int s = 0; s < S; s++) {
            const u32x4* c = cur + kg * kGroupUnits + s * MT * 128 + lane;
            V ah[MT], al[MT];
#pragma unroll
            for (int m = 0; m < MT; m++) {
                ah[m] = __builtin_bit_cast(V, c[(m * 2 + 0) * 64]);
                al[m] = __builtin_bit_cast(V, c[(m * 2 + 1) * 64]);
            }
            V nh, nl;
            form(&nh, &nl);                             // the next step's basis
            advance();
#pragma unroll
            for (int m = 0; m < MT; m++) acc[m] = mfma(ah[m], bh, acc[m]);
#pragma unroll
            for (int m = 0; m < MT; m++) acc[m] = mfma(ah[m], bl, acc[m]);
#pragma unroll
            for (int m = 0; m < MT; m++) acc[m] = mfma(al[m], bh, acc[m]);
            if constexpr (decltype(lowToo)::value) {
#pragma unroll
                for (int m = 0; m < MT; m++) acc[m] = mfma(al[m], bl, acc[m]);
            }
            bh = nh;
            bl = nl;
        }
        if (--left == 0) {                              // uniform
            left = flush;
#pragma unroll
            for (int m = 0; m < MT; m++)
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    tot[m][r] += acc[m][r];
                    acc[m][r] = 0.0f;
                }
        }
        // the other buffer was last read before the previous barrier
        if (u + 1 < nStages) stash(nxt);
        __syncthreads();
    };
    auto stages = [&](int64_t u0, int64_t u1, auto even, auto odd) {              // u0 even
        for (int64_t u = u0; u < u1; u += 2) {
            stage(u, panA, panB, even);
            if (u + 1 < nStages) stage(u + 1, panB, panA, odd);
        }
    };
    const std::true_type with{};
    const std::false_type without{};
    if constexpr (!std::is_same<V, b8>::value) {
        stages(0, nStages, without, without);
    } else if constexpr (KG == 1) {
        int64_t low = (nStages + 2 * kLatLowPart - 1) / (2 * kLatLowPart) * 2;
        if (low > nStages) low = nStages;
        stages(0, low, with, with);
        stages(low, nStages, without, without);
    } else {
        stages(0, nStages, with, without);
    }
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int r = 0; r < 16; r++) tot[m][r] += acc[m][r];
    // group 0 adds the others' sums, one group at a time through panel space
    float* x = reinterpret_cast<float*>(panA);
    static_assert(KG == 1 || W * 64 * 16 * MT * sizeof(float) <= (size_t)lat_units(KG) * 16, "sums of one group");
    for (int g = 1; g < KG; g++) {
        if (kg == g) {
#pragma unroll
            for (int m = 0; m < MT; m++)
#pragma unroll
                for (int r = 0; r < 16; r++) x[((pw * MT + m) * 16 + r) * 64 + lane] = tot[m][r];
        }
        __syncthreads();
        if (kg == 0) {
#pragma unroll
            for (int m = 0; m < MT; m++)
#pragma unroll
                for (int r = 0; r < 16; r++) tot[m][r] += x[((pw * MT + m) * 16 + r) * 64 + lane];
        }
        __syncthreads();
    }
    if (kg != 0 || pt >= a.i1) return;
    store_tiles<MT>(a, tot, outScale, pt, mt0, h);
}

template <typename V, int D, int MT, int W, int KG>
__global__ __launch_bounds__(64 * W * KG) __attribute__((amdgpu_waves_per_eu(4)))
void k_lat(rf_sum_args a, rf_lat_dev L, int mtTotal, const u32x4* __restrict__ panels, float outScale) {
    __shared__ u32x4 panA[lat_units(KG)];
    __shared__ u32x4 panB[lat_units(KG)];
    extern __shared__ float2 lat_tab[];
    lat_block<V, D, MT, W, KG>(a, L, mtTotal, panels, outScale, a.i0 + (int64_t)blockIdx.x * (32 * W),
                               blockIdx.y * kLatMT, panA, panB, lat_tab);
}

// A batch of independent fields on one lattice (requests of a serving batch,
// all of one shape): block b of a launch from tile0 runs tile tile0 + b = (field, 32 W points, up to kLatMT
// M-tiles); the per-point operation order is that of k_lat.
template <typename V, int W, int KG>
__global__ __launch_bounds__(64 * W * KG) __attribute__((amdgpu_waves_per_eu(4)))
void k_group_lat(const rf_group_req* __restrict__ reqs, int nReq, rf_lat_dev L, int64_t tile0) {
    __shared__ u32x4 panA[lat_units(KG)];
    __shared__ u32x4 panB[lat_units(KG)];
    extern __shared__ float2 lat_tab[];
    const int64_t b = tile0 + blockIdx.x;
    const rf_group_req& q = reqs[group_find(reqs, nReq, b)];
    const int nSub = (q.mtTotal + kLatMT - 1) / kLatMT;
    const int64_t local = b - q.tile0;
    const int64_t pt0 = (local / nSub) * (32 * W);
    const int mt0 = (int)(local % nSub) * kLatMT;
    const rf_sum_args a = q.a;
    const u32x4* P = static_cast<const u32x4*>(q.ops0);
    if (q.mtTotal - mt0 >= 2) lat_block<V, 3, 2, W, KG>(a, L, q.mtTotal, P, q.outScale, pt0, mt0, panA, panB, lat_tab);
    else lat_block<V, 3, 1, W, KG>(a, L, q.mtTotal, P, q.outScale, pt0, mt0, panA, panB, lat_tab);
}

// Coefficient panels [step][mtile][hilo][lane][8]: one thread per (step, mtile,
// lane) folds the blocks of its lattice point(s) for one realization.  Phases
// 2 pi U from phase[r][b kNu + j], or, phase NULL, from the uniforms of
// elements r kNr + b kNu + j of stream (seed, tag 2); amplitudes
// amp[r ampStrideR + b kNu + j] * scale.
template <typename T>
__global__ __launch_bounds__(256) void k_lat_prep(int D, rf_lat_dev L, int Nmc, int mtTotal,
                                                  const double* __restrict__ phase, uint64_t seed,
                                                  const double* __restrict__ amp, int64_t ampStrideR, double scale,
                                                  T* __restrict__ panels) {
    typedef T t8 __attribute__((ext_vector_type(8)));
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= L.nSteps * mtTotal * 64) return;
    const int lane = (int)(e & 63), h = lane >> 5;
    const int64_t sm = e >> 6;
    const int mt = (int)(sm % mtTotal);
    const int64_t step = sm / mtTotal;
    const int t = (int)(step % L.TS);
    const int64_t row = step / L.TS;
    const int j2 = (int)(row % L.n2);
    const int64_t j3 = row / L.n2;
    const int r = mt * 32 + (lane & 31);
    const int nb = 1 << (D - 1);
    const int64_t kNu = (int64_t)L.n1 * L.n2 * L.n3;
    double v[8];
#pragma unroll
    for (int i = 0; i < 8; i++) v[i] = 0.0;
    // block b of lattice point j: its cosine and sine coefficients
    auto coef = [&](int64_t j, int b, double* C, double* Sn) {
        const int64_t s = b * kNu + j;
        const double A = amp[(int64_t)r * ampStrideR + s] * scale;
        const int64_t src = (int64_t)r * nb * kNu + s;
        const double ph = phase ? phase[src] : 2.0 * RF_PI_REF * rf_uniform(seed, 2u, (uint64_t)src);
        double sp, cp;
        sincos(ph, &sp, &cp);
        *C = A * cp;
        *Sn = -A * sp;
    };
    if (r < Nmc && j3 < L.n3) {
        const int64_t base = (j3 * L.n2 + j2) * L.n1;
        if (D == 3) {
            const int j1 = 2 * t + h;
            if (j1 < L.n1) {
#pragma unroll
                for (int b = 0; b < 4; b++) {
                    double C, S;
                    coef(base + j1, b, &C, &S);
                    const double s2 = b & 2 ? -1.0 : 1.0, s3 = b & 1 ? -1.0 : 1.0;
                    v[0] += C;              // c c c
                    v[1] += s3 * S;         // c c s
                    v[2] += s2 * S;         // c s c
                    v[3] -= s2 * s3 * C;    // c s s
                    v[4] += S;              // s c c
                    v[5] -= s3 * C;         // s c s
                    v[6] -= s2 * C;         // s s c
                    v[7] -= s2 * s3 * S;    // s s s
                }
            }
        } else {
#pragma unroll
            for (int u = 0; u < 2; u++) {
                const int j1 = 4 * t + 2 * h + u;
                if (j1 < L.n1) {
#pragma unroll
                    for (int b = 0; b < 2; b++) {
                        double C, S;
                        coef(base + j1, b, &C, &S);
                        const double s2 = b & 1 ? -1.0 : 1.0;
                        v[4 * u + 0] += C;          // c c
                        v[4 * u + 1] += s2 * S;     // c s
                        v[4 * u + 2] += S;          // s c
                        v[4 * u + 3] -= s2 * C;     // s s
                    }
                }
            }
        }
    }
    t8 hi, lo;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const T x = (T)(float)v[i];
        hi[i] = x;
        lo[i] = (T)(float)(v[i] - (double)(float)x);
    }
    t8* pan = reinterpret_cast<t8*>(panels) + (step * mtTotal + mt) * 128;
    pan[lane] = hi;
    pan[64 + lane] = lo;
}

size_t table_bytes(const rf_lat_dev& L, int W) { return (size_t)(L.P1 + L.n2) * 32 * W * sizeof(float2); }

// Kernels whose tables pass the default dynamic LDS limit ask for theirs, on
// each device that runs them (the limit belongs to the function on a device).
template <typename K>
hipError_t allow_lds(K* f, rf_per_device* asked) {
    int device = 0;
    const hipError_t e = hipGetDevice(&device);
    if (e != hipSuccess) return e;
    return asked->once(device, [&]() {
        return hipFuncSetAttribute(reinterpret_cast<const void*>(f), hipFuncAttributeMaxDynamicSharedMemorySize,
                                   kLatTableMax);
    });
}

template <typename V, int D, int MT, int W, int KG>
hipError_t launch(const rf_sum_args& a, const rf_lat_dev& L, int mtTotal, const void* B, float sc, hipStream_t s) {
    static rf_per_device asked;
    const hipError_t e = allow_lds(k_lat<V, D, MT, W, KG>, &asked);
    if (e != hipSuccess) return e;
    const int64_t blocks = (a.i1 - a.i0 + 32 * W - 1) / (32 * W);
    return rf_block_ranges(blocks, 64 * W * KG, [&](int64_t first, unsigned n) {
        rf_sum_args q = a;
        q.i0 += first * (32 * W);
        hipLaunchKernelGGL((k_lat<V, D, MT, W, KG>), dim3(n, (unsigned)((mtTotal + kLatMT - 1) / kLatMT)),
                           dim3(64 * W * KG), table_bytes(L, W), s, q, L, mtTotal, static_cast<const u32x4*>(B), sc);
        return hipGetLastError();
    });
}

template <typename V, int D>
hipError_t launch_d(const rf_sum_args& a, const rf_lat_dev& L, int mtTotal, const void* B, float sc, hipStream_t s) {
    if (rf_lat_small(L, a.N))
        return mtTotal == 1 ? launch<V, D, 1, 4, 4>(a, L, mtTotal, B, sc, s)
                            : launch<V, D, 2, 4, 4>(a, L, mtTotal, B, sc, s);
    return mtTotal == 1 ? launch<V, D, 1, 8, 1>(a, L, mtTotal, B, sc, s) : launch<V, D, 2, 8, 1>(a, L, mtTotal, B, sc, s);
}

template <typename V, int W, int KG>
hipError_t launch_group(const rf_lat_dev& L, const rf_group_req* d_reqs, int nReq, int64_t nTiles, hipStream_t s) {
    static rf_per_device asked;
    const hipError_t e = allow_lds(k_group_lat<V, W, KG>, &asked);
    if (e != hipSuccess) return e;
    return rf_block_ranges(nTiles, 64 * W * KG, [&](int64_t first, unsigned n) {
        hipLaunchKernelGGL((k_group_lat<V, W, KG>), dim3(n), dim3(64 * W * KG), table_bytes(L, W), s, d_reqs, nReq, L, first);
        return hipGetLastError();
    });
}

}  // namespace

bool rf_lat_describe(int nDim, const int32_t* kNStep, const double* kDelta, rf_lat_dev* L) {
    if (nDim < 2 || nDim > 3) return false;
    *L = rf_lat_dev{};
    L->n1 = kNStep[0];
    L->n2 = kNStep[1];
    L->n3 = nDim == 3 ? kNStep[2] : 1;
    const int per = nDim == 3 ? 2 : 4;                  // axis-1 points of a K-step
    L->TS = (L->n1 + per - 1) / per;
    L->P1 = L->TS * per;
    const int64_t steps = (int64_t)L->TS * L->n2 * L->n3;
    L->nSteps = (steps + 15) / 16 * 16;            // four groups of whole stages
    for (int d = 0; d < nDim; d++) L->kd[d] = kDelta[d] * RF_INV_TWO_PI;
    return table_bytes(*L, 4) <= (size_t)kLatTableMax;
}

// The shape of a field: by its N, and W = 8 only where its tables fit the LDS.
bool rf_lat_small(const rf_lat_dev& L, int64_t N) {
    return N <= kLatSmallN || table_bytes(L, 8) > (size_t)kLatTableMax;
}

size_t rf_lat_bbytes(const rf_lat_dev& L, int Npad) { return (size_t)L.nSteps * (Npad / 32) * 128 * 16; }

hipError_t rf_launch_lat_prep(int form, int nDim, const rf_lat_dev& L, int Nmc, int Npad, const double* d_phase,
                              uint64_t seed, const double* d_amp, int64_t ampStrideR, double scale, void* d_B,
                              hipStream_t s) {
    const int mtTotal = Npad / 32;
    const int64_t grid = (L.nSteps * mtTotal * 64 + 255) / 256;
    if (grid > rf_max_blocks(256)) return hipErrorInvalidValue;
    if (form == RF_FORM_MFMA_BF16)
        hipLaunchKernelGGL(k_lat_prep<__bf16>, dim3((unsigned)grid), dim3(256), 0, s, nDim, L, Nmc, mtTotal, d_phase, seed,
                           d_amp, ampStrideR, scale, static_cast<__bf16*>(d_B));
    else
        hipLaunchKernelGGL(k_lat_prep<_Float16>, dim3((unsigned)grid), dim3(256), 0, s, nDim, L, Nmc, mtTotal, d_phase,
                           seed, d_amp, ampStrideR, scale, static_cast<_Float16*>(d_B));
    return hipGetLastError();
}

// An even number of M-tiles, or one (rf_mfma_npad).
hipError_t rf_launch_sum_lat(int form, const rf_sum_args& a, const rf_lat_dev& L, int Npad, const void* d_B,
                             double outScale, hipStream_t s) {
    if (a.i1 <= a.i0) return hipSuccess;
    const int mtTotal = Npad / 32;
    const float sc = (float)outScale;
    const bool bf = form == RF_FORM_MFMA_BF16;
    if (a.nDim == 2)
        return bf ? launch_d<b8, 2>(a, L, mtTotal, d_B, sc, s) : launch_d<h8, 2>(a, L, mtTotal, d_B, sc, s);
    return bf ? launch_d<b8, 3>(a, L, mtTotal, d_B, sc, s) : launch_d<h8, 3>(a, L, mtTotal, d_B, sc, s);
}

hipError_t rf_launch_group_lat(int form, int small, const rf_lat_dev& L, const rf_group_req* d_reqs, int nReq,
                               int64_t nTiles, hipStream_t s) {
    if (nTiles <= 0 || nReq <= 0) return hipSuccess;
    const bool bf = form == RF_FORM_MFMA_BF16;
    if (small)
        return bf ? launch_group<b8, 4, 4>(L, d_reqs, nReq, nTiles, s) : launch_group<h8, 4, 4>(L, d_reqs, nReq, nTiles, s);
    return bf ? launch_group<b8, 8, 1>(L, d_reqs, nReq, nTiles, s) : launch_group<h8, 8, 1>(L, d_reqs, nReq, nTiles, s);
}
