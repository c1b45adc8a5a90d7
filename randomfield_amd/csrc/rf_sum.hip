// rf_sum.hip -- direct spectral sums u_r(x) = ampMult * sum_j a_rj cos(k_j.x + phi_rj)
// (randomFieldND.f90:184-337 methods 2/3, :368-514 method 1).
//
// Two precision forms:
//  * FP64: one sine and cosine per (point, wavevector), shared by all
//    realizations of a chunk, cos(t + phi) = cos t cos phi - sin t sin phi; the
//    wavevectors of a point are split over its block or, few wavevectors or many
//    points, taken by one lane.
//  * FP32: one thread per point holding R realization accumulators.  The
//    argument k.x is formed in FP64, reduced to revolutions in [-1/2, 1/2)
//    once per (point, k) and reused for all R realizations; each term is then
//    one FP32 add, one hardware cosine (v_cos_f32 takes revolutions) and one
//    FMA.  Wavevector, phase and amplitude operands are wave-uniform and come
//    through scalar loads, so the inner loop is pure VALU/transcendental work.
//    With per-realization directions the arguments come from the FP64 matrix cores.
#include <algorithm>

#include "rf_internal.h"

namespace {

constexpr int kBlock = 256;

template <typename T>
__device__ inline void store_out(void* out, int64_t idx, T v, int dtype) {
    if (dtype == RF_DTYPE_F64) static_cast<double*>(out)[idx] = (double)v;
    else static_cast<float*>(out)[idx] = (float)v;
}

// randomFieldND.f90:171-176 fused after the sum.
__device__ inline double epilogue64(double u, const rf_epilogue& e) {
#pragma clang fp contract(off)
    if (e.margi == RF_FOM_NONE) return u;
    const double y = u * e.scale + e.shift;
    return (e.margi == RF_FOM_LOGNORMAL) ? exp(y) : y;
}
__device__ inline float epilogue32(float u, const rf_epilogue& e) {
    if (e.margi == RF_FOM_NONE) return u;
    const float y = fmaf(u, (float)e.scale, (float)e.shift);
    return (e.margi == RF_FOM_LOGNORMAL) ? expf(y) : y;
}

// ---------------------------------------------------------------- FP64 form
// sin t and cos t for |t| < 2^30: t = n pi/2 + r with pi/2 in two doubles (the
// FMAs keep n P1 exact, so r is good to half an ulp and n 2^-107), then the
// minimax polynomials of sin r / r and cos r on |r| <= pi/4 (with the coefficients
// rounded to FP64 2^-57 and 2^-59.9; from a Remez exchange in 50-digit arithmetic).  Branch-free: ~28
// FP64 instructions against the library call's ~100 with its range tests.
__device__ __forceinline__ void sincos_fast(double t, double* sn, double* cs) {
    // n = rint(2 t / pi) by the rounding of an addition: the low word of the
    // sum holds n (two's complement)
    const double m = fma(t, 0.6366197723675814, 6755399441055744.0);   // 1.5 2^52
    const unsigned q = (unsigned)__builtin_bit_cast(uint64_t, m);
    const double n = m - 6755399441055744.0;
    double r = fma(-n, 0x1.921fb54442d18p+0, t);
    r = fma(-n, 0x1.1a62633145c07p-54, r);
    const double z = r * r;
    double ps = 1.5896795644221148e-10, pc = -1.1359647777745982e-11;
    ps = fma(ps, z, -2.5050758115096302e-08);
    pc = fma(pc, z, 2.087572327278296e-09);
    ps = fma(ps, z, 2.7557313691916818e-06);
    pc = fma(pc, z, -2.755731435233002e-07);
    ps = fma(ps, z, -0.00019841269829807805);
    pc = fma(pc, z, 2.4801587289482178e-05);
    ps = fma(ps, z, 0.008333333333322413);
    pc = fma(pc, z, -0.0013888888888874125);
    ps = fma(ps, z, -0.16666666666666632);
    pc = fma(pc, z, 0.0416666666666666);
    const double s = fma(r * z, ps, r);
    const double c = fma(z, fma(z, pc, -0.5), 1.0);
    const double ss = (q & 1) ? c : s, cc = (q & 1) ? s : c;
    const uint64_t fs = (uint64_t)((q << 30) & 0x80000000u) << 32;
    const uint64_t fc = (uint64_t)(((q << 30) + 0x40000000u) & 0x80000000u) << 32;
    *sn = __builtin_bit_cast(double, __builtin_bit_cast(uint64_t, ss) ^ fs);
    *cs = __builtin_bit_cast(double, __builtin_bit_cast(uint64_t, cc) ^ fc);
}

constexpr int kF64Waves = 8;     // waves of a block
constexpr int kF64Q = 4;         // points of a lane
constexpr int kF64Points = 16;   // points of a block: 4 lanes' worth
constexpr int kF64Shares = kF64Waves * 16;

// One block: 16 points, R realizations, all wavevectors.  The wavevectors are
// dealt to 128 shares (16 per wave, j = share mod 128), a lane takes one share
// and four points.  CS holds (a cos phi, -a sin phi): [j][Rpad] for a shared
// wavevector table, [r][j] with per-realization directions (ISO, R = 1).  A
// term costs the FP64 VALU 3 FMAs for k.x, ~28 instructions of sine and cosine
// and 2 FMAs per realization; that rate bounds it.  Why this split: with one
// point per lane the operands (24 + 16 R bytes per term) bound it instead, by
// latency as scalar loads (523 us) or by the vector memory path (575 us); four
// points per load leave the VALU busy, and small blocks spread 20,000 points
// evenly over the CUs.  20,000 points x 10,976 wavevectors x 4 realizations:
// 366 us (before: one thread per point and realization, a library cosine
// per term: 4159 us).  The shares are added in a fixed order.
// bound: max |k component|, for the block-uniform choice of the sine.
template <int D, int R, bool ISO>
__global__ __launch_bounds__(64 * kF64Waves) void k_sum_fp64(rf_sum_args a, const double* __restrict__ k,
                                                             double bound, const uint8_t* __restrict__ calc,
                                                             const double2* __restrict__ CS, int Rpad) {
    constexpr int Q = kF64Q, P = kF64Points;
    __shared__ double red[kF64Waves][R][P];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, pl = lane & 3;
    const int64_t p0 = a.i0 + (int64_t)blockIdx.x * P;
    const int r0 = blockIdx.y * R;
    double xn[Q][D];
    bool slow = false;
#pragma unroll
    for (int q = 0; q < Q; q++) {
        const int64_t i = p0 + pl * Q + q, ic = i < a.i1 ? i : a.i1 - 1;
        double reach = 0.0;
#pragma unroll
        for (int d = 0; d < D; d++) {
            xn[q][d] = a.x[ic * D + d] / a.corrL[d];   // :59
            reach += fabs(xn[q][d]);
        }
        // arguments past the fast sine's range, infinities, NaN: library sine
        slow |= !(reach * bound < 1073741824.0);
    }
    const bool fast = !__syncthreads_or(slow);
    double acc[Q][R];
#pragma unroll
    for (int q = 0; q < Q; q++)
#pragma unroll
        for (int r = 0; r < R; r++) acc[q][r] = 0.0;
    const double* kr = k + (ISO ? (int64_t)r0 * a.kN * D : 0);
    const double2* C = CS + (ISO ? (int64_t)r0 * a.kN : (int64_t)r0);
    const int64_t cStep = ISO ? 1 : Rpad;
    auto sweep = [&](auto sc) {
        for (int64_t j = w * 16 + (lane >> 2); j < a.kN; j += kF64Shares) {
            double kj[D];
#pragma unroll
            for (int d = 0; d < D; d++) kj[d] = kr[j * D + d];
            double sn[Q], cs[Q];
#pragma unroll
            for (int q = 0; q < Q; q++) {
                double t = kj[0] * xn[q][0];
#pragma unroll
                for (int d = 1; d < D; d++) t = fma(kj[d], xn[q][d], t);
                sc(t, &sn[q], &cs[q]);
            }
#pragma unroll
            for (int r = 0; r < R; r++) {
                const double2 c = C[j * cStep + r];
#pragma unroll
                for (int q = 0; q < Q; q++) acc[q][r] = fma(c.x, cs[q], fma(c.y, sn[q], acc[q][r]));
            }
        }
    };
    if (fast) sweep([](double t, double* s, double* c) { sincos_fast(t, s, c); });
    else sweep([](double t, double* s, double* c) { sincos(t, s, c); });
#pragma unroll
    for (int q = 0; q < Q; q++)
#pragma unroll
        for (int r = 0; r < R; r++) {
            double v = acc[q][r];
#pragma unroll
            for (int o = 4; o < 64; o <<= 1) v += __shfl_xor(v, o);
            if (lane < 4) red[w][r][pl * Q + q] = v;
        }
    __syncthreads();
    for (int e = threadIdx.x; e < R * P; e += 64 * kF64Waves) {
        const int r = e / P, p = e % P;
        const int64_t ip = p0 + p;
        if (ip >= a.i1 || r0 + r >= a.Nmc) continue;
        double s = red[0][r][p];
#pragma unroll
        for (int v = 1; v < kF64Waves; v++) s += red[v][r][p];
        // a realization the caller masks is zero at every point
        const double u = epilogue64(calc[r0 + r] ? a.ampMult * s : 0.0, a.epi);   // :330
        store_out(a.out, (int64_t)(r0 + r) * a.N + ip, u, a.outDtype);
    }
}

// The same sum with one point per lane, every wavevector in order, the operands
// wave-uniform (scalar loads): no reduction and no idle share, so it is the
// faster one where the wavevectors are few (a block above spends 3 .. 56 ns of the
// chip on its set-up and reduction, R = 1 .. 16) or the points many, and with
// per-realization directions, whose chunks hold one realization.  Bound by the
// latency of its loads and sine up to two waves per SIMD, then by the FP64 VALU.
// One term and realization at a time with the library cosine / shares / lane:
// 1M points x 13 wavevectors x 1: 29 / 296 / 17 us; 1M x 392 x 4: 2947 / 1083 /
// 461; isotropic 100,000 x 61 x 17: 207 / 727 / 106; 20,000 x 2,048 x 4: 765 / 73 /
// 445.  The accumulators go to running sums every kF64Flush terms, so that the
// rounding does not grow over that of the shares.
constexpr int kF64LaneBlock = 256;
constexpr int kF64Flush = 32;
template <int D, int R, bool ISO>
__global__ __launch_bounds__(kF64LaneBlock) void k_sum_fp64_lane(rf_sum_args a, const double* __restrict__ k,
                                                                 double bound, const uint8_t* __restrict__ calc,
                                                                 const double2* __restrict__ CS, int Rpad) {
    const int64_t i = a.i0 + (int64_t)blockIdx.x * kF64LaneBlock + threadIdx.x;
    if (i >= a.i1) return;
    const int r0 = blockIdx.y * R;
    double xn[D], reach = 0.0;
#pragma unroll
    for (int d = 0; d < D; d++) {
        xn[d] = a.x[i * D + d] / a.corrL[d];   // :59
        reach += fabs(xn[d]);
    }
    double acc[R];
#pragma unroll
    for (int r = 0; r < R; r++) acc[r] = 0.0;
    const double* kr = k + (ISO ? (int64_t)r0 * a.kN * D : 0);
    const double2* C = CS + (ISO ? (int64_t)r0 * a.kN : (int64_t)r0);
    const int64_t cStep = ISO ? 1 : Rpad;
    auto sweep = [&](auto sc) {
        for (int64_t j0 = 0; j0 < a.kN; j0 += kF64Flush) {
            const int64_t j1 = j0 + kF64Flush < a.kN ? j0 + kF64Flush : a.kN;
            double part[R];
#pragma unroll
            for (int r = 0; r < R; r++) part[r] = 0.0;
            for (int64_t j = j0; j < j1; j++) {
                double t = kr[j * D] * xn[0];
#pragma unroll
                for (int d = 1; d < D; d++) t = fma(kr[j * D + d], xn[d], t);
                double sn, cs;
                sc(t, &sn, &cs);
#pragma unroll
                for (int r = 0; r < R; r++) {
                    const double2 c = C[j * cStep + r];
                    part[r] = fma(c.x, cs, fma(c.y, sn, part[r]));
                }
            }
#pragma unroll
            for (int r = 0; r < R; r++) acc[r] += part[r];
        }
    };
    // per wave: arguments past the fast sine's range, infinities, NaN
    if (!__any(!(reach * bound < 1073741824.0))) sweep([](double t, double* s, double* c) { sincos_fast(t, s, c); });
    else sweep([](double t, double* s, double* c) { sincos(t, s, c); });
#pragma unroll
    for (int r = 0; r < R; r++) {
        if (r0 + r >= a.Nmc) break;
        // a realization the caller masks is zero at every point
        const double u = epilogue64(calc[r0 + r] ? a.ampMult * acc[r] : 0.0, a.epi);   // :330
        store_out(a.out, (int64_t)(r0 + r) * a.N + i, u, a.outDtype);
    }
}

// (a cos phi, -a sin phi) of the FP64 form from phases and amplitudes [r][j]:
// [j][Rpad], zero for padded realizations, or [r][j] (ISO).
__global__ __launch_bounds__(kBlock) void k_prep_fp64(int64_t kN, int Nmc, int Rpad, int iso,
                                                      const double* __restrict__ phase,
                                                      const double* __restrict__ amp, double2* __restrict__ CS) {
    for (int64_t e = (int64_t)blockIdx.x * kBlock + threadIdx.x; e < kN * Rpad; e += (int64_t)gridDim.x * kBlock) {
        const int64_t j = iso ? e % kN : e / Rpad;
        const int r = (int)(iso ? e / kN : e - j * Rpad);
        double2 v = {0.0, 0.0};
        if (r < Nmc) {
            const double A = amp[(int64_t)r * kN + j];
            double sn, cs;
            sincos(phase[(int64_t)r * kN + j], &sn, &cs);
            v.x = A * cs;
            v.y = -A * sn;
        }
        CS[e] = v;
    }
}

// ---------------------------------------------------------------- FP32 form
template <int D, int R>
__global__ __launch_bounds__(kBlock) void k_sum_fp32(rf_sum_args a, const double* __restrict__ kRev,
                                                     const float* __restrict__ phT,
                                                     const float* __restrict__ aT, int Rpad) {
    const int64_t i = a.i0 + (int64_t)blockIdx.x * kBlock + threadIdx.x;
    const int r0 = blockIdx.y * R;
    if (i >= a.i1) return;
    double xn[D];
#pragma unroll
    for (int d = 0; d < D; d++) xn[d] = a.x[i * D + d] / a.corrL[d];
    float acc[R];
#pragma unroll
    for (int r = 0; r < R; r++) acc[r] = 0.0f;
    const float* ph = phT + r0;
    const float* am = aT + r0;
    for (int64_t j = 0; j < a.kN; j++) {
        const double* kj = kRev + j * D;
        double t = kj[0] * xn[0];
#pragma unroll
        for (int d = 1; d < D; d++) t = fma(kj[d], xn[d], t);
        t = t - rint(t);                 // k.x mod 2pi, in revolutions
        const float tf = (float)t;
        const float* phj = ph + j * Rpad;
        const float* amj = am + j * Rpad;
#pragma unroll
        for (int r = 0; r < R; r++)
            acc[r] = fmaf(amj[r], __builtin_amdgcn_cosf(tf + phj[r]), acc[r]);
    }
#pragma unroll
    for (int r = 0; r < R; r++) {
        if (r0 + r < a.Nmc)
            store_out(a.out, (int64_t)(r0 + r) * a.N + i, epilogue32(acc[r], a.epi), a.outDtype);
    }
}

// FP32 form of the isotropic sum with per-realization directions: no argument
// is shared between realizations, so every term forms its own FP64 k.x + phi --
// on the FP64 matrix cores.  A row of v_mfma_f64_16x16x4_f64's A operand is one
// (wavevector, realization): (kx, ky, kz, phi) in revolutions; a column of B is one
// point: (x, y, z, 1).  The 16 rows are 16 / Rp wavevectors x Rp realizations, Rp
// the power of two (at most 16) that holds Nmc; larger Nmc in chunks of 16.
// The accumulator starts at 1.5 2^20, whose last place is 2^-32: the low word of
// D is then the argument modulo one revolution in 2^-32 (signed), converted and
// scaled for v_cos_f32.  A term costs four VALU instructions and a sixteenth of
// an MFMA of 64 cycles, which the VALU does not overlap; k.x by FMAs, v_fract_f64 and
// the phase cost eight (36 cycles either way), so what is gained is the
// packing of few realizations and waves of 32 points where a field is small:
// 200,000 points x 16 realizations, 286 shells 375 -> 284 us (error 1.9e-7 -> 1.8e-7);
// large fields of full rows take k_sum_fp32_iso_fma.  One instruction less -- v_alignbit of the word to a
// float 1 + argument of 23 bits -- gave 254 us and 8.66 ms with an error of 2.1e-7.
// Arguments that may reach 2^19 revolutions (or are not finite) take a zero
// accumulator and v_fract_f64; the choice is per wave.
// kA [block][4][16], aA [block][row % 4][row / 4], block = wavevector block x chunks
// + chunk; padded rows have zero amplitude.  Q groups of 16 points per wave: 2
// spread 200,000 points over the CUs more evenly than 4, whose operand loads and
// loop weigh half.
typedef double d4v __attribute__((ext_vector_type(4)));
typedef const double __attribute__((address_space(1))) gdbl;
typedef float f4v __attribute__((ext_vector_type(4)));
typedef const f4v __attribute__((address_space(1))) gf4;
constexpr int kIsoQ = 2;                               // 16-point groups of a wave, small fields and batches
static_assert(kGroupIsoPts == kBlock / 64 * 16 * kIsoQ, "points of a block");

constexpr double kIsoBias = 1572864.0;                 // 1.5 2^20
__device__ __forceinline__ float iso_turn(double t) {
    return (float)(int)(unsigned)__builtin_bit_cast(uint64_t, t) * 0x1p-32f;
}

template <int Q>
__device__ __forceinline__ void iso_block(const rf_sum_args& a, gdbl* __restrict__ kA, gf4* __restrict__ aA, int64_t nJ,
                                          int nChunk, int chunk, int Rp, double kMax, int64_t p0, float (*red)[16 * Q]) {
    constexpr int P = 16 * Q;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c = lane & 15, g = lane >> 4;
    const int64_t pw = p0 + wave * P;
    double b[Q];
    bool far = false;
#pragma unroll
    for (int q = 0; q < Q; q++) {
        const int64_t i = pw + 16 * q + c, ic = i < a.i1 ? i : a.i1 - 1;
        b[q] = g == 3 ? 1.0 : g < a.nDim ? a.x[ic * a.nDim + g] / a.corrL[g] : 0.0;
        far |= !(3.0 * kMax * fabs(b[q]) + 1.0 < 524288.0);
    }
    float acc[Q][4];
#pragma unroll
    for (int q = 0; q < Q; q++)
#pragma unroll
        for (int e = 0; e < 4; e++) acc[q][e] = 0.0f;
    auto sweep = [&](double c0, auto turn) {
        const d4v C = {c0, c0, c0, c0};
        gdbl* kp = kA + (int64_t)chunk * 64 + lane;
        gf4* ap = aA + (int64_t)chunk * 4 + g;
        auto terms = [&](double kj, const f4v& aj) {
#pragma unroll
            for (int q = 0; q < Q; q++) {
                const d4v t = __builtin_amdgcn_mfma_f64_16x16x4f64(kj, b[q], C, 0, 0, 0);
#pragma unroll
                for (int e = 0; e < 4; e++) acc[q][e] = fmaf(aj[e], __builtin_amdgcn_cosf(turn(t[e])), acc[q][e]);
            }
        };
        double kn = *kp;
        f4v an = *ap;
        for (int64_t j = 0; j < nJ; j++) {
            const double kj = kn;
            const f4v aj = an;
            if (j + 1 < nJ) {                          // one block ahead
                kp += nChunk * 64;
                ap += nChunk * 4;
                kn = *kp;
                an = *ap;
            }
            terms(kj, aj);
        }
    };
    if (!__any(far))
        sweep(kIsoBias, [](double t) { return iso_turn(t); });
    else
        sweep(0.0, [](double t) { return (float)__builtin_amdgcn_fract(t); });
    // D: column c, rows 4 e + g; the wavevectors of a block added in row order
#pragma unroll
    for (int q = 0; q < Q; q++)
#pragma unroll
        for (int e = 0; e < 4; e++) red[wave * 16 + 4 * e + g][16 * q + c] = acc[q][e];
    __syncthreads();
    for (int idx = lane; idx < Rp * P; idx += 64) {
        const int r = idx / P, p = idx % P, R = chunk * 16 + r;
        if (R >= a.Nmc || pw + p >= a.i1) continue;
        float s = 0.0f;
        for (int row = r; row < 16; row += Rp) s += red[wave * 16 + row][p];
        store_out(a.out, (int64_t)R * a.N + pw + p, epilogue32(s, a.epi), a.outDtype);
    }
}

template <int Q>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(Q > 2 ? 6 : 8))) void k_sum_fp32_iso(
    rf_sum_args a, const double* __restrict__ kA, const float* __restrict__ aA, int64_t nJ, int Rp, double kMax) {
    __shared__ float red[kBlock / 64 * 16][16 * Q];
    iso_block<Q>(a, (gdbl*)kA, (gf4*)aA, nJ, gridDim.y, blockIdx.y, Rp, kMax, a.i0 + (int64_t)blockIdx.x * (kBlock / 4 * Q),
                 red);
}

// The same sum by FMAs, one point per lane and 16 realizations of a chunk (Rp 16: one
// wavevector per operand block): large fields, whose waves of 64 points fill the chip
// and whose rows the matrix cores' packing has nothing to gain on.  The argument is
// formed on the same bias in the same order and read the same way: the same bits.
// Operands wave-uniform; the phase is added on its own because a VALU instruction
// reads one scalar operand (as the addend of an FMA it took two moves more, 10 %).
// 16 realizations: 2-D, 1M points, 116 shells 383 us (MFMA form 488), 3-D, 300,000 points,
// 146 shells 195 (207), 1M 545 (612).
template <int D>
__global__ __launch_bounds__(kBlock) void k_sum_fp32_iso_fma(rf_sum_args a, const double* __restrict__ kA,
                                                             const float* __restrict__ aA, int64_t nJ, double kMax) {
    const int64_t i = a.i0 + (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= a.i1) return;
    double x[D];
    bool far = false;
#pragma unroll
    for (int d = 0; d < D; d++) {
        x[d] = a.x[i * D + d] / a.corrL[d];
        far |= !(3.0 * kMax * fabs(x[d]) + 1.0 < 524288.0);
    }
    const int chunk = blockIdx.y, nChunk = gridDim.y;
    float acc[16];
#pragma unroll
    for (int r = 0; r < 16; r++) acc[r] = 0.0f;
    auto sweep = [&](double c0, auto turn) {
        for (int64_t j = 0; j < nJ; j++) {
            const double* k = kA + (j * nChunk + chunk) * 64;
            const float* am = aA + (j * nChunk + chunk) * 16;
#pragma unroll
            for (int r = 0; r < 16; r++) {
                double t = c0;
#pragma unroll
                for (int d = 0; d < D; d++) t = fma(k[16 * d + r], x[d], t);
                t += k[48 + r];
                acc[r] = fmaf(am[(r & 3) * 4 + (r >> 2)], __builtin_amdgcn_cosf(turn(t)), acc[r]);
            }
        }
    };
    if (!__any(far)) sweep(kIsoBias, [](double t) { return iso_turn(t); });
    else sweep(0.0, [](double t) { return (float)__builtin_amdgcn_fract(t); });
#pragma unroll
    for (int r = 0; r < 16; r++) {
        const int R = chunk * 16 + r;
        if (R < a.Nmc) store_out(a.out, (int64_t)R * a.N + i, epilogue32(acc[r], a.epi), a.outDtype);
    }
}

// Grouped form: block b of a launch from tile0 runs tile tile0 + b = (field, kGroupIsoPts points, chunk of
// 16 realizations), found by binary search over the fields' first tiles; same
// per-point operation order as k_sum_fp32_iso.
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(8))) void k_group_iso(
    const rf_group_req* __restrict__ reqs, int nReq, int64_t tile0) {
    __shared__ float red[kBlock / 64 * 16][16 * kIsoQ];
    const int64_t b = tile0 + blockIdx.x;
    int lo = 0, hi = nReq - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (reqs[mid].tile0 <= b) lo = mid;
        else hi = mid - 1;
    }
    const rf_group_req& q = reqs[lo];
    const rf_iso_shape sh = rf_iso_rows(q.a.kN, q.a.Nmc);
    const int64_t local = b - q.tile0;
    iso_block<kIsoQ>(q.a, (gdbl*)q.ops0, (gf4*)q.ops1, sh.nJ, sh.nChunk, (int)(local % sh.nChunk), sh.Rp, q.kMax,
              (local / sh.nChunk) * kGroupIsoPts, red);
}

// Shares or one point per lane: the smaller of what the two were measured to
// take (us) over 1 .. 1M points, 13 .. 6,912 wavevectors, 1 .. 64 realizations.
// Shares: start-up + per turn of 128 wavevectors, per block, chip-wide, and not below
// 9 us for 16 realizations (one block's reduction).  Lane: per wavevector, a
// latency up to about two waves per SIMD, then a rate per wave of a SIMD.
bool f64_lane(int64_t points, int64_t kN, int chunks, int R) {
    constexpr double kStart[5] = {2.6e-3, 4.2e-3, 9e-3, 26e-3, 51e-3}, kTurn[5] = {2.17e-3, 2.3e-3, 2.5e-3, 4.8e-3, 5.5e-3};
    constexpr double kLatency[5] = {0.18, 0.195, 0.225, 0.24, 0.267}, kRate[5] = {0.07, 0.072, 0.085, 0.105, 0.135};
    constexpr double kLeast[5] = {0.0, 0.0, 0.0, 0.0, 9.0};
    int i = 0;
    while ((1 << i) < R) i++;
    const double blocks = (double)((points + kF64Points - 1) / kF64Points) * chunks;
    const double turns = (double)((kN + kF64Shares - 1) / kF64Shares);
    const double perSimd = (double)(((points + 63) / 64 * chunks + 1023) / 1024);
    const double shares = std::max(kLeast[i], blocks * (kStart[i] + kTurn[i] * turns));
    return (double)kN * std::max(kLatency[i], perSimd * kRate[i]) < shares;
}

template <int D, int R, bool ISO>
hipError_t launch_fp64_r(const rf_sum_args& a, const double* k, double bound, const uint8_t* calc,
                         const double2* CS, int Rpad, hipStream_t s) {
    if (f64_lane(a.i1 - a.i0, a.kN, Rpad / R, R)) {
        const int64_t all = (a.i1 - a.i0 + kF64LaneBlock - 1) / kF64LaneBlock;
        return rf_block_ranges(all, kF64LaneBlock, [&](int64_t first, unsigned n) {
            rf_sum_args q = a;
            q.i0 += first * kF64LaneBlock;
            hipLaunchKernelGGL((k_sum_fp64_lane<D, R, ISO>), dim3(n, (unsigned)(Rpad / R)), dim3(kF64LaneBlock), 0, s, q, k,
                               bound, calc, CS, Rpad);
            return hipGetLastError();
        });
    }
    // 32 work-items per point: fields of 2^27 points and more in several launches
    const int64_t blocks = (a.i1 - a.i0 + kF64Points - 1) / kF64Points;
    return rf_block_ranges(blocks, 64 * kF64Waves, [&](int64_t first, unsigned n) {
        rf_sum_args q = a;
        q.i0 += first * kF64Points;
        hipLaunchKernelGGL((k_sum_fp64<D, R, ISO>), dim3(n, (unsigned)(Rpad / R)), dim3(64 * kF64Waves), 0, s, q, k, bound,
                           calc, CS, Rpad);
        return hipGetLastError();
    });
}

template <int D>
hipError_t launch_fp64(const rf_sum_args& a, const double* k, int iso, double bound, const uint8_t* calc,
                       const double2* CS, int Rpad, hipStream_t s) {
    if (iso) return launch_fp64_r<D, 1, true>(a, k, bound, calc, CS, Rpad, s);
    switch (rf_fp64_rchunk(a.Nmc)) {
        case 1: return launch_fp64_r<D, 1, false>(a, k, bound, calc, CS, Rpad, s);
        case 2: return launch_fp64_r<D, 2, false>(a, k, bound, calc, CS, Rpad, s);
        case 4: return launch_fp64_r<D, 4, false>(a, k, bound, calc, CS, Rpad, s);
        case 8: return launch_fp64_r<D, 8, false>(a, k, bound, calc, CS, Rpad, s);
        default: return launch_fp64_r<D, 16, false>(a, k, bound, calc, CS, Rpad, s);
    }
}

}  // namespace

// Realization chunk of the FP32 kernels (accumulators per thread).
constexpr int kRChunk = 16;

// Realizations per block of the FP64 kernel: the power of two that holds Nmc,
// at most 16 (the sine of a term is then shared by all of them).
int rf_fp64_rchunk(int Nmc) {
    int r = 1;
    while (r < Nmc && r < 16) r <<= 1;
    return r;
}

int rf_fp64_rpad(int Nmc, int iso) {
    const int c = rf_fp64_rchunk(Nmc);
    return iso ? Nmc : (Nmc + c - 1) / c * c;
}

hipError_t rf_launch_prep_fp64(int64_t kN, int Nmc, int Rpad, int iso, const double* d_phase, const double* d_amp,
                               double2* d_CS, hipStream_t s) {
    const int64_t n = kN * Rpad;
    if (n <= 0) return hipSuccess;
    const int64_t blocks = std::min((n + kBlock - 1) / kBlock, rf_max_blocks(kBlock));
    hipLaunchKernelGGL(k_prep_fp64, dim3((unsigned)blocks), dim3(kBlock), 0, s, kN, Nmc, Rpad, iso, d_phase, d_amp, d_CS);
    return hipGetLastError();
}

hipError_t rf_launch_sum_fp64(const rf_sum_args& a, const double* d_k, int iso, double bound, const uint8_t* d_calc,
                              const double2* d_CS, int Rpad, hipStream_t s) {
    if (a.i1 <= a.i0) return hipSuccess;
    switch (a.nDim) {
        case 1: return launch_fp64<1>(a, d_k, iso, bound, d_calc, d_CS, Rpad, s);
        case 2: return launch_fp64<2>(a, d_k, iso, bound, d_calc, d_CS, Rpad, s);
        default: return launch_fp64<3>(a, d_k, iso, bound, d_calc, d_CS, Rpad, s);
    }
}

hipError_t rf_launch_sum_fp32(const rf_sum_args& a, const double* d_kRev, const float* d_phT,
                              const float* d_aT, int Rpad, hipStream_t s) {
    if (a.i1 <= a.i0) return hipSuccess;
    const int64_t n = a.i1 - a.i0;
    dim3 grid((unsigned)((n + kBlock - 1) / kBlock), (unsigned)(Rpad / kRChunk));
    switch (a.nDim) {
        case 1:
            hipLaunchKernelGGL((k_sum_fp32<1, kRChunk>), grid, dim3(kBlock), 0, s, a, d_kRev, d_phT, d_aT, Rpad);
            break;
        case 2:
            hipLaunchKernelGGL((k_sum_fp32<2, kRChunk>), grid, dim3(kBlock), 0, s, a, d_kRev, d_phT, d_aT, Rpad);
            break;
        default:
            hipLaunchKernelGGL((k_sum_fp32<3, kRChunk>), grid, dim3(kBlock), 0, s, a, d_kRev, d_phT, d_aT, Rpad);
            break;
    }
    return hipGetLastError();
}

hipError_t rf_launch_sum_fp32_iso_t(const rf_sum_args& a, const double* d_kA, const float* d_aA, double kMax,
                                    hipStream_t s) {
    if (a.i1 <= a.i0) return hipSuccess;
    const rf_iso_shape sh = rf_iso_rows(a.kN, a.Nmc);
    if (sh.nChunk > 65535) return hipErrorInvalidValue;
    // FMA form, full rows: by (point, chunk) pairs in units of one wave per SIMD, 65,536.
    // Time against the MFMA form, whose waves hold 32 points: 3-D 1.3-1.4 at 80,000, 1.11
    // at 200,000, 0.90-0.96 at 300,000, 0.88 at 2M; 2-D, a quarter of whose MFMA multiplies
    // zeros, 0.83-0.93 at 100,000 and 131,000, 1.06 at 140,000 (a third round), 0.99 at
    // 200,000, 0.77 at 2M.
    const int64_t pairs = (a.i1 - a.i0) * sh.nChunk;
    const bool fma2 = pairs >= 3 * 65536 || (2 * pairs >= 3 * 65536 && pairs <= 2 * 65536), fma3 = 2 * pairs >= 9 * 65536;
    if (sh.Rp == 16 && (a.nDim == 2 ? fma2 : fma3)) {
        const int64_t all = (a.i1 - a.i0 + kBlock - 1) / kBlock;
        return rf_block_ranges(all, kBlock, [&](int64_t first, unsigned n) {
            rf_sum_args q = a;
            q.i0 += first * kBlock;
            const dim3 grid(n, (unsigned)sh.nChunk);
            if (a.nDim == 2) hipLaunchKernelGGL(k_sum_fp32_iso_fma<2>, grid, dim3(kBlock), 0, s, q, d_kA, d_aA, sh.nJ, kMax);
            else hipLaunchKernelGGL(k_sum_fp32_iso_fma<3>, grid, dim3(kBlock), 0, s, q, d_kA, d_aA, sh.nJ, kMax);
            return hipGetLastError();
        });
    }
    // 64 points per wave where that still gives every SIMD about sixteen waves
    // (the operand loads and the loop weigh half), else 32.  At the line, 1,048,575 and
    // 1,048,576 points, 146 shells: one realization 51.8 and 48.0 us, five 320 and 307
    const bool wide = (a.i1 - a.i0) / 64 * sh.nChunk >= 16384;
    const int pts = kBlock / 4 * (wide ? 4 : kIsoQ);
    const int64_t blocks = (a.i1 - a.i0 + pts - 1) / pts;
    return rf_block_ranges(blocks, kBlock, [&](int64_t first, unsigned n) {
        rf_sum_args q = a;
        q.i0 += first * pts;
        const dim3 grid(n, (unsigned)sh.nChunk);
        if (wide) hipLaunchKernelGGL(k_sum_fp32_iso<4>, grid, dim3(kBlock), 0, s, q, d_kA, d_aA, sh.nJ, sh.Rp, kMax);
        else hipLaunchKernelGGL(k_sum_fp32_iso<kIsoQ>, grid, dim3(kBlock), 0, s, q, d_kA, d_aA, sh.nJ, sh.Rp, kMax);
        return hipGetLastError();
    });
}

int rf_fp32_rchunk() { return kRChunk; }

hipError_t rf_launch_group_iso(const rf_group_req* d_reqs, int nReq, int64_t nTiles, hipStream_t s) {
    if (nTiles <= 0 || nReq <= 0) return hipSuccess;
    return rf_block_ranges(nTiles, kBlock, [&](int64_t first, unsigned n) {
        hipLaunchKernelGGL(k_group_iso, dim3(n), dim3(kBlock), 0, s, d_reqs, nReq, first);
        return hipGetLastError();
    });
}
