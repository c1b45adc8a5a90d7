// rf_grid.hip -- Shinozuka sums on structured grids by axis-wise contraction.
//
// On a grid x = o + (i1, i2, i3) * step (x fastest, setGrid order,
// math_RF.f90:70-88) and the Shinozuka lattice -- per sign block b the tensor
// product k = (s1 k1_j1, s2 k2_j2, s3 k3_j3) of 1-D lattices k_a,j = j dk_a
// (spectra_RF.f90:88-133) -- the sum of randomFieldND.f90:276-330 factorises:
//
//   u_r(x) = Re sum_b sum_j3 E3^{s3}[j3][x3] sum_j2 E2^{s2}[j2][x2]
//                        sum_j1 E1[j1][x1] C_r[b][j3][j2][j1],
//   E_a[j][x] = exp(i k_a,j x_a),  C = ampMult A exp(i phi),
//
// three small batched complex GEMMs instead of N * N_k cosines
// (O(n N_k + n^2 N_k^(2/3) + n^3 N_k^(1/3)) per realization and block).
// Every stage is one tiled complex GEMM on the matrix cores,
// D[m][n] = sum_k A[m][k] B[k][n] with per-stage strides: operands split
// into FP16 hi + lo halves (power-of-two scaled into range), three
// v_mfma_f32_32x32x16_f16 products with FP32 accumulation (strip GEMMs,
// rf_strip.hip);
// an FP32-operand MFMA tile (v_mfma_f32_32x32x2_f32) serves shapes whose K would
// leave the FP16 range or whose strides a strip's 32-bit offsets.
// The negative sign blocks are folded into the first contraction
// (conjugated tables and coefficients).  The phase tables are formed in FP64
// and rounded to FP32; accumulation is FP32 over <= 4*N_k^(1/3) terms.
//
// The isotropic method (randomFieldND.f90:368-514) has no lattice, but on a
// grid each of its terms still factorises over the axes: per realization one
// real-part GEMM over the shells whose operands are per-axis phase tables
// (k_iso_tables, the isotropic strip GEMM).
#include "rf_grid_dev.h"

namespace {

constexpr int kTM = 64, kTN = 64, kTK = 16;   // block tile; 256 threads, 4x4 each

__device__ inline float epi32(float u, const rf_epilogue& e) {
    if (e.margi == RF_FOM_NONE) return u;
    const float y = fmaf(u, (float)e.scale, (float)e.shift);
    return (e.margi == RF_FOM_LOGNORMAL) ? expf(y) : y;
}

// One 64 x 64 output tile (complex rows m0.., columns n0.., batch) of
// D = A B on the matrix cores in FP32 (v_mfma_f32_32x32x2_f32): the complex
// product is the real GEMM
//   [Re D; Im D] = [[Re A, -Im A], [Im A, Re A]] [Re B; Im B]
// with the real rows interleaved (2m: Re, 2m+1: Im), one complex k per
// instruction (lanes 0-31 take the k' = 2k column, 32-63 the k' = 2k+1
// column).  RealOnly forms Re D only: [Re A, -Im A] [Re B; Im B].  Operand
// tiles of 16 complex k are staged in LDS as FP32 complex, as loaded.
// Waves: complex output 128 real rows x 64 columns, wave w owns real rows
// 32w.. and both 32-column halves; RealOnly 64 x 64, wave w one 32 x 32 tile.
template <bool RealOnly>
__device__ __forceinline__ void gemm_tile(const rf_gemm_desc& g, int m0, int n0, int batch,
                                          float2 (*sA)[kTM + 1], float2 (*sB)[kTN + 1]) {
    const int tid = threadIdx.x;
    const int wave = tid >> 6, lane = tid & 63, half = lane >> 5, l32 = lane & 31;
    const float2* A = g.A + (int64_t)((batch / g.aDiv) % g.aMod) * g.aStrideB;
    const float2* B = g.B + (int64_t)batch * g.bStrideB;
    f32x16 acc0, acc1;
#pragma unroll
    for (int i = 0; i < 16; i++) {
        acc0[i] = 0.0f;
        acc1[i] = 0.0f;
    }
    // RealOnly tile of this wave
    const int rt = wave >> 1, ct = wave & 1;
    // operand chunks of kTK complex k: each thread fetches kPer elements of
    // A and of B into registers one chunk ahead (zero outside the matrices)
    constexpr int kPer = kTM * kTK / 256;
    static_assert(kTM * kTK == kTK * kTN && kPer * 256 == kTM * kTK, "staging split");
    float2 ra[kPer], rb[kPer];
    auto fetch = [&](int k0) {
#pragma unroll
        for (int i = 0; i < kPer; i++) {
            const int e = tid + i * 256;
            const int mm = e / kTK, ka = e % kTK;
            const int m = m0 + mm, k = k0 + ka;
            ra[i] = (m < g.M && k < g.K) ? A[m * g.aSm + k * g.aSk] : make_float2(0.f, 0.f);
            const int kb = e / kTN, nn = e % kTN;
            const int n = n0 + nn, k2 = k0 + kb;
            rb[i] = (n < g.N && k2 < g.K) ? B[k2 * g.bSk + col_b(g, n)] : make_float2(0.f, 0.f);
        }
    };
    auto stash = [&]() {
#pragma unroll
        for (int i = 0; i < kPer; i++) {
            const int e = tid + i * 256;
            sA[e % kTK][e / kTK] = ra[i];
            sB[e / kTN][e % kTN] = rb[i];
        }
    };
    fetch(0);
    for (int k0 = 0; k0 < g.K; k0 += kTK) {
        stash();
        __syncthreads();
        if (k0 + kTK < g.K) fetch(k0 + kTK);      // in flight during the MFMAs
        // 32 x 32 sub-tiles entirely outside D are skipped (wave-uniform), so
        // edge tiles of the ~130-point grid axes cost only their valid part
        if (!RealOnly) {
            if (m0 + wave * 16 < g.M) {
                if (n0 + 32 < g.N) {
#pragma unroll 4
                    for (int kk = 0; kk < kTK; kk++) {
                        const float2 a = sA[kk][wave * 16 + (l32 >> 1)];
                        // row part (l32 & 1): 0 -> Re row (Re A, -Im A), 1 -> Im row (Im A, Re A)
                        const float av = (l32 & 1) ? (half ? a.x : a.y) : (half ? -a.y : a.x);
                        const float2 b0 = sB[kk][l32], b1 = sB[kk][32 + l32];
                        acc0 = __builtin_amdgcn_mfma_f32_32x32x2f32(av, half ? b0.y : b0.x, acc0, 0, 0, 0);
                        acc1 = __builtin_amdgcn_mfma_f32_32x32x2f32(av, half ? b1.y : b1.x, acc1, 0, 0, 0);
                    }
                } else {
#pragma unroll 4
                    for (int kk = 0; kk < kTK; kk++) {
                        const float2 a = sA[kk][wave * 16 + (l32 >> 1)];
                        const float av = (l32 & 1) ? (half ? a.x : a.y) : (half ? -a.y : a.x);
                        const float2 b0 = sB[kk][l32];
                        acc0 = __builtin_amdgcn_mfma_f32_32x32x2f32(av, half ? b0.y : b0.x, acc0, 0, 0, 0);
                    }
                }
            }
        } else if (m0 + rt * 32 < g.M && n0 + ct * 32 < g.N) {
#pragma unroll 4
            for (int kk = 0; kk < kTK; kk++) {
                const float2 a = sA[kk][rt * 32 + l32];
                const float2 b = sB[kk][ct * 32 + l32];
                acc0 = __builtin_amdgcn_mfma_f32_32x32x2f32(half ? -a.y : a.x, half ? b.y : b.x, acc0, 0, 0, 0);
            }
        }
        __syncthreads();
    }
    // D layout of a 32x32 tile: lane column l32, rows 8*(i/4) + 4*half + i%4
    if (!RealOnly) {
#pragma unroll
        for (int i = 0; i < 16; i += 2) {
            const int r = 8 * (i >> 2) + 4 * half + (i & 3);       // even: the Re row
            const int m = m0 + wave * 16 + (r >> 1);
            if (m >= g.M) continue;
#pragma unroll
            for (int c = 0; c < 2; c++) {
                const int n = n0 + c * 32 + l32;
                if (n >= g.N) continue;
                const int64_t o = (int64_t)batch * g.dStrideB + m * g.dSm + col_d(g, n);
                static_cast<float2*>(g.D)[o] = c ? make_float2(acc1[i] * g.outScale, acc1[i + 1] * g.outScale)
                                                 : make_float2(acc0[i] * g.outScale, acc0[i + 1] * g.outScale);
            }
        }
    } else {
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const int m = m0 + rt * 32 + 8 * (i >> 2) + 4 * half + (i & 3);
            const int n = n0 + ct * 32 + l32;
            if (m >= g.M || n >= g.N) continue;
            const int64_t o = (int64_t)batch * g.dStrideB + m * g.dSm + col_d(g, n);
            const float u = epi32(acc0[i] * g.outScale, g.epi);
            if (g.outDtype == RF_DTYPE_F64) static_cast<double*>(g.D)[o] = (double)u;
            else static_cast<float*>(g.D)[o] = u;
        }
    }
}

struct FStage {
    float2 a[kTK][kTM + 1];
    float2 b[kTK][kTN + 1];
};

// An FP32-operand tile: row tiles fastest (they share a column slab of B).
template <bool RealOnly>
__device__ __forceinline__ void run_tile(const rf_gemm_desc& g, int64_t local, char* smem) {
    const int ntN = (g.N + kTN - 1) / kTN, ntM = (g.M + kTM - 1) / kTM;
    const int mI = (int)(local % ntM);
    const int64_t r = local / ntM;
    FStage* f = reinterpret_cast<FStage*>(smem);
    gemm_tile<RealOnly>(g, mI * kTM, (int)(r % ntN) * kTN, (int)(r / ntN), f->a, f->b);
}

// The FP32-operand tile (a first contraction whose K would leave the FP16
// range).
template <bool RealOnly>
__global__ __launch_bounds__(256) void k_cgemm(rf_gemm_desc g, int64_t nTiles) {
    __shared__ __attribute__((aligned(16))) char smem[sizeof(FStage)];
    const int64_t L = xcd_tile(blockIdx.x, nTiles);
    if (L >= nTiles) return;
    run_tile<RealOnly>(g, L, smem);
}
template <bool RealOnly>
__global__ __launch_bounds__(256) void k_cgemm_group(const rf_gemm_desc* __restrict__ gs, int nG, int64_t nTiles) {
    __shared__ __attribute__((aligned(16))) char smem[sizeof(FStage)];
    const int64_t L = xcd_tile(blockIdx.x, nTiles);
    if (L >= nTiles) return;
    const rf_gemm_desc g = gs[gemm_find(gs, nG, L)];
    run_tile<RealOnly>(g, L - g.tile0, smem);
}

// Isotropic phase tables of the grid's axes, in FP64 then rounded: axis 0
// carries the coefficient, W = c a e^{i(k_x x + phi)} (c: ampMult times a power of
// two), the others e^{i k_a x}; k runs to kP (kN rounded up to whole steps), zero
// past kN.  The last axis goes to Z in the strip GEMM's fragment order, split into
// FP16 hi + lo ([r][k / 8][x / 32][hi, lo][re, im][x % 32][k % 8]), the others to T0
// and T1 as [r][k / 4][x][k % 4]; a thread's position runs along what it writes.
struct rf_iso_tables {
    int nDim, Nmc;
    int64_t kN, kP;
    int n[3], w[3];                // points; entries written (the last axis: whole tiles)
    double o[3], st[3], inv[3], coef;
    const double* kIso; const double* amp; const double* phase;
    float2* T[2];
    _Float16* Z;
};
__global__ __launch_bounds__(256) void k_iso_tables(rf_iso_tables t) {
    const int64_t per = t.kP * (t.w[0] + t.w[1] + t.w[2]);       // of a realization
    int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= t.Nmc * per) return;
    const int64_t r = e / per;
    e -= r * per;
    int a = 0;
    while (a + 1 < t.nDim && e >= t.kP * t.w[a]) e -= t.kP * t.w[a++];
    const bool last = a == t.nDim - 1;
    int64_t k;
    int idx;
    if (last) {
        const int nT = t.w[a] / 32;
        const int64_t st = e >> 8;                               // step * nT + tile
        k = st / nT * 8 + (e & 7);
        idx = (int)(st % nT) * 32 + ((int)(e >> 3) & 31);
    } else {
        const int64_t c = e / (4 * t.w[a]);
        k = 4 * c + (e & 3);
        idx = (int)((e - c * 4 * t.w[a]) >> 2);
    }
    float2 v = make_float2(0.f, 0.f);
    if (k < t.kN && idx < t.n[a]) {
        const int64_t rk = r * t.kN + k;
        const double x = (t.o[a] + t.st[a] * (double)idx) * t.inv[a];
        double th = t.kIso[rk * t.nDim + a] * x;
        if (a == 0) th += t.phase[rk];
        double sn, cs;
        sincos(th, &sn, &cs);
        const double m = a == 0 ? t.amp[rk] * t.coef : 1.0;
        v = make_float2((float)(m * cs), (float)(m * sn));
    }
    if (!last) {
        t.T[a][r * t.kP * t.w[a] + e] = v;
        return;
    }
    _Float16* F = t.Z + (r * t.kP * t.w[a] + (e & ~(int64_t)255)) * 4 + (e & 255);
    asm("" : "+v"(v.x), "+v"(v.y));
    const _Float16 ch = (_Float16)v.x, sh = (_Float16)v.y;
    F[0] = ch;
    F[256] = sh;
    F[512] = (_Float16)(v.x - (float)ch);
    F[768] = (_Float16)(v.y - (float)sh);
}

// The tables of all axes of one execution (one launch: a grid of 129 x 129
// points spent three launches of 5-9 us on what this does in one).  Axis a's
// blocks start at block0[a].
//   Shinozuka: E[v][j][x] = exp(i s_v k_j x), k_j = j dk, x = (o + i step) / L,
//     in FP64; variant v = 0 plain, v = 1 conjugate (negative sign).
//   Method 4: E[v][j][i] = (w_j cos(pi j (2i+1) / (2n)), 0), w_0 = 1, w_j = 2: the
//     REDFT01 (DCT-III) of FFTW that gen_Std_Gauss_FFT applies along each axis
//     (randomFieldND.f90:694-735), as a matrix; both variants equal.
//   frag: in the strip GEMM's fragment order instead, split into FP16 hi + lo:
//     K entry k is entry k % nk of variant k / nk, [step k / 8][tile x / 32][hi,
//     lo][re, im][x % 32][k % 8], zero past K and past nx.
struct rf_table_args {
    int dct, nAx, frag;
    int nk[3], nx[3], K[3];
    unsigned block0[3];
    double dk[3], o[3], step[3], invL[3];
    void* E[3];
};
__global__ __launch_bounds__(256) void k_axis_tables(rf_table_args t) {
    int a = 0;
    while (a + 1 < t.nAx && blockIdx.x >= t.block0[a + 1]) a++;
    const int64_t e = (int64_t)(blockIdx.x - t.block0[a]) * 256 + threadIdx.x;
    const int nx = t.nx[a];
    if (t.frag) {
        const int nT = (nx + 31) / 32;
        const int64_t st = e >> 8;                       // step * nT + tile
        const int64_t s = st / nT;
        if (s >= (t.K[a] + 7) / 8) return;
        const int row = (int)(e >> 3) & 31, q = (int)e & 7;
        const int k = (int)(8 * s) + q, i = (int)(st - s * nT) * 32 + row;
        const int v = k / t.nk[a], j = k - v * t.nk[a];
        double c = 0.0, sn = 0.0;
        if (k < t.K[a] && i < nx) {
            if (t.dct) {
                c = (j == 0 ? 1.0 : 2.0) * cos(3.14159265358979323846 * (double)j * (2.0 * i + 1.0) / (2.0 * nx));
            } else {
                sincos((t.dk[a] * (double)j) * ((t.o[a] + t.step[a] * (double)i) * t.invL[a]), &sn, &c);
                if (v) sn = -sn;
            }
        }
        // rounded to FP32 first, then split (opaque: the two conversions would be
        // folded into one)
        float cf = (float)c, sf = (float)sn;
        asm("" : "+v"(cf), "+v"(sf));
        const _Float16 ch = (_Float16)cf, sh = (_Float16)sf;
        _Float16* F = static_cast<_Float16*>(t.E[a]) + st * 1024 + row * 8 + q;
        F[0] = ch;
        F[256] = sh;
        F[512] = (_Float16)(cf - (float)ch);
        F[768] = (_Float16)(sf - (float)sh);
        return;
    }
    const int64_t cnt = (int64_t)t.nk[a] * nx;
    if (e >= cnt) return;
    const int j = (int)(e / nx), i = (int)(e % nx);
    float2* E = static_cast<float2*>(t.E[a]);
    if (t.dct) {
        const double w = j == 0 ? 1.0 : 2.0;
        const double c = w * cos(3.14159265358979323846 * (double)j * (2.0 * i + 1.0) / (2.0 * nx));
        E[e] = make_float2((float)c, 0.0f);
        E[cnt + e] = make_float2((float)c, 0.0f);
        return;
    }
    const double x = (t.o[a] + t.step[a] * (double)i) * t.invL[a];
    const double th = (t.dk[a] * (double)j) * x;
    double s, c;
    sincos(th, &s, &c);
    E[e] = make_float2((float)c, (float)s);
    E[cnt + e] = make_float2((float)c, (float)-s);
}

// Sign-block folding.  The field is Re of the sum, and the tables of a
// negative sign are conjugates, Re(E3^- E2^s2 T) = Re(E3^+ E2^-s2 conj(T)):
// each block with s3 = - folds onto s3 = + with its stage-1 result
// conjugated, and conj(sum_j1 E1 C) = sum_j1 conj(E1) conj(C).  In 3-D
// (blocks b = 2 f2 + f3, f = 1 for a negative sign):
//   V_q[j3][j2][x1] = sum_{h,j1} E1^{h}[j1][x1] Cv[j3][q][j2][h][j1],
//     q = 0: Cv[.][0] = C_0, Cv[.][1] = conj(C_3);  q = 1: C_2, conj(C_1)
//   W[j3][x2][x1] = sum_{q,j2} E2^{q}[j2][x2] V_q[j3][j2][x1]
//   u[x3][x2][x1] = Re sum_j3 E3^+[j3][x3] W[j3][x2][x1]
// In 2-D: V[j2][x1] = sum_{h,j1} E1^h (C_0 | conj(C_1)), u = Re sum_j2 E2^+ V.
// The middle intermediate W is a quarter of the per-block one and the last
// contraction runs over nk3 instead of 4 nk3.  Without sign blocks (method 4)
// Cv = C.
//
// Cv[r][j3][q][j2][h][j1] = (conj if h) ampMult amp[r][b][j][j1] exp(i phase),
// stored K-major: element (row m = (r, j3, q, j2), k = (h, j1)) at k * rows + m,
// so the first contraction's operand loads run along rows (whole cache lines
// per wave) instead of 16 rows of 32 bytes each.
// ph == NULL: real coefficients (method 4), no phase factor.
// One block per 64 x 64 tile of (row m, k): the coefficients are formed in
// the source order (k fastest: the amplitude and phase reads are contiguous
// along j1) into LDS and written out K-major (m fastest).
// The phase is 2 pi U with U the phase uniform [r][src] (randomFieldND.f90:
// 278-279), or, Draw, element (*draw * Nmc + r) * kNr + src of the device
// stream (seed, tag 2) -- the uniform the plan's generator would have drawn.
// ampStrideR 0: every realization has the amplitudes of row 0.
constexpr int kFoldM = 64, kFoldK = 32;   // coefficient-fold tile: rows x k


// One 64-row x 32-k tile of the folded coefficients, transposed through LDS
// to the K-major layout C[k * rows + m]; rows < 2^31 (checked by the launchers).
template <bool Draw>
__device__ __forceinline__ void fold_tile(const rf_fold_desc& f, int bx, int by, uint64_t seed, int64_t drawBase,
                                          float2 (*tile)[kFoldM + 1]) {
#pragma clang fp contract(off)
    const int rows = (int)f.rows;
    const int m0 = bx * kFoldM;
    const int k0 = by * kFoldK;
    const unsigned nk1 = (unsigned)f.nk1, nk2 = (unsigned)f.nk2, nk3 = (unsigned)f.nk3;
    const unsigned Q = (f.fold && f.nDim == 3) ? 2u : 1u;
    // a thread keeps one k (256 is a multiple of kFoldK) and walks rows
    // mm0, mm0 + 8, ...: the row's digits (j2, q, j3, r) advance by carries
    // instead of a division per element
    static_assert(256 % kFoldK == 0, "one k per thread");
    constexpr int kRowStep = 256 / kFoldK;
    const int kk = threadIdx.x % kFoldK, mm0 = threadIdx.x / kFoldK;
    const int k = k0 + kk;
    if (k < f.K) {
        const unsigned j1 = (unsigned)k % nk1;
        const unsigned h = (unsigned)k / nk1;
        unsigned rem = (unsigned)(m0 + mm0);
        unsigned j2 = rem % nk2; rem /= nk2;
        unsigned q = rem % Q; rem /= Q;
        unsigned j3 = f.nDim == 3 ? rem % nk3 : 0u;
        unsigned r = f.nDim == 3 ? rem / nk3 : rem;
        for (int mm = mm0; mm < kFoldM; mm += kRowStep) {
            const int m = m0 + mm;
            if (m >= rows) break;
            if (Draw) {
                tile[kk][mm] = fold_coef_draw(f, r, j3, q, j2, j1, h, seed, drawBase);
            } else {
                unsigned b = 0;
                if (f.fold) b = f.nDim == 3 ? (q == 0 ? (h ? 3u : 0u) : (h ? 1u : 2u)) : h;
                const int64_t jb = (int64_t)b * f.kNu + ((int64_t)j3 * nk2 + j2) * nk1 + j1;   // b kNu + j
                const int64_t src = (int64_t)r * f.kNr + jb;
                const double a = f.amp[(int64_t)r * f.ampStrideR + jb] * f.ampMult;
                if (!f.uni) {
                    tile[kk][mm] = make_float2((float)a, 0.0f);
                } else {
                    float cs, sn;
                    cis_rev(f.uni[src], &cs, &sn);
                    tile[kk][mm] = make_float2((float)(a * (double)cs), (float)(h ? -(a * (double)sn) : a * (double)sn));
                }
            }
            // next row m + kRowStep: j2 fastest, then q, then j3 (3-D), then r
            j2 += kRowStep;
            while (j2 >= nk2) {
                j2 -= nk2;
                if (++q == Q) {
                    q = 0;
                    if (f.nDim != 3) {
                        ++r;
                    } else if (++j3 == nk3) {
                        j3 = 0;
                        ++r;
                    }
                }
            }
        }
    }
    __syncthreads();
    for (int e = threadIdx.x; e < kFoldM * kFoldK; e += 256) {
        const int mm = e % kFoldM, kk = e / kFoldM;
        const int m = m0 + mm;
        const int k = k0 + kk;
        if (m < rows && k < f.K) f.C[(int64_t)k * rows + m] = tile[kk][mm];
    }
}

// The coefficients of one grid execution from the plan's phase uniforms
// (f.uni) or, method 4, the real DCT coefficients (f.uni NULL).
__global__ __launch_bounds__(256) void k_coeffs_fold(rf_fold_desc f) {
    __shared__ float2 tile[kFoldK][kFoldM + 1];
    fold_tile<false>(f, blockIdx.x, blockIdx.y, 0, 0, tile);
}

// Every field of a batch in one launch, phases drawn in place: field i owns
// blocks block0 .. block0 + nbx * nby - 1 (ascending in i), block -> field by
// binary search; realizations *draw * Nmc .. of the field's stream.  Logical
// blocks are placed per XCD (xcd_tile): each XCD folds a contiguous run of
// fields, so a field's amplitudes are fetched into one L2, not eight.
__global__ __launch_bounds__(256) void k_coeffs_fold_draw(const rf_fold_item* __restrict__ items, int n,
                                                          const int64_t* __restrict__ draw, int64_t nBlocks) {
    __shared__ float2 tile[kFoldK][kFoldM + 1];
    const int64_t blk = xcd_tile(blockIdx.x, nBlocks);
    if (blk >= nBlocks) return;
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (items[mid].block0 <= blk) lo = mid; else hi = mid - 1;
    }
    const rf_fold_item& it = items[lo];
    const int lb = (int)(blk - it.block0);
    const int64_t drawBase = (*draw) * (int64_t)it.Nmc * it.f.kNr;
    fold_tile<true>(it.f, lb % it.nbx, lb / it.nbx, it.seed, drawBase, tile);
}

inline unsigned blocks_for(int64_t n) { return (unsigned)((n + 255) / 256); }

}  // namespace

// Logical tiles of a GEMM: blocks of strips x table groups, or FP32 tiles.
int64_t rf_gemm_tiles(const rf_gemm_desc& g, int mt) {
    mt &= ~kStripShort;
    if (mt > 0)
        return (int64_t)(((g.M + 31) / 32 + mt - 1) / mt) * (((int64_t)g.N + kStripL - 1) / kStripL) * g.batches;
    return (int64_t)((g.N + kTN - 1) / kTN) * ((g.M + kTM - 1) / kTM) * g.batches;
}

// blocks of a launch over nTiles logical tiles (a multiple of the XCD count)
inline int64_t xcd_blocks(int64_t nTiles) { return (nTiles + kXcd - 1) / kXcd * kXcd; }

namespace {
// One GEMM (g) or a group of them (d_gs, nG), all of one kind: strips of
// mt tiles or, mt 0, FP32-operand tiles.
hipError_t launch_any(int kind, int mt, const rf_gemm_desc* g, const rf_gemm_desc* d_gs, int nG, int64_t nTiles,
                      hipStream_t s) {
    if (nTiles <= 0) return hipSuccess;
    const int64_t nb = xcd_blocks(nTiles);
    if (nb > rf_max_blocks(256) || mt < 0 || (mt & ~kStripShort) > kStripMaxMT) return hipErrorInvalidValue;
    const unsigned blocks = (unsigned)nb;
    if (kind == RF_GEMM_ISO) return rf_strip_launch_iso(mt, g, d_gs, nG, nTiles, blocks, s);
    if (mt > 0 && g && g->real) {
        if (kind == RF_GEMM_FIRST) return rf_strip_launch_first_real(mt, g, d_gs, nG, nTiles, blocks, s);
        if (kind == RF_GEMM_MIDDLE) return rf_strip_launch_middle_real(mt, g, d_gs, nG, nTiles, blocks, s);
        return rf_strip_launch_last_real(mt, g, d_gs, nG, nTiles, blocks, s);
    }
    if (mt > 0) {
        if (kind == RF_GEMM_FIRST) return rf_strip_launch_first(mt, g, d_gs, nG, nTiles, blocks, s);
        if (kind == RF_GEMM_MIDDLE) return rf_strip_launch_middle(mt, g, d_gs, nG, nTiles, blocks, s);
        return rf_strip_launch_last(mt, g, d_gs, nG, nTiles, blocks, s);
    }
    if (kind == RF_GEMM_LAST) {
        if (g) hipLaunchKernelGGL(k_cgemm<true>, dim3(blocks), dim3(256), 0, s, *g, nTiles);
        else hipLaunchKernelGGL(k_cgemm_group<true>, dim3(blocks), dim3(256), 0, s, d_gs, nG, nTiles);
    } else {
        if (g) hipLaunchKernelGGL(k_cgemm<false>, dim3(blocks), dim3(256), 0, s, *g, nTiles);
        else hipLaunchKernelGGL(k_cgemm_group<false>, dim3(blocks), dim3(256), 0, s, d_gs, nG, nTiles);
    }
    return hipGetLastError();
}

// MT of a strip GEMM: all of the table axis in one wave (up to kStripMaxMT
// tiles) so that every streamed value is read and converted once, unless the
// launch would then leave SIMDs without a wave.  The last contraction, whose
// stores bound it, takes at most 3 tiles: 32 fields of ~131^3 x 16 (K 44, short
// form) on 4 / 3 / 2 / 1 tiles: 2.15 / 1.96 / 2.18 / 2.67 ms, in chunks 2.31 / 2.29 /
// 2.29 / 2.66; 135 x 131 x 131 x 4 in chunks on 5 / 3: 24.8 / 20.6 us (a batch tunes it).
int strip_choose(const rf_gemm_desc& g) {
    const int mt = (g.M + 31) / 32;
    const int64_t strips = (((int64_t)g.N + 31) / 32) * g.batches;
    const int most = g.kind == RF_GEMM_LAST ? 3 : kStripMaxMT;
    int gr = (mt + most - 1) / most;
    while (gr < mt && strips * gr < kStripFill) gr++;
    return (mt + gr - 1) / gr | (rf_strip_short(g) ? kStripShort : 0);
}
}  // namespace

hipError_t rf_launch_gemm_group(int kind, int mt, const rf_gemm_desc* d_gs, int nG, int64_t nTiles, hipStream_t s) {
    if (nG <= 0) return hipSuccess;
    return launch_any(kind, mt, nullptr, d_gs, nG, nTiles, s);
}

// Room for an axis' table in either layout (float2 elements; fragment order:
// K entries to whole steps, 32-entry tiles; 256-byte aligned).
static int64_t table_elems(int nk, int n) {
    const int64_t frag = (2LL * nk + 7) / 8 * 8 * (((int64_t)n + 31) / 32 * 32), plain = 2LL * nk * n;
    return ((frag > plain ? frag : plain) + 31) / 32 * 32;
}

// Scratch for one grid execution (float2 elements): tables (both sign
// variants per axis), folded coefficients, V and (3-D) W.
size_t rf_grid_scratch_elems(int nDim, const int32_t* kNStep, int nb, int Nmc, const int32_t* n) {
    const int fold = nb > 1, Q = (fold && nDim == 3) ? 2 : 1;
    int64_t tables = 0;
    for (int a = 0; a < nDim; a++) tables += table_elems(kNStep[a], n[a]);
    int64_t coeff = (int64_t)nb * Nmc;
    for (int a = 0; a < nDim; a++) coeff *= kNStep[a];
    int64_t v = (int64_t)Nmc * Q * n[0];
    for (int a = 1; a < nDim; a++) v *= kNStep[a];
    const int64_t w = nDim == 3 ? (int64_t)Nmc * kNStep[2] * n[1] * n[0] : 0;
    return (size_t)(tables + coeff + v + w);
}

// Builds the phase tables and coefficients in scratch (launches on s) and
// describes the GEMM stages: stage 1 rows (r, b, j_d..j_2) x j1 -> x1;
// stage 2 (3-D) per (r, b, j3): x2 x j2 times j2 x x1; last stage per r:
// x_d x (b, j_d) times (b, j_d) x plane, real part, epilogue, into d_out.
hipError_t rf_grid_prepare(int kind, int nDim, int Nmc, const int32_t* kNStep, const double* kDelta, int nb,
                           const double* origin, const double* step, const int32_t* n,
                           const double* corrL, const double* d_amp, int ampShared, const double* d_unif,
                           double ampMult, double coefMax, const rf_epilogue& epi, void* d_out, int outDtype,
                           float2* scratch, hipStream_t s, rf_grid_stages* st, rf_grid_coef* coef) {
    // power-of-two scales for the FP16 operands: coefficients into [1/2, 1),
    // the middle contraction's output below 2^14 (|V| <= eMax K1 and
    // |W| <= eMax^2 K1 K2 for |table| <= eMax); the last stage undoes both
    const int fold = nb > 1 ? 1 : 0;
    const int H = fold ? 2 : 1, Q = (fold && nDim == 3) ? 2 : 1;
    const double eMax = kind == 1 ? 2.0 : 1.0;
    double sc = 1.0;
    if (coefMax > 0.0 && std::isfinite(coefMax)) {
        int e = 0;
        std::frexp(coefMax, &e);
        sc = std::ldexp(1.0, -e);
    }
    const int K1 = H * kNStep[0];
    const int K2 = nDim == 3 ? Q * kNStep[1] : kNStep[1];
    const double bound1 = eMax * K1;
    const double bound2 = nDim == 3 ? eMax * eMax * K1 * (double)K2 : bound1;
    int m2 = 0;
    while (nDim == 3 && std::ldexp(bound2, -m2) > 16384.0) m2++;
    int split = bound1 <= 16384.0 ? 1 : 0;

    // the strip GEMM addresses eight k of a strip's lines in 32-bit bytes and a
    // tile of D in 32-bit elements
    {
        const int64_t lim = (int64_t)1 << 29;
        int64_t rows1 = (int64_t)Nmc * Q, plane = n[0];
        for (int a = 1; a < nDim; a++) rows1 *= kNStep[a];
        if (nDim == 3) plane *= n[1];
        int64_t span = 8 * rows1;                                       // first: K-major coefficients
        if (8LL * n[0] > span) span = 8LL * n[0];                       // first: D (32 lines), a quarter
        if (8 * plane > span) span = 8 * plane;                         // last: streamed, D
        if (nDim == 3 && ((int64_t)K2 + 8) * n[0] > span) span = ((int64_t)K2 + 8) * n[0];      // middle: streamed
        if (nDim == 3 && 40LL * n[0] + plane > span) span = 40LL * n[0] + plane;                // middle: D
        if (span >= lim) split = 0;
    }

    float2* p = scratch;
    void* E[3];
    rf_table_args ta{};
    ta.dct = kind == 1;
    ta.nAx = nDim;
    ta.frag = split;
    unsigned tabBlocks = 0;
    for (int a = 0; a < nDim; a++) {
        E[a] = p; p += table_elems(kNStep[a], n[a]);
        ta.nk[a] = kNStep[a];
        ta.nx[a] = n[a];
        // the last axis has no sign variants left (folded)
        ta.K[a] = a == nDim - 1 ? kNStep[a] : a == 0 ? K1 : K2;
        ta.block0[a] = tabBlocks;
        tabBlocks += split ? (unsigned)((ta.K[a] + 7) / 8) * (unsigned)((n[a] + 31) / 32)
                           : blocks_for((int64_t)kNStep[a] * n[a]);
        ta.dk[a] = kDelta[a]; ta.o[a] = origin[a]; ta.step[a] = step[a]; ta.invL[a] = 1.0 / corrL[a];
        ta.E[a] = E[a];
    }
    hipLaunchKernelGGL(k_axis_tables, dim3(tabBlocks), dim3(256), 0, s, ta);
    int64_t kNu = 1;
    for (int a = 0; a < nDim; a++) kNu *= kNStep[a];
    const int64_t nC = (int64_t)Nmc * nb * kNu;          // = Nmc x nk3 x Q x nk2 x H x nk1
    float2* Cf = p; p += nC;
    // a caller-owned coefficient buffer is reused while its scale matches
    // (the coefficients depend only on the plan and the scale).  Method 4 of a
    // plan: its real amplitudes go into the first contraction as they are (no
    // fold, 50 us of 128^3 x 8), on real operands throughout
    const bool real = coef && split && kind == 1;
    bool fresh = real;
    if (coef && coef->buf) {
        Cf = coef->buf;
        fresh = fresh || coef->key == ampMult * sc;
        coef->key = ampMult * sc;
    }
    *st = rf_grid_stages{};
    rf_fold_desc& fd = st->fold;
    fd.rows = nC / K1; fd.K = K1; fd.nDim = nDim; fd.fold = fold;
    fd.nk1 = kNStep[0]; fd.nk2 = nDim > 1 ? kNStep[1] : 1; fd.nk3 = nDim > 2 ? kNStep[2] : 1;
    fd.kNu = kNu; fd.kNr = (int64_t)nb * kNu;
    fd.amp = d_amp; fd.ampStrideR = ampShared ? 0 : fd.kNr;
    fd.uni = kind == 1 ? nullptr : d_unif;
    fd.ampMult = ampMult * sc; fd.C = Cf;
    if (fd.rows > INT32_MAX) return hipErrorInvalidValue;
    if (!fresh)
        hipLaunchKernelGGL(k_coeffs_fold,
                           dim3((unsigned)((fd.rows + kFoldM - 1) / kFoldM), (unsigned)((K1 + kFoldK - 1) / kFoldK)),
                           dim3(256), 0, s, fd);
    // stage 1: rows (r, j3, q, j2) x K (h, j1) -> V[r][j3][q][j2][x1].  FP32
    // tiles: A = the coefficients, B = the table; strips: the table x1 x K
    // against the lines (r, j3, q, j2) of the K-major coefficients
    const int64_t rows1 = nC / K1;
    float2* V = p; p += rows1 * n[0];
    auto table = [&](rf_gemm_desc& q, int a) {       // the table operand of axis a, rows x
        if (split) q.T = E[a];
        else {
            q.A = static_cast<const float2*>(E[a]);
            q.aSm = 1; q.aSk = n[a];
        }
        q.aDiv = 1; q.aMod = 1;
        q.M = n[a]; q.dSm = 1;
    };
    rf_gemm_desc& g = st->g[st->n++];
    g.kind = RF_GEMM_FIRST;
    if (split) {
        table(g, 0);
        g.B = Cf; g.bSk = rows1; g.bSn = 1;          // K-major
        g.D = V; g.dSn = n[0];
        g.N = (int)rows1;
    } else {
        g.A = Cf; g.aSm = 1; g.aSk = rows1; g.aDiv = 1; g.aMod = 1;
        g.B = static_cast<const float2*>(E[0]); g.bSk = n[0]; g.bSn = 1;     // K (h, j1): variant h of E1
        g.D = V; g.dSm = n[0]; g.dSn = 1;
        g.M = (int)rows1; g.N = n[0];
    }
    g.K = K1; g.batches = 1;
    g.gen = fd;
    if (real) {
        // lines (r, j3, j2) of the amplitudes, k contiguous (no sign blocks)
        g.B = reinterpret_cast<const float2*>(d_amp);
        g.bSk = 1; g.bSn = kNStep[0];
    }
    g.outScale = 1.0f;
    const float2* last = V;
    int64_t plane = n[0];                      // points already resolved
    int64_t lastStrideB = (int64_t)kNStep[1] * n[0];
    if (nDim == 3) {
        // stage 2, batch r, columns (j3, x1):
        // W[j3][x2][x1] = sum_{q,j2} E2^q[j2][x2] V[j3][q][j2][x1]
        float2* W = p; p += (int64_t)Nmc * kNStep[2] * n[1] * n[0];
        rf_gemm_desc& h = st->g[st->n++];
        h.kind = RF_GEMM_MIDDLE;
        table(h, 1);
        h.B = V; h.bSk = n[0]; h.bSn = 1; h.bStrideB = (int64_t)kNStep[2] * K2 * n[0];
        h.D = W; h.dSm = n[0]; h.dSn = 1; h.dStrideB = (int64_t)kNStep[2] * n[1] * n[0];
        h.nLo = n[0]; h.bSnHi = (int64_t)K2 * n[0]; h.dSnHi = (int64_t)n[1] * n[0];
        h.N = kNStep[2] * n[0]; h.K = K2; h.batches = Nmc;
        h.outScale = (float)std::ldexp(1.0, -m2);
        last = W;
        plane = (int64_t)n[0] * n[1];
        lastStrideB = (int64_t)kNStep[2] * plane;
    }
    // last stage per realization: u[x_d][plane] = Re sum_j E_d^+[j][x_d] last[j][plane]
    const int ad = nDim - 1;
    rf_gemm_desc& f = st->g[st->n++];
    f.kind = RF_GEMM_LAST;
    table(f, ad);
    f.B = last; f.bSk = plane; f.bSn = 1; f.bStrideB = lastStrideB;
    f.D = d_out; f.dSm = plane; f.dSn = 1; f.dStrideB = plane * n[ad];
    f.N = (int)plane; f.K = kNStep[ad]; f.batches = Nmc;
    f.outDtype = outDtype; f.epi = epi;
    f.outScale = (float)(1.0 / (sc * std::ldexp(1.0, -m2)));
    for (int i = 0; i < st->n; i++) {
        st->g[i].mt = split ? strip_choose(st->g[i]) : 0;
        st->g[i].real = real;
    }
    return hipGetLastError();
}

int rf_fold_item_blocks(const rf_fold_desc& f) {
    return (int)(((f.rows + kFoldM - 1) / kFoldM) * ((f.K + kFoldK - 1) / kFoldK));
}

void rf_fold_item_init(rf_fold_item* it, const rf_fold_desc& f, int Nmc, uint64_t seed, int64_t block0) {
    it->f = f;
    it->seed = seed;
    it->Nmc = Nmc;
    it->nbx = (int)((f.rows + kFoldM - 1) / kFoldM);
    it->block0 = block0;
}

hipError_t rf_launch_refold_draw(const rf_fold_item* d_items, int n, int64_t blocks, const int64_t* d_draw,
                                 hipStream_t s) {
    if (n <= 0 || blocks <= 0) return hipSuccess;
    if (!d_items || !d_draw || xcd_blocks(blocks) > rf_max_blocks(256)) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_coeffs_fold_draw, dim3((unsigned)xcd_blocks(blocks)), dim3(256), 0, s, d_items, n, d_draw,
                       blocks);
    return hipGetLastError();
}

namespace {
__global__ void k_draw_counter(int64_t* st, int64_t value, int gen) {
    if (threadIdx.x != 0) return;
    if (value >= 0) {
        st[0] = value;
        st[1] = value;
    } else if (value == -1) {
        st[1] = st[0];
        st[0] = st[0] + 1;
    } else if (value == -2) {
        st[0] = 1;
        st[1] = 0;
    }
    st[2] = gen;
}
}  // namespace

hipError_t rf_launch_draw_counter(int64_t* d_state, int64_t value, int gen, hipStream_t s) {
    hipLaunchKernelGGL(k_draw_counter, dim3(1), dim3(64), 0, s, d_state, value, gen);
    return hipGetLastError();
}

hipError_t rf_grid_run(const rf_grid_stages& st, hipStream_t s) {
    for (int i = 0; i < st.n; i++) {
        const rf_gemm_desc& g = st.g[i];
        const hipError_t e = launch_any(g.kind, g.mt, &g, nullptr, 0, rf_gemm_tiles(g, g.mt), s);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

static int64_t iso_k_padded(int64_t kN) { return (kN + 7) / 8 * 8; }

// the last axis' table in whole 32-entry tiles
size_t rf_iso_grid_scratch_elems(int nDim, int64_t kN, int Nmc, const int32_t* n) {
    int64_t t = 0;
    for (int a = 0; a < nDim; a++) t += a == nDim - 1 ? ((int64_t)n[a] + 31) / 32 * 32 : n[a];
    return (size_t)(Nmc * iso_k_padded(kN) * t);
}

hipError_t rf_launch_iso_grid(const rf_iso_grid_args& a, hipStream_t s) {
    if (a.nDim < 2 || a.nDim > 3 || a.Nmc < 1 || a.kN < 1) return hipErrorInvalidValue;
    // coefficients into [1/2, 1) by a power of two, undone by the epilogue
    double sc = 1.0;
    if (a.coefMax > 0.0 && std::isfinite(a.coefMax)) {
        int e = 0;
        std::frexp(a.coefMax, &e);
        sc = std::ldexp(1.0, -e);
    }
    const int64_t kP = iso_k_padded(a.kN);
    rf_iso_tables t{};
    t.nDim = a.nDim; t.Nmc = a.Nmc; t.kN = a.kN; t.kP = kP;
    t.kIso = a.kIso; t.amp = a.amp; t.phase = a.phase;
    t.coef = a.ampMult * sc;
    const int ad = a.nDim - 1;
    float2* p = a.scratch;
    for (int d = 0; d < a.nDim; d++) {
        t.n[d] = a.n[d];
        t.w[d] = d == ad ? (a.n[d] + 31) / 32 * 32 : a.n[d];
        t.o[d] = a.origin[d]; t.st[d] = a.step[d]; t.inv[d] = a.invL[d];
        if (d == ad) t.Z = reinterpret_cast<_Float16*>(p);
        else t.T[d] = p;
        p += a.Nmc * kP * t.w[d];
    }
    const int64_t cnt = a.Nmc * kP * ((int64_t)t.w[0] + t.w[1] + t.w[2]);
    if ((cnt + 255) / 256 > rf_max_blocks(256)) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_iso_tables, dim3(blocks_for(cnt)), dim3(256), 0, s, t);
    rf_gemm_desc g{};
    g.kind = RF_GEMM_ISO;
    g.T = t.Z; g.M = a.n[ad]; g.K = (int)kP; g.batches = a.Nmc;
    g.B = t.T[0]; g.bStrideB = kP * a.n[0]; g.isoNx = a.n[0]; g.isoNy = 1;
    g.N = a.n[0];
    if (a.nDim == 3) {
        g.isoY = t.T[1]; g.isoNy = a.n[1]; g.isoYStrideB = kP * a.n[1];
        g.N = a.n[0] * a.n[1];
    }
    g.D = a.d_out; g.dSm = g.N; g.dSn = 1; g.dStrideB = (int64_t)g.M * g.N;
    g.outDtype = a.outDtype;
    g.epi = a.epi;
    g.outScale = (float)(1.0 / sc);
    g.mt = strip_choose(g);
    return launch_any(g.kind, g.mt, &g, nullptr, 0, rf_gemm_tiles(g, g.mt), s);
}
