// rf_post.hip -- HBM-bound kernels around the spectral sum:
//   marginal map        multiVariateTransformation (randomFieldND.f90:139-178)
//   FP64 moments        calculate_average_and_stdVar_MPI (statistics_RF.f90:18-87)
//   normalisation       normalize_randField (randomFieldND.f90:820-926)
//   overlap blend       add_RF_to_Group + generateUnityPartition_Matrix + the
//                       boundary correction (localization_RF.f90:199-263,705-857;
//                       calls_RF.f90:324-369), in gather form: every group point
//                       reads its <= 2^d covering subdomains, no atomics.
#include "rf_internal.h"
#include "rf_blend.h"

#include <algorithm>
#include <climits>
#include <type_traits>

namespace {

constexpr int kBlock = 256;

template <typename T>
__global__ __launch_bounds__(kBlock) void k_marginal(int margi, double scale, double shift,
                                                     T* __restrict__ d, int64_t n) {
#pragma clang fp contract(off)
    constexpr int U = 4;                  // independent loads in flight per thread
    const int64_t stride = (int64_t)gridDim.x * kBlock;
    for (int64_t e = (int64_t)blockIdx.x * kBlock + threadIdx.x; e < n; e += U * stride) {
        T v[U];
#pragma unroll
        for (int u = 0; u < U; u++) v[u] = (e + u * stride < n) ? d[e + u * stride] : T(0);
#pragma unroll
        for (int u = 0; u < U; u++)
            if (e + u * stride < n) {
                const double y = (double)v[u] * scale + shift;                  // :171
                d[e + u * stride] = (T)((margi == RF_FOM_LOGNORMAL) ? exp(y) : y);  // :175
            }
    }
}

// The same map over 16-byte vectors (4 floats or 2 doubles per load): nVec
// vectors from d, which must be 16-byte aligned; the tail goes to k_marginal.
template <typename T>
__global__ __launch_bounds__(kBlock) void k_marginal_vec(int margi, double scale, double shift,
                                                         T* __restrict__ d, int64_t nVec) {
#pragma clang fp contract(off)
    constexpr int L = 16 / sizeof(T);
    typedef T vec __attribute__((ext_vector_type(L)));
    vec* v = reinterpret_cast<vec*>(d);
    const int64_t stride = (int64_t)gridDim.x * kBlock;
    for (int64_t e = (int64_t)blockIdx.x * kBlock + threadIdx.x; e < nVec; e += 2 * stride) {
        vec a = v[e];
        vec b = (e + stride < nVec) ? v[e + stride] : a;
#pragma unroll
        for (int l = 0; l < L; l++) {
            const double ya = (double)a[l] * scale + shift;
            const double yb = (double)b[l] * scale + shift;
            a[l] = (T)((margi == RF_FOM_LOGNORMAL) ? exp(ya) : ya);
            b[l] = (T)((margi == RF_FOM_LOGNORMAL) ? exp(yb) : yb);
        }
        v[e] = a;
        if (e + stride < nVec) v[e + stride] = b;
    }
}

// Partial sums of u and u^2 of each realization in FP64; grid (nPart, Nmc).  Bound by
// the read: two independent 16-byte loads per thread and turn where every
// realization starts on a 16-byte boundary (VEC), one element otherwise
// (128^3 x 16 FP32: 27 -> 22 us, 6.0 TB/s).
template <typename T, bool VEC>
__global__ __launch_bounds__(kBlock) void k_moments_partial(const T* __restrict__ d, int64_t N,
                                                            double* __restrict__ part) {
    constexpr int L = VEC ? 16 / sizeof(T) : 1;
    typedef T vec __attribute__((ext_vector_type(L)));
    __shared__ double s1[kBlock], s2[kBlock];
    const int r = blockIdx.y;
    const T* col = d + (int64_t)r * N;
    double a = 0.0, b = 0.0, a2 = 0.0, b2 = 0.0;
    const int64_t stride = (int64_t)gridDim.x * kBlock;
    const int64_t nV = N / L;
    int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (VEC) {
        const vec* cv = reinterpret_cast<const vec*>(col);
        for (; i + stride < nV; i += 2 * stride) {
            const vec v = cv[i], w = cv[i + stride];
#pragma unroll
            for (int l = 0; l < L; l++) {
                const double x = (double)v[l], y = (double)w[l];
                a += x;
                b = fma(x, x, b);
                a2 += y;
                b2 = fma(y, y, b2);
            }
        }
        if (i < nV) {
            const vec v = cv[i];
#pragma unroll
            for (int l = 0; l < L; l++) {
                const double x = (double)v[l];
                a += x;
                b = fma(x, x, b);
            }
        }
        i = nV * L + (int64_t)blockIdx.x * kBlock + threadIdx.x;   // the last N % L elements
    }
    for (; i < N; i += stride) {
        const double v = (double)col[i];
        a += v;
        b = fma(v, v, b);
    }
    s1[threadIdx.x] = a + a2;
    s2[threadIdx.x] = b + b2;
    __syncthreads();
    for (int w = kBlock / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) {
            s1[threadIdx.x] += s1[threadIdx.x + w];
            s2[threadIdx.x] += s2[threadIdx.x + w];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        part[((int64_t)r * gridDim.x + blockIdx.x) * 2 + 0] = s1[0];
        part[((int64_t)r * gridDim.x + blockIdx.x) * 2 + 1] = s2[0];
    }
}

// Partial sums of u and u^2 over the box lo..hi (0-based, inclusive) of
// realization 0 of a grid field (x fastest); grid (nPart).  The summed box is
// the window normalize_randField reads through its RF_2D / RF_3D views of
// column 1 (randomFieldND.f90:857-862).
template <typename T>
__global__ __launch_bounds__(kBlock) void k_window_moments_partial(const T* __restrict__ d, rf_window w,
                                                                   double* __restrict__ part) {
    __shared__ double s1[kBlock], s2[kBlock];
    double a = 0.0, b = 0.0;
    const int64_t stride = (int64_t)gridDim.x * kBlock;
    for (int64_t q = (int64_t)blockIdx.x * kBlock + threadIdx.x; q < w.count; q += stride) {
        const int64_t i0 = q % w.ext[0];
        const int64_t r = q / w.ext[0];
        const int64_t i1 = r % w.ext[1];
        const int64_t i2 = r / w.ext[1];
        const int64_t off = (w.lo[0] + i0) + w.n[0] * ((w.lo[1] + i1) + w.n[1] * (w.lo[2] + i2));
        const double v = (double)d[off];
        a += v;
        b = fma(v, v, b);
    }
    s1[threadIdx.x] = a;
    s2[threadIdx.x] = b;
    __syncthreads();
    for (int k = kBlock / 2; k > 0; k >>= 1) {
        if ((int)threadIdx.x < k) {
            s1[threadIdx.x] += s1[threadIdx.x + k];
            s2[threadIdx.x] += s2[threadIdx.x + k];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        part[(int64_t)blockIdx.x * 2 + 0] = s1[0];
        part[(int64_t)blockIdx.x * 2 + 1] = s2[0];
    }
}

// Sum over a wave, the same order on every run; the result is in every lane.
__device__ inline double wave_sum(double v) {
#pragma unroll
    for (int w = 32; w > 0; w >>= 1) v += __shfl_xor(v, w);
    return v;
}

// Fixed-order final reduction of the partials: sums[r] = (sum u, sum u^2),
// one wave per realization (a serial chain over the 256 partials of a large
// field took 26 us; 3 us so).
__global__ __launch_bounds__(64) void k_moments_final(const double* __restrict__ part, int nPart,
                                                      double* __restrict__ sums) {
    const int r = blockIdx.x;
    double a = 0.0, b = 0.0;
    for (int p = threadIdx.x; p < nPart; p += 64) {
        a += part[((int64_t)r * nPart + p) * 2 + 0];
        b += part[((int64_t)r * nPart + p) * 2 + 1];
    }
    a = wave_sum(a);
    b = wave_sum(b);
    if (threadIdx.x == 0) {
        sums[2 * r + 0] = a;
        sums[2 * r + 1] = b;
    }
}

// u <- (u - shift_r) * mul_r
template <typename T>
__global__ void k_affine(T* __restrict__ d, int64_t N, const double* __restrict__ shift,
                         const double* __restrict__ mul) {
    const int r = blockIdx.y;
    T* col = d + (int64_t)r * N;
    const double m = shift[r], s = mul[r];
    const int64_t stride = (int64_t)gridDim.x * kBlock;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < N; i += stride)
        col[i] = (T)(((double)col[i] - m) * s);
}

// ------------------------------------------------- directional correlation
// rebuild_Sk_FFT (statistics_RF.f90:262-409) restated as the circular
// autocorrelation it computes: for lag m (grid y) the sum over all points of
// v(x) v(x + m e_a mod n_a), v = (u - avg)/std, in FP64; partials per block
// (grid x), reduced in fixed order by k_corr_final.
template <typename T>
__global__ __launch_bounds__(kBlock) void k_corr_partial(const T* __restrict__ u, int64_t N, int64_t strideA,
                                                         int nA, double avg, double std,
                                                         double* __restrict__ part) {
    __shared__ double sh[kBlock];
    const int m = blockIdx.y;
    double acc = 0.0;
    const int64_t stride = (int64_t)gridDim.x * kBlock;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < N; i += stride) {
        const int64_t ia = (i / strideA) % nA;
        int64_t ja = ia + m;
        if (ja >= nA) ja -= nA;
        const int64_t j = i + (ja - ia) * strideA;
        const double vi = ((double)u[i] - avg) / std;
        const double vj = ((double)u[j] - avg) / std;
        acc = fma(vi, vj, acc);
    }
    sh[threadIdx.x] = acc;
    __syncthreads();
    for (int w = kBlock / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[(int64_t)m * gridDim.x + blockIdx.x] = sh[0];
}

// One wave per lag (grid x), partials in fixed order.
__global__ __launch_bounds__(64) void k_corr_final(const double* __restrict__ part, int nPart, double invN,
                                                   double* __restrict__ R) {
    const int m = blockIdx.x;
    double s = 0.0;
    for (int p = threadIdx.x; p < nPart; p += 64) s += part[(int64_t)m * nPart + p];
    s = wave_sum(s);
    if (threadIdx.x == 0) R[m] = s * invN;
}

// The same correlations through the FP64 matrix cores.  With v_l the
// normalised values of line l along the axis, G = sum_l v_l v_l^T holds every
// product of two points of a line; the lag m is the sum of G over j - i = m and
// j - i = m - n.  One pass over the field gives all lags, where the lag
// sweep above reads it twice per lag.  A block holds the tile pair (SI, SJ),
// SI <= SJ, of 64 positions each, and a share of the lines: 16 accumulator
// tiles of v_mfma_f64_16x16x4_f64 per wave, whose A and B operands have the
// same lane layout (position l % 16, line l / 16), so the fragments come
// straight from global memory and one load serves a row and a column of
// tiles.  The four lines of lane group g and step t are 4 g + t: 16
// neighbouring lines per turn, contiguous for every axis but the first.  Bound
// by the matrix cores (16 MFMAs of 64 cycles per 8 fragments); all axes of a
// field share one launch.  128^3 FP32: 3 x 307 us (the sweep) -> 56 us.
typedef double d4v __attribute__((ext_vector_type(4)));
constexpr int kCorrT = 64;                 // positions per side of a tile pair
constexpr int kCorrDiag = 2 * kCorrT;      // partial sums per block: j - i + 63 in 0 .. 126

template <typename T>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(2, 2)))
void k_corr_gram(rf_corr_gram q, const T* __restrict__ u, double avg, double std, double* __restrict__ part) {
    __shared__ double tile[4][7 * 256];
    __shared__ double diag[4][kCorrDiag];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int c = lane & 15, g = lane >> 4;
    int ax = 0;
    while (ax + 1 < q.nAx && (int)blockIdx.x >= q.ax[ax + 1].block0) ax++;
    const rf_corr_axis A = q.ax[ax];
    const int local = (int)blockIdx.x - A.block0;
    const int chunk = local % A.chunks;
    // tile pair: distance-major, pair(D, SI) = sum_{k < D} (nS - k) + SI
    int SI = local / A.chunks, D = 0;
    while (SI >= A.nS - D) {
        SI -= A.nS - D;
        D++;
    }
    const int SJ = SI + D;
    const int pi = SI * kCorrT + c, pj = SJ * kCorrT + c;

    // the lane's four lines, as (offset of the line's first point, index along
    // the faster axes); 64 * chunks lines further on every turn
    const int64_t S = A.stride, hop = S * (A.n - 1);
    const int64_t dq = (int64_t)64 * A.chunks;
    const int64_t dO = dq / S, dX = dq - dO * S;
    int64_t line = (int64_t)(chunk * 4 + wave) * 16 + 4 * g;
    int64_t x[4], base[4];
#pragma unroll
    for (int t = 0; t < 4; t++) {
        const int64_t o = (line + t) / S;
        x[t] = (line + t) - o * S;
        base[t] = o * S * A.n + x[t];
    }
    d4v acc[4][4];
#pragma unroll
    for (int I = 0; I < 4; I++)
#pragma unroll
        for (int J = 0; J < 4; J++) acc[I][J] = d4v{0.0, 0.0, 0.0, 0.0};

    const int64_t turns = (A.nLines - (int64_t)(chunk * 4 + wave) * 16 + dq - 1) / dq;   // wave-uniform
    for (int64_t it = 0; it < turns; it++) {
        T a[4][4], b[4][4];
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const bool in = line + t < A.nLines;
            const T* p = u + (in ? base[t] : 0);
#pragma unroll
            for (int I = 0; I < 4; I++) {
                const int i = pi + 16 * I, j = pj + 16 * I;
                a[t][I] = p[in && i < A.n ? i * S : 0];
                b[t][I] = D == 0 ? a[t][I] : p[in && j < A.n ? j * S : 0];
            }
        }
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const bool in = line + t < A.nLines;
            double va[4], vb[4];
#pragma unroll
            for (int I = 0; I < 4; I++) {
                va[I] = in && pi + 16 * I < A.n ? ((double)a[t][I] - avg) / std : 0.0;
                if (D == 0) vb[I] = va[I];
                else vb[I] = in && pj + 16 * I < A.n ? ((double)b[t][I] - avg) / std : 0.0;
            }
#pragma unroll
            for (int I = 0; I < 4; I++)
#pragma unroll
                for (int J = 0; J < 4; J++)
                    if (I <= J || D != 0)
                        acc[I][J] = __builtin_amdgcn_mfma_f64_16x16x4f64(va[I], vb[J], acc[I][J], 0, 0, 0);
        }
#pragma unroll
        for (int t = 0; t < 4; t++) {
            x[t] += dX;
            base[t] += dO * S * A.n + dX;
            if (x[t] >= S) {
                x[t] -= S;
                base[t] += hop;
            }
        }
        line += dq;
    }

    // tiles of equal J - I added up, then each diagonal of the wave's sums.
    // Positions past the axis end enter no diagonal (a product with a value
    // that is not finite is not zero there).
    for (int k = -3; k <= 3; k++) {
        d4v s = {0.0, 0.0, 0.0, 0.0};
        if (k >= 0 || D != 0) {
#pragma unroll
            for (int I = 0; I < 4; I++)
#pragma unroll
                for (int J = 0; J < 4; J++)
                    if (J - I == k) {
#pragma unroll
                        for (int e = 0; e < 4; e++)
                            if (pi - c + 16 * I + 4 * e + g < A.n && pj + 16 * J < A.n) s[e] += acc[I][J][e];
                    }
        }
#pragma unroll
        for (int e = 0; e < 4; e++) tile[wave][(k + 3) * 256 + (4 * e + g) * 16 + c] = s[e];   // row 4 e + g, column c
    }
    __syncthreads();
    for (int t = lane; t < kCorrDiag - 1; t += 64) {
        const int d = t - (kCorrT - 1);
        const int k = (d + 64) / 16 - 4, rem = d - 16 * k;            // d = 16 k + rem, 0 <= rem < 16
        double s = 0.0;
        if (d >= 0 || D != 0) {
            if (k >= -3)
                for (int r = 0; r + rem < 16; r++) s += tile[wave][(k + 3) * 256 + r * 16 + r + rem];
            if (rem > 0 && k + 1 <= 3)
                for (int r = 16 - rem; r < 16; r++) s += tile[wave][(k + 4) * 256 + r * 16 + r + rem - 16];
        }
        diag[wave][t] = s;
    }
    __syncthreads();
    for (int t = threadIdx.x; t < kCorrDiag - 1; t += kBlock)
        part[(int64_t)blockIdx.x * kCorrDiag + t] = ((diag[0][t] + diag[1][t]) + diag[2][t]) + diag[3][t];
}

// R[m] of every axis from the blocks' diagonals: one wave per lag, fixed order.
__global__ __launch_bounds__(64) void k_corr_gram_final(rf_corr_gram q, const double* __restrict__ part,
                                                        double invN, double* __restrict__ R) {
    int ax = 0;
    while (ax + 1 < q.nAx && (int)blockIdx.x >= q.ax[ax + 1].lag0) ax++;
    const rf_corr_axis A = q.ax[ax];
    const int m = (int)blockIdx.x - A.lag0;
    double s = 0.0;
    for (int h = 0; h < (m > 0 ? 2 : 1); h++) {
        const int d = h ? A.n - m : m;                  // j - i = d, lag m or n - m
        for (int D = d / kCorrT; D <= (d + kCorrT - 1) / kCorrT && D < A.nS; D++) {
            const int64_t b0 = A.block0 + (int64_t)(D * A.nS - D * (D - 1) / 2) * A.chunks;
            const int64_t nB = (int64_t)(A.nS - D) * A.chunks;
            const int t = d - D * kCorrT + kCorrT - 1;
            for (int64_t b = threadIdx.x; b < nB; b += 64) s += part[(b0 + b) * kCorrDiag + t];
        }
    }
    s = wave_sum(s);
    if (threadIdx.x == 0) R[A.out0 + m] = s * invN;
}

// ------------------------------------------------ interpolation to nodes
// interpolateToMesh (sample_RF.f90:872-1106) for every realization: one
// thread per node and chunk of realizations (grid y).  1-based cell
// position c = (x - xMin)/xStep + 1 in FP64, cell floor(c) moved down one on
// the upper border (:1024), corners in the reference's order (:996-1013),
// weight prod(1 - |c - corner|), sum in corner order (:1072-1086).  Nodes
// outside the grid get NaN and raise *flag.
// The grid in memory may be a box of a larger grid: global indices lo..hi
// (1-based, hi = lo + nstep - 1), positions still measured from the larger
// grid's xMin, and hi is the border of the cell rule, as the reference reads
// the bounding box of the nodes (:936-975).
struct rf_interp_dev {
    int nDim, Nmc;
    int nstep[3];
    int lo[3], hi[3];
    double xMin[3], xStep[3];
    int64_t Ng, nNodes;
};
constexpr int kInterpR = 2;      // realizations in flight together on the direct path

// Two neighbouring grid values along the first axis: the corners of a cell come
// in such pairs.
template <typename T>
struct interp_pair { T a, b; };
template <typename T, int align>
struct __attribute__((packed, aligned(align))) interp_load { T a, b; };
typedef __attribute__((address_space(3))) void interp_lds;

// One block: NT consecutive nodes, RC realizations (grid y).  The gather's
// bound is the address rate of the vector memory path: ~33 cycles per wave
// load and cell corner, whatever the cache does.  Nodes in mesh order are close
// to each other, so a block finds the box of cells its nodes lie in and, where
// it fits the LDS (interp_k elements per thread), copies it there realization
// by realization, coalesced and straight to LDS, and gathers from LDS.  Other blocks read the corners directly,
// 2^(D-1) pairs per node.  Blocks of an XCD take one contiguous run of nodes.
// 4M nodes in mesh order from a 256 x 256 x 128 grid, 16 realizations, FP32:
// direct single loads 530 us, direct pairs 480-500 us at any block size and
// chunk, from LDS 345 us (1.2 GB of HBM traffic, 3.5 TB/s; the grid is read
// 1.2 times).  Two blocks of 1024 per CU (64 VGPRs) share more of the planes
// in their XCD's L2 than one with the next realization held in registers
// (500 us); chunks of realizations repeat the set-up: 8 +20 %, 4 +60 %.
constexpr int interp_k(int NT, int size) { return NT == 256 && size == 4 ? 24 : 12; }

template <typename TG, typename TO, int D, int NT>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(sizeof(TG) == 4 ? 8 : 4))) void k_interp(rf_interp_dev q, const TG* __restrict__ grid,
                                               const double* __restrict__ x, TO* __restrict__ out,
                                               int* __restrict__ flag, int64_t nBlocks, int RC) {
#pragma clang fp contract(off)
    constexpr int kX = 8;                          // XCDs, blocks dealt round them
    constexpr int K = interp_k(NT, sizeof(TG));
    __shared__ TG box[K * NT];
    __shared__ int lim[6];
    const int64_t per = (nBlocks + kX - 1) / kX;
    const int64_t blk = (int64_t)(blockIdx.x % kX) * per + blockIdx.x / kX;
    if (blk >= nBlocks || blockIdx.x / kX >= per) return;      // whole block
    const int64_t i = blk * NT + threadIdx.x;
    const int r0 = blockIdx.y * RC;
    const int r1 = r0 + RC < q.Nmc ? r0 + RC : q.Nmc;
    const int64_t ic = i < q.nNodes ? i : q.nNodes - 1;
    double c[D];
    int64_t ci[D];
    bool inside = i < q.nNodes;
#pragma unroll
    for (int a = 0; a < D; a++) {
        c[a] = (x[ic * D + a] - q.xMin[a]) / q.xStep[a] + 1.0;
        ci[a] = (int64_t)floor(c[a]);
        if (ci[a] == q.hi[a]) ci[a] -= 1;
        if (ci[a] < q.lo[a] || ci[a] + 1 > q.hi[a]) inside = false;
    }
    if (threadIdx.x < 6) lim[threadIdx.x] = threadIdx.x < 3 ? INT_MAX : -1;
    __syncthreads();
    int cell[3] = {0, 0, 0};                       // from the first grid point of each axis
    if (inside) {
#pragma unroll
        for (int a = 0; a < D; a++) cell[a] = (int)(ci[a] - q.lo[a]);
    } else if (i < q.nNodes) {
        flag[0] = 1;
        for (int r = r0; r < r1; r++) out[(int64_t)r * q.nNodes + i] = (TO)NAN;
    }
    // the box of the block's cells: per wave, then over the waves
#pragma unroll
    for (int a = 0; a < D; a++) {
        int lo = inside ? cell[a] : INT_MAX, hi = inside ? cell[a] : -1;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            lo = min(lo, __shfl_xor(lo, o));
            hi = max(hi, __shfl_xor(hi, o));
        }
        if ((threadIdx.x & 63) == 0) {
            atomicMin(&lim[a], lo);
            atomicMax(&lim[3 + a], hi);
        }
    }
    __syncthreads();
    if (lim[3] < 0) return;                        // no node of the block is inside
    const int64_t s1 = q.nstep[0], s2 = (int64_t)q.nstep[0] * q.nstep[1];
    // corners in the reference's order: 3-D (:996-1013), 2-D, 1-D
    constexpr int nc = 1 << D, nP = nc / 2;
    constexpr int o3[8][3] = {{0, 0, 0}, {1, 0, 0}, {0, 1, 0}, {0, 0, 1}, {1, 1, 0}, {0, 1, 1}, {1, 0, 1}, {1, 1, 1}};
    constexpr int o2[4][3] = {{0, 0, 0}, {1, 0, 0}, {0, 1, 0}, {1, 1, 0}};
    double w[nc];
#pragma unroll
    for (int j = 0; j < nc; j++) {
        double wj = 1.0;
#pragma unroll
        for (int a = 0; a < D; a++) {
            const int off = D == 3 ? o3[j][a] : (D == 2 ? o2[j & 3][a] : j);
            wj = wj * (1.0 - fabs(c[a] - (double)(ci[a] + off)));
        }
        w[j] = wj;
    }
    auto one = [&](const interp_pair<TG>* v) {
        double acc = 0.0;
#pragma unroll
        for (int j = 0; j < nc; j++) {
            const int ox = D == 3 ? o3[j][0] : (D == 2 ? o2[j & 3][0] : j);
            const int pr = D == 3 ? o3[j][1] + 2 * o3[j][2] : (D == 2 ? o2[j & 3][1] : 0);
            acc = acc + (double)(ox ? v[pr].b : v[pr].a) * w[j];
        }
        return acc;
    };
    TO* o = out + (int64_t)r0 * q.nNodes + i;

    const int W = lim[3] - lim[0] + 2;             // grid points: cells + 1
    const int H = D > 1 ? lim[4] - lim[1] + 2 : 1, P = D > 2 ? lim[5] - lim[2] + 2 : 1;
    const int64_t vol = (int64_t)W * H * P;
    if (vol <= (int64_t)K * NT && s2 * P * (int64_t)sizeof(TG) < INT_MAX) {
        // copied in 4-byte words, straight to LDS (word e of the box to word e)
        constexpr int KW = K * (int)sizeof(TG) / 4, E = (int)sizeof(TG) / 4;
        const int n = (int)vol * E;
        const TG* g = grid + (int64_t)r0 * q.Ng + lim[0] + (D > 1 ? lim[1] * s1 : 0) + (D > 2 ? lim[2] * s2 : 0);
        // quotients by W and H through a 32-bit reciprocal, exact for the
        // elements of a box (el < 2^15 and el * divisor < 2^32); a divisor of 1
        // has none
        static_assert(K * NT < 1 << 15, "reciprocal range");
        const unsigned mW = 0xffffffffu / (unsigned)W + 1, mH = 0xffffffffu / (unsigned)H + 1;
        const int sW = (int)s1 - W, sH = (int)s2 - H * (int)s1;
        int off[KW];
#pragma unroll
        for (int k = 0; k < KW; k++) {
            const int e = (int)threadIdx.x + k * NT, el = e / E;
            const int row = W > 1 ? (int)__umulhi((unsigned)el, mW) : el;
            const int z = H > 1 ? (int)__umulhi((unsigned)row, mH) : row;
            off[k] = e < n ? (el + row * sW + z * sH) * E + e % E : 0;   // el - row W + (row - z H) s1 + z s2
        }
        const int wave0 = (int)threadIdx.x & ~63;
        const int c0 = (cell[0] - lim[0]) + (D > 1 ? (cell[1] - lim[1]) * W : 0) + (D > 2 ? (cell[2] - lim[2]) * W * H : 0);
        const TG* b = box + (inside ? c0 : 0);
        for (int r = r0; r < r1; r++) {
            const uint32_t* gw = reinterpret_cast<const uint32_t*>(g);
            uint32_t* bw = reinterpret_cast<uint32_t*>(box);
#pragma unroll
            for (int k = 0; k < KW; k++)
                if (k * NT < n)                            // uniform
                    __builtin_amdgcn_global_load_lds((const void*)(gw + off[k]), (interp_lds*)(bw + wave0 + k * NT), 4, 0, 0);
            __builtin_amdgcn_s_waitcnt(0x0F70);            // vmcnt(0): the copies have landed
            __syncthreads();
            if (inside) {
                interp_pair<TG> u[nP];
#pragma unroll
                for (int k = 0; k < nP; k++) {
                    const TG* p = b + (k & 1 ? W : 0) + (k & 2 ? W * H : 0);
                    u[k].a = p[0];
                    u[k].b = p[1];
                }
                *o = (TO)one(u);
            }
            o += q.nNodes;
            g += q.Ng;
            __syncthreads();
        }
        return;
    }
    if (!inside) return;
    const TG* g = grid + (int64_t)r0 * q.Ng + cell[0] + (D > 1 ? cell[1] * s1 : 0) + (D > 2 ? cell[2] * s2 : 0);
    auto load = [&](const TG* p, interp_pair<TG>* v) {
#pragma unroll
        for (int k = 0; k < nP; k++) {
            const auto t = *reinterpret_cast<const interp_load<TG, sizeof(TG)>*>(p + (k & 1 ? s1 : 0) + (k & 2 ? s2 : 0));
            v[k].a = t.a;
            v[k].b = t.b;
        }
    };
    int r = r0;
    for (; r + kInterpR <= r1; r += kInterpR) {
        interp_pair<TG> v[kInterpR][nP];
#pragma unroll
        for (int u = 0; u < kInterpR; u++) load(g + u * q.Ng, v[u]);
#pragma unroll
        for (int u = 0; u < kInterpR; u++) o[u * q.nNodes] = (TO)one(v[u]);
        g += kInterpR * q.Ng;
        o += kInterpR * q.nNodes;
    }
    for (; r < r1; r++) {
        interp_pair<TG> v[nP];
        load(g, v);
        *o = (TO)one(v);
        g += q.Ng;
        o += q.nNodes;
    }
}

// ----------------------------------------------------------------- blend
// One thread per group point and chunk of kBlendR realizations (grid y), so
// the blocks in flight sweep the points of a few realizations at a time (few
// pages per wave) and the loads of a chunk are independent.  Sums run in FP64
// in ascending subdomain order (the reference's loop over fields,
// calls_RF.f90:237), each term v * PU then + (localization_RF.f90:228,253).
constexpr int kBlendR = 4;

template <typename T>
__global__ __launch_bounds__(kBlock) void k_blend(rf_blend_dev b, T* __restrict__ group) {
#pragma clang fp contract(off)
    const int64_t g = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (g >= b.groupTot) return;
    int gi[3];
    {
        int64_t rem = g;
        gi[0] = (int)(rem % b.groupN[0]);
        rem /= b.groupN[0];
        gi[1] = (int)(rem % b.groupN[1]);
        gi[2] = (int)(rem / b.groupN[1]);
    }
    int cell = b.seg[0][gi[0]];
    if (b.nDim > 1) cell += b.nSeg[0] * b.seg[1][gi[1]];
    if (b.nDim > 2) cell += b.nSeg[0] * b.nSeg[1] * b.seg[2][gi[2]];
    const int e0 = b.cellOff[cell];
    const int nh = b.cellOff[cell + 1] - e0;
    const T* F[kBlendMaxEntries];
    int64_t rs[kBlendMaxEntries], loc[kBlendMaxEntries];
    double w[kBlendMaxEntries];
#pragma unroll
    for (int h = 0; h < kBlendMaxEntries; h++) {
        F[h] = nullptr;
        rs[h] = 0;
        loc[h] = 0;
        w[h] = 0.0;
        if (h < nh) {
            const rf_blend_entry& E = b.entries[e0 + h];
            F[h] = static_cast<const T*>(E.field);
            rs[h] = E.subTot;
            loc[h] = E.base + gi[0] + (int64_t)gi[1] * E.stride1 + (int64_t)gi[2] * E.stride2;
            // PU product in the reference's order: lower faces of axes 1..d,
            // then upper faces (localization_RF.f90:755-851)
            // (all six factor loads issued together; axes beyond nDim read
            // entry 0 and multiply by an exact 1.0)
            const double* lf = b.lowF + (int64_t)E.s * 3 * b.maxSize;
            const double* uf = b.upF + (int64_t)E.s * 3 * b.maxSize;
            double fl[3], fu[3];
#pragma unroll
            for (int a = 0; a < 3; a++) {
                const int pos = a < b.nDim ? gi[a] - E.o[a] : 0;
                fl[a] = lf[a * b.maxSize + pos];
                fu[a] = uf[a * b.maxSize + pos];
            }
            double pu = 1.0;
#pragma unroll
            for (int a = 0; a < 3; a++) pu = pu * (a < b.nDim ? fl[a] : 1.0);
#pragma unroll
            for (int a = 0; a < 3; a++) pu = pu * (a < b.nDim ? fu[a] : 1.0);
            w[h] = pu;
        }
    }
    double pu1 = 1.0;
    if (b.mode == RF_REF_COMPAT) {
        for (int a = 0; a < b.nDim; a++) pu1 = pu1 * b.pu1Low[a][gi[a]];
        for (int a = 0; a < b.nDim; a++) pu1 = pu1 * b.pu1Up[a][gi[a]];
    }
    {
        const int r0 = blockIdx.y * kBlendR;
        double acc[kBlendR];
#pragma unroll
        for (int j = 0; j < kBlendR; j++) acc[j] = 0.0;
        // the chunk's loads are unconditional (realization index clamped), so
        // they issue together instead of one branch and wait per load
#pragma unroll
        for (int h = 0; h < kBlendMaxEntries; h++) {
            if (h < nh) {
                T v[kBlendR];
#pragma unroll
                for (int j = 0; j < kBlendR; j++) v[j] = F[h][(int64_t)min(r0 + j, b.Nmc - 1) * rs[h] + loc[h]];
#pragma unroll
                for (int j = 0; j < kBlendR; j++) acc[j] = (double)v[j] * w[h] + acc[j];
            }
        }
#pragma unroll
        for (int j = 0; j < kBlendR; j++)
            if (r0 + j < b.Nmc) {
                double u = acc[j];
                if (b.mode == RF_REF_COMPAT && r0 + j == 0) u = u / pu1;   // calls_RF.f90:355
                group[(int64_t)(r0 + j) * b.groupTot + g] = (T)u;
            }
    }
}

// Separable form: one thread per group point, all realizations; the <= 2^d
// contributions come from the per-axis tables.  FP64 sums, each term v * PU
// then + (localization_RF.f90:228,253); the PU product is taken per axis
// (a reordering of the reference's lower-then-upper face product, equal up
// to rounding) and contributions are added in interval order.
//
// Every field load is unconditional (realization index clamped, absent
// contributions read a dummy address with stride 0 and are masked out of
// the sum): a load under a per-element condition becomes a branch that waits
// for its value before the next load issues, which leaves one load in
// flight per wave.  A wave whose points have at most two contributions
// takes a straight-line path chosen wave-uniformly (16 realizations of
// loads in flight for one contribution, 2 x 8 for two); larger counts (the
// corners where 3-D overlaps meet) take the general loop.
template <typename T>
__device__ __forceinline__ void blend_store(T* p, double u) {
    __builtin_nontemporal_store((T)u, p);   // written once, read by the next kernel
}

// Where field S holds its value at local position (p0, p1, p2) (s0, s1: its
// first two extents): a first-axis overlap band array of a fused batch, or
// the field itself; *st: the realization stride.
// Written with selects: an if-return form of this lookup was compiled (ROCm
// 7.2, gfx950) so that lanes leaving the high-band test for the field kept
// the band width as their stride.
template <typename T>
__device__ __forceinline__ const T* blend_locate(const rf_blend_sub& S, int64_t p0, int64_t p1, int64_t p2,
                                                 int64_t s0, int64_t s1, int64_t* st) {
    const int64_t row = p1 + p2 * s1;
    const int64_t wLo = S.wLo, wHi = S.wHi;
    const int64_t tLo = S.bandLoTot, tHi = S.bandHiTot, tF = S.subTot;
    const T* bLo = static_cast<const T*>(S.bandLo);
    const T* bHi = static_cast<const T*>(S.bandHi);
    const T* bF = static_cast<const T*>(S.field);
    const bool lo = bLo != nullptr && p0 < wLo;
    const bool hi = !lo && bHi != nullptr && p0 >= s0 - wHi;
    const int64_t offField = p0 + row * s0, offLo = row * wLo + p0, offHi = row * wHi + (p0 - (s0 - wHi));
    *st = lo ? tLo : (hi ? tHi : tF);
    return lo ? bLo + offLo : (hi ? bHi + offHi : bF + offField);
}

// One group point (gi0, gi1, gi2) of the separable blend, every realization.
template <typename T>
__device__ __forceinline__ void blend_sep_point(const rf_blend_sep& b, int gi0, int gi1, int gi2,
                                                T* __restrict__ group) {
#pragma clang fp contract(off)
    const int64_t g = gi0 + (int64_t)b.groupN[0] * (gi1 + (int64_t)b.groupN[1] * gi2);
    const rf_blend_axis A0 = b.ax[0][gi0];
    const rf_blend_axis A1 = b.ax[1][gi1];
    const rf_blend_axis A2 = b.ax[2][gi2];
    const double pu1 = (A0.pu1 * A1.pu1) * A2.pu1;
    const bool fix0 = b.mode == RF_REF_COMPAT;      // realization 0 divided by pu1 (calls_RF.f90:355)
    const int Nmc = b.Nmc;
    // the interval combinations covering this point (bit k: interval k & 1 of
    // axis 0, (k >> 1) & 1 of axis 1, k >> 2 of axis 2)
    uint32_t live = 0;
#pragma unroll
    for (int k = 0; k < 8; k++) {
        const int i0 = (k & 1) ? A0.iv[1] : A0.iv[0];
        const int i1 = ((k >> 1) & 1) ? A1.iv[1] : A1.iv[0];
        const int i2 = (k >> 2) ? A2.iv[1] : A2.iv[0];
        if (i0 >= 0 && i1 >= 0 && i2 >= 0) live |= 1u << k;
    }
    // the first two contributions in interval order; absent ones read the
    // axis-0 table entry with stride 0
    const T* dummy = reinterpret_cast<const T*>(b.ax[0]);
    const T* F0 = dummy; const T* F1 = dummy;
    int64_t st0 = 0, st1 = 0;
    double w0 = 0.0, w1 = 0.0;
    int n = 0;
    for (uint32_t lm = live; lm; lm &= lm - 1) {
        const int k = __builtin_ctz(lm);
        // selects, not indexing: the tables stay in registers
        const bool c0 = k & 1, c1 = (k >> 1) & 1, c2 = k >> 2;
        const int i0 = c0 ? A0.iv[1] : A0.iv[0];
        const int i1 = c1 ? A1.iv[1] : A1.iv[0];
        const int i2 = c2 ? A2.iv[1] : A2.iv[0];
        const rf_blend_sub S = b.sub[i0 + b.nInt[0] * (i1 + b.nInt[1] * i2)];
        if (!S.field) continue;
        if (n == 2) { n = 3; break; }
        const int64_t s0 = c0 ? A0.sz[1] : A0.sz[0], s1 = c1 ? A1.sz[1] : A1.sz[0];
        const int64_t p0 = c0 ? A0.pos[1] : A0.pos[0], p1 = c1 ? A1.pos[1] : A1.pos[0];
        const int64_t p2 = c2 ? A2.pos[1] : A2.pos[0];
        int64_t st;
        const T* F = blend_locate<T>(S, p0, p1, p2, s0, s1, &st);
        const double w = ((c0 ? A0.f[1] : A0.f[0]) * (c1 ? A1.f[1] : A1.f[0])) * (c2 ? A2.f[1] : A2.f[0]);
        if (n == 0) { F0 = F; st0 = st; w0 = w; }
        else { F1 = F; st1 = st; w1 = w; }
        n++;
    }
    if (b.skipSingle && n == 1) return;            // written by the fused last contraction
    if (!__any(n > 2)) {
        if (!__any(n > 1)) {
            constexpr int RB = 16;
            for (int r0 = 0; r0 < Nmc; r0 += RB) {
                T v[RB];
#pragma unroll
                for (int j = 0; j < RB; j++) v[j] = F0[(int64_t)min(r0 + j, Nmc - 1) * st0];
#pragma unroll
                for (int j = 0; j < RB; j++)
                    if (r0 + j < Nmc) {
                        double u = 0.0;
                        if (n == 1) u = (double)v[j] * w0 + u;
                        if (fix0 && r0 + j == 0) u = u / pu1;
                        blend_store(group + (int64_t)(r0 + j) * b.groupTot + g, u);
                    }
            }
        } else {
            constexpr int RB = 8;
            for (int r0 = 0; r0 < Nmc; r0 += RB) {
                T v0[RB], v1[RB];
#pragma unroll
                for (int j = 0; j < RB; j++) {
                    const int64_t r = min(r0 + j, Nmc - 1);
                    v0[j] = F0[r * st0];
                    v1[j] = F1[r * st1];
                }
#pragma unroll
                for (int j = 0; j < RB; j++)
                    if (r0 + j < Nmc) {
                        double u = 0.0;
                        if (n >= 1) u = (double)v0[j] * w0 + u;
                        if (n >= 2) u = (double)v1[j] * w1 + u;
                        if (fix0 && r0 + j == 0) u = u / pu1;
                        blend_store(group + (int64_t)(r0 + j) * b.groupTot + g, u);
                    }
            }
        }
        return;
    }
    // general loop: every contribution, 8 realizations per pass
    constexpr int RB = 8;
    for (int r0 = 0; r0 < Nmc; r0 += RB) {
        double acc[RB];
#pragma unroll
        for (int j = 0; j < RB; j++) acc[j] = 0.0;
        for (uint32_t lm = live; lm; lm &= lm - 1) {
            const int k = __builtin_ctz(lm);
            const bool c0 = k & 1, c1 = (k >> 1) & 1, c2 = k >> 2;
            const int i0 = c0 ? A0.iv[1] : A0.iv[0];
            const int i1 = c1 ? A1.iv[1] : A1.iv[0];
            const int i2 = c2 ? A2.iv[1] : A2.iv[0];
            const rf_blend_sub S = b.sub[i0 + b.nInt[0] * (i1 + b.nInt[1] * i2)];
            if (!S.field) continue;
            const int64_t s0 = c0 ? A0.sz[1] : A0.sz[0], s1 = c1 ? A1.sz[1] : A1.sz[0];
            const int64_t p0 = c0 ? A0.pos[1] : A0.pos[0], p1 = c1 ? A1.pos[1] : A1.pos[0];
            const int64_t p2 = c2 ? A2.pos[1] : A2.pos[0];
            int64_t st;
            const T* F = blend_locate<T>(S, p0, p1, p2, s0, s1, &st);
            const double w = ((c0 ? A0.f[1] : A0.f[0]) * (c1 ? A1.f[1] : A1.f[0])) * (c2 ? A2.f[1] : A2.f[0]);
            T v[RB];
#pragma unroll
            for (int j = 0; j < RB; j++) v[j] = F[(int64_t)min(r0 + j, Nmc - 1) * st];
#pragma unroll
            for (int j = 0; j < RB; j++) acc[j] = (double)v[j] * w + acc[j];
        }
#pragma unroll
        for (int j = 0; j < RB; j++)
            if (r0 + j < Nmc) {
                double u = acc[j];
                if (fix0 && r0 + j == 0) u = u / pu1;
                blend_store(group + (int64_t)(r0 + j) * b.groupTot + g, u);
            }
    }
}

// 7 waves per SIMD (at most 72 VGPRs, no spills; unconstrained the
// allocation is 81 VGPRs, 5 waves)
// block (x segment, gi1, gi2): the axis-1 and axis-2 entries are
// block-uniform (scalar loads), one axis-0 entry per thread
template <typename T>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(7))) void k_blend_sep(rf_blend_sep b, T* __restrict__ group) {
    const int gi0 = blockIdx.x * kBlock + threadIdx.x;
    if (gi0 >= b.groupN[0]) return;
    blend_sep_point<T>(b, gi0, blockIdx.y, blockIdx.z, group);
}

// The overlap bands only (the fused blend: the last contraction stored the
// points one subdomain covers): boxes of group indices, box k covering
// points first .. first + n0 n1 n2 - 1 of the launch, x fastest.
template <typename T>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(5))) void k_blend_boxes(
        rf_blend_sep b, const rf_blend_box* __restrict__ boxes, int nBoxes, int64_t total, T* __restrict__ group) {
    const int64_t e = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (e >= total) return;
    int k = 0;
    while (k + 1 < nBoxes && boxes[k + 1].first <= e) k++;
    const rf_blend_box& x = boxes[k];
    const int64_t q = e - x.first;
    const int i0 = (int)(q % x.n[0]);
    const int64_t r = q / x.n[0];
    blend_sep_point<T>(b, x.lo[0] + i0, x.lo[1] + (int)(r % x.n[1]), x.lo[2] + (int)(r / x.n[1]), group);
}

}  // namespace

hipError_t rf_launch_marginal(int margi, double scale, double shift, void* d, int64_t count,
                              int dtype, hipStream_t s) {
    if (count <= 0) return hipSuccess;
    const size_t esz = dtype == RF_DTYPE_F64 ? 8 : 4;
    int64_t head = 0;                        // elements done by the vector kernel
    if (((uintptr_t)d & 15) == 0) {
        const int64_t L = (int64_t)(16 / esz);
        const int64_t nVec = count / L;
        if (nVec > 0) {
            int64_t blocks = (nVec + 2 * kBlock - 1) / (2 * kBlock);
            if (blocks > 65536) blocks = 65536;
            if (dtype == RF_DTYPE_F64)
                hipLaunchKernelGGL(k_marginal_vec<double>, dim3((unsigned)blocks), dim3(kBlock), 0, s,
                                   margi, scale, shift, static_cast<double*>(d), nVec);
            else
                hipLaunchKernelGGL(k_marginal_vec<float>, dim3((unsigned)blocks), dim3(kBlock), 0, s,
                                   margi, scale, shift, static_cast<float*>(d), nVec);
            head = nVec * L;
        }
    }
    const int64_t rest = count - head;
    if (rest > 0) {
        int64_t blocks = (rest + 4 * kBlock - 1) / (4 * kBlock);
        if (blocks > 65536) blocks = 65536;
        if (dtype == RF_DTYPE_F64)
            hipLaunchKernelGGL(k_marginal<double>, dim3((unsigned)blocks), dim3(kBlock), 0, s, margi,
                               scale, shift, static_cast<double*>(d) + head, rest);
        else
            hipLaunchKernelGGL(k_marginal<float>, dim3((unsigned)blocks), dim3(kBlock), 0, s, margi,
                               scale, shift, static_cast<float*>(d) + head, rest);
    }
    return hipGetLastError();
}

int rf_moments_parts(int64_t N) {
    int64_t p = (N + kBlock * 8 - 1) / (kBlock * 8);
    if (p < 1) p = 1;
    if (p > 256) p = 256;
    return (int)p;
}

hipError_t rf_launch_moments(const void* d, int64_t N, int Nmc, int dtype, double* d_part,
                             int nPart, double* d_sums, hipStream_t s) {
    dim3 grid((unsigned)nPart, (unsigned)Nmc);
    const size_t esz = dtype == RF_DTYPE_F64 ? 8 : 4;
    const bool vec = (uintptr_t)d % 16 == 0 && (Nmc == 1 || (size_t)N * esz % 16 == 0);
    if (dtype == RF_DTYPE_F64 && vec)
        hipLaunchKernelGGL((k_moments_partial<double, true>), grid, dim3(kBlock), 0, s, static_cast<const double*>(d), N, d_part);
    else if (dtype == RF_DTYPE_F64)
        hipLaunchKernelGGL((k_moments_partial<double, false>), grid, dim3(kBlock), 0, s, static_cast<const double*>(d), N, d_part);
    else if (vec)
        hipLaunchKernelGGL((k_moments_partial<float, true>), grid, dim3(kBlock), 0, s, static_cast<const float*>(d), N, d_part);
    else
        hipLaunchKernelGGL((k_moments_partial<float, false>), grid, dim3(kBlock), 0, s, static_cast<const float*>(d), N, d_part);
    hipLaunchKernelGGL(k_moments_final, dim3((unsigned)Nmc), dim3(64), 0, s, d_part, nPart, d_sums);
    return hipGetLastError();
}

hipError_t rf_launch_window_moments(const void* d, int dtype, const rf_window& w, double* d_part, int nPart,
                                    double* d_sums, hipStream_t s) {
    if (dtype == RF_DTYPE_F64)
        hipLaunchKernelGGL(k_window_moments_partial<double>, dim3((unsigned)nPart), dim3(kBlock), 0, s,
                           static_cast<const double*>(d), w, d_part);
    else
        hipLaunchKernelGGL(k_window_moments_partial<float>, dim3((unsigned)nPart), dim3(kBlock), 0, s,
                           static_cast<const float*>(d), w, d_part);
    hipLaunchKernelGGL(k_moments_final, dim3(1), dim3(64), 0, s, d_part, nPart, d_sums);
    return hipGetLastError();
}

hipError_t rf_launch_affine(void* d, int64_t N, int Nmc, int dtype, const double* d_shift,
                            const double* d_mul, hipStream_t s) {
    int64_t bx = (N + kBlock - 1) / kBlock;
    if (bx > 4096) bx = 4096;
    dim3 grid((unsigned)bx, (unsigned)Nmc);
    if (dtype == RF_DTYPE_F64)
        hipLaunchKernelGGL(k_affine<double>, grid, dim3(kBlock), 0, s, static_cast<double*>(d), N,
                           d_shift, d_mul);
    else
        hipLaunchKernelGGL(k_affine<float>, grid, dim3(kBlock), 0, s, static_cast<float*>(d), N,
                           d_shift, d_mul);
    return hipGetLastError();
}

hipError_t rf_launch_blend_dev(const rf_blend_dev& b, void* d_group, int dtype, hipStream_t s) {
    const dim3 grid((unsigned)((b.groupTot + kBlock - 1) / kBlock), (unsigned)((b.Nmc + kBlendR - 1) / kBlendR));
    if (grid.y > 65535) return hipErrorInvalidValue;
    if (dtype == RF_DTYPE_F64)
        hipLaunchKernelGGL(k_blend<double>, grid, dim3(kBlock), 0, s, b, static_cast<double*>(d_group));
    else
        hipLaunchKernelGGL(k_blend<float>, grid, dim3(kBlock), 0, s, b, static_cast<float*>(d_group));
    return hipGetLastError();
}

int rf_corr_parts(int64_t N) {
    int64_t p = (N + kBlock * 16 - 1) / (kBlock * 16);
    if (p < 1) p = 1;
    if (p > 512) p = 512;
    return (int)p;
}

hipError_t rf_launch_corr(const void* u, int dtype, int64_t N, int64_t strideA, int nA, int M, double avg,
                          double std, double* d_part, int nPart, double* d_R, hipStream_t s) {
    if (M <= 0) return hipSuccess;
    const dim3 grid((unsigned)nPart, (unsigned)M);
    if (dtype == RF_DTYPE_F64)
        hipLaunchKernelGGL(k_corr_partial<double>, grid, dim3(kBlock), 0, s, static_cast<const double*>(u), N,
                           strideA, nA, avg, std, d_part);
    else
        hipLaunchKernelGGL(k_corr_partial<float>, grid, dim3(kBlock), 0, s, static_cast<const float*>(u), N,
                           strideA, nA, avg, std, d_part);
    hipLaunchKernelGGL(k_corr_final, dim3((unsigned)M), dim3(64), 0, s, d_part, nPart, 1.0 / (double)N, d_R);
    return hipGetLastError();
}

bool rf_corr_gram_add(rf_corr_gram* q, int n, int64_t stride, int64_t N, int out0) {
    const int64_t nLines = N / n;
    const int nS = (n + kCorrT - 1) / kCorrT;
    if (n < 2 || n > kCorrGramMaxN || nLines < kCorrGramMinLines) return false;
    rf_corr_axis& A = q->ax[q->nAx++];
    A.n = n;
    A.stride = stride;
    A.nLines = nLines;
    A.nS = nS;
    A.pairs = nS * (nS + 1) / 2;
    A.out0 = out0;
    return true;
}

// Shares of the lines per tile pair: about 512 blocks in all (two 4-wave
// blocks per CU), at least four turns of 64 lines per block.  Axes of unequal
// length: no block of more than twice an even share of all turns (2048 x 64 x 4: the
// 528 pairs of the long axis left one block for the 131,072 lines of the short one,
// 6199 us; 123 now, a sweep per lag 1232).
size_t rf_corr_gram_plan(rf_corr_gram* q) {
    int pairs = 0;
    int64_t turns = 0;
    for (int a = 0; a < q->nAx; a++) {
        pairs += q->ax[a].pairs;
        turns += q->ax[a].pairs * ((q->ax[a].nLines + 63) / 64);
    }
    const int64_t share = std::max<int64_t>(4, (turns + 511) / 512);
    q->blocks = q->lags = 0;
    for (int a = 0; a < q->nAx; a++) {
        rf_corr_axis& A = q->ax[a];
        const int64_t most = (A.nLines + 255) / 256;
        const int64_t even = std::max<int64_t>(512 / pairs, ((A.nLines + 63) / 64 + 2 * share - 1) / (2 * share));
        A.chunks = (int)(most < even ? most : even);
        A.block0 = q->blocks;
        A.lag0 = q->lags;
        q->blocks += A.pairs * A.chunks;
        q->lags += A.n / 2;
    }
    return (size_t)q->blocks * kCorrDiag;
}

hipError_t rf_launch_corr_gram(const rf_corr_gram& q, const void* u, int dtype, int64_t N, double avg, double std,
                               double* d_part, double* d_R, hipStream_t s) {
    if (q.blocks <= 0) return hipSuccess;
    if (dtype == RF_DTYPE_F64)
        hipLaunchKernelGGL(k_corr_gram<double>, dim3((unsigned)q.blocks), dim3(kBlock), 0, s, q,
                           static_cast<const double*>(u), avg, std, d_part);
    else
        hipLaunchKernelGGL(k_corr_gram<float>, dim3((unsigned)q.blocks), dim3(kBlock), 0, s, q,
                           static_cast<const float*>(u), avg, std, d_part);
    hipLaunchKernelGGL(k_corr_gram_final, dim3((unsigned)q.lags), dim3(64), 0, s, q, d_part, 1.0 / (double)N, d_R);
    return hipGetLastError();
}

hipError_t rf_launch_interp(int nDim, const int32_t* nstep, const int32_t* lo, const double* xMin,
                            const double* xStep, int Nmc, const void* grid, int gridDtype, const double* x,
                            int64_t nNodes, void* out, int outDtype, int* d_flag, hipStream_t s) {
    if (nNodes <= 0) return hipSuccess;
    rf_interp_dev q{};
    q.nDim = nDim;
    q.Nmc = Nmc;
    q.Ng = 1;
    for (int a = 0; a < 3; a++) {
        q.nstep[a] = a < nDim ? nstep[a] : 1;
        q.lo[a] = (a < nDim && lo) ? lo[a] : 1;
        q.hi[a] = q.lo[a] + q.nstep[a] - 1;
        q.xMin[a] = a < nDim ? xMin[a] : 0.0;
        q.xStep[a] = a < nDim ? xStep[a] : 1.0;
        q.Ng *= q.nstep[a];
    }
    q.nNodes = nNodes;
    // Many nodes, at most six grid points to a node: all realizations in a block
    // (cells and weights formed once); else four, so that small calls fill the
    // chip and a block's scattered corners stay in L2 (256 x 256 x 128, 600,000 nodes, 16
    // realizations FP32: 281 us all together in blocks of 1024, 195 in blocks of 256, 181
    // in fours).  FP32 grids in blocks of 1024 nodes (the most compact boxes) down to
    // four grid points to a node, a few realizations down to six (4M nodes 345 us;
    // 2M nodes, 4.2 points to a node, 16 realizations 395 us against 287 in blocks of
    // 256, one realization 52 against 71).  FP64 grids in blocks of 256: five waves per
    // SIMD whose set-ups cover each other, 251 x 151 x 32, 3.3M nodes, 1 / 4 / 16
    // realizations 99 / 127 / 348 us against 118 / 154 / 365 in blocks of 512.
    const bool wide = nNodes >= 512 * 1024 && q.Ng <= 6 * nNodes;
    const int RC = wide ? Nmc : 4;
    const bool g64 = gridDtype == RF_DTYPE_F64, o64 = outDtype == RF_DTYPE_F64;
    const bool large = wide && !g64 && (Nmc <= 4 || q.Ng <= 4 * nNodes);
    const int NT = large ? 1024 : 256;
    const int64_t nBlocks = (nNodes + NT - 1) / NT;
    if ((nBlocks + 7) / 8 * 8 > rf_max_blocks(NT)) return hipErrorInvalidValue;
    const dim3 grid2((unsigned)((nBlocks + 7) / 8 * 8), (unsigned)((Nmc + RC - 1) / RC));
    if (grid2.y > 65535) return hipErrorInvalidValue;
    auto run = [&](auto dim, auto* g, auto* o) {
        typedef std::remove_const_t<std::remove_pointer_t<decltype(g)>> TG;
        typedef std::remove_pointer_t<decltype(o)> TO;
        constexpr int D = decltype(dim)::value;
        if constexpr (sizeof(TG) == 4) {
            if (large) {
                hipLaunchKernelGGL((k_interp<TG, TO, D, 1024>), grid2, dim3(NT), 0, s, q, g, x, o, d_flag, nBlocks, RC);
                return;
            }
        }
        hipLaunchKernelGGL((k_interp<TG, TO, D, 256>), grid2, dim3(NT), 0, s, q, g, x, o, d_flag, nBlocks, RC);
    };
    auto go = [&](auto* g, auto* o) {
        if (nDim == 3) run(std::integral_constant<int, 3>(), g, o);
        else if (nDim == 2) run(std::integral_constant<int, 2>(), g, o);
        else run(std::integral_constant<int, 1>(), g, o);
    };
    if (g64 && o64) go(static_cast<const double*>(grid), static_cast<double*>(out));
    else if (g64) go(static_cast<const double*>(grid), static_cast<float*>(out));
    else if (o64) go(static_cast<const float*>(grid), static_cast<double*>(out));
    else go(static_cast<const float*>(grid), static_cast<float*>(out));
    return hipGetLastError();
}

hipError_t rf_launch_blend_boxes(const rf_blend_sep& b, const rf_blend_box* d_boxes, int nBoxes, int64_t total,
                                 void* d_group, int dtype, hipStream_t s) {
    if (total <= 0) return hipSuccess;
    const unsigned grid = (unsigned)((total + kBlock - 1) / kBlock);
    if (dtype == RF_DTYPE_F64)
        hipLaunchKernelGGL(k_blend_boxes<double>, dim3(grid), dim3(kBlock), 0, s, b, d_boxes, nBoxes, total,
                           static_cast<double*>(d_group));
    else
        hipLaunchKernelGGL(k_blend_boxes<float>, dim3(grid), dim3(kBlock), 0, s, b, d_boxes, nBoxes, total,
                           static_cast<float*>(d_group));
    return hipGetLastError();
}

hipError_t rf_launch_blend_sep(const rf_blend_sep& b, void* d_group, int dtype, hipStream_t s) {
    if (b.groupN[1] > 65535 || b.groupN[2] > 65535) return hipErrorInvalidValue;
    const dim3 grid((unsigned)((b.groupN[0] + kBlock - 1) / kBlock), (unsigned)b.groupN[1], (unsigned)b.groupN[2]);
    if (dtype == RF_DTYPE_F64)
        hipLaunchKernelGGL(k_blend_sep<double>, grid, dim3(kBlock), 0, s, b, static_cast<double*>(d_group));
    else
        hipLaunchKernelGGL(k_blend_sep<float>, grid, dim3(kBlock), 0, s, b, static_cast<float*>(d_group));
    return hipGetLastError();
}
