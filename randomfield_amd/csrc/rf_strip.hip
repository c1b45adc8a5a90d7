// rf_strip.hip -- the strip GEMM: every contraction of the grid form with FP16
// operands.  Compiled once per kind and operand type (RF_STRIP_PART: rf_gemm_kind, +3
// real operands; 6 isotropic).
//
// One operand of each contraction is a small phase table shared by the whole
// launch (M entries of an axis x K), the other -- the coefficients or the
// previous contraction's output -- is streamed, N lines of K complex values.
// A wave owns 32 lines and MT 32-entry tiles of the table axis (with MT * 32 >=
// M every streamed value is read from memory and converted once in the whole
// launch).  Operands are split into FP16 hi + lo halves; three
// v_mfma_f32_32x32x16_f16 products (hi hi, hi lo, lo hi) with FP32 accumulation.
//
// A K-step is 8 complex k = 16 MFMA K entries: the re parts in lane half 0, the
// im parts in half 1.  A lane loads k = 8 s + 4 h + (0..3) of its own line straight
// to registers (no LDS), splits them and trades with the other half
// (v_permlane32_swap).  Re D pairs table (re, im) with streamed (re, -im); Im D pairs
// (im, re) with (re, im) -- the lane reads the other half's slot -- or, in the
// first contraction, (re, im) with (im, re).  The table is stored in HBM pre-split
// in fragment order [step][tile][hi, lo][lane][8] (k_axis_tables) and goes to LDS by
// direct loads, shared by the block's waves.
//
// Replaces 64..160-wide block tiles that staged and split both operands in LDS
// per 16 k, re-reading and re-splitting the streamed one per table tile, two
// barriers per 16 k.  32 fields of ~131^3 x 16 realizations: first contraction
// (with its draws) 1.48 -> 1.44 ms, middle 1.93 -> 1.26, last 3.1 -> 2.3-2.4; 128^3
// x 8 of method 4: 104 / 88 / 73 -> 68 / 63 / 55 us, on real operands 63 / 35 / 42.  Same bits.  By counters the
// first is bound by its draws (VALU 63 % of the cycles, matrix cores 21 %), the
// middle moves 5.3 GB at 4.2 TB/s (matrix cores 38 %), the last 8.4 GB at 3.5.
//
// Isotropic sum on a grid, per-realization directions.  With x = o + i step per
// axis, e^{i(k.x + phi)} factorises over the axes, so per realization r
//   u_r[l][(i, j)] = Re sum_k Z_k[l] B_k[(i, j)],   B_k[(i, j)] = W_k[i] Y_k[j],
//   W_k[i] = a_k e^{i(k_x x_i + phi_k)},  Y_k[j] = e^{i k_y y_j},  Z_k[l] = e^{i k_z z_l}
// (2-D: u_r[j][i] = Re sum_k Y_k[j] W_k[i]): the table is Z, one per realization,
// the lines are the points of the plane and a streamed value is the product of
// two table entries, formed as it is split.  128^3 x 64 lognormal, 286 shells: 570 us
// of kernel (128 x 128 block tiles with both operands staged 620); the matrix
// cores are busy 41 % of the cycles, the VALU 48 % (a third of it the exponentials).
//
// D orientation: the table is the A operand (lanes run along lines) where D
// is stored with lines contiguous, the B operand (lanes run along the table
// axis) in the first contraction, whose D has the table axis contiguous.
//
// A block is kStripW waves; the table goes to LDS kStripCS steps at a time in a
// double buffer, one barrier per chunk.  A last contraction of at most
// kStripShortCS steps (kStripShort) loads everything -- table and lines -- at once
// instead: it is bound by its loads and stores, and every chunk exposed one more
// memory latency.  The last contraction above 2.29 -> 1.96 ms to the fields, 2.45 ->
// 2.40 into the group grid.
#include "rf_grid_dev.h"

#include <type_traits>

#ifndef RF_STRIP_PART
#error "rf_strip.hip is compiled once per RF_STRIP_PART (0..6)"
#endif

namespace {

constexpr bool kIso = RF_STRIP_PART == 6;
constexpr int kKind = kIso ? RF_GEMM_ISO : RF_STRIP_PART % 3;
// real operands throughout (method 4): the im halves are zero, intermediates float
constexpr bool kRealOps = RF_STRIP_PART >= 3 && !kIso;
constexpr bool kFirst = kKind == RF_GEMM_FIRST, kLast = kKind == RF_GEMM_LAST || kIso;
constexpr bool kReal = kLast || kRealOps;   // Re D only
constexpr int NA = kReal ? 1 : 2;       // accumulators per tile: Re, Im
constexpr unsigned kElem = kRealOps && !kFirst ? 4u : 8u;   // bytes of a streamed element (real first: FP64)
constexpr int NV = kIso ? 8 : 4;        // values of a lane per step (isotropic: two factors)
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) void lds_void;
typedef const char __attribute__((address_space(1))) gch;
constexpr int strip_units(int MT, int CS) { return CS * MT * 128; }   // 16-byte units of a chunk

// x and y hold k = 4 h + (0..3) in lane half h: half 0's x for all eight k in
// half 0, half 1's y for all eight in half 1.
__device__ __forceinline__ u32x4 half_swap(const hv4& x, const hv4& y) {
    const u32x2 a = __builtin_bit_cast(u32x2, x), b = __builtin_bit_cast(u32x2, y);
    const u32x2 p = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane32_swap(a.x, b.x, false, false));
    const u32x2 q = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane32_swap(a.y, b.y, false, false));
    return u32x4{p.x, q.x, p.y, q.y};
}

// One strip: lines n0 .. n0 + 31 of a batch (n0 < N; lines past N re-read the
// last one and are not stored).
struct strip {
    // streamed operand: wave-uniform base, 32-bit lane offset (the launcher
    // keeps a strip's span below 2^27 elements).  Global address space: the
    // descriptor of a grouped launch is read from memory, and generic (flat)
    // loads would also count against the LDS wait counter.
    gch* S;
    gch* Y;                               // isotropic: the lane's values of the second factor (S: of the first)
    unsigned lo0;
    int batch, n0;
    unsigned gr, gj3, gq, gj2;            // drawn coefficients: the line's digits
};

__device__ __forceinline__ strip strip_at(const rf_gemm_desc& g, int batch, int n0, bool gen, int l32) {
    strip p;
    p.batch = batch;
    p.n0 = n0;
    const int nc = n0 + l32 < g.N ? n0 + l32 : g.N - 1;
    p.Y = nullptr;
    p.gr = p.gj3 = p.gq = p.gj2 = 0;
    if constexpr (kIso) {
        // tables [k / 4][index][k % 4]: a lane's four k are 32 bytes
        const int64_t half = (threadIdx.x >> 5) & 1;
        p.S = (gch*)(g.B + (int64_t)batch * g.bStrideB) + 32 * (nc % g.isoNx + half * g.isoNx);
        p.Y = (gch*)(g.isoY + (int64_t)batch * g.isoYStrideB) + 32 * (nc / g.isoNx + half * g.isoNy);
        p.lo0 = 0;
        return p;
    }
    const int64_t col0 = col_b(g, n0);
    p.S = (gch*)g.B + ((int64_t)batch * g.bStrideB + col0) * (int64_t)kElem;
    p.lo0 = (unsigned)(col_b(g, nc) - col0) * kElem;
    if (kFirst && gen) {
        const unsigned Q = (g.gen.fold && g.gen.nDim == 3) ? 2u : 1u;
        unsigned rem = (unsigned)nc;
        p.gj2 = rem % (unsigned)g.gen.nk2; rem /= (unsigned)g.gen.nk2;
        p.gq = rem % Q; rem /= Q;
        p.gj3 = g.gen.nDim == 3 ? rem % (unsigned)g.gen.nk3 : 0u;
        p.gr = g.gen.nDim == 3 ? rem / (unsigned)g.gen.nk3 : rem;
    }
    return p;
}

// The values of steps CS c .. of this lane (a step past the last repeats it);
// past K the table is zero and the last valid value is read again.  gen: a
// batch's fresh realizations, the coefficients of the current draw formed here
// (fold_coef_draw, as the fold would store them) instead of read.  Real first
// contraction: the plan's FP64 amplitudes as they are (strip_split scales them),
// k contiguous.
template <int CS>
__device__ __forceinline__ void strip_fetch(const rf_gemm_desc& g, const strip& p, int c, int nSteps, bool gen,
                                            int64_t drawBase, int half, f2v (*v)[NV]) {
    const unsigned kb = (unsigned)g.bSk * kElem;      // bytes per k
#pragma unroll
    for (int st = 0; st < CS; st++) {
        const int s = CS * c + st < nSteps ? CS * c + st : nSteps - 1;
        if constexpr (kIso) {
            auto run = [&](gch* t, int n, f2v* o) {
                const gf4* q = (const gf4*)(t + (int64_t)(2 * s) * n * 32);
                const f4v a = q[0], b = q[1];
                o[0] = f2v{a.x, a.y};
                o[1] = f2v{a.z, a.w};
                o[2] = f2v{b.x, b.y};
                o[3] = f2v{b.z, b.w};
            };
            run(p.S, g.isoNx, v[st]);
            if (g.isoY) {
                run(p.Y, g.isoNy, v[st] + 4);
            } else {
#pragma unroll
                for (int i = 4; i < NV; i++) v[st][i] = f2v{1.f, 0.f};
            }
        } else if constexpr (kFirst && kRealOps) {
            struct __attribute__((packed, aligned(8))) pair { f2v a, b; };
            typedef const pair __attribute__((address_space(1))) gpair;
            gch* b = p.S + (p.lo0 + 64u * (unsigned)s);
            const int left = g.K - 1 - 8 * s;
            if (left >= 7) {                                                      // uniform
#pragma unroll
                for (int i = 0; i < 4; i += 2) {
                    const gpair* e = (const gpair*)(b + 8 * (4 * half + i));
                    v[st][i] = e->a;
                    v[st][i + 1] = e->b;
                }
            } else {
#pragma unroll
                for (int i = 0; i < 4; i++) v[st][i] = *(gf2*)(b + 8 * (4 * half + i < left ? 4 * half + i : left));
            }
        } else if (kFirst && gen) {
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int k = 8 * s + 4 * half + i;
                if (k < g.K) {
                    const unsigned h = k >= g.gen.nk1 ? 1u : 0u;
                    const float2 x = fold_coef_draw(g.gen, p.gr, p.gj3, p.gq, p.gj2, (unsigned)(k - (h ? g.gen.nk1 : 0)), h,
                                                    g.genSeed, drawBase);
                    v[st][i] = f2v{x.x, x.y};
                } else {
                    v[st][i] = f2v{0.f, 0.f};
                }
            }
        } else {
            gch* b = p.S + (int64_t)(8 * s) * kb;
            const int left = g.K - 1 - 8 * s;         // >= 0
#pragma unroll
            for (int i = 0; i < 4; i++) {
                int k = 4 * half + i;
                if (left < 7) k = k < left ? k : left;                            // uniform: the last step
                gch* e = b + (p.lo0 + (unsigned)k * kb);
                if constexpr (kElem == 4) v[st][i] = f2v{*(const gfo*)e, 0.0f};
                else v[st][i] = *(gf2*)e;
            }
        }
    }
}

template <int CS>
__device__ __forceinline__ void strip_split(const f2v (*r)[NV], double scale, unsigned sgn, u32x4 (*fh)[NA],
                                            u32x4 (*fl)[NA]) {
#pragma clang fp contract(off)
#pragma unroll
    for (int st = 0; st < CS; st++) {
        float re[4], im[4];
        hv4 rh, rl, ih, il;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if constexpr (kIso) {
                const f2v w = r[st][i], y = r[st][4 + i];
                re[i] = fmaf(w.x, y.x, -w.y * y.y);
                im[i] = fmaf(w.x, y.y, w.y * y.x);
                continue;
            }
            re[i] = kFirst && kRealOps ? (float)(__builtin_bit_cast(double, r[st][i]) * scale) : r[st][i].x;
            im[i] = r[st][i].y;
        }
        split4(re, &rh, &rl);
        if (kRealOps) ih = il = hv4{0, 0, 0, 0};
        else split4(im, &ih, &il);
        const u32x4 h = half_swap(rh, ih), l = half_swap(rl, il);                 // (Re, Im)
        fh[st][0] = h ^ sgn;
        fl[st][0] = l ^ sgn;
        if (kFirst && !kReal) {
            fh[st][NA - 1] = half_swap(ih, rh);                                   // (Im, Re)
            fl[st][NA - 1] = half_swap(il, rl);
        } else if (!kReal) {
            fh[st][NA - 1] = h;
            fl[st][NA - 1] = l;
        }
    }
}

// One step's products: tiles 0 .. MT - 1 at tab (one step of the table).
template <int MT>
__device__ __forceinline__ void strip_step(const u32x4* tab, const u32x4* fh, const u32x4* fl, int lane,
                                           f32x16 (*acc)[NA]) {
    auto mm = [](const u32x4& x, const u32x4& y, const f32x16& d) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(hv8, x), __builtin_bit_cast(hv8, y), d, 0, 0, 0);
    };
#pragma unroll
    for (int t = 0; t < MT; t++) {
        u32x4 th[NA], tl[NA];
        th[0] = tab[(2 * t) * 64 + lane];
        tl[0] = tab[(2 * t + 1) * 64 + lane];
        if (!kReal && !kFirst) {
            th[NA - 1] = tab[(2 * t) * 64 + (lane ^ 32)];
            tl[NA - 1] = tab[(2 * t + 1) * 64 + (lane ^ 32)];
        } else {
            th[NA - 1] = th[0];
            tl[NA - 1] = tl[0];
        }
        // A hi B hi, A hi B lo, A lo B hi
#pragma unroll
        for (int a = 0; a < NA; a++) acc[t][a] = kFirst ? mm(fh[a], th[a], acc[t][a]) : mm(th[a], fh[a], acc[t][a]);
#pragma unroll
        for (int a = 0; a < NA; a++) acc[t][a] = kFirst ? mm(fh[a], tl[a], acc[t][a]) : mm(th[a], fl[a], acc[t][a]);
#pragma unroll
        for (int a = 0; a < NA; a++) acc[t][a] = kFirst ? mm(fl[a], th[a], acc[t][a]) : mm(tl[a], fh[a], acc[t][a]);
    }
}

template <int MT>
__device__ __forceinline__ void strip_zero(f32x16 (*acc)[NA]) {
#pragma unroll
    for (int t = 0; t < MT; t++)
#pragma unroll
        for (int a = 0; a < NA; a++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc[t][a][i] = 0.0f;
}

// Strip p's tiles t0 .. t0 + MT - 1 to D.  Layout of a 32x32 tile: lane column
// l32 (B operand), rows 8*(i/4) + 4*half + i%4 (A operand).
template <int MT>
__device__ __forceinline__ void strip_store(const rf_gemm_desc& g, const strip& p, int t0, int half, int l32,
                                            f32x16 (*acc)[NA]) {
    const float os = g.outScale;
    const int n0 = p.n0, n = n0 + l32;
    const int dSm = (int)g.dSm, dSn = (int)g.dSn, rows = g.M;
    // an intermediate's element type, address and value
    auto at = [&](int64_t e) {
        if constexpr (kRealOps) return (gfo*)(static_cast<float*>(g.D) + e);
        else return (gf2o*)(static_cast<float2*>(g.D) + e);
    };
    auto val = [&](int t, int i) {
        if constexpr (kRealOps) return acc[t][0][i] * os;
        else return f2v{acc[t][0][i] * os, acc[t][NA - 1][i] * os};
    };
    if constexpr (kFirst) {
        // lane: table entry 32 (t0 + t) + l32; rows: lines
        auto* D = at((int64_t)p.batch * g.dStrideB + (int64_t)n0 * g.dSn);
#pragma unroll
        for (int t = 0; t < MT; t++) {
            const int m = 32 * (t0 + t) + l32;
            if (m >= rows) continue;
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const int line = 8 * (i >> 2) + 4 * half + (i & 3);
                if (n0 + line < g.N) D[line * dSn + m] = val(t, i);
            }
        }
    } else if constexpr (!kLast) {
        if (n >= g.N) return;
        const int64_t d0 = col_d(g, n0);
        auto* D = at((int64_t)p.batch * g.dStrideB + d0 + (int64_t)(32 * t0) * g.dSm);
        const int oc = (int)(col_d(g, n) - d0);
#pragma unroll
        for (int t = 0; t < MT; t++)
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const int m = 32 * t + 8 * (i >> 2) + 4 * half + (i & 3);
                if (32 * t0 + m < rows) D[m * dSm + oc] = val(t, i);
            }
    } else {
        // the epilogue's map, in place
        const float sc = (float)g.epi.scale, sh = (float)g.epi.shift;
        auto each = [&](auto map) {
#pragma unroll
            for (int t = 0; t < MT; t++)
#pragma unroll
                for (int i = 0; i < 16; i++) acc[t][0][i] = map(acc[t][0][i] * os);
        };
        if (g.epi.margi == RF_FOM_NONE) each([](float u) { return u; });
        else if (g.epi.margi == RF_FOM_LOGNORMAL) each([=](float u) { return expf(fmaf(u, sc, sh)); });
        else each([=](float u) { return fmaf(u, sc, sh); });
        const int64_t dBase = (int64_t)p.batch * g.dStrideB + (int64_t)n0 * g.dSn;
        const bool nIn = n < g.N;
        auto store = [&](auto* D, auto* G, auto* BL, auto* BH, auto one) {
            typedef decltype(one) T;
            typedef std::conditional_t<kIso, int64_t, int> index;     // (isotropic planes of any size)
            if (kIso || !g.grp) {
#pragma unroll
                for (int t = 0; t < MT; t++) {
                    const int R0 = 32 * (t0 + t);
                    if (R0 >= rows) break;                                        // uniform
                    auto* d = D + (int64_t)R0 * dSm;
                    const bool whole = R0 + 32 <= rows;                           // uniform
#pragma unroll
                    for (int i = 0; i < 16; i++) {
                        const int m = 8 * (i >> 2) + 4 * half + (i & 3);
                        if (nIn && (whole || R0 + m < rows)) d[(index)m * dSm + l32] = (T)acc[t][0][i];
                    }
                }
                return;
            }
            // fused blend: a lane's column goes to the group grid (rows zLo ..
            // zHi - 1 of it, the others to the field), to a first-axis band array
            // or to the field: one pointer and row stride per lane, so that a tile
            // inside zLo .. zHi costs an address addition per store (a choice per
            // value: 22 VALU instructions each, 44 % of the kernel's issue slots)
            if (!nIn) return;
            const int64_t gc = grp_col(g, n);
            int bside = 0, bst = 0;
            const int64_t bo = gc < 0 ? band_col(g, n, p.batch, &bside, &bst) : -1;
            const bool inG = gc >= 0, inB = bo >= 0;
            auto* f = D + l32;
            auto* q = inG ? G + (g.grpRow0 + gc) : inB ? (bside ? BH : BL) + bo : f;
            const int64_t qs = inG ? g.grpPlaneG : inB ? (int64_t)bst : (int64_t)dSm;
            q += (32 * t0 + 4 * half) * qs;
#pragma unroll
            for (int t = 0; t < MT; t++) {
                const int R0 = 32 * (t0 + t);
                if (R0 >= rows) break;                                            // uniform
                const bool inside = R0 >= g.grpZlo && R0 + 32 <= g.grpZhi;        // uniform
                auto* r = q;
#pragma unroll
                for (int a = 0; a < 4; a++) {
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const int M = R0 + 8 * a + 4 * half + i;
                        if (inside || (M < rows && (!inG || (M >= g.grpZlo && M < g.grpZhi)))) *r = (T)acc[t][0][4 * a + i];
                        else if (M < rows) f[(int64_t)M * dSm] = (T)acc[t][0][4 * a + i];
                        r += qs;
                    }
                    r += 4 * qs;
                }
                q += 32 * qs;
            }
        };
        if (g.outDtype == RF_DTYPE_F64)
            store((gdo*)(static_cast<double*>(g.D) + dBase),
                  (gdo*)(static_cast<double*>(g.grp) + (int64_t)p.batch * g.grpStrideB),
                  (gdo*)static_cast<double*>(g.bandLo), (gdo*)static_cast<double*>(g.bandHi), 0.0);
        else
            store((gfo*)(static_cast<float*>(g.D) + dBase), (gfo*)(static_cast<float*>(g.grp) + (int64_t)p.batch * g.grpStrideB),
                  (gfo*)static_cast<float*>(g.bandLo), (gfo*)static_cast<float*>(g.bandHi), 0.0f);
    }
}

// Logical tile `local` = (table group fastest -- the groups share
// the streamed lines --, block of kStripW strips, batch).
template <int MT, int CS>
__device__ __forceinline__ void strip_tile(const rf_gemm_desc& g, int64_t local, u32x4* ldsA, u32x4* ldsB) {
    const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5, l32 = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int mtTot = (g.M + 31) / 32, nGr = (mtTot + MT - 1) / MT;
    const int t0 = (int)(local % nGr) * MT;
    const int64_t rest = local / nGr;
    const int nSB = (int)(((int64_t)g.N + kStripL - 1) / kStripL);
    const int batch = (int)(rest / nSB);
    const int64_t first = (rest % nSB) * kStripL + wave * 32;
    const bool active = first < g.N;                  // uniform
    const int nSteps = (g.K + 7) / 8, nChunks = (nSteps + CS - 1) / CS;
    const unsigned sgn = half ? 0x80008000u : 0u;
    const bool gen = kFirst && !kRealOps && g.genState != nullptr && g.genState[2] != 0;
    const int64_t drawBase = gen ? g.genState[1] * (int64_t)g.genNmc * g.gen.kNr : 0;
    const strip p = strip_at(g, batch, active ? (int)first : 0, gen, l32);

    f32x16 acc[MT][NA];
    strip_zero<MT>(acc);
    f2v r[CS][NV];
    // chunk c of the table (steps CS c ..): 1 KB pieces over the waves; tiles
    // and steps past the table re-read its last ones, whose products are never
    // stored, resp. never formed
    const u32x4* T = static_cast<const u32x4*>(g.T) + (kIso ? (int64_t)batch * nSteps * mtTot * 128 : 0);
    auto dma = [&](int c, u32x4* dst) {
        constexpr int kPieces = CS * MT * 2;
#pragma unroll
        for (int i = 0; i < (kPieces + kStripW - 1) / kStripW; i++) {
            const int q = wave + i * kStripW;
            if (kPieces % kStripW == 0 || q < kPieces) {
                const int st = q / (2 * MT), u = q % (2 * MT);
                const int s = CS * c + st < nSteps ? CS * c + st : nSteps - 1;
                const int t = t0 + (u >> 1) < mtTot ? t0 + (u >> 1) : mtTot - 1;
                __builtin_amdgcn_global_load_lds((const void*)(T + (((int64_t)s * mtTot + t) * 2 + (u & 1)) * 64 + lane),
                                                 (lds_void*)&dst[q * 64], 16, 0, 0);
            }
        }
    };
    auto chunk = [&](int c, const u32x4* cur, u32x4* nxt) {
        // fragments of this chunk's streamed values, then the loads of the next
        // (all of K in one chunk: step by step, for the registers)
        constexpr bool kAll = CS == kStripCS;
        const double scale = kFirst ? g.gen.ampMult : 1.0;
        u32x4 fh[kAll ? CS : 1][NA], fl[kAll ? CS : 1][NA];
        if constexpr (kAll) strip_split<CS>(r, scale, sgn, fh, fl);
        if (CS == kStripCS && c + 1 < nChunks) {      // in flight during the MFMAs
            dma(c + 1, nxt);
            strip_fetch<CS>(g, p, c + 1, nSteps, gen, drawBase, half, r);
        }
#pragma unroll
        for (int st = 0; st < CS; st++) {
            if (!active || CS * c + st >= nSteps) break;                          // uniform
            if constexpr (!kAll) strip_split<1>(r + st, scale, sgn, fh, fl);
            strip_step<MT>(cur + st * MT * 128, fh[kAll ? st : 0], fl[kAll ? st : 0], lane, acc);
        }
        if (CS != kStripCS) return;                   // all of K in one chunk
        // this wave's direct loads are complete (vmcnt(0)) before the barrier
        // publishes them
        __builtin_amdgcn_s_waitcnt(0x0F70);
        __syncthreads();
    };
    dma(0, ldsA);
    strip_fetch<CS>(g, p, 0, nSteps, gen, drawBase, half, r);
    __builtin_amdgcn_s_waitcnt(0x0F70);
    __syncthreads();
    for (int c = 0; c < nChunks; c += 2) {
        chunk(c, ldsA, ldsB);
        if (c + 1 < nChunks) chunk(c + 1, ldsB, ldsA);
    }
    if (active) strip_store<MT>(g, p, t0, half, l32, acc);
}

// Registers: 16 MT accumulators per lane (32 MT complex) decide the waves per
// SIMD; the compiler then keeps them in VGPRs without spills.
constexpr int strip_waves(int MT, int CS) {
    if (CS != kStripCS) return MT >= 4 ? 2 : 3;
    return NA == 1 ? (MT >= 3 ? 3 : 4) : (MT >= 3 ? 2 : MT == 2 ? 3 : 4);
}

template <int MT, int CS, int KIND, bool REAL>
__global__ __launch_bounds__(64 * kStripW) __attribute__((amdgpu_waves_per_eu(strip_waves(MT, CS))))
void k_strip(rf_gemm_desc g, int64_t nTiles) {
    __shared__ u32x4 ldsA[strip_units(MT, CS)];
    __shared__ u32x4 ldsB[CS == kStripCS ? strip_units(MT, CS) : 1];
    const int64_t L = xcd_tile(blockIdx.x, nTiles);
    if (L >= nTiles) return;
    strip_tile<MT, CS>(g, L, ldsA, ldsB);
}

template <int MT, int CS, int KIND, bool REAL>
__global__ __launch_bounds__(64 * kStripW) __attribute__((amdgpu_waves_per_eu(strip_waves(MT, CS))))
void k_strip_group(const rf_gemm_desc* __restrict__ gs, int nG, int64_t nTiles) {
    __shared__ u32x4 ldsA[strip_units(MT, CS)];
    __shared__ u32x4 ldsB[CS == kStripCS ? strip_units(MT, CS) : 1];
    const int64_t L = xcd_tile(blockIdx.x, nTiles);
    if (L >= nTiles) return;
    const rf_gemm_desc g = gs[gemm_find(gs, nG, L)];   // uniform: scalar registers
    strip_tile<MT, CS>(g, L - g.tile0, ldsA, ldsB);
}

template <int MT, int CS>
hipError_t launch_cs(const rf_gemm_desc* g, const rf_gemm_desc* d_gs, int nG, int64_t n, unsigned blocks, hipStream_t s) {
    if (g) hipLaunchKernelGGL((k_strip<MT, CS, kKind, kRealOps>), dim3(blocks), dim3(64 * kStripW), 0, s, *g, n);
    else if constexpr (kRealOps || kIso) return hipErrorInvalidValue;
    else hipLaunchKernelGGL((k_strip_group<MT, CS, kKind, kRealOps>), dim3(blocks), dim3(64 * kStripW), 0, s, d_gs, nG, n);
    return hipGetLastError();
}

template <int MT>
hipError_t launch(bool brief, const rf_gemm_desc* g, const rf_gemm_desc* d_gs, int nG, int64_t n, unsigned blocks,
                  hipStream_t s) {
    if constexpr (kKind == RF_GEMM_LAST) {
        if (brief) return launch_cs<MT, kStripShortCS>(g, d_gs, nG, n, blocks, s);
    }
    return launch_cs<MT, kStripCS>(g, d_gs, nG, n, blocks, s);
}

}  // namespace

#if RF_STRIP_PART == 0
#define RF_STRIP_LAUNCH rf_strip_launch_first
#elif RF_STRIP_PART == 1
#define RF_STRIP_LAUNCH rf_strip_launch_middle
#elif RF_STRIP_PART == 2
#define RF_STRIP_LAUNCH rf_strip_launch_last
#elif RF_STRIP_PART == 3
#define RF_STRIP_LAUNCH rf_strip_launch_first_real
#elif RF_STRIP_PART == 4
#define RF_STRIP_LAUNCH rf_strip_launch_middle_real
#elif RF_STRIP_PART == 5
#define RF_STRIP_LAUNCH rf_strip_launch_last_real
#else
#define RF_STRIP_LAUNCH rf_strip_launch_iso
#endif
hipError_t RF_STRIP_LAUNCH(int mt, const rf_gemm_desc* g, const rf_gemm_desc* d_gs, int nG, int64_t n, unsigned blocks,
                           hipStream_t s) {
    const bool brief = mt & kStripShort;
    switch (mt & ~kStripShort) {
        case 1: return launch<1>(brief, g, d_gs, nG, n, blocks, s);
        case 2: return launch<2>(brief, g, d_gs, nG, n, blocks, s);
        case 3: return launch<3>(brief, g, d_gs, nG, n, blocks, s);
        case 4: return launch<4>(brief, g, d_gs, nG, n, blocks, s);
        default: return launch<kStripMaxMT>(brief, g, d_gs, nG, n, blocks, s);
    }
}
