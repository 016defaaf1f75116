// zj_tri_frag.hpp -- the triangle kernels' dense operator products on the
// matrix cores (gfx950).
//
// A wave owns groups of four elements.  The 16 columns of a product are the
// four elements' four conservative variables, its rows the solution or flux
// points, in blocks of four: lane l holds row 4 b + l/16 of block b, of
// element (l/4) mod 4 and variable l mod 4.  That is at once the B operand
// and the result layout of v_mfma_f64_16x16x4 and v_mfma_f64_4x4x4_4b (four
// blocks: one element each), and, with the operator's rows permuted within a
// tile, of v_mfma_f32_16x16x4: a product's result feeds the next product as
// it stands, and state, gradient and fluxes stay one value per lane and block.
//
// Why: applied row by row with scalar operator entries, the same products
// took two thirds of the kernels' VALU issue, waited on scalar loads, and
// held every point of an element in one lane (132 VGPRs, one wave per SIMD).
// The matrix cores run FP64 at the VALU's rate (71 TFLOP/s measured for both
// shapes) and FP32 at twice it, beside the VALU.  FP64 rows beyond the last
// whole tile of 16 take the 4x4x4 shape, at the same rate, so no 16-row
// padding is paid; FP32 has no such shape and pads.
//
// Operator rows beyond the matrix are zero; the columns' rows beyond it must
// be given as zero too (0 x NaN would spread).
#pragma once

#include "zj_kernels.hpp"
#include "zj_tri_ops.hpp"

#include <hip/hip_runtime.h>

#include <type_traits>
#include <vector>

namespace zj {
namespace tri {

// Table of an operator of MB row blocks and KB column blocks: whole tiles of
// four row blocks as [tile][column block][64], lane order, then (FP64) the
// other row blocks as [block][column block][16], (column, row) order.
template <typename R, int MB, int KB> struct FragTab {
    static constexpr bool F64 = std::is_same<R, double>::value;
    static constexpr int TILES = F64 ? MB / 4 : (MB + 3) / 4, SINGLES = F64 ? MB % 4 : 0;
    static constexpr int WORDS = TILES * KB * 64 + SINGLES * KB * 16;
};

// Fills a table from at(row, column), zero outside the matrix.
template <typename R, int MB, int KB, typename F> void frag_fill(R* t, F&& at) {
    using T = FragTab<R, MB, KB>;
    for (int i = 0; i < T::TILES; ++i)
        for (int k = 0; k < KB; ++k)
            for (int l = 0; l < 64; ++l) {
                const int r = l % 16;  // FP32 results hold rows 4 (l/16) + register: permuted to 4 register + l/16
                const int row = 16 * i + (T::F64 ? r : 4 * (r % 4) + r / 4);
                t[(i * KB + k) * 64 + l] = row < 4 * MB ? R(at(row, 4 * k + l / 16)) : R(0);
            }
    t += T::TILES * KB * 64;
    for (int s = 0; s < T::SINGLES; ++s)
        for (int k = 0; k < KB; ++k)
            for (int l = 0; l < 16; ++l)
                t[(s * KB + k) * 16 + l] = R(at(16 * T::TILES + 4 * s + l % 4, 4 * k + l / 4));
}

typedef double v4d __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
template <typename R> struct Vec4;
template <> struct Vec4<double> { using type = v4d; };
template <> struct Vec4<float> { using type = v4f; };
__device__ __forceinline__ v4d mma16(double a, double b, v4d c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ v4f mma16(float a, float b, v4f c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// acc[g] += table . b[g] for G column groups, each operator word loaded once.
// ZERO: acc starts at zero.
template <bool ZERO, typename R, int G, int MB, int KB>
__device__ __forceinline__ void frag_mma(const R* t, const R (&b)[G][KB], R (&acc)[G][MB]) {
    using T = FragTab<R, MB, KB>;
    using V = typename Vec4<R>::type;
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int i = 0; i < T::TILES; ++i) {
        V c[G];
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
            for (int r = 0; r < 4; ++r) c[g][r] = ZERO || 4 * i + r >= MB ? R(0) : acc[g][4 * i + r < MB ? 4 * i + r : 0];
#pragma unroll
        for (int k = 0; k < KB; ++k) {
            const R a = t[(i * KB + k) * 64 + lane];
#pragma unroll
            for (int g = 0; g < G; ++g) c[g] = mma16(a, b[g][k], c[g]);
        }
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (4 * i + r < MB) acc[g][4 * i + r < MB ? 4 * i + r : 0] = c[g][r];
    }
    if constexpr (T::SINGLES > 0) {
        const R* s = t + T::TILES * KB * 64 + (lane >> 4) * 4 + (lane & 3);
#pragma unroll
        for (int i = 0; i < T::SINGLES; ++i) {
            constexpr int M0 = 4 * T::TILES;
#pragma unroll
            for (int k = 0; k < KB; ++k) {
                const R a = s[(i * KB + k) * 16];
#pragma unroll
                for (int g = 0; g < G; ++g)
                    acc[g][M0 + i] = __builtin_amdgcn_mfma_f64_4x4x4f64(a, b[g][k], ZERO && k == 0 ? R(0) : acc[g][M0 + i],
                                                                        0, 0, 0);
            }
        }
    }
}

// Four block-diagonal operators on the flux points at once, one (p+1) x (p+1)
// block per edge: a tile's four row blocks are one row block of each operator,
// and only the 4 x 4 blocks that meet an edge's block are kept, [block][64].
template <int P> struct DiagTab {
    static constexpr int FP = P + 1, NFP = 3 * FP, FB = (NFP + 3) / 4;
    static constexpr bool nz(int m, int k) {
        const int m1 = 4 * m + 3 < NFP ? 4 * m + 3 : NFP - 1, k1 = 4 * k + 3 < NFP ? 4 * k + 3 : NFP - 1;
        return 4 * m / FP <= k1 / FP && 4 * k / FP <= m1 / FP;
    }
    static constexpr int before(int m, int k) {  // kept blocks before block (m, k)
        int n = 0;
        for (int i = 0; i < FB; ++i)
            for (int j = 0; j < FB; ++j)
                if (i < m || (i == m && j < k)) n += nz(i, j);
        return n;
    }
    static constexpr int WORDS = 64 * before(FB, 0);
};
// at(operator, row, column)
template <typename R, int P, typename F> void diag_fill(R* t, F&& at) {
    using T = DiagTab<P>;
    for (int m = 0; m < T::FB; ++m)
        for (int k = 0; k < T::FB; ++k)
            for (int l = 0; l < 64 && T::nz(m, k); ++l) {
                const int r = l % 16, row = std::is_same<R, double>::value ? r : 4 * (r % 4) + r / 4;
                t[T::before(m, k) * 64 + l] = R(at(row / 4, 4 * m + row % 4, 4 * k + l / 16));
            }
}
// acc[g][operator] = operator . b[g]
template <typename R, int P, int G, int FB>
__device__ __forceinline__ void diag_mma(const R* t, const R (&b)[G][FB], R (&acc)[G][4][FB]) {
    using T = DiagTab<P>;
    using V = typename Vec4<R>::type;
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int m = 0; m < FB; ++m) {
        V c[G];
#pragma unroll
        for (int g = 0; g < G; ++g) c[g] = V{R(0), R(0), R(0), R(0)};
#pragma unroll
        for (int k = 0; k < FB; ++k) {
            if (!T::nz(m, k)) continue;
            const R a = t[T::before(m, k) * 64 + lane];
#pragma unroll
            for (int g = 0; g < G; ++g) c[g] = mma16(a, b[g][k], c[g]);
        }
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
            for (int o = 0; o < 4; ++o) acc[g][o][m] = c[g][o];
    }
}

// The sum of the four operators' transposes, each of its own columns:
// acc[g] = sum_o operator_o^T . b[g][o].  FP64: the kept 4 x 4 blocks as
// [row block][column block][operator][16]; FP32: whole tiles of rows.
template <typename R, int P> struct DiagTTab {
    using T = DiagTab<P>;
    static constexpr bool F64 = std::is_same<R, double>::value;
    static constexpr int FB = T::FB, WORDS = F64 ? 4 * 16 * T::before(FB, 0) : FragTab<R, FB, 4 * FB>::WORDS;
};
template <typename R, int P, typename F> void diag_fill_t(R* t, F&& at) {
    using T = DiagTab<P>;
    constexpr int FB = T::FB;
    auto tr = [&](int row, int o, int col) { return at(o, col, row); };
    if constexpr (DiagTTab<R, P>::F64) {
        for (int m = 0; m < FB; ++m)
            for (int k = 0; k < FB; ++k)
                for (int l = 0; l < 64 && T::nz(m, k); ++l)
                    t[T::before(m, k) * 64 + l] = R(tr(4 * m + l % 4, l / 16, 4 * k + l / 4 % 4));
    } else {
        frag_fill<R, FB, 4 * FB>(t, [&](int row, int c) { return tr(row, c / (4 * FB), c % (4 * FB)); });
    }
}
template <typename R, int P, int G, int FB>
__device__ __forceinline__ void diag_mma_t(const R* t, const R (&b)[G][4][FB], R (&acc)[G][FB]) {
    using T = DiagTab<P>;
    if constexpr (DiagTTab<R, P>::F64) {
        const int lane = threadIdx.x & 63;
        const R* s = t + (lane >> 4) * 4 + (lane & 3);
#pragma unroll
        for (int m = 0; m < FB; ++m) {
#pragma unroll
            for (int g = 0; g < G; ++g) acc[g][m] = R(0);
#pragma unroll
            for (int k = 0; k < FB; ++k) {
                if (!T::nz(m, k)) continue;
#pragma unroll
                for (int o = 0; o < 4; ++o) {
                    const R a = s[T::before(m, k) * 64 + o * 16];
#pragma unroll
                    for (int g = 0; g < G; ++g)
                        acc[g][m] = __builtin_amdgcn_mfma_f64_4x4x4f64(a, b[g][o][k], acc[g][m], 0, 0, 0);
                }
            }
        }
    } else {
        R f[G][4 * FB];
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
            for (int o = 0; o < 4; ++o)
#pragma unroll
                for (int k = 0; k < FB; ++k) f[g][o * FB + k] = b[g][o][k];
        frag_mma<true, R, G, FB, 4 * FB>(t, f, acc);
    }
}

// Orders LDS writes of a wave's lanes before its other lanes' later reads (a
// wave's LDS operations execute in order; the compiler must keep them so).
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Words between two elements of an LDS array [element][rows][4], at least
// 4 rows and a multiple of 4, such that a lane group's four elements (FP64),
// or two rows of them (FP32), fall on different banks.
template <typename R> constexpr int elem_stride(int rows) {
    return std::is_same<R, double>::value ? 4 * (rows | 1) : (4 * rows + 7) / 16 * 16 + 8;
}

// The operators of order P as tables, one after the other; row and column
// blocks of solution points (PB), flux points (FB) and of both contravariant
// fluxes' points (CB, rows of F_r then F_s):
//   D   gradient: Dr, Ds                                   2 PB x PB
//   I   interpolation to the flux points                     FB x PB
//   G   traces of the gradient: I Dr, I Ds                 2 FB x PB
//   F   divergence Dr F_r + Ds F_s, then the transformed normal fluxes
//       -I F_s, I (F_r + F_s), -I F_r of edges 0, 1, 2     PB + FB x CB
// then, per correction family (DG, SD = GA, HU):
//   L   lifting                                              PB x FB
//   LF  face liftings (block-diagonal on the flux points): one edge's jumps
//       at that edge's own points, and, for each of a neighbour's edges 0, 1,
//       2, the neighbour's face lifting of the same jumps by this side's
//       points (slots run the other way along a shared edge)
// and for the adjoint (after the families, its own family parts last):
//   FT  F backwards: cotangents of F_r, F_s (PB blocks each) from those of
//       the divergence and of the flux differences      2 PB x (PB + FB)
//   GT  traces of U and of its gradient's r and s parts backwards  PB x 3 FB
//   DT  gradient backwards                                       PB x 2 PB
//   LT  lifting backwards                                          FB x PB
//   LFT face liftings backwards
template <typename R, int P> struct FragOps {
    static constexpr int NP = (P + 1) * (P + 2) / 2, FP = P + 1, NFP = 3 * FP;
    static constexpr int PB = (NP + 3) / 4, FB = (NFP + 3) / 4, CB = (2 * NP + 3) / 4;
    static constexpr int D = 0;
    static constexpr int I = D + FragTab<R, 2 * PB, PB>::WORDS;
    static constexpr int G = I + FragTab<R, FB, PB>::WORDS;
    static constexpr int F = G + FragTab<R, 2 * FB, PB>::WORDS;
    static constexpr int COMMON = F + FragTab<R, PB + FB, CB>::WORDS;
    static constexpr int L = 0;
    static constexpr int LF = L + FragTab<R, PB, FB>::WORDS;
    static constexpr int FAMILY = LF + DiagTab<P>::WORDS;
    static constexpr int FT = 0;
    static constexpr int GT = FT + FragTab<R, 2 * PB, PB + FB>::WORDS;
    static constexpr int DT = GT + FragTab<R, PB, 3 * FB>::WORDS;
    static constexpr int ADJ = DT + FragTab<R, PB, 2 * PB>::WORDS;
    static constexpr int LT = 0;
    static constexpr int LFT = LT + FragTab<R, FB, PB>::WORDS;
    static constexpr int ADJ_FAMILY = LFT + DiagTTab<R, P>::WORDS;
    static constexpr int ADJ0 = COMMON + 3 * FAMILY;          // where they begin
    static constexpr int ADJ_FAM0 = ADJ0 + ADJ;
    static constexpr int WORDS = ADJ_FAM0 + 3 * ADJ_FAMILY;
    static_assert(F % 4 == 0 && ADJ % 4 == 0 && ADJ_FAMILY % 4 == 0, "copied by four words");
    static_assert(COMMON % 4 == 0 && FAMILY % 4 == 0, "copied by four words");
};
template <typename R> constexpr int frag_offset(int P) {
    return (P > 1 ? FragOps<R, 1>::WORDS : 0) + (P > 2 ? FragOps<R, 2>::WORDS : 0) +
           (P > 3 ? FragOps<R, 3>::WORDS : 0) + (P > 4 ? FragOps<R, 4>::WORDS : 0) + (P > 5 ? FragOps<R, 5>::WORDS : 0);
}

// Tables of order P from the operators of the families DG, SD (= GA), HU.
template <typename R, int P> void frag_build(R* t, const Operators* fam) {
    using O = FragOps<R, P>;
    constexpr int NP = O::NP, FP = O::FP, NFP = O::NFP, PB = O::PB, FB = O::FB, CB = O::CB;
    const Operators& A = fam[0];
    auto dr = [&](int i, int m) { return i < NP && m < NP ? A.Dr[(size_t)i * NP + m] : 0.0; };
    auto ds = [&](int i, int m) { return i < NP && m < NP ? A.Ds[(size_t)i * NP + m] : 0.0; };
    auto in = [&](int j, int m) { return j < NFP && m < NP ? A.interp[(size_t)j * NP + m] : 0.0; };
    auto in_d = [&](bool r, int j, int m) {
        long double s = 0;
        for (int i = 0; i < NP; ++i) s += (long double)in(j, i) * (r ? dr(i, m) : ds(i, m));
        return (double)s;
    };
    frag_fill<R, 2 * PB, PB>(t + O::D, [&](int r, int m) { return r < 4 * PB ? dr(r, m) : ds(r - 4 * PB, m); });
    frag_fill<R, FB, PB>(t + O::I, in);
    frag_fill<R, 2 * FB, PB>(t + O::G, [&](int r, int m) { return r < 4 * FB ? in_d(true, r, m) : in_d(false, r - 4 * FB, m); });
    frag_fill<R, PB + FB, CB>(t + O::F, [&](int r, int c) {
        const bool s = c >= NP;  // a column of F_s
        const int m = s ? c - NP : c;
        if (r < 4 * PB) return s ? ds(r, m) : dr(r, m);
        const int j = r - 4 * PB;
        if (j < FP) return s ? -in(j, m) : 0.0;
        return j < 2 * FP ? in(j, m) : (s ? 0.0 : -in(j, m));
    });
    for (int k = 0; k < 3; ++k) {
        R* f = t + O::COMMON + k * O::FAMILY;
        auto lift = [&](int i, int j) { return i < NP && j < NFP ? fam[k].lift[(size_t)i * NFP + j] : 0.0; };
        auto lf = [&](int a, int b) {  // flux points a, b of one edge
            double s = 0;
            for (int i = 0; i < NP; ++i) s += in(a, i) * lift(i, b);
            return s;
        };
        auto same = [&](int a, int b) { return a < NFP && b < NFP && a / FP == b / FP; };
        frag_fill<R, PB, FB>(f + O::L, lift);
        auto faces = [&](int o, int a, int b) {
            if (!same(a, b)) return 0.0;
            return o == 0 ? lf(a, b) : lf((o - 1) * FP + (P - a % FP), (o - 1) * FP + (P - b % FP));
        };
        diag_fill<R, P>(f + O::LF, faces);
        R* fa = t + O::ADJ_FAM0 + k * O::ADJ_FAMILY;
        frag_fill<R, FB, PB>(fa + O::LT, [&](int j, int i) { return lift(i, j); });
        diag_fill_t<R, P>(fa + O::LFT, faces);
    }
    R* ad = t + O::ADJ0;
    frag_fill<R, 2 * PB, PB + FB>(ad + O::FT, [&](int r, int c) {
        const bool s = r >= 4 * PB;  // a row of F_s
        const int m = s ? r - 4 * PB : r;
        if (c < 4 * PB) return s ? ds(c, m) : dr(c, m);
        const int j = c - 4 * PB;  // flux difference = scaled common flux minus normal flux
        if (j < FP) return s ? in(j, m) : 0.0;
        return j < 2 * FP ? -in(j, m) : (s ? 0.0 : in(j, m));
    });
    frag_fill<R, PB, 3 * FB>(ad + O::GT, [&](int m, int c) {
        const int j = c % (4 * FB);
        return c < 4 * FB ? in(j, m) : in_d(c < 8 * FB, j, m);
    });
    frag_fill<R, PB, 2 * PB>(ad + O::DT, [&](int m, int c) { return c < 4 * PB ? dr(c, m) : ds(c - 4 * PB, m); });
}

}  // namespace tri
}  // namespace zj
