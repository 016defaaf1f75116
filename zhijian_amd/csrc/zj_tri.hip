// zj_tri.hip -- flux reconstruction on straight-sided triangles (textbook
// scheme) and its SSP-RK3 step: one fused kernel per stage, C ABI zj_tri_*
// (include/zhijian_amd.h).
//
// The reference has no triangle semantics to follow: FROperators::initTriangle
// leaves every table zero (src/basis/basis.cpp:615-669) and FRSolver assumes
// quadrilaterals (src/solver/fr_solver.cpp:138-140).  The scheme is the one its
// settings name on simplices: nodal FR with an energy-stable correction field
// (Castonguay, Vincent & Jameson 2012; the L2 lifting for DG, c = 0, and its
// (M + K)^-1 M filtering for SD = GA and HU, zj_tri_ops.hpp), transformed
// fluxes through the constant affine metric, one common flux per face point
// from the configured Riemann solver (include/physics/euler.hpp:204-375).
//
//   dU/dt = -(Dr Fr + Ds Fs) - sum_j lift[:, j] (F^I_j s_j - Fn_j)
//   Fr = r_x F + r_y G,  Fs = s_x F + s_y G   (contravariant fluxes)
//   s_j = |e|/(2J) of flux point j's edge:  |grad s|, |grad r + grad s|, |grad r|
//   Fn_j = interpolated transformed normal flux: -Fs, Fr + Fs, -Fr on edges 0, 1, 2
//   F^I_j = Riemann flux along the face normal, outward on each side
//
// Work mapping: the stage and the Navier-Stokes kernels apply the operators on
// the matrix cores (zj_tri_frag.hpp).  The scalar forms (large P1 and P2
// meshes) and the inviscid adjoint take one lane per (element, conservative
// variable); the four lanes of an element form a DPP quad.  A lane keeps its variable at every solution
// point in registers and applies the dense operators as sums of outer
// products whose entries are wave-uniform, read from constant memory through
// scalar loads: no operator or state traffic through LDS.  The Euler flux of
// point m gathers the point's four variables across the quad by DPP.  LDS
// holds only the element tile's flux-point traces (for the Riemann solves of
// in-tile faces) and the common fluxes on their way back to their variables.
//
// Device layout (one GPU holds the whole mesh):
//   U, W, R  state in blocks of 16 elements: [E/16][Np][16][4] FP64, so the 64
//            lanes of a wave (16 elements x 4 variables) touch 512 contiguous
//            bytes per solution point (W = U1, then U2 in place)
//   T[3]     flux-point traces [E][3(p+1)][4] in the compute precision;
//            only edges whose neighbour lies in another tile (of 32 elements,
//            64 in the scalar forms) are written (a neighbour in the same tile
//            is read from LDS), rotating as the quadrilateral path's: stage 1
//            T0->T1, 2 T1->T2, 3 T2->T0
//   geo      [E][10]: r_x, r_y, s_x, s_y, then the face normal (as the face's
//            left element sees it) of edges 0, 1, 2
//   edge     [E][3][2]: |e|/(2J) of each edge and of the neighbour's side of it
//            (0 on a boundary), for the matrix-core kernels; apart from geo,
//            whose words the others read alone
//   links    [E][3] int2: x = neighbour element (-1 on a boundary), y = packed
//            neighbour edge (or BC type) | role << 3 | BC data index << 6
//   ops      constant memory, per order: Dr, Ds [Np][Np], interp [3(p+1)][Np],
//            lift [Np][3(p+1)]
#include "zhijian_amd.h"
#include "zj_device.hpp"
#include "zj_host_math.hpp"
#include "zj_kernels.hpp"
#include "zj_riemann_vjp.hpp"
#include "zj_tri_frag.hpp"
#include "zj_tri_ops.hpp"
#include "zj_viscous.hpp"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstring>
#include <mutex>
#include <string>
#include <new>
#include <vector>

using namespace zj;

namespace {

template <int P>
struct TriShape {
    static constexpr int NP = (P + 1) * (P + 2) / 2;        // solution points
    static constexpr int FP = P + 1;                        // flux points per edge
    static constexpr int NFP = 3 * FP;
};

constexpr int TILE = BLOCK / NV;  // elements per workgroup (one lane per element and variable)
constexpr int EB = 16;            // elements per block of the state and trace layouts
constexpr int GEO = 10;           // geometry words per element
constexpr int EDG = 6;            // edge factors per element: own and the neighbour's, edge by edge

// Operator tables of order P in constant memory, laid out for wide scalar
// loads in the kernels' loops:
//   A  for each solution point m: column m of Dr, of Ds (NP each) and of the
//      interpolation to the flux points (NFP), contiguous -- the point loop of
//      the volume phase reads one such block per iteration;
//   B  the lifting matrix by columns: column j (NP values) contiguous;
//   C  the interpolation matrix by rows (row j: NP values), for the traces;
//   D  the lifting matrices of the SD (= GA) and HU correction fields, laid
//      out as B, one after the other.
// The kernel reads the lifting matrix at a per-handle offset (B or D).
template <int P> struct TriOps {
    static constexpr int NP = (P + 1) * (P + 2) / 2, NFP = 3 * (P + 1);
    static constexpr int CA = 2 * NP + NFP;         // words per block of A
    static constexpr int B = NP * CA, C = B + NFP * NP, D = C + NFP * NP;
};
constexpr int ops_words(int P) {
    return 2 * ((P + 1) * (P + 2) / 2) * ((P + 1) * (P + 2) / 2) + 5 * 3 * (P + 1) * ((P + 1) * (P + 2) / 2);
}
// Offset of a correction family's lifting matrix within the order-P block.
inline int lift_offset(int P, int family) {
    const int np = (P + 1) * (P + 2) / 2, nfp = 3 * (P + 1), b = np * (2 * np + nfp);
    if (family == ZJ_CORR_DG) return b;
    const int d = b + 2 * nfp * np;
    return family == ZJ_CORR_HU ? d + nfp * np : d;   // SD and GA share one field
}
constexpr int ops_offset(int P) {
    int o = 0;
    for (int q = 1; q < P; ++q) o += ops_words(q);
    return o;
}
constexpr int OPS_TOTAL = ops_offset(6);

__constant__ double c_ops64[OPS_TOTAL];
__constant__ float c_ops32[OPS_TOTAL];

// BR2 face liftings, per order and correction family (DG, SD = GA, HU):
// LF_k = interp(edge k rows) . lift(edge k columns), [3][FP][FP] -- the lifting
// of one edge's jumps evaluated at that edge's own flux points.  For the scalar
// forms, which exist at P1 and P2.
constexpr int lf_words(int P) { return 9 * (P + 1) * (P + 1); }
constexpr int lf_offset(int P) {
    int o = 0;
    for (int q = 1; q < P; ++q) o += 3 * lf_words(q);
    return o;
}
constexpr int LF_ORDERS = 2, LF_TOTAL = lf_offset(LF_ORDERS + 1);
inline int lf_family(int corr) { return corr == ZJ_CORR_DG ? 0 : (corr == ZJ_CORR_HU ? 2 : 1); }
__constant__ double c_lf64[LF_TOTAL];
__constant__ float c_lf32[LF_TOTAL];
template <typename R> __device__ __forceinline__ R clf(int k);
template <> __device__ __forceinline__ double clf<double>(int k) { return c_lf64[k]; }
template <> __device__ __forceinline__ float clf<float>(int k) { return c_lf32[k]; }

// The same operators as matrix-core tables, in device memory (vector loads).
__device__ double d_frag64[tri::frag_offset<double>(6)];
__device__ float d_frag32[tri::frag_offset<float>(6)];
template <typename R> __device__ __forceinline__ const R* frag_ops();
template <> __device__ __forceinline__ const double* frag_ops<double>() { return d_frag64; }
template <> __device__ __forceinline__ const float* frag_ops<float>() { return d_frag32; }

template <typename R> __device__ __forceinline__ R cop(int k);
template <> __device__ __forceinline__ double cop<double>(int k) { return c_ops64[k]; }
template <> __device__ __forceinline__ float cop<float>(int k) { return c_ops32[k]; }

// value of lane W of this lane's quad
template <int W> __device__ __forceinline__ double quad_get(double x) { return dpp_mov<W * 0x55>(x); }
template <int W> __device__ __forceinline__ float quad_get(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), W * 0x55, 0xF, 0xF, false));
}

// offset of variable 0 of (element e, point j) in a [E/16][n][16][4] array
__device__ __forceinline__ int64_t blk(int e, int j, int n) {
    return ((int64_t)(e >> 4) * n + j) * (EB * NV) + (e & (EB - 1)) * NV;
}
// offset of variable 0 of (element e, flux point j) in the [E][n][4] trace
// array: the p+1 points of an edge share one 128-byte line (FP64, p = 3)
__device__ __forceinline__ int64_t trix(int e, int j, int n) { return ((int64_t)e * n + j) * NV; }

// A wave's rows of point values in the [E/16][NP][16][4] layout, G groups of
// four elements from element e0 + 4 G wave: at(p, q, b) is row 4 b + lane/16 of
// this lane's element and variable in group q.  The base is uniform, the
// lane's part 32 bits (a scalar base and an offset in the load, instead of
// 64-bit address arithmetic per value).  Rows and groups beyond the mesh are
// clamped to the last ones; elements beyond it in the last group of four are
// the layout's padding.
template <int NP, int G> struct PointRows {
    static constexpr int PB = (NP + 3) / 4;
    int first, last;   // this wave's first element, the mesh's last group of four
    unsigned lo, hi;   // byte offsets of the lane: rows of a whole block, of the last block
    __device__ __forceinline__ PointRows(int e0, int wave, int lane, int E) {
        first = e0 + __builtin_amdgcn_readfirstlane(wave) * 4 * G;
        last = (E - 1) & ~3;
        const int row = lane >> 4;
        lo = (unsigned)(row * EB * NV + (lane & 15)) * 8u;
        hi = (unsigned)(min(4 * (PB - 1) + row, NP - 1) * EB * NV + (lane & 15)) * 8u;
    }
    template <typename T> __device__ __forceinline__ T* at(T* p, int q, int b) const {
        static_assert(sizeof(T) == 8, "state arrays are FP64");
        using C = typename std::conditional<std::is_const<T>::value, const char, char>::type;
        C* const base = reinterpret_cast<C*>(p + blk(min(first + 4 * q, last), 0, NP));
        return reinterpret_cast<T*>(base + (b < PB - 1 ? 4 * b * EB * NV * 8 + lo : hi));
    }
};

template <typename R>
struct TriArgs {
    int E;
    const double* U_in;   // stage input
    const double* U0;     // U^n (stages 2, 3)
    double* U_out;        // stage output (may alias U_in or U0 lane-locally)
    double* R_out;        // residual (MODE_RESIDUAL)
    const R* geo;
    const R* edge;
    const int2* links;
    const R* T_in;
    R* T_out;
    const double* bc_data;
    const double* dt_ptr;
    double* l2_partial;   // per tile sum of R^2, or nullptr
    double gamma;
    int riemann;
    int xcd_groups;
    int lift_off;         // the correction family's lifting matrix in the order's operator block
    // Navier-Stokes terms (tri_visc_stage_kernel): mu = 1/Re, kappa, BR2 penalty,
    // and the family's face liftings in c_lf
    double mu, kappa, eta;
    int lf_off;
    int family;           // of the correction: DG, SD = GA, HU
};

__device__ __forceinline__ int link_edge(int info) { return info & 7; }
__device__ __forceinline__ int link_role(int info) { return (info >> 3) & 3; }
__device__ __forceinline__ int link_bc(int info) { return info >> 6; }

// 1/x: a Newton-refined hardware reciprocal in FP64 (within 2 ulp), the
// hardware reciprocal in FP32.
template <typename R> __device__ __forceinline__ R fast_rcp(R x);
template <> __device__ __forceinline__ double fast_rcp<double>(double x) { return rcp_refined(x); }
template <> __device__ __forceinline__ float fast_rcp<float>(float x) { return __builtin_amdgcn_rcpf(x); }

// The stage of large meshes at P1 and P2: lanes one per (element, variable),
// the operators as scalar operands (see the file's head); higher orders and
// small meshes take tri_stage_kernel below (TriTile has the rules; residuals
// alone come here at other orders, too).  us a stage, this / that: P1 FP64
// 51,200 elements 11.7 / 15.7, 16,200 7.6 / 7.2, 7,200 7.5 / 5.5; P2 FP64
// 500,000 166 / 182, 51,200 24 / 21; P2 FP32 80,000 17 / 18, 51,200 14 / 14,
// 32,768 11 / 9.5.
template <typename R, int P, int MODE>
__global__ __launch_bounds__(BLOCK, (sizeof(R) == 8 && P == 3 ? 3 : 1)) void tri_scalar_kernel(TriArgs<R> a) {
    using S = TriShape<P>;
    constexpr int NP = S::NP, FP = S::FP, NFP = S::NFP;
    constexpr int NW = NP > NFP ? NP : NFP;
    using OP = TriOps<P>;
    constexpr int O0 = ops_offset(P), CA = OP::CA, OI = O0 + OP::C;
    const int OLT = O0 + a.lift_off;
    __shared__ R sT[TILE * NFP * NV];  // own traces
    __shared__ R sW[TILE * NW * NV];   // the stage input state, then the transformed normal fluxes,
                                       // then the flux differences
    __shared__ double sred[BLOCK / 64];
    __shared__ R sEdge[TILE * 3];                // |a| of every element edge of the tile
    __shared__ unsigned char sList[TILE * 3];    // edges whose face points this tile solves (el * 3 + edge)
    __shared__ int sCnt[BLOCK / 64];             // such edges per wave

    const int tid = threadIdx.x, el = tid >> 2, v = tid & 3;
    const int tile = tile_of_block(a.xcd_groups);
    const int e0 = tile * TILE, e = e0 + el;
    const bool live = e < a.E;
    const R g = R(a.gamma);
    const int64_t base = blk(e, 0, NP) + v;  // this lane's variable at point 0; point i at + i*EB*NV

    double u[NP];
    R div[NP];
    R rx = R(0), ry = R(0), sx = R(0), sy = R(0);
    int2 L[3] = {make_int2(0, 0), make_int2(0, 0), make_int2(0, 0)};

    // ---- 0: this lane's variable at every solution point (one coalesced
    // 512-byte row per point and wave), kept for the stage update
    if (live) {
#pragma unroll
        for (int m = 0; m < NP; ++m) u[m] = a.U_in[base + (int64_t)m * EB * NV];
        const R* G = a.geo + (int64_t)e * GEO;
        rx = G[0]; ry = G[1]; sx = G[2]; sy = G[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) L[k] = a.links[(int64_t)e * 3 + k];
#pragma unroll
        for (int m = 0; m < NP; ++m) sW[(el * NP + m) * NV + v] = R(u[m]);
        if (v < 3) {  // a: the metric gradient normal to edge v (-Fs on edge 0, Fr + Fs on 1, -Fr on 2)
            const R ax = v == 0 ? sx : (v == 1 ? rx + sx : rx), ay = v == 0 ? sy : (v == 1 ? ry + sy : ry);
            sEdge[el * 3 + v] = sqrtR(ax * ax + ay * ay);
        }
    }
    // Lane v < 3 of an element stands for its edge v.  An in-tile face is
    // solved by its left element only; an edge on a boundary or shared with
    // another tile by its own element.
    bool owned = false;
    if (live && v < 3) {
        const int2 Lv = v == 0 ? L[0] : (v == 1 ? L[1] : L[2]);
        const int nl = Lv.x - e0;
        owned = !(link_role(Lv.y) == ROLE_RIGHT && nl >= 0 && nl < TILE);
    }
    const unsigned long long own_mask = __ballot(owned);
    const int lane = tid & 63, wave = tid >> 6;
    if (lane == 0) sCnt[wave] = __popcll(own_mask);
    __syncthreads();

    // ---- 1: fluxes, divergence, traces and interpolated normal fluxes, as
    // sums over the solution points m of outer products with wave-uniform
    // operator columns
    R fn[NFP];
    if (live) {
#pragma unroll
        for (int i = 0; i < NP; ++i) div[i] = R(0);
#pragma unroll
        for (int j = 0; j < NFP; ++j) fn[j] = R(0);
#pragma unroll 1
        for (int m = 0; m < NP; ++m) {
            const R um = sW[(el * NP + m) * NV + v];
            const R q0 = quad_get<0>(um), q1 = quad_get<1>(um), q2 = quad_get<2>(um), q3 = quad_get<3>(um);
            const R inv = fast_rcp(q0);
            const R ux = q1 * inv, uy = q2 * inv;
            const R p = (g - R(1)) * (q3 - R(0.5) * (q1 * ux + q2 * uy));
            const R fx = v == 0 ? q1 : (v == 1 ? q1 * ux + p : (v == 2 ? q1 * uy : (q3 + p) * ux));
            const R fy = v == 0 ? q2 : (v == 1 ? q2 * ux : (v == 2 ? q2 * uy + p : (q3 + p) * uy));
            const R fr = rx * fx + ry * fy, fs = sx * fx + sy * fy, frs = fr + fs;
#pragma unroll
            for (int i = 0; i < NP; ++i)
                div[i] = fmaR(cop<R>(O0 + m * CA + NP + i), fs, fmaR(cop<R>(O0 + m * CA + i), fr, div[i]));
#pragma unroll
            for (int j = 0; j < NFP; ++j)
                fn[j] = fmaR(cop<R>(O0 + m * CA + 2 * NP + j), j < FP ? fs : (j < 2 * FP ? frs : fr), fn[j]);
        }
        // traces in a second pass, so that they and the fluxes' sums are not live together
        R ut[NFP];
#pragma unroll
        for (int j = 0; j < NFP; ++j) ut[j] = R(0);
#pragma unroll 1
        for (int m = 0; m < NP; ++m) {
            const R um = sW[(el * NP + m) * NV + v];
#pragma unroll
            for (int j = 0; j < NFP; ++j) ut[j] = fmaR(cop<R>(O0 + m * CA + 2 * NP + j), um, ut[j]);
        }
#pragma unroll
        for (int j = 0; j < NFP; ++j) sT[(el * NFP + j) * NV + v] = ut[j];
    }
    if (owned) {  // compact the solved edges, in element order
        int pos = __popcll(own_mask & ((1ull << lane) - 1));
        for (int w = 0; w < wave; ++w) pos += sCnt[w];
        sList[pos] = (unsigned char)(el * 3 + v);
    }
    __syncthreads();  // traces in place, state reads done
    // transformed normal fluxes to their flux points' slots in sW:
    // -Fs on edge 0, Fr + Fs on edge 1, -Fr on edge 2
    if (live) {
#pragma unroll
        for (int j = 0; j < NFP; ++j) sW[(el * NFP + j) * NV + v] = (j >= FP && j < 2 * FP) ? fn[j] : -fn[j];
    }
    __syncthreads();

    // ---- 2: common fluxes over the tile's solved edges, spread evenly over
    // the workgroup: the flux difference sc F^I - Fn of this side, and of the
    // in-tile neighbour's side with the same common flux (both elements store
    // the face normal of the left element, so the neighbour would have solved
    // the same problem).  sc = +-|a|, negative on the right.
    {
        int nsolved = 0;
#pragma unroll
        for (int w = 0; w < BLOCK / 64; ++w) nsolved += sCnt[w];
#pragma unroll 1
        for (int t = tid; t < nsolved * FP; t += BLOCK) {
            const int c = sList[t / FP], f = t - (t / FP) * FP;
            const int elt = c / 3, kk = c - elt * 3, j = kk * FP + f;
            const int2 Lk = a.links[(int64_t)(e0 + elt) * 3 + kk];
            const int role = link_role(Lk.y);
            const R nx = a.geo[(int64_t)(e0 + elt) * GEO + 4 + 2 * kk];
            const R ny = a.geo[(int64_t)(e0 + elt) * GEO + 5 + 2 * kk];
            R own[NV], oth[NV], UL[NV], UR[NV], Fc[NV];
#pragma unroll
            for (int w = 0; w < NV; ++w) own[w] = sT[(elt * NFP + j) * NV + w];
            int nl = -1, oj = 0;
            if (role == ROLE_BOUNDARY) {
                ghost_state(own, nx, ny, link_edge(Lk.y), a.bc_data + (int64_t)link_bc(Lk.y) * 8, g, oth);
            } else {
                nl = Lk.x - e0;
                oj = link_edge(Lk.y) * FP + (P - f);
                if (nl >= 0 && nl < TILE) {
#pragma unroll
                    for (int w = 0; w < NV; ++w) oth[w] = sT[(nl * NFP + oj) * NV + w];
                } else {
                    load4(a.T_in + trix(Lk.x, oj, NFP), oth);
                    nl = -1;
                }
            }
            const bool right = role == ROLE_RIGHT;
#pragma unroll
            for (int w = 0; w < NV; ++w) { UL[w] = right ? oth[w] : own[w]; UR[w] = right ? own[w] : oth[w]; }
            riemann_by_kind(a.riemann, UL, UR, nx, ny, g, Fc);
            {
                const R sc = right ? -sEdge[c] : sEdge[c];
                R* d = sW + (elt * NFP + j) * NV;
#pragma unroll
                for (int w = 0; w < NV; ++w) d[w] = sc * Fc[w] - d[w];
            }
            if (nl >= 0) {  // the in-tile neighbour, whose side is the right one
                const R sc = -sEdge[nl * 3 + link_edge(Lk.y)];
                R* d = sW + (nl * NFP + oj) * NV;
#pragma unroll
                for (int w = 0; w < NV; ++w) d[w] = sc * Fc[w] - d[w];
            }
        }
    }
    __syncthreads();

    // ---- 3: lifted flux differences, RK stage update
    double l2 = 0.0;
    double un[NP];
    if (live) {
#pragma unroll 1
        for (int j = 0; j < NFP; ++j) {
            const R d = sW[(el * NFP + j) * NV + v];
#pragma unroll
            for (int i = 0; i < NP; ++i) div[i] = fmaR(cop<R>(OLT + j * NP + i), d, div[i]);
        }
        const double dt = MODE == MODE_RESIDUAL ? 0.0 : *a.dt_ptr;
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const double res = -double(div[i]);
            const int64_t gi = base + (int64_t)i * EB * NV;
            if (MODE == MODE_RESIDUAL) {
                a.R_out[gi] = res;
                l2 += res * res;
            } else {
                if (MODE == MODE_STAGE1) {
                    un[i] = u[i] + dt * res;
                } else {
                    const double u0 = a.U0[gi];
                    un[i] = MODE == MODE_STAGE2 ? 0.75 * u0 + 0.25 * (u[i] + dt * res)
                                                : (1.0 / 3.0) * u0 + (2.0 / 3.0) * (u[i] + dt * res);
                    if (MODE == MODE_STAGE3) l2 += res * res;
                }
                a.U_out[gi] = un[i];
            }
        }
    }
    if ((MODE == MODE_RESIDUAL || MODE == MODE_STAGE3) && a.l2_partial) {
        const double s = block_reduce<OpSum>(l2, sred);
        if (tid == 0) a.l2_partial[tile] = s;
    }
    if (MODE == MODE_RESIDUAL || !live) return;

    // ---- 4: traces of the new stage state on edges another tile reads
#pragma unroll
    for (int kk = 0; kk < 3; ++kk) {
        const int nl = L[kk].x - e0;
        if (link_role(L[kk].y) == ROLE_BOUNDARY || (nl >= 0 && nl < TILE)) continue;
#pragma unroll 1
        for (int j = kk * FP; j < kk * FP + FP; ++j) {
            R t = R(0);
#pragma unroll
            for (int m = 0; m < NP; ++m) t = fmaR(cop<R>(OI + j * NP + m), R(un[m]), t);
            a.T_out[trix(e, j, NFP) + v] = t;
        }
    }
}

// The stage on the matrix cores: lanes as zj_tri_frag.hpp has them (a wave
// owns G groups of four elements, one point row per lane), one lane per point
// for the Euler fluxes and one per solved face point for the common fluxes,
// through LDS; loads carry no branches.  Bounded by LDS latency and VALU
// issue, then memory.  500,000 elements, P3, HLLC, us a stage, one lane per
// element and variable with scalar operands -> this: FP64
// 214 / 260 / 264 -> 225 / 232 / 238, FP32 123 / 162 / 167 -> 127 / 150 / 155;
// on 7,200, whose tiles of 64 left half the CUs idle, 17 -> 7.8 and 14 -> 6.2.
template <typename R, int P> struct TriTile {
    static constexpr int NP = (P + 1) * (P + 2) / 2, NFP = 3 * (P + 1);
    static constexpr int PB = (NP + 3) / 4, FB = (NFP + 3) / 4, CB = (2 * NP + 3) / 4;
    static constexpr bool BIG = sizeof(R) == 8 && P == 5;
    static constexpr int G = BIG ? 1 : 2, WV = BIG ? 8 : 4, value = 4 * G * WV, WPE = sizeof(R) == 8 && P >= 4 ? 2 : 3;
    // P1 and P2 meshes of at least SCALAR_FROM elements take the scalar form.  So do P2 meshes from HALF_FROM to
    // HALF_TO elements where it gives the busiest of the 256 CUs half as many of its tiles of 64 as the matrix-core
    // form gives of 32: only a last round of fewer makes the latter the quicker there.  us a step, scalar / matrix
    // cores: FP64 26,912 elements 45.5 / 46.2 (2 against 4 tiles), 39,200 56.4 / 54.6 (3, 5), 43,808 57.9 / 61.8
    // (3, 6), 49,928 76.8 / 69.0 (4, 7), 60,552 81.3 / 76.6 (4, 8); FP32 39,200 41.7 / 37.9, 43,808 42.8 / 44.5,
    // 52,488 48.7 / 49.1, 60,552 50.5 / 52.9
    static constexpr int SCALAR_FROM = P == 1 ? 24576 : (P == 2 ? 65536 : INT_MAX);
    static constexpr int HALF_FROM = P == 2 ? (sizeof(R) == 8 ? 24576 : 40960) : INT_MAX;
    static constexpr int HALF_TO = sizeof(R) == 8 ? 49152 : SCALAR_FROM;
    static constexpr int per_cu(int E, int t) { return ((E + t - 1) / t + 255) / 256; }
    static constexpr bool scalar(int E) {
        return E >= SCALAR_FROM || (E >= HALF_FROM && E <= HALF_TO && 2 * per_cu(E, TILE) <= per_cu(E, value));
    }
    static constexpr int tile(int E) { return scalar(E) ? TILE : value; }
    // A residual alone reads no U^n, which is what the scalar form's FP64 stages 2 and 3 wait for: large meshes
    // take it for that (its tiles of 64 are whole tiles of the other's, so the traces it needs are there).  us, with
    // the conversion of the result, scalar / matrix cores: P1 FP32 20,000 elements 9.5 / 10.0; P2 FP64 60,552
    // 27.7 / 30.6, FP32 52,488 21.1 / 22.4; P3 FP32 500,000 166 / 175, 180,000 64 / 63; P5 FP64 500,000 635 / 722
    // (572 in builds whose operator table falls well into the scalar cache), 180,000 248 / 267, 80,000 115 / 115; P5 FP32 500,000 380 / 410, 259,200 221 / 224; P4 500,000 434 / 424
    static constexpr int RESIDUAL_FROM =
        P == 1 ? 16384 : P == 2 ? HALF_FROM : P == 3 ? 200000 : P == 5 ? (sizeof(R) == 8 ? 100000 : 200000) : INT_MAX;
    static constexpr bool scalar_residual(int E) { return scalar(E) || E >= RESIDUAL_FROM; }
    static constexpr int residual_tile(int E) { return scalar_residual(E) ? TILE : value; }
    // rows of an element: traces of U; then U, later F_r, and F_s, later the common fluxes and the
    // other tiles' traces
    static constexpr int RU = 4 * FB, RO = RU + NFP;
    static constexpr int ROWS = RU + 4 * CB > RO + 4 * FB ? RU + 4 * CB : RO + 4 * FB;
    static constexpr int ESX = tri::elem_stride<R>(ROWS);
};

template <typename R, int P, int MODE>
__global__ __launch_bounds__((64 * TriTile<R, P>::WV), (TriTile<R, P>::WPE)) void tri_stage_kernel(TriArgs<R> a) {
    using TV = TriTile<R, P>;
    using FO = tri::FragOps<R, P>;
    constexpr int NP = FO::NP, FP = FO::FP, NFP = FO::NFP, PB = FO::PB, FB = FO::FB, CB = FO::CB;
    constexpr int G = TV::G, NWV = TV::WV, NB = 64 * NWV, TT = TV::value, ESX = TV::ESX, RU = TV::RU, RO = TV::RO;
    constexpr int OI = 0, OF = tri::FragTab<R, FB, PB>::WORDS, OL = OF + tri::FragTab<R, PB + FB, CB>::WORDS, OW = OL + tri::FragTab<R, PB, FB>::WORDS;
    __shared__ R ops[OW];            // the operator tables I, F, L
    __shared__ R sX[TT * ESX];
    __shared__ double sred[NWV];
    __shared__ R sGeo[TT * 4];       // r_x, r_y, s_x, s_y
    __shared__ R sNs[TT * 3 * 4];    // per edge: face normal, own factor +-|e|/(2J), the partner's -+|e|/(2J)
    __shared__ int4 sPa[TT * 3];     // per edge: partner's element and slot P of its edge in the tile (the edge's own
                                     // else); 0 in the tile, 1 across tiles, 2 boundary; then the row of slot P in
                                     // the trace array, or BC type and data index
    __shared__ unsigned char sList[TT * 3];
    __shared__ int sCnt[NWV];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int row = lane >> 4, v = lane & 3;
    const int tile = tile_of_block(a.xcd_groups);
    const int e0 = tile * TT;
    const R g = R(a.gamma);
    auto elg = [&](int q) { return (wave * G + q) * 4 + ((lane >> 2) & 3); };  // this lane's element of group q
    auto sx_ = [](int elx, int r) { return elx * ESX + r * NV; };

    const PointRows<NP, G> rows(e0, wave, lane, a.E);

    // ---- 0: state, operators, edges
    double u[G][PB];
    R ur[G][PB];
#pragma unroll
    for (int q = 0; q < G; ++q)
#pragma unroll
        for (int b = 0; b < PB; ++b) u[q][b] = *rows.at(a.U_in, q, b);
    {
        const R* const src = frag_ops<R>() + tri::frag_offset<R>(P);
        for (int t = 4 * tid; t < OW; t += 4 * NB) {
            R w[4];
            load4(src + (t < OF ? FO::I + t : t < OL ? FO::F + t - OF : FO::COMMON + a.family * FO::FAMILY + t - OL), w);
            store4(ops + t, w);
        }
    }
    static_assert(TT * 3 <= NB, "one lane per edge of the tile");
    bool owned = false;
    if (tid < TT * 3) {
        const int el = tid / 3, k = tid - el * 3, e = min(e0 + el, a.E - 1);
        const R* Ge = a.geo + (int64_t)e * GEO;
        const int2 Lk = a.links[(int64_t)e * 3 + k];
        const int nl = Lk.x - e0, ek = link_edge(Lk.y), role = link_role(Lk.y);
        const bool right = role == ROLE_RIGHT, live = e0 + el < a.E, bnd = role == ROLE_BOUNDARY;
        const bool in = !bnd && nl >= 0 && nl < TT;
        const R s = a.edge[(int64_t)e * EDG + 2 * k], sn = a.edge[(int64_t)e * EDG + 2 * k + 1], nx = Ge[4 + 2 * k], ny = Ge[5 + 2 * k];
        const R ns[4] = {nx, ny, right ? -s : s, right ? sn : -sn};
        store4(sNs + 4 * tid, ns);
        const bool self = !live || !in;
        sPa[tid] = make_int4(self ? el : nl, (self ? k : ek) * FP + P, !live || in ? 0 : (bnd ? 2 : 1),
                             !live || in ? P : (bnd ? ek | link_bc(Lk.y) << 3 : (int)((unsigned)Lk.x * NFP + ek * FP + P)));
        owned = live && !(right && in);
    }
    if (tid < TT) {
        const R* Ge = a.geo + (int64_t)min(e0 + tid, a.E - 1) * GEO;
        const R w[4] = {Ge[0], Ge[1], Ge[2], Ge[3]};
        store4(sGeo + 4 * tid, w);
    }
    const unsigned long long own_mask = __ballot(owned);
    if (lane == 0) sCnt[wave] = __popcll(own_mask);
#pragma unroll
    for (int q = 0; q < G; ++q)
#pragma unroll
        for (int b = 0; b < PB; ++b) {
            ur[q][b] = 4 * b + row < NP ? R(u[q][b]) : R(0);
            sX[sx_(elg(q), RU + 4 * b + row) + v] = ur[q][b];
        }
    __syncthreads();  // operators and edges in place

    // ---- 1: the other tiles' traces on their way, own traces, contravariant
    // fluxes (one lane per point of the wave's elements, in place of U)
    R oth[G][FB];
    unsigned cross = 0;  // one bit per slot: an edge another tile reads
#pragma unroll
    for (int q = 0; q < G; ++q)
#pragma unroll
        for (int b = 0; b < FB; ++b) {
            const int j = min(4 * b + row, NFP - 1);
            const int4 pa = sPa[elg(q) * 3 + j / FP];
            cross |= (unsigned)(pa.z == 1 && 4 * b + row < NFP) << (q * FB + b);
            oth[q][b] = a.T_in[(pa.z == 1 ? (int64_t)(unsigned)pa.w - j % FP : (int64_t)0) * NV + v];
        }
    {
        R tu[G][FB];
        tri::frag_mma<true, R, G, FB, PB>(ops + OI, ur, tu);
#pragma unroll
        for (int q = 0; q < G; ++q)
#pragma unroll
            for (int b = 0; b < FB; ++b) sX[sx_(elg(q), 4 * b + row) + v] = tu[q][b];
    }
    if (owned) {
        int pos = __popcll(own_mask & ((1ull << lane) - 1));
        for (int w = 0; w < wave; ++w) pos += sCnt[w];
        sList[pos] = (unsigned char)tid;
    }
    tri::wave_lds_fence();
#pragma unroll 1
    for (int t = lane; t < 4 * G * NP; t += 64) {
        const int el = wave * 4 * G + t / NP, m = t % NP;
        R U4[NV], FR[NV], FS[NV], ge[4];
        load4(sX + sx_(el, RU + m), U4);
        load4(sGeo + 4 * el, ge);
        const R inv = fast_rcp(U4[0]);
        const R ux = U4[1] * inv, uy = U4[2] * inv;
        const R p = (g - R(1)) * (U4[3] - R(0.5) * (U4[1] * ux + U4[2] * uy));
        const R fx[NV] = {U4[1], U4[1] * ux + p, U4[1] * uy, (U4[3] + p) * ux};
        const R fy[NV] = {U4[2], U4[2] * ux, U4[2] * uy + p, (U4[3] + p) * uy};
#pragma unroll
        for (int w = 0; w < NV; ++w) {
            FR[w] = ge[0] * fx[w] + ge[1] * fy[w];
            FS[w] = ge[2] * fx[w] + ge[3] * fy[w];
        }
        store4(sX + sx_(el, RU + m), FR);
        store4(sX + sx_(el, RU + NP + m), FS);
    }
    tri::wave_lds_fence();

    // ---- 2: divergence and transformed normal fluxes
    R dv[G][PB + FB];
    {
        R f[G][CB];
#pragma unroll
        for (int q = 0; q < G; ++q)
#pragma unroll
            for (int b = 0; b < CB; ++b) {
                const R w = sX[sx_(elg(q), RU + 4 * b + row) + v];
                f[q][b] = 4 * b + row < 2 * NP ? w : R(0);
            }
        tri::frag_mma<true, R, G, PB + FB, CB>(ops + OF, f, dv);
    }
    tri::wave_lds_fence();  // every read of the point fluxes done
#pragma unroll
    for (int q = 0; q < G; ++q)
#pragma unroll
        for (int b = 0; b < FB; ++b) sX[sx_(elg(q), RO + 4 * b + row) + v] = oth[q][b];
    double u0[G][PB];
    if (MODE == MODE_STAGE2 || MODE == MODE_STAGE3) {
#pragma unroll
        for (int q = 0; q < G; ++q)
#pragma unroll
            for (int b = 0; b < PB; ++b) u0[q][b] = *rows.at(a.U0, q, b);
    }
    __syncthreads();
    int nsolved = 0;
#pragma unroll
    for (int w = 0; w < NWV; ++w) nsolved += sCnt[w];

    // ---- 3: common fluxes of the solved face points, scaled by each side's
    // +-|e|/(2J), at both sides' slots (an in-tile face by its left element;
    // without a partner in the tile both are the edge's own, written last)
#pragma unroll 1
    for (int t = tid; t < nsolved * FP; t += NB) {
        const int c = sList[t / FP], f = t - (t / FP) * FP;
        const int el = c / 3, j = (c - el * 3) * FP + f;
        const int4 pc = sPa[c];
        R own[NV], ot[NV], ns[4], UL[NV], UR[NV], Fc[NV], d[NV], dn[NV];
        load4(sX + sx_(el, j), own);
        load4(sX + (pc.z == 0 ? sx_(pc.x, pc.y - f) : sx_(el, RO + j)), ot);
        load4(sNs + 4 * c, ns);
        if (pc.z == 2) ghost_state(own, ns[0], ns[1], pc.w & 7, a.bc_data + (int64_t)(pc.w >> 3) * 8, g, ot);
        const bool right = ns[2] < R(0);
#pragma unroll
        for (int w = 0; w < NV; ++w) {
            UL[w] = right ? ot[w] : own[w];
            UR[w] = right ? own[w] : ot[w];
        }
        riemann_by_kind(a.riemann, UL, UR, ns[0], ns[1], g, Fc);
#pragma unroll
        for (int w = 0; w < NV; ++w) {
            d[w] = ns[2] * Fc[w];
            dn[w] = ns[3] * Fc[w];
        }
        store4(sX + (pc.z == 0 ? sx_(pc.x, RU + pc.y - f) : sx_(el, RU + j)), dn);
        tri::wave_lds_fence();
        store4(sX + sx_(el, RU + j), d);
    }
    __syncthreads();

    // ---- 4: lifted flux differences, RK stage update
    {
        R d[G][FB], div[G][PB];
#pragma unroll
        for (int q = 0; q < G; ++q) {
#pragma unroll
            for (int b = 0; b < FB; ++b) {
                const R w = sX[sx_(elg(q), RU + 4 * b + row) + v];
                d[q][b] = 4 * b + row < NFP ? w - dv[q][PB + b] : R(0);
            }
#pragma unroll
            for (int b = 0; b < PB; ++b) div[q][b] = dv[q][b];
        }
        tri::frag_mma<false, R, G, PB, FB>(ops + OL, d, div);
        const double dt = MODE == MODE_RESIDUAL ? 0.0 : *a.dt_ptr;
        double l2 = 0.0;
#pragma unroll
        for (int q = 0; q < G; ++q) {
            const int e = e0 + elg(q);
#pragma unroll
            for (int b = 0; b < PB; ++b) {
                const int i = 4 * b + row;
                const bool ok = i < NP && e < a.E;
                const double res = -double(div[q][b]);
                double un = res;
                if (MODE == MODE_STAGE1) un = u[q][b] + dt * res;
                if (MODE == MODE_STAGE2) un = 0.75 * u0[q][b] + 0.25 * (u[q][b] + dt * res);
                if (MODE == MODE_STAGE3) un = (1.0 / 3.0) * u0[q][b] + (2.0 / 3.0) * (u[q][b] + dt * res);
                if (ok) *rows.at(MODE == MODE_RESIDUAL ? a.R_out : a.U_out, q, b) = un;
                if (MODE == MODE_RESIDUAL || MODE == MODE_STAGE3) l2 += ok ? res * res : 0.0;
                ur[q][b] = i < NP ? R(un) : R(0);
            }
        }
        if ((MODE == MODE_RESIDUAL || MODE == MODE_STAGE3) && a.l2_partial) {
            const double s2 = block_reduce_n<OpSum, NWV>(l2, sred);
            if (tid == 0) a.l2_partial[tile] = s2;
        }
    }
    if (MODE == MODE_RESIDUAL) return;

    // ---- 5: traces of the new stage state on edges another tile reads
    R tn[G][FB];
    tri::frag_mma<true, R, G, FB, PB>(ops + OI, ur, tn);
#pragma unroll
    for (int q = 0; q < G; ++q)
#pragma unroll
        for (int b = 0; b < FB; ++b)
            if (cross >> (q * FB + b) & 1) a.T_out[trix(e0 + elg(q), 4 * b + row, NFP) + v] = tn[q][b];
}

// ------------------------------------------------------------ Navier-Stokes terms
// The stage with the compressible Navier-Stokes viscous terms, BR2 (textbook
// scheme; Bassi-Rebay 2 on the triangle's FR correction field), periodic
// meshes:
//   U^C = (U_own + U_nbr)/2 at every face point, jump U^C - U_own
//   Q = grad U + sum_j lift[:, j] s_j n_j (U^C - U_own)_j   (corrected gradient)
//   F = F_inv(U) - F_v(U, Q) at the points (F_v: ViscousFlux, mu = 1/Re)
//   F^I = Riemann(U_L, U_R) - F_v(U^C, Qbar) . n, Qbar the mean of both sides'
//       trace of grad U plus eta times the lifting of this face's jumps
//       alone at the face's points (LF_k = interp . lift of edge k)
//   dU/dt = -(Dr Fr + Ds Fs) - sum_j lift[:, j] (s_j F^I_j - Fn_j)
// Lanes as zj_tri_frag.hpp has them: a wave owns G groups of four elements,
// lane l holds row 4 b + l/16 (solution or flux point) of element (l/4) mod 4,
// variable l mod 4.  The operators are matrix-core products over such
// fragments; what needs the four variables of a point together (the fluxes)
// takes one lane per point or face point through LDS.  Traces across tiles
// carry 12 words per flux point ([E][3(p+1)][12]: U, dU/dx, dU/dy).
//
// What bounds it is the latency of LDS and memory at two (FP64) or three
// (FP32 P2, P3) waves per SIMD, then VALU issue (about 1,400 instructions per wave of
// eight elements) beside 4,400 (FP64) cycles of matrix-core work.  Hence no
// branches around loads (rows in excess, in-tile edges and elements beyond
// the mesh read a valid address and select afterwards: branches had split
// the LDS reads into some 60 waits a wave), the operator tables in LDS (read
// from memory they took a quarter of the kernel's time), the neighbours'
// traces fetched a phase ahead, and two element groups per wave per operator
// word.  500,000 elements, P3, HLLC, us a stage, scalar operands and one lane
// per element and variable -> this: FP64 670 / 771 / 771 -> 430, FP32
// 354 / 390 / 384 -> 241 / 272 / 277 (1.9 TB/s of the stage's traffic).
constexpr int TWV = 12;

// The workgroup: WV waves of G groups each, 4 G WV elements.
// LDS per element: the traces of U, then one region that holds U with the
// corrected gradient, the point fluxes in its place, and at last both traces
// of the BR2 gradient, whose x part the face fluxes replace.
template <typename R, int P> struct TriViscTile {
    static constexpr int NP = (P + 1) * (P + 2) / 2, NFP = 3 * (P + 1), PB = (NP + 3) / 4, FB = (NFP + 3) / 4;
    static constexpr bool BIG = sizeof(R) == 8 && P == 5;
    static constexpr int G = BIG ? 1 : 2, WV = BIG ? 8 : 4;
    static constexpr int value = 4 * G * WV;
    // P1 and FP32 P2 meshes of at least this many elements take the scalar form, in tiles of 64 (FP64 P1: two
    // workgroups fit on a CU, so at 32 elements each the 256 CUs hold 16,384 elements at a time)
    static constexpr int SCALAR_FROM = P == 1 ? (sizeof(R) == 8 ? 16384 : 24576) : (P == 2 && sizeof(R) == 4 ? 32768 : INT_MAX);
    static constexpr int tile(int E) { return E >= SCALAR_FROM ? TILE : value; }
    // rows of an element's region: Q_x, then F_r, at 0; Q_y, then F_s, at NP; U at RU; then the
    // gradient traces x (later the common fluxes) at 0 and y at NFP, the partner's U traces at
    // 2 NFP.  Arrays are stored whole blocks of four rows at a time, in the order of their rows,
    // so that the next array overwrites the rows in excess.
    static constexpr int RU = NP + 4 * PB;
    static constexpr int ROWS = RU + 4 * PB > 2 * NFP + 4 * FB ? RU + 4 * PB : 2 * NFP + 4 * FB;
    static constexpr int ESF = tri::elem_stride<R>(4 * FB), ESX = tri::elem_stride<R>(ROWS);
    static_assert(value * (ESF + ESX) * (int)sizeof(R) <= 122880, "the tile exceeds the LDS");
};

template <typename R, int P, int MODE>
__global__ __launch_bounds__((64 * TriViscTile<R, P>::WV), 2) void tri_visc_stage_kernel(TriArgs<R> a) {
    using S = TriShape<P>;
    using TV = TriViscTile<R, P>;
    using FO = tri::FragOps<R, P>;
    constexpr int NP = S::NP, FP = S::FP, NFP = S::NFP, PB = FO::PB, FB = FO::FB, CB = FO::CB;
    constexpr int G = TV::G, NWV = TV::WV, NB = 64 * NWV, TT = TV::value, ESF = TV::ESF, ESX = TV::ESX;
    constexpr int RU = TV::RU, RY = NFP, RO = 2 * NFP;  // rows of U, the y gradient traces, the partner's U traces
    __shared__ R ops[FO::COMMON + FO::FAMILY];  // the operator tables
    const R* const fam = ops + FO::COMMON;
    __shared__ R sTu[TT * ESF];      // traces of U
    __shared__ R sX[TT * ESX];
    __shared__ double sred[NWV];
    __shared__ R sGeo[TT * 4];       // r_x, r_y, s_x, s_y
    __shared__ R sEw[TT * 3 * 4];    // per edge: jump weights x, y (outward normal times |e|/(2J)), the partner's
                                     // weights of its face lifting x, y
    __shared__ R sNs[TT * 3 * 4];    // per edge: face normal, own factor +-|e|/(2J), the partner's -+|e|/(2J)
    __shared__ int4 sPa[TT * 3];     // per edge, where its partner's slots are (point f faces slot P - f): element
                                     // and slot P of its edge in the tile (the edge's own if across tiles), the
                                     // partner's edge if across tiles (else 3), the row of slot P in the trace array
    __shared__ unsigned char sList[TT * 3];
    __shared__ int sCnt[NWV];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int row = lane >> 4, v = lane & 3;
    const int tile = tile_of_block(a.xcd_groups);
    const int e0 = tile * TT;
    const R g = R(a.gamma), mu = R(a.mu), kappa = R(a.kappa), eta = R(a.eta);
    auto elg = [&](int q) { return (wave * G + q) * 4 + ((lane >> 2) & 3); };  // this lane's element of group q
    auto st = [](int elx, int j) { return elx * ESF + j * NV; };                 // trace slots
    auto sx_ = [](int elx, int r) { return elx * ESX + r * NV; };              // rows of the other region

    const PointRows<NP, G> rows(e0, wave, lane, a.E);

    // ---- 0: state, gradient, traces of U
    double u[G][PB];
    R ur[G][PB];
#pragma unroll
    for (int q = 0; q < G; ++q)
#pragma unroll
        for (int b = 0; b < PB; ++b) u[q][b] = *rows.at(a.U_in, q, b);
    {
        const R* const src = frag_ops<R>() + tri::frag_offset<R>(P);
        for (int t = 4 * tid; t < FO::COMMON + FO::FAMILY; t += 4 * NB) {
            R w[4];
            load4(src + (t < FO::COMMON ? t : t + a.family * FO::FAMILY), w);
            store4(ops + t, w);
        }
    }
    // one lane per edge of the tile; an in-tile face is solved by its left element only
    static_assert(TT * 3 <= NB, "one lane per edge of the tile");
    bool owned = false;
    if (tid < TT * 3) {
        const int el = tid / 3, k = tid - el * 3, e = min(e0 + el, a.E - 1);
        const R* Ge = a.geo + (int64_t)e * GEO;
        const int2 Lk = a.links[(int64_t)e * 3 + k];
        const int nl = Lk.x - e0, ek = link_edge(Lk.y);
        const bool right = link_role(Lk.y) == ROLE_RIGHT, live = e0 + el < a.E;
        const bool in = !live || (nl >= 0 && nl < TT);  // beyond the mesh: its own neighbour
        const R s = a.edge[(int64_t)e * EDG + 2 * k], sn = a.edge[(int64_t)e * EDG + 2 * k + 1], nx = Ge[4 + 2 * k], ny = Ge[5 + 2 * k];
        const R w = right ? -s : s, wn = right ? -eta * sn : eta * sn;
        const R we[4] = {w * nx, w * ny, wn * nx, wn * ny}, ns[4] = {nx, ny, w, right ? sn : -sn};
        store4(sEw + 4 * tid, we);
        store4(sNs + 4 * tid, ns);
        const bool self = !live || !in;
        sPa[tid] = make_int4(self ? el : nl, (self ? k : ek) * FP + P, in ? 3 : ek,
                             in ? P : (int)((unsigned)Lk.x * NFP + ek * FP + P));  // row < 2^32
        owned = live && !(right && in);
    }
    if (tid < TT) {
        const R* Ge = a.geo + (int64_t)min(e0 + tid, a.E - 1) * GEO;
        const R w[4] = {Ge[0], Ge[1], Ge[2], Ge[3]};
        store4(sGeo + 4 * tid, w);
    }
    const unsigned long long own_mask = __ballot(owned);
    if (lane == 0) sCnt[wave] = __popcll(own_mask);
#pragma unroll
    for (int q = 0; q < G; ++q)
#pragma unroll
        for (int b = 0; b < PB; ++b) {
            ur[q][b] = 4 * b + row < NP ? R(u[q][b]) : R(0);
            sX[sx_(elg(q), RU + 4 * b + row) + v] = ur[q][b];
        }
    __syncthreads();  // operators and edges in place
    // the neighbours' U traces across tiles (lanes of in-tile edges read one line in common)
    auto partner = [&](int q, int b) { return sPa[elg(q) * 3 + min(4 * b + row, NFP - 1) / FP]; };
    auto remote = [&](int w, int b) { return ((int64_t)(unsigned)w - min(4 * b + row, NFP - 1) % FP) * TWV + v; };
    R oth[G][FB];
    unsigned edges = 0;  // two bits per slot: the partner's edge, 3 in the tile
#pragma unroll
    for (int q = 0; q < G; ++q)
#pragma unroll
        for (int b = 0; b < FB; ++b) {
            const int4 pa = partner(q, b);
            edges |= (unsigned)pa.z << 2 * (q * FB + b);
            oth[q][b] = a.T_in[remote(pa.w, b)];
        }
    auto edge_of = [&](int q, int b) { return (int)(edges >> 2 * (q * FB + b)) & 3; };
    static_assert(G * FB <= 16, "two bits per slot");
    R tu[G][FB], gd[G][2 * PB];
    tri::frag_mma<true, R, G, FB, PB>(ops + FO::I, ur, tu);
#pragma unroll
    for (int q = 0; q < G; ++q)
#pragma unroll
        for (int b = 0; b < FB; ++b) sTu[st(elg(q), 4 * b + row) + v] = tu[q][b];
    tri::frag_mma<true, R, G, 2 * PB, PB>(ops + FO::D, ur, gd);
    if (owned) {
        int pos = __popcll(own_mask & ((1ull << lane) - 1));
        for (int w = 0; w < wave; ++w) pos += sCnt[w];
        sList[pos] = (unsigned char)tid;
    }
    __syncthreads();

    // ---- 1: jumps, corrected gradient (the jumps' lifting along the outward normals)
    R jmp[G][FB];
    {
        R jw[2 * G][FB], Q[2 * G][PB], ti[G][FB];
#pragma unroll
        for (int q = 0; q < G; ++q)
#pragma unroll
            for (int b = 0; b < FB; ++b) {
                const int4 pa = partner(q, b);
                ti[q][b] = sTu[st(pa.x, pa.y - min(4 * b + row, NFP - 1) % FP) + v];
            }
#pragma unroll
        for (int q = 0; q < G; ++q) {
            R ge[4];
            load4(sGeo + 4 * elg(q), ge);
#pragma unroll
            for (int b = 0; b < PB; ++b) {
                Q[2 * q][b] = ge[0] * gd[q][b] + ge[2] * gd[q][PB + b];
                Q[2 * q + 1][b] = ge[1] * gd[q][b] + ge[3] * gd[q][PB + b];
            }
#pragma unroll
            for (int b = 0; b < FB; ++b) {
                const int j = 4 * b + row;
                const R* w = sEw + 4 * (elg(q) * 3 + min(j, NFP - 1) / FP);
                oth[q][b] = edge_of(q, b) == 3 ? ti[q][b] : oth[q][b];
                const R d = R(0.5) * (tu[q][b] + oth[q][b]) - tu[q][b];
                jmp[q][b] = j < NFP ? d : R(0);
                jw[2 * q][b] = w[0] * jmp[q][b];
                jw[2 * q + 1][b] = w[1] * jmp[q][b];
            }
        }
        tri::frag_mma<false, R, 2 * G, PB, FB>(fam + FO::L, jw, Q);
#pragma unroll
        for (int q = 0; q < G; ++q)
#pragma unroll
            for (int b = 0; b < PB; ++b) sX[sx_(elg(q), 4 * b + row) + v] = Q[2 * q][b];
        tri::wave_lds_fence();
#pragma unroll
        for (int q = 0; q < G; ++q)
#pragma unroll
            for (int b = 0; b < PB; ++b) sX[sx_(elg(q), NP + 4 * b + row) + v] = Q[2 * q + 1][b];
    }
    tri::wave_lds_fence();  // U and Q of the wave's elements in place

    // ---- 2: contravariant total fluxes, one lane per point of the wave's
    // elements, in place of Q; the partner's gradient traces on their way
    R ox[G][FB], oy[G][FB];
#pragma unroll
    for (int q = 0; q < G; ++q)
#pragma unroll
        for (int b = 0; b < FB; ++b) {
            const R* T = a.T_in + remote(partner(q, b).w, b);
            ox[q][b] = T[NV];
            oy[q][b] = T[2 * NV];
        }
#pragma unroll 1
    for (int t = lane; t < 4 * G * NP; t += 64) {
        const int el = wave * 4 * G + t / NP, m = t % NP;
        R U4[NV], X4[NV], Y4[NV], FR[NV], FS[NV], Fv[NV], Gv[NV], ge[4];
        load4(sX + sx_(el, RU + m), U4);
        load4(sX + sx_(el, m), X4);
        load4(sX + sx_(el, NP + m), Y4);
        load4(sGeo + 4 * el, ge);
        const R inv = fast_rcp(U4[0]);
        const R ux = U4[1] * inv, uy = U4[2] * inv;
        const R p = (g - R(1)) * (U4[3] - R(0.5) * (U4[1] * ux + U4[2] * uy));
        visc_flux(U4, X4, Y4, g, mu, kappa, Fv, Gv);
        const R fx[NV] = {U4[1], U4[1] * ux + p, U4[1] * uy, (U4[3] + p) * ux};
        const R fy[NV] = {U4[2], U4[2] * ux, U4[2] * uy + p, (U4[3] + p) * uy};
#pragma unroll
        for (int w = 0; w < NV; ++w) {
            const R Fx = fx[w] - Fv[w], Fy = fy[w] - Gv[w];
            FR[w] = ge[0] * Fx + ge[1] * Fy;
            FS[w] = ge[2] * Fx + ge[3] * Fy;
        }
        store4(sX + sx_(el, m), FR);
        store4(sX + sx_(el, NP + m), FS);
    }
    tri::wave_lds_fence();

    // ---- 3: divergence and transformed normal fluxes; then the traces of
    // the gradient plus the BR2 lifting of each edge's own jumps (across
    // tiles the mean of both sides), in place of the point values
    R dv[G][PB + FB];
    {
        R f[G][CB];
#pragma unroll
        for (int q = 0; q < G; ++q)
#pragma unroll
            for (int b = 0; b < CB; ++b) {
                const R w = sX[sx_(elg(q), 4 * b + row) + v];
                f[q][b] = 4 * b + row < 2 * NP ? w : R(0);
            }
        tri::frag_mma<true, R, G, PB + FB, CB>(ops + FO::F, f, dv);
    }
    tri::wave_lds_fence();  // every read of the point fluxes done
    {
        R tg[G][2 * FB], lo[G][4][FB], gyv[G][FB];
        tri::frag_mma<true, R, G, 2 * FB, PB>(ops + FO::G, ur, tg);
        tri::diag_mma<R, P>(fam + FO::LF, jmp, lo);
#pragma unroll
        for (int q = 0; q < G; ++q) {
            const int el = elg(q);
            R ge[4];
            load4(sGeo + 4 * el, ge);
#pragma unroll
            for (int b = 0; b < FB; ++b) {
                const int j = 4 * b + row, ek = edge_of(q, b);
                R w[4];
                load4(sEw + 4 * (el * 3 + min(j, NFP - 1) / FP), w);
                const R own = eta * lo[q][0][b];
                R gx = ge[0] * tg[q][b] + ge[2] * tg[q][FB + b] + w[0] * own;
                R gy = ge[1] * tg[q][b] + ge[3] * tg[q][FB + b] + w[1] * own;
                // the partner's jumps and outward normal are minus this side's
                const R ln = ek == 0 ? lo[q][1][b] : (ek == 1 ? lo[q][2][b] : lo[q][3][b]);
                gx = ek == 3 ? gx : R(0.5) * (gx + (ox[q][b] + w[2] * ln));
                gy = ek == 3 ? gy : R(0.5) * (gy + (oy[q][b] + w[3] * ln));
                sX[sx_(el, j) + v] = gx;
                gyv[q][b] = gy;
            }
        }
        tri::wave_lds_fence();
#pragma unroll
        for (int q = 0; q < G; ++q)
#pragma unroll
            for (int b = 0; b < FB; ++b) sX[sx_(elg(q), RY + 4 * b + row) + v] = gyv[q][b];
        tri::wave_lds_fence();
#pragma unroll
        for (int q = 0; q < G; ++q)
#pragma unroll
            for (int b = 0; b < FB; ++b) sX[sx_(elg(q), RO + 4 * b + row) + v] = oth[q][b];
    }
    double u0[G][PB];
    if (MODE == MODE_STAGE2 || MODE == MODE_STAGE3) {
#pragma unroll
        for (int q = 0; q < G; ++q)
#pragma unroll
            for (int b = 0; b < PB; ++b) u0[q][b] = *rows.at(a.U0, q, b);
    }
    __syncthreads();
    int nsolved = 0;
#pragma unroll
    for (int w = 0; w < NWV; ++w) nsolved += sCnt[w];

    // ---- 4: common fluxes of the solved face points, scaled by each side's
    // +-|e|/(2J): Riemann minus the BR2 viscous flux, in place of both sides'
    // x gradient traces (each slot's is read by the lane that solves it
    // alone).  Across tiles the partner's slot is the edge's own, which holds
    // the mean, and whose flux is written last.
#pragma unroll 1
    for (int t = tid; t < nsolved * FP; t += NB) {
        const int c = sList[t / FP], f = t - (t / FP) * FP;
        const int el = c / 3, j = (c - el * 3) * FP + f;
        const int4 pc = sPa[c];
        const int so = sx_(el, j), sn = pc.z == 3 ? sx_(pc.x, pc.y - f) : so;
        R own[NV], ot[NV], ns[4], Qbx[NV], Qby[NV], gx[NV], gy[NV];
        load4(sTu + st(el, j), own);
        load4(sX + sx_(el, RO + j), ot);
        load4(sNs + 4 * c, ns);
        load4(sX + so, Qbx);
        load4(sX + sn, gx);
        load4(sX + so + RY * NV, Qby);
        load4(sX + sn + RY * NV, gy);
        const bool right = ns[2] < R(0);
        R Uc[NV], UL[NV], UR[NV], Fc[NV], Fv[NV], Gv[NV];
#pragma unroll
        for (int w = 0; w < NV; ++w) {
            Uc[w] = R(0.5) * (own[w] + ot[w]);
            Qbx[w] = R(0.5) * (Qbx[w] + gx[w]);
            Qby[w] = R(0.5) * (Qby[w] + gy[w]);
            UL[w] = right ? ot[w] : own[w];
            UR[w] = right ? own[w] : ot[w];
        }
        visc_flux(Uc, Qbx, Qby, g, mu, kappa, Fv, Gv);
        riemann_by_kind(a.riemann, UL, UR, ns[0], ns[1], g, Fc);
        R d[NV], dn[NV];
#pragma unroll
        for (int w = 0; w < NV; ++w) {
            Fc[w] -= Fv[w] * ns[0] + Gv[w] * ns[1];
            d[w] = ns[2] * Fc[w];
            dn[w] = ns[3] * Fc[w];
        }
        store4(sX + sn, dn);
        tri::wave_lds_fence();
        store4(sX + so, d);
    }
    __syncthreads();

    // ---- 5: lifted flux differences, RK stage update
    {
        R d[G][FB], div[G][PB];
#pragma unroll
        for (int q = 0; q < G; ++q) {
#pragma unroll
            for (int b = 0; b < FB; ++b) {
                const R w = sX[sx_(elg(q), 4 * b + row) + v];
                d[q][b] = 4 * b + row < NFP ? w - dv[q][PB + b] : R(0);
            }
#pragma unroll
            for (int b = 0; b < PB; ++b) div[q][b] = dv[q][b];
        }
        tri::frag_mma<false, R, G, PB, FB>(fam + FO::L, d, div);
        const double dt = MODE == MODE_RESIDUAL ? 0.0 : *a.dt_ptr;
        double l2 = 0.0;
#pragma unroll
        for (int q = 0; q < G; ++q) {
            const int e = e0 + elg(q);
#pragma unroll
            for (int b = 0; b < PB; ++b) {
                const int i = 4 * b + row;
                const bool ok = i < NP && e < a.E;
                const double res = -double(div[q][b]);
                double un = res;
                if (MODE == MODE_STAGE1) un = u[q][b] + dt * res;
                if (MODE == MODE_STAGE2) un = 0.75 * u0[q][b] + 0.25 * (u[q][b] + dt * res);
                if (MODE == MODE_STAGE3) un = (1.0 / 3.0) * u0[q][b] + (2.0 / 3.0) * (u[q][b] + dt * res);
                if (ok) *rows.at(MODE == MODE_RESIDUAL ? a.R_out : a.U_out, q, b) = un;
                if (MODE == MODE_RESIDUAL || MODE == MODE_STAGE3) l2 += ok ? res * res : 0.0;
                ur[q][b] = i < NP ? R(un) : R(0);
            }
        }
        if ((MODE == MODE_RESIDUAL || MODE == MODE_STAGE3) && a.l2_partial) {
            const double s2 = block_reduce_n<OpSum, NWV>(l2, sred);
            if (tid == 0) a.l2_partial[tile] = s2;
        }
    }
    if (MODE == MODE_RESIDUAL) return;

    // ---- 6: traces of the new stage state and of its gradient on edges
    // another tile reads
    R tn[G][FB], tg[G][2 * FB];
    tri::frag_mma<true, R, G, FB, PB>(ops + FO::I, ur, tn);
    tri::frag_mma<true, R, G, 2 * FB, PB>(ops + FO::G, ur, tg);
#pragma unroll
    for (int q = 0; q < G; ++q) {
        R ge[4];
        load4(sGeo + 4 * elg(q), ge);
#pragma unroll
        for (int b = 0; b < FB; ++b) {
            if (edge_of(q, b) == 3 || 4 * b + row >= NFP) continue;
            R* T = a.T_out + ((int64_t)(e0 + elg(q)) * NFP + 4 * b + row) * TWV + v;
            T[0] = tn[q][b];
            T[NV] = ge[0] * tg[q][b] + ge[2] * tg[q][FB + b];
            T[2 * NV] = ge[1] * tg[q][b] + ge[3] * tg[q][FB + b];
        }
    }
}

// The stage of large meshes at the lowest orders (P1, and P2 in FP32): lanes
// as in tri_scalar_kernel, one per element and variable, the operators as
// scalar operands.  A point has few operator entries there, and padding to
// blocks of four costs the matrix-core form a third of its rows; but its
// tiles of 64 leave a small mesh's CUs idle.  us a stage, this / matrix cores:
// P1 FP64 32,768 elements 13 / 17, 16,200 10.5 / 9.5, 7,200 10 / 7; P1 FP32
// 80,000 20 / 22, 16,200 9 / 7; P2 FP32 80,000 36 / 37, 32,768 16.7 / 17.1,
// 16,200 14 / 10 (P2 FP64 80,000 85 / 59).  Whole steps: P1 FP64 24,200
// elements 43 / 47, 20,000 42 / 45.5, 16,200 35 / 32; P1 FP32 24,200 35.4 /
// 32.9, 25,088 35.0 / 35.7, 51,200 44 / 56; P2 FP32 32,768 54.9 / 56.5, 51,200
// 96 / 84, 125,000 164 / 171, 500,000 634 / 623: within 5% on either side
// but for 50,000 to 65,000 elements.  The point values (U, then Q) live in
// LDS, each lane reads a point's four variables there.
template <typename R, int P, int MODE>
__global__ __launch_bounds__(BLOCK) void tri_visc_scalar_kernel(TriArgs<R> a) {
    using S = TriShape<P>;
    constexpr int NP = S::NP, FP = S::FP, NFP = S::NFP;
    constexpr int TT = TILE, NB = BLOCK, NWV = NB / 64;
    static_assert(2 * NP >= NFP, "point-array layout");
    using OP = TriOps<P>;
    constexpr int O0 = ops_offset(P), CA = OP::CA, OI = O0 + OP::C;
    const int OLT = O0 + a.lift_off;
    const int LFO = lf_offset(P) + a.lf_off;
    __shared__ R sTu[TT * NFP * NV], sTx[TT * NFP * NV], sTy[TT * NFP * NV];
    __shared__ R sU[TT * NP * NV];       // the stage input, later the stage output
    __shared__ R sQ[2 * TT * NP * NV];   // Qx, Qy; later the flux differences [TT][NFP][NV]
    __shared__ double sred[NWV];
    __shared__ R sEdge[TT * 3];
    __shared__ int2 sLink[TT * 3];  // the tile's edge links and face normals
    __shared__ R sNrm[TT * 3 * 2];
    __shared__ unsigned char sList[TT * 3];
    __shared__ int sCnt[NWV];
    R* const sQx = sQ;
    R* const sQy = sQ + TT * NP * NV;
    R* const sD = sQ;

    const int tid = threadIdx.x, el = tid >> 2, v = tid & 3;
    const int tile = tile_of_block(a.xcd_groups);
    const int e0 = tile * TT, e = e0 + el;
    const bool live = e < a.E;
    const R g = R(a.gamma), mu = R(a.mu), kappa = R(a.kappa), eta = R(a.eta);
    const int64_t base = blk(e, 0, NP) + v;
    auto sl = [](int elx, int j, int w) { return (elx * NFP + j) * NV + w; };   // trace slots
    auto sp = [](int elx, int m, int w) { return (elx * NP + m) * NV + w; };    // point slots

    // physical gradient of this lane's variable at the points, from sU into gx,
    // gy (every point's sums advance together: 2 NP independent FMA chains)
    auto gradient_of = [&](R rx_, R ry_, R sx_, R sy_, R* gx, R* gy) __attribute__((always_inline)) {
        R gr[NP], gs[NP];
#pragma unroll
        for (int i = 0; i < NP; ++i) { gr[i] = R(0); gs[i] = R(0); }
#pragma unroll
        for (int m = 0; m < NP; ++m) {
            const R um = sU[sp(el, m, v)];
#pragma unroll
            for (int i = 0; i < NP; ++i) {
                gr[i] = fmaR(cop<R>(O0 + m * CA + i), um, gr[i]);
                gs[i] = fmaR(cop<R>(O0 + m * CA + NP + i), um, gs[i]);
            }
        }
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            gx[sp(el, i, v)] = rx_ * gr[i] + sx_ * gs[i];
            gy[sp(el, i, v)] = ry_ * gr[i] + sy_ * gs[i];
        }
    };
    // traces of U, gx, gy (this lane's variable) at the FP points of edge kk
    // (3 FP independent FMA chains), for each through out(j, tu, tx, ty)
    auto edge_traces = [&](int kk, int op_row, const R* gx, const R* gy, auto&& out) __attribute__((always_inline)) {
        R tu[FP], tx[FP], ty[FP];
#pragma unroll
        for (int f = 0; f < FP; ++f) { tu[f] = R(0); tx[f] = R(0); ty[f] = R(0); }
#pragma unroll
        for (int m = 0; m < NP; ++m) {
            const R um = sU[sp(el, m, v)], xm = gx[sp(el, m, v)], ym = gy[sp(el, m, v)];
#pragma unroll
            for (int f = 0; f < FP; ++f) {
                const int j = kk * FP + f;
                const R w = op_row ? cop<R>(OI + j * NP + m) : cop<R>(O0 + m * CA + 2 * NP + j);
                tu[f] = fmaR(w, um, tu[f]);
                tx[f] = fmaR(w, xm, tx[f]);
                ty[f] = fmaR(w, ym, ty[f]);
            }
        }
#pragma unroll
        for (int f = 0; f < FP; ++f) out(kk * FP + f, tu[f], tx[f], ty[f]);
    };

    // ---- 0: state, gradient, traces of U and grad U
    R rx = R(0), ry = R(0), sx = R(0), sy = R(0);
    int2 L[3] = {make_int2(0, 0), make_int2(0, 0), make_int2(0, 0)};
    if (live) {
#pragma unroll
        for (int m = 0; m < NP; ++m) sU[sp(el, m, v)] = R(a.U_in[base + (int64_t)m * EB * NV]);
        const R* G = a.geo + (int64_t)e * GEO;
        rx = G[0]; ry = G[1]; sx = G[2]; sy = G[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) L[k] = a.links[(int64_t)e * 3 + k];
        if (v < 3) {
            const R ax = v == 0 ? sx : (v == 1 ? rx + sx : rx), ay = v == 0 ? sy : (v == 1 ? ry + sy : ry);
            sEdge[el * 3 + v] = sqrtR(ax * ax + ay * ay);
            // the edge's link and normal, for whichever lane solves its face points
            sLink[el * 3 + v] = v == 0 ? L[0] : (v == 1 ? L[1] : L[2]);
            sNrm[(el * 3 + v) * 2] = G[4 + 2 * v];
            sNrm[(el * 3 + v) * 2 + 1] = G[5 + 2 * v];
        }
        gradient_of(rx, ry, sx, sy, sQx, sQy);
#pragma unroll 1
        for (int kk = 0; kk < 3; ++kk)
            edge_traces(kk, 0, sQx, sQy, [&](int j, R tu, R tx, R ty) __attribute__((always_inline)) {
                sTu[sl(el, j, v)] = tu;
                sTx[sl(el, j, v)] = tx;
                sTy[sl(el, j, v)] = ty;
            });
    }
    bool owned = false;
    if (live && v < 3) {
        const int2 Lv = v == 0 ? L[0] : (v == 1 ? L[1] : L[2]);
        const int nl = Lv.x - e0;
        owned = !(link_role(Lv.y) == ROLE_RIGHT && nl >= 0 && nl < TT);
    }
    const unsigned long long own_mask = __ballot(owned);
    const int lane = tid & 63, wave = tid >> 6;
    if (lane == 0) sCnt[wave] = __popcll(own_mask);
    __syncthreads();

    // ---- 1: corrected gradient: the lifted jumps along the outward normals
    if (live) {
        R jwx[NFP], jwy[NFP];
#pragma unroll
        for (int kk = 0; kk < 3; ++kk) {
            const int2 Lk = L[kk];
            const R sg = link_role(Lk.y) == ROLE_RIGHT ? R(-1) : R(1);
            const R s = sEdge[el * 3 + kk];
            const R wx = sg * s * a.geo[(int64_t)e * GEO + 4 + 2 * kk];
            const R wy = sg * s * a.geo[(int64_t)e * GEO + 5 + 2 * kk];
            const int nl = Lk.x - e0;
            const bool in = nl >= 0 && nl < TT;
            const int ek = link_edge(Lk.y);
#pragma unroll
            for (int f = 0; f < FP; ++f) {
                const int j = kk * FP + f, oj = ek * FP + (P - f);
                const R own = sTu[sl(el, j, v)];
                R oth;
                if (in) oth = sTu[sl(nl, oj, v)];
                else oth = a.T_in[((int64_t)Lk.x * NFP + oj) * TWV + v];
                const R jmp = R(0.5) * (own + oth) - own;
                jwx[j] = wx * jmp;
                jwy[j] = wy * jmp;
            }
        }
#pragma unroll 2
        for (int i = 0; i < NP; ++i) {
            R qx = sQx[sp(el, i, v)], qy = sQy[sp(el, i, v)];
#pragma unroll
            for (int j = 0; j < NFP; ++j) {
                const R l = cop<R>(OLT + j * NP + i);
                qx = fmaR(l, jwx[j], qx);
                qy = fmaR(l, jwy[j], qy);
            }
            sQx[sp(el, i, v)] = qx;
            sQy[sp(el, i, v)] = qy;
        }
    }
    if (owned) {
        int pos = __popcll(own_mask & ((1ull << lane) - 1));
        for (int w = 0; w < wave; ++w) pos += sCnt[w];
        sList[pos] = (unsigned char)(el * 3 + v);
    }
    __syncthreads();  // Q of every variable in place

    // ---- 2: total fluxes at the points, each point's four components formed
    // once: this lane takes points v, v + 4, ... of its element and leaves
    // their contravariant fluxes where Q was; then every lane accumulates its
    // own component's divergence and interpolated normal fluxes
    constexpr int MPL = (NP + NV - 1) / NV;  // points per lane
    R FR[MPL][NV], FS[MPL][NV];
    if (live) {
#pragma unroll
        for (int q = 0; q < MPL; ++q) {
            const int m = v + NV * q;
            if (m >= NP) break;
            R U4[NV], X4[NV], Y4[NV];
#pragma unroll
            for (int w = 0; w < NV; ++w) {
                U4[w] = sU[sp(el, m, w)];
                X4[w] = sQx[sp(el, m, w)];
                Y4[w] = sQy[sp(el, m, w)];
            }
            const R inv = fast_rcp(U4[0]);
            const R ux = U4[1] * inv, uy = U4[2] * inv;
            const R p = (g - R(1)) * (U4[3] - R(0.5) * (U4[1] * ux + U4[2] * uy));
            R Fv[NV], Gv[NV];
            visc_flux(U4, X4, Y4, g, mu, kappa, Fv, Gv);
            const R fx[NV] = {U4[1], U4[1] * ux + p, U4[1] * uy, (U4[3] + p) * ux};
            const R fy[NV] = {U4[2], U4[2] * ux, U4[2] * uy + p, (U4[3] + p) * uy};
#pragma unroll
            for (int w = 0; w < NV; ++w) {
                const R Fx = fx[w] - Fv[w], Fy = fy[w] - Gv[w];
                FR[q][w] = rx * Fx + ry * Fy;
                FS[q][w] = sx * Fx + sy * Fy;
            }
        }
    }
    __syncthreads();  // every read of Q done: the contravariant fluxes take its place
    if (live) {
#pragma unroll
        for (int q = 0; q < MPL; ++q) {
            const int m = v + NV * q;
            if (m >= NP) break;
#pragma unroll
            for (int w = 0; w < NV; ++w) {
                sQx[sp(el, m, w)] = FR[q][w];
                sQy[sp(el, m, w)] = FS[q][w];
            }
        }
    }
    __syncthreads();
    R div[NP], fn[NFP];
#pragma unroll
    for (int i = 0; i < NP; ++i) div[i] = R(0);
#pragma unroll
    for (int j = 0; j < NFP; ++j) fn[j] = R(0);
    if (live) {
#pragma unroll 1
        for (int m = 0; m < NP; ++m) {
            const R fr = sQx[sp(el, m, v)], fs = sQy[sp(el, m, v)], frs = fr + fs;
#pragma unroll
            for (int i = 0; i < NP; ++i)
                div[i] = fmaR(cop<R>(O0 + m * CA + NP + i), fs, fmaR(cop<R>(O0 + m * CA + i), fr, div[i]));
#pragma unroll
            for (int j = 0; j < NFP; ++j)
                fn[j] = fmaR(cop<R>(O0 + m * CA + 2 * NP + j), j < FP ? fs : (j < 2 * FP ? frs : fr), fn[j]);
        }
    }
    __syncthreads();  // every read of the point fluxes done: the flux differences take their place
    if (live) {
#pragma unroll
        for (int j = 0; j < NFP; ++j) sD[sl(el, j, v)] = (j >= FP && j < 2 * FP) ? fn[j] : -fn[j];
    }
    __syncthreads();
    int nsolved = 0;
#pragma unroll
    for (int w = 0; w < NWV; ++w) nsolved += sCnt[w];

    // ---- 3: common fluxes of the solved face points: Riemann minus the BR2
    // viscous flux; flux differences of both sides (in-tile partner included)
#pragma unroll 1
    for (int t = tid; t < nsolved * FP; t += NB) {
        const int c = sList[t / FP], f = t - (t / FP) * FP;
        const int elt = c / 3, kk = c - elt * 3, j = kk * FP + f;
        const int2 Lk = sLink[elt * 3 + kk];
        const bool right = link_role(Lk.y) == ROLE_RIGHT;
        const R nx = sNrm[(elt * 3 + kk) * 2];
        const R ny = sNrm[(elt * 3 + kk) * 2 + 1];
        const int ek = link_edge(Lk.y), oj = ek * FP + (P - f);
        const int nl = Lk.x - e0;
        const bool in = nl >= 0 && nl < TT;
        const R* Tn = a.T_in + (int64_t)Lk.x * NFP * TWV;  // the partner's traces (across tiles)
        R own[NV], oth[NV], gxo[NV], gyo[NV], gxn[NV], gyn[NV];
#pragma unroll
        for (int w = 0; w < NV; ++w) {
            own[w] = sTu[sl(elt, j, w)];
            gxo[w] = sTx[sl(elt, j, w)];
            gyo[w] = sTy[sl(elt, j, w)];
        }
        if (in) {
#pragma unroll
            for (int w = 0; w < NV; ++w) {
                oth[w] = sTu[sl(nl, oj, w)];
                gxn[w] = sTx[sl(nl, oj, w)];
                gyn[w] = sTy[sl(nl, oj, w)];
            }
        } else {
            load4(Tn + (int64_t)oj * TWV, oth);
            load4(Tn + (int64_t)oj * TWV + NV, gxn);
            load4(Tn + (int64_t)oj * TWV + 2 * NV, gyn);
        }
        // each side's edge factor |e|/(2J)
        const R so = sEdge[elt * 3 + kk];
        R sn;
        if (in) {
            sn = sEdge[nl * 3 + ek];
        } else {
            const R* Gn = a.geo + (int64_t)Lk.x * GEO;
            const R ax = ek == 0 ? Gn[2] : (ek == 1 ? Gn[0] + Gn[2] : Gn[0]);
            const R ay = ek == 0 ? Gn[3] : (ek == 1 ? Gn[1] + Gn[3] : Gn[1]);
            sn = sqrtR(ax * ax + ay * ay);
        }
        // liftings of this face's jumps at both sides' points; the partner's
        // jump at its slot P-f2 is minus this side's at f2
        R lo[NV] = {R(0), R(0), R(0), R(0)}, ln[NV] = {R(0), R(0), R(0), R(0)};
#pragma unroll 2
        for (int f2 = 0; f2 < FP; ++f2) {
            const int j2 = kk * FP + f2, o2 = ek * FP + (P - f2);
            R uo[NV], un[NV];
#pragma unroll
            for (int w = 0; w < NV; ++w) uo[w] = sTu[sl(elt, j2, w)];
            if (in) {
#pragma unroll
                for (int w = 0; w < NV; ++w) un[w] = sTu[sl(nl, o2, w)];
            } else {
                load4(Tn + (int64_t)o2 * TWV, un);
            }
            const R wo = clf<R>(LFO + (kk * FP + f) * FP + f2);
            const R wn = clf<R>(LFO + (ek * FP + (P - f)) * FP + (P - f2));
#pragma unroll
            for (int w = 0; w < NV; ++w) {
                const R jo = R(0.5) * (uo[w] + un[w]) - uo[w];
                lo[w] = fmaR(wo, jo, lo[w]);
                ln[w] = fmaR(wn, jo, ln[w]);
            }
        }
        const R sg = right ? R(-1) : R(1);
        const R nox = sg * nx, noy = sg * ny;  // this side's outward normal
        R Uc[NV], Qbx[NV], Qby[NV], UL[NV], UR[NV], Fc[NV], Fv[NV], Gv[NV];
#pragma unroll
        for (int w = 0; w < NV; ++w) {
            Uc[w] = R(0.5) * (own[w] + oth[w]);
            Qbx[w] = R(0.5) * ((gxo[w] + eta * so * nox * lo[w]) + (gxn[w] + eta * sn * nox * ln[w]));
            Qby[w] = R(0.5) * ((gyo[w] + eta * so * noy * lo[w]) + (gyn[w] + eta * sn * noy * ln[w]));
            UL[w] = right ? oth[w] : own[w];
            UR[w] = right ? own[w] : oth[w];
        }
        visc_flux(Uc, Qbx, Qby, g, mu, kappa, Fv, Gv);
        riemann_by_kind(a.riemann, UL, UR, nx, ny, g, Fc);
        {
            const R sc = right ? -so : so;
#pragma unroll
            for (int w = 0; w < NV; ++w) {
                const R fi = Fc[w] - (Fv[w] * nx + Gv[w] * ny);
                sD[sl(elt, j, w)] = sc * fi - sD[sl(elt, j, w)];
            }
        }
        if (in) {  // the in-tile partner, whose side is the right one
            const R sc = -sEdge[nl * 3 + ek];
#pragma unroll
            for (int w = 0; w < NV; ++w) {
                const R fi = Fc[w] - (Fv[w] * nx + Gv[w] * ny);
                sD[sl(nl, oj, w)] = sc * fi - sD[sl(nl, oj, w)];
            }
        }
    }
    __syncthreads();

    // ---- 4: lifted flux differences, RK stage update (the stage input read
    // again from memory); the stage output to sU for its traces
    double l2 = 0.0;
    if (live) {
#pragma unroll 1
        for (int j = 0; j < NFP; ++j) {
            const R d = sD[sl(el, j, v)];
#pragma unroll
            for (int i = 0; i < NP; ++i) div[i] = fmaR(cop<R>(OLT + j * NP + i), d, div[i]);
        }
        const double dt = MODE == MODE_RESIDUAL ? 0.0 : *a.dt_ptr;
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const double res = -double(div[i]);
            const int64_t gi = base + (int64_t)i * EB * NV;
            if (MODE == MODE_RESIDUAL) {
                a.R_out[gi] = res;
                l2 += res * res;
            } else {
                const double q = a.U_in[gi];
                double un;
                if (MODE == MODE_STAGE1) {
                    un = q + dt * res;
                } else {
                    const double u0 = a.U0[gi];
                    un = MODE == MODE_STAGE2 ? 0.75 * u0 + 0.25 * (q + dt * res)
                                             : (1.0 / 3.0) * u0 + (2.0 / 3.0) * (q + dt * res);
                    if (MODE == MODE_STAGE3) l2 += res * res;
                }
                a.U_out[gi] = un;
                sU[sp(el, i, v)] = R(un);  // only this lane reads its variable's points back
            }
        }
    }
    if ((MODE == MODE_RESIDUAL || MODE == MODE_STAGE3) && a.l2_partial) {
        const double s2 = block_reduce_n<OpSum, NWV>(l2, sred);
        if (tid == 0) a.l2_partial[tile] = s2;
    }
    if (MODE == MODE_RESIDUAL) return;
    __syncthreads();  // every read of the flux differences done: their space is reused below
    if (!live) return;

    // ---- 5: traces of the new stage state and of its gradient on edges
    // another tile reads (the gradient into the Q arrays, own variable only)
    bool any_out = false;
#pragma unroll
    for (int kk = 0; kk < 3; ++kk) {
        const int nl = L[kk].x - e0;
        any_out = any_out || !(nl >= 0 && nl < TT);
    }
    if (!any_out) return;
    R* const gx = sQx;  // each lane reads only its own variable's slots from here on
    R* const gy = sQy;
    gradient_of(rx, ry, sx, sy, gx, gy);
#pragma unroll
    for (int kk = 0; kk < 3; ++kk) {
        const int nl = L[kk].x - e0;
        if (nl >= 0 && nl < TT) continue;
        edge_traces(kk, 1, gx, gy, [&](int j, R tu, R tx, R ty) __attribute__((always_inline)) {
            R* T = a.T_out + ((int64_t)e * NFP + j) * TWV;
            T[v] = tu;
            T[NV + v] = tx;
            T[2 * NV + v] = ty;
        });
    }
}

// The traces of a new state and the completion of a cotangent, below: waves of
// G groups of four elements, four waves a workgroup.
constexpr int TRACE_G = 2, TRACE_TILE = BLOCK / 64 * 4 * TRACE_G;

// Traces of U and grad U on every edge (after a new state is set).  Bound by
// writing them: 1.1 KB an element at P3 FP64 against 0.3 read.  The operator
// tables are read into LDS once for 32 elements, and a group's rows leave
// through LDS in whole lines; with the tables from memory and 32-byte pieces
// stored from the products, set_state took, us, one lane per element and
// variable with scalar operands / that / this, at 500,000 elements: P3 FP64
// 312 / 350 / 214, P1 FP64 112 / 142 / 98, P5 FP64 544 / 638 / 424, P3 FP32
// 245 / 220 / 158.
// The bound of two waves per SIMD keeps the products' results out of the
// accumulation registers: with some of them there, hipcc 7.2 merged their LDS
// stores with the others' at wrong offsets (FP32).
template <typename R, int P>
__global__ __launch_bounds__(BLOCK, 2) void tri_visc_trace_kernel(int E, const double* U, const R* geo, R* T_out) {
    using FO = tri::FragOps<R, P>;
    constexpr int NP = FO::NP, NFP = FO::NFP, PB = FO::PB, FB = FO::FB, G = TRACE_G;
    __shared__ R ops[FO::F - FO::I];  // the operator tables I, G
    __shared__ R sOut[BLOCK / 64 * 4 * NFP * TWV];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, row = lane >> 4, v = lane & 3;
    const int e0 = blockIdx.x * TRACE_TILE;
    auto elg = [&](int q) { return e0 + (wave * G + q) * 4 + ((lane >> 2) & 3); };
    const PointRows<NP, G> rows(e0, wave, lane, E);
    double u0[G][PB];
    R ge[G][4];
#pragma unroll
    for (int q = 0; q < G; ++q) {
#pragma unroll
        for (int b = 0; b < PB; ++b) u0[q][b] = *rows.at(U, q, b);
#pragma unroll
        for (int c = 0; c < 4; ++c) ge[q][c] = geo[(int64_t)min(elg(q), E - 1) * GEO + c];
    }
    {
        const R* const src = frag_ops<R>() + tri::frag_offset<R>(P) + FO::I;
        for (int t = 4 * threadIdx.x; t < FO::F - FO::I; t += 4 * BLOCK) {
            R w[4];
            load4(src + t, w);
            store4(ops + t, w);
        }
    }
    R u[G][PB], tu[G][FB], tg[G][2 * FB];
#pragma unroll
    for (int q = 0; q < G; ++q)
#pragma unroll
        for (int b = 0; b < PB; ++b) u[q][b] = 4 * b + row < NP ? R(u0[q][b]) : R(0);
    __syncthreads();
    tri::frag_mma<true, R, G, FB, PB>(ops, u, tu);
    tri::frag_mma<true, R, G, 2 * FB, PB>(ops + (FO::G - FO::I), u, tg);
    // a group's rows are one run of memory: through LDS, so that a store's lanes write whole lines of it
    R* const out = sOut + wave * (4 * NFP * TWV);
#pragma unroll
    for (int q = 0; q < G; ++q) {
        const int first = e0 + (wave * G + q) * 4;
        tri::wave_lds_fence();
#pragma unroll
        for (int b = 0; b < FB; ++b) {
            if (4 * b + row >= NFP) continue;
            R* T = out + (((lane >> 2) & 3) * NFP + 4 * b + row) * TWV + v;
            T[0] = tu[q][b];
            T[NV] = ge[q][0] * tg[q][b] + ge[q][2] * tg[q][FB + b];
            T[2 * NV] = ge[q][1] * tg[q][b] + ge[q][3] * tg[q][FB + b];
        }
        tri::wave_lds_fence();
        const int n = min(4, E - first) * NFP * TWV;  // words; none beyond the mesh
        using V = typename std::conditional<sizeof(R) == 8, double2, float4>::type;  // one lane's 16 bytes
        constexpr int W = sizeof(V) / sizeof(R);
        for (int t = W * lane; t < n; t += W * 64)
            *reinterpret_cast<V*>(T_out + (int64_t)first * NFP * TWV + t) = *reinterpret_cast<const V*>(out + t);
    }
}

// ------------------------------------------------------------ adjoint
// Vector-Jacobian product of one triangle stage u_n = a U^n + b q + c dt R(q)
// (MODE_STAGE1..3), or of the residual alone (MODE_RESIDUAL).  The forward
// values are recomputed as tri_scalar_kernel forms them; then, per lane
// (element, variable):
//   R1  cotangent of u_out: its partial value plus the transposed trace
//       operator on the edge cotangents other tiles left (cross-tile edges);
//       the RK combination's cotangents of U^n, q and dt
//   R2  the lifting transposed: the flux differences' cotangents (LDS)
//   R3  per solved face point (as the forward solves them): the common flux's
//       cotangent from both sides' differences, the Riemann solver's VJP, to
//       this side's trace cotangent (LDS), an in-tile neighbour's (LDS) or a
//       cross-tile neighbour's (HBM, at its slot) or through the ghost state
//   R4  per solution point: Dr, Ds and the interpolated normal flux
//       transposed, the metric, the Euler flux Jacobian (the four variables'
//       cotangents gathered across the element's DPP quad), and the
//       transposed trace operator
template <typename R>
struct TriVjpArgs {
    int E;
    const double* U_in;     // q
    const double* U0;       // U^n (stages 2, 3)
    const R* geo;
    const R* edge;
    const int2* links;
    const R* T_in;          // traces of q on edges read across tiles
    const double* bc_data;
    const double* dt_ptr;
    const double* Ub_in;    // partial cotangent of u_out, or of R
    const R* Tb_in;         // cross-tile edge cotangents completing Ub_in (nullptr: none)
    double* Ub_out;         // partial cotangent of q (may alias Ub_in)
    R* Tb_out;              // cross-tile edge cotangents of q, at the neighbour's slots
    double* U0b;            // cotangent of U^n: stage 3 writes, stage 2 adds, stage 1 reads
    double* dtb_partial;    // per-tile sum of c R . du_n (nullptr: skip)
    double gamma;
    int riemann;
    int xcd_groups;
    int lift_off;
    double mu, kappa, eta;  // Navier-Stokes terms (tri_visc_vjp_kernel)
    int lf_off;
    int family;             // of the correction: DG, SD = GA, HU
    const double* R_in;     // residual at q, with dtb_partial (tri_visc_vjp_kernel)
};

template <typename R, int P, int MODE>
__global__ __launch_bounds__(BLOCK) void tri_vjp_kernel(TriVjpArgs<R> a) {
    using S = TriShape<P>;
    constexpr int NP = S::NP, FP = S::FP, NFP = S::NFP;
    constexpr int NW = NP > NFP ? NP : NFP;
    using OP = TriOps<P>;
    constexpr int O0 = ops_offset(P), CA = OP::CA, OI = O0 + OP::C;
    constexpr double ca = MODE == MODE_STAGE2 ? 0.75 : (MODE == MODE_STAGE3 ? 1.0 / 3.0 : 0.0);
    constexpr double cb = MODE == MODE_STAGE2 ? 0.25 : (MODE == MODE_STAGE3 ? 2.0 / 3.0 : 1.0);
    constexpr double cc = MODE == MODE_STAGE2 ? 0.25 : (MODE == MODE_STAGE3 ? 2.0 / 3.0 : 1.0);
    const int OLT = O0 + a.lift_off;
    __shared__ R sT[TILE * NFP * NV];   // own traces
    __shared__ R sW[TILE * NW * NV];    // q, then Fn, then the flux differences d, then their cotangents
    __shared__ R sTb[TILE * NFP * NV];  // trace cotangents
    __shared__ double sred[BLOCK / 64];
    __shared__ R sEdge[TILE * 3];
    __shared__ unsigned char sList[TILE * 3];
    __shared__ int sCnt[BLOCK / 64];

    const int tid = threadIdx.x, el = tid >> 2, v = tid & 3;
    const int tile = tile_of_block(a.xcd_groups);
    const int e0 = tile * TILE, e = e0 + el;
    const bool live = e < a.E;
    const R g = R(a.gamma);
    const int64_t base = blk(e, 0, NP) + v;

    double q[NP];
    R rx = R(0), ry = R(0), sx = R(0), sy = R(0);
    int2 L[3] = {make_int2(0, 0), make_int2(0, 0), make_int2(0, 0)};
    if (live) {
#pragma unroll
        for (int m = 0; m < NP; ++m) q[m] = a.U_in[base + (int64_t)m * EB * NV];
        const R* G = a.geo + (int64_t)e * GEO;
        rx = G[0]; ry = G[1]; sx = G[2]; sy = G[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) L[k] = a.links[(int64_t)e * 3 + k];
#pragma unroll
        for (int m = 0; m < NP; ++m) sW[(el * NP + m) * NV + v] = R(q[m]);
        if (v < 3) {
            const R ax = v == 0 ? sx : (v == 1 ? rx + sx : rx), ay = v == 0 ? sy : (v == 1 ? ry + sy : ry);
            sEdge[el * 3 + v] = sqrtR(ax * ax + ay * ay);
        }
    } else {
#pragma unroll
        for (int m = 0; m < NP; ++m) q[m] = 0.0;
    }
    bool owned = false;
    if (live && v < 3) {
        const int2 Lv = v == 0 ? L[0] : (v == 1 ? L[1] : L[2]);
        const int nl = Lv.x - e0;
        owned = !(link_role(Lv.y) == ROLE_RIGHT && nl >= 0 && nl < TILE);
    }
    const unsigned long long own_mask = __ballot(owned);
    const int lane = tid & 63, wave = tid >> 6;
    if (lane == 0) sCnt[wave] = __popcll(own_mask);
    __syncthreads();

    // ---- forward 1: divergence, interpolated normal fluxes, traces
    R div[NP], fn[NFP];
    if (live) {
#pragma unroll
        for (int i = 0; i < NP; ++i) div[i] = R(0);
#pragma unroll
        for (int j = 0; j < NFP; ++j) fn[j] = R(0);
#pragma unroll 1
        for (int m = 0; m < NP; ++m) {
            const R um = sW[(el * NP + m) * NV + v];
            const R q0 = quad_get<0>(um), q1 = quad_get<1>(um), q2 = quad_get<2>(um), q3 = quad_get<3>(um);
            const R inv = fast_rcp(q0);
            const R ux = q1 * inv, uy = q2 * inv;
            const R p = (g - R(1)) * (q3 - R(0.5) * (q1 * ux + q2 * uy));
            const R fx = v == 0 ? q1 : (v == 1 ? q1 * ux + p : (v == 2 ? q1 * uy : (q3 + p) * ux));
            const R fy = v == 0 ? q2 : (v == 1 ? q2 * ux : (v == 2 ? q2 * uy + p : (q3 + p) * uy));
            const R fr = rx * fx + ry * fy, fs = sx * fx + sy * fy, frs = fr + fs;
#pragma unroll
            for (int i = 0; i < NP; ++i)
                div[i] = fmaR(cop<R>(O0 + m * CA + NP + i), fs, fmaR(cop<R>(O0 + m * CA + i), fr, div[i]));
#pragma unroll
            for (int j = 0; j < NFP; ++j)
                fn[j] = fmaR(cop<R>(O0 + m * CA + 2 * NP + j), j < FP ? fs : (j < 2 * FP ? frs : fr), fn[j]);
        }
        R ut[NFP];
#pragma unroll
        for (int j = 0; j < NFP; ++j) ut[j] = R(0);
#pragma unroll 1
        for (int m = 0; m < NP; ++m) {
            const R um = sW[(el * NP + m) * NV + v];
#pragma unroll
            for (int j = 0; j < NFP; ++j) ut[j] = fmaR(cop<R>(O0 + m * CA + 2 * NP + j), um, ut[j]);
        }
#pragma unroll
        for (int j = 0; j < NFP; ++j) sT[(el * NFP + j) * NV + v] = ut[j];
    }
    if (owned) {
        int pos = __popcll(own_mask & ((1ull << lane) - 1));
        for (int w = 0; w < wave; ++w) pos += sCnt[w];
        sList[pos] = (unsigned char)(el * 3 + v);
    }
    __syncthreads();
    if (live) {
#pragma unroll
        for (int j = 0; j < NFP; ++j) sW[(el * NFP + j) * NV + v] = (j >= FP && j < 2 * FP) ? fn[j] : -fn[j];
    }
    __syncthreads();
    int nsolved = 0;
#pragma unroll
    for (int w = 0; w < BLOCK / 64; ++w) nsolved += sCnt[w];

    // ---- forward 2: flux differences d = sc F^I - Fn of both sides of every solved face point
#pragma unroll 1
    for (int t = tid; t < nsolved * FP; t += BLOCK) {
        const int c = sList[t / FP], f = t - (t / FP) * FP;
        const int elt = c / 3, kk = c - elt * 3, j = kk * FP + f;
        const int2 Lk = a.links[(int64_t)(e0 + elt) * 3 + kk];
        const int role = link_role(Lk.y);
        const R nx = a.geo[(int64_t)(e0 + elt) * GEO + 4 + 2 * kk];
        const R ny = a.geo[(int64_t)(e0 + elt) * GEO + 5 + 2 * kk];
        R own[NV], oth[NV], UL[NV], UR[NV], Fc[NV];
#pragma unroll
        for (int w = 0; w < NV; ++w) own[w] = sT[(elt * NFP + j) * NV + w];
        int nl = -1, oj = 0;
        if (role == ROLE_BOUNDARY) {
            ghost_state(own, nx, ny, link_edge(Lk.y), a.bc_data + (int64_t)link_bc(Lk.y) * 8, g, oth);
        } else {
            nl = Lk.x - e0;
            oj = link_edge(Lk.y) * FP + (P - f);
            if (nl >= 0 && nl < TILE) {
#pragma unroll
                for (int w = 0; w < NV; ++w) oth[w] = sT[(nl * NFP + oj) * NV + w];
            } else {
                load4(a.T_in + trix(Lk.x, oj, NFP), oth);
                nl = -1;
            }
        }
        const bool right = role == ROLE_RIGHT;
#pragma unroll
        for (int w = 0; w < NV; ++w) { UL[w] = right ? oth[w] : own[w]; UR[w] = right ? own[w] : oth[w]; }
        riemann_by_kind(a.riemann, UL, UR, nx, ny, g, Fc);
        {
            const R sc = right ? -sEdge[c] : sEdge[c];
            R* d = sW + (elt * NFP + j) * NV;
#pragma unroll
            for (int w = 0; w < NV; ++w) d[w] = sc * Fc[w] - d[w];
        }
        if (nl >= 0) {
            const R sc = -sEdge[nl * 3 + link_edge(Lk.y)];
            R* d = sW + (nl * NFP + oj) * NV;
#pragma unroll
            for (int w = 0; w < NV; ++w) d[w] = sc * Fc[w] - d[w];
        }
    }
    __syncthreads();

    // ---- forward 3: residual; R1: cotangent of the stage output, RK combination
    double rsum = 0.0;
    R divb[NP];
    double qb[NP];
    if (live) {
#pragma unroll 1
        for (int j = 0; j < NFP; ++j) {
            const R d = sW[(el * NFP + j) * NV + v];
#pragma unroll
            for (int i = 0; i < NP; ++i) div[i] = fmaR(cop<R>(OLT + j * NP + i), d, div[i]);
        }
        // incoming edge cotangents of u_out on this element's cross-tile edges
        R tin[NFP];
#pragma unroll
        for (int j = 0; j < NFP; ++j) tin[j] = R(0);
        if (MODE != MODE_RESIDUAL && a.Tb_in) {
#pragma unroll
            for (int kk = 0; kk < 3; ++kk) {
                const int nl = L[kk].x - e0;
                const int role = link_role(L[kk].y);
                if (role == ROLE_BOUNDARY || (nl >= 0 && nl < TILE)) continue;
#pragma unroll
                for (int f = 0; f < FP; ++f) tin[kk * FP + f] = a.Tb_in[trix(e, kk * FP + f, NFP) + v];
            }
        }
        const double dt = MODE == MODE_RESIDUAL ? 0.0 : *a.dt_ptr;
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const int64_t gi = base + (int64_t)i * EB * NV;
            double rb;
            if (MODE == MODE_RESIDUAL) {
                rb = a.Ub_in[gi];
                qb[i] = 0.0;
            } else {
                R tsum = R(0);
#pragma unroll
                for (int j = 0; j < NFP; ++j) tsum = fmaR(cop<R>(OI + j * NP + i), tin[j], tsum);
                const double unb = a.Ub_in[gi] + double(tsum);
                if (MODE == MODE_STAGE3) a.U0b[gi] = ca * unb;
                if (MODE == MODE_STAGE2) a.U0b[gi] += ca * unb;
                qb[i] = cb * unb;
                rb = cc * dt * unb;
                rsum += cc * (-double(div[i])) * unb;
            }
            divb[i] = R(-rb);  // R = -div
        }
    } else {
#pragma unroll
        for (int i = 0; i < NP; ++i) { divb[i] = R(0); qb[i] = 0.0; }
    }
    if (a.dtb_partial) {
        const double s = block_reduce<OpSum>(rsum, sred);
        if (tid == 0) a.dtb_partial[tile] = s;
    }
    __syncthreads();  // every lane's reads of sW (forward 3) are done

    // ---- R2: the lifting transposed, d_j's cotangent into sW; trace cotangents cleared
    if (live) {
#pragma unroll 1
        for (int j = 0; j < NFP; ++j) {
            R acc = R(0);
#pragma unroll
            for (int i = 0; i < NP; ++i) acc = fmaR(cop<R>(OLT + j * NP + i), divb[i], acc);
            sW[(el * NFP + j) * NV + v] = acc;
            sTb[(el * NFP + j) * NV + v] = R(0);
        }
    }
    __syncthreads();

    // ---- R3: the common flux of every solved face point, backwards
#pragma unroll 1
    for (int t = tid; t < nsolved * FP; t += BLOCK) {
        const int c = sList[t / FP], f = t - (t / FP) * FP;
        const int elt = c / 3, kk = c - elt * 3, j = kk * FP + f;
        const int2 Lk = a.links[(int64_t)(e0 + elt) * 3 + kk];
        const int role = link_role(Lk.y);
        const R nx = a.geo[(int64_t)(e0 + elt) * GEO + 4 + 2 * kk];
        const R ny = a.geo[(int64_t)(e0 + elt) * GEO + 5 + 2 * kk];
        R own[NV], oth[NV], UL[NV], UR[NV], Fcb[NV];
#pragma unroll
        for (int w = 0; w < NV; ++w) own[w] = sT[(elt * NFP + j) * NV + w];
        int nl = -1, oj = 0;
        bool cross = false;
        const double* bcd = a.bc_data + (int64_t)(role == ROLE_BOUNDARY ? link_bc(Lk.y) : 0) * 8;
        if (role == ROLE_BOUNDARY) {
            ghost_state(own, nx, ny, link_edge(Lk.y), bcd, g, oth);
        } else {
            nl = Lk.x - e0;
            oj = link_edge(Lk.y) * FP + (P - f);
            if (nl >= 0 && nl < TILE) {
#pragma unroll
                for (int w = 0; w < NV; ++w) oth[w] = sT[(nl * NFP + oj) * NV + w];
            } else {
                load4(a.T_in + trix(Lk.x, oj, NFP), oth);
                nl = -1;
                cross = true;
            }
        }
        const bool right = role == ROLE_RIGHT;
        const R sc = right ? -sEdge[c] : sEdge[c];
#pragma unroll
        for (int w = 0; w < NV; ++w) {
            UL[w] = right ? oth[w] : own[w];
            UR[w] = right ? own[w] : oth[w];
            Fcb[w] = sc * sW[(elt * NFP + j) * NV + w];
        }
        if (nl >= 0) {
            const R scn = -sEdge[nl * 3 + link_edge(Lk.y)];
#pragma unroll
            for (int w = 0; w < NV; ++w) Fcb[w] += scn * sW[(nl * NFP + oj) * NV + w];
        }
        R ULb[NV] = {R(0), R(0), R(0), R(0)}, URb[NV] = {R(0), R(0), R(0), R(0)};
        riemann_by_kind_vjp(a.riemann, UL, UR, nx, ny, g, Fcb, ULb, URb);
        R ownb[NV], othb[NV];
#pragma unroll
        for (int w = 0; w < NV; ++w) {
            ownb[w] = right ? URb[w] : ULb[w];
            othb[w] = right ? ULb[w] : URb[w];
        }
        if (role == ROLE_BOUNDARY) {
            ghost_state_vjp(own, nx, ny, link_edge(Lk.y), bcd, g, othb, ownb);
        } else if (nl >= 0) {
#pragma unroll
            for (int w = 0; w < NV; ++w) sTb[(nl * NFP + oj) * NV + w] = othb[w];
        } else if (cross) {
            store4(a.Tb_out + trix(Lk.x, oj, NFP), othb);
        }
#pragma unroll
        for (int w = 0; w < NV; ++w) sTb[(elt * NFP + j) * NV + w] = ownb[w];
    }
    __syncthreads();

    // ---- R4: volume terms at the solution points, transposed traces; cotangent of q
    if (!live) return;
#pragma unroll 1
    for (int m = 0; m < NP; ++m) {
        R frb = R(0), fsb = R(0);
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            frb = fmaR(cop<R>(O0 + m * CA + i), divb[i], frb);
            fsb = fmaR(cop<R>(O0 + m * CA + NP + i), divb[i], fsb);
        }
        R tb = R(0);
#pragma unroll
        for (int j = 0; j < NFP; ++j) {
            const R im = cop<R>(O0 + m * CA + 2 * NP + j);
            // Fn = -fn (edges 0, 2), +fn (edge 1); d = sc F^I - Fn; fn_j = sum_m interp[j][m] X_m
            // with X = fs, fr + fs, fr on edges 0, 1, 2
            const R db = sW[(el * NFP + j) * NV + v];
            const R fnb = (j >= FP && j < 2 * FP) ? -db : db;
            if (j >= FP) frb = fmaR(im, fnb, frb);
            if (j < 2 * FP) fsb = fmaR(im, fnb, fsb);
            tb = fmaR(im, sTb[(el * NFP + j) * NV + v], tb);
        }
        const R fxb = rx * frb + sx * fsb, fyb = ry * frb + sy * fsb;
        const R um = R(q[m]);
        const R Uq[NV] = {quad_get<0>(um), quad_get<1>(um), quad_get<2>(um), quad_get<3>(um)};
        const R A[NV] = {quad_get<0>(fxb), quad_get<1>(fxb), quad_get<2>(fxb), quad_get<3>(fxb)};
        const R B[NV] = {quad_get<0>(fyb), quad_get<1>(fyb), quad_get<2>(fyb), quad_get<3>(fyb)};
        R Ub[NV] = {R(0), R(0), R(0), R(0)};
        euler_flux_vjp(Uq, g, A, B, Ub);
        const R mine = v == 0 ? Ub[0] : (v == 1 ? Ub[1] : (v == 2 ? Ub[2] : Ub[3]));
        const int64_t gi = base + (int64_t)m * EB * NV;
        double out = qb[m] + double(mine) + double(tb);
        if (MODE == MODE_STAGE1) out += a.U0b[gi];
        a.Ub_out[gi] = out;
    }
}

// Completion of a cotangent: U_bar plus the transposed traces of the
// cross-tile edge cotangents that the last adjoint launch left for this tile.
template <typename R, int P>
__global__ __launch_bounds__(BLOCK) void tri_complete_kernel(int E, const int2* __restrict__ links,
                                                             const double* __restrict__ Ub, const R* __restrict__ Tb,
                                                             double* __restrict__ out, int xcd_groups) {
    using S = TriShape<P>;
    constexpr int NP = S::NP, FP = S::FP, NFP = S::NFP;
    constexpr int OI = ops_offset(P) + TriOps<P>::C;
    const int tid = threadIdx.x, el = tid >> 2, v = tid & 3;
    const int e0 = tile_of_block(xcd_groups) * TILE, e = e0 + el;
    if (e >= E) return;
    const int64_t base = blk(e, 0, NP) + v;
    R tin[NFP];
#pragma unroll
    for (int j = 0; j < NFP; ++j) tin[j] = R(0);
    if (Tb) {
#pragma unroll
        for (int kk = 0; kk < 3; ++kk) {
            const int2 Lk = links[(int64_t)e * 3 + kk];
            const int nl = Lk.x - e0;
            if (link_role(Lk.y) == ROLE_BOUNDARY || (nl >= 0 && nl < TILE)) continue;
#pragma unroll
            for (int f = 0; f < FP; ++f) tin[kk * FP + f] = Tb[trix(e, kk * FP + f, NFP) + v];
        }
    }
#pragma unroll
    for (int i = 0; i < NP; ++i) {
        R tsum = R(0);
#pragma unroll
        for (int j = 0; j < NFP; ++j) tsum = fmaR(cop<R>(OI + j * NP + i), tin[j], tsum);
        const int64_t gi = base + (int64_t)i * EB * NV;
        out[gi] = Ub[gi] + double(tsum);
    }
}

// ------------------------------------------------------------ adjoint, BR2
// Vector-Jacobian product of one triangle stage with the Navier-Stokes terms
// (tri_visc_stage_kernel), or of its residual alone; lanes and operator
// products as there.  Of the forward values it recomputes the traces, the
// corrected gradient and both sides' BR2 gradients; the residual, needed for
// the time step's cotangent alone, comes from a residual launch (R_in).  Then
//   R1  cotangent of u_out: its partial value plus, on cross-tile edges, the
//       transposed traces of U and of its gradient; the RK combination
//   R2  the lifting transposed: the flux differences' cotangents
//   R4  the divergence and the interpolated normal fluxes transposed; then one
//       lane per point (all four variables): the Euler and viscous flux VJPs,
//       the cotangents of U and of the corrected gradient at the point
//   R5  the corrected gradient's lifted jumps transposed
//   R3  per solved face point: the common flux's cotangent, the Riemann and
//       viscous flux VJPs at the face, the cotangents of both sides' traces
//       (of U and of the gradient) at their slots
//   R7  the face liftings transposed; every edge point's jump cotangent
//   R6  the traces and the gradient transposed: cotangent of q.  Across tiles
//       the partner's 12 words go to its slot in memory
// Bounds as the stage kernel's, with one (FP64) or two waves per SIMD.  80,000
// elements, P3, us a launch (operators as scalar operands, the residual
// recomputed in every launch -> this): FP64 480 -> 175, FP32 210 -> 90; a step
// backwards 1719 -> 665 and 820 -> 356.
template <typename R, int P> struct TriViscVjpTile {
    static constexpr int NP = (P + 1) * (P + 2) / 2, NFP = 3 * (P + 1), PB = (NP + 3) / 4, FB = (NFP + 3) / 4;
    static constexpr bool BIG = sizeof(R) == 8 && P == 5;
    static constexpr int G = BIG ? 1 : 2, WV = P == 1 ? 8 : 4;
    // FP32 meshes of at least this many elements have tiles of 64, as the scalar stage form has (so that no trace
    // is formed again), and take the scalar form below: P1 always, P2 where dJ/d(dt) is asked for (else eight
    // waves of the matrix-core form)
    static constexpr int LARGE_FROM = sizeof(R) == 8 || P > 2 ? INT_MAX : P == 1 ? 16384 : 24576;
    static constexpr int tile(int E) { return E >= LARGE_FROM ? TILE : 4 * G * WV; }
    // waves per SIMD asked for: in FP64 the face points' VJPs take more than the 256 VGPRs of two (P2:
    // 584 us a step at one wave, 707 at two with scratch), P5's LDS allows one workgroup.  FP64 P1 at two keeps 180
    // bytes a lane in scratch and is the quicker of them on large meshes: 500,000 elements 2139 us a step, tiles of
    // 32 at one wave without scratch 2522 (80,000 322 / 383, 16,200 77 / 79, 800 58 / 44)
    static constexpr int WPE = (sizeof(R) == 8 ? P == 1 : P < 5) ? 2 : 1;
    // rows of an element's region: Q_x, Q_y, the point fluxes' cotangents x, y, U (RU); later the
    // gradient traces x and y, the partner's U traces and the flux differences' cotangents
    static constexpr int RU = 3 * NP + 4 * PB;
    static constexpr int ROWS = RU + 4 * PB > 3 * NFP + 4 * FB ? RU + 4 * PB : 3 * NFP + 4 * FB;
    static constexpr int ESF = tri::elem_stride<R>(4 * FB), ESX = tri::elem_stride<R>(ROWS);
};

template <typename R, int P, int MODE, int NWV>
__global__ __launch_bounds__(64 * NWV, (TriViscVjpTile<R, P>::WPE)) void tri_visc_vjp_kernel(TriVjpArgs<R> a) {
    using S = TriShape<P>;
    using TV = TriViscVjpTile<R, P>;
    using FO = tri::FragOps<R, P>;
    constexpr int NP = S::NP, FP = S::FP, NFP = S::NFP, PB = FO::PB, FB = FO::FB;
    constexpr int G = TV::G, NB = 64 * NWV, TT = 4 * G * NWV, ESF = TV::ESF, ESX = TV::ESX;
    constexpr int RU = TV::RU, RA = 2 * NP, RB = 3 * NP;       // point rows
    constexpr int RY = NFP, RO = 2 * NFP, RD = 3 * NFP;         // trace rows
    constexpr double ca = MODE == MODE_STAGE2 ? 0.75 : (MODE == MODE_STAGE3 ? 1.0 / 3.0 : 0.0);
    constexpr double cb = MODE == MODE_STAGE2 ? 0.25 : (MODE == MODE_STAGE3 ? 2.0 / 3.0 : 1.0);
    constexpr double cc = MODE == MODE_STAGE2 ? 0.25 : (MODE == MODE_STAGE3 ? 2.0 / 3.0 : 1.0);
    constexpr int N0 = FO::F, N1 = FO::FAMILY, N2 = FO::ADJ, N3 = FO::ADJ_FAMILY;  // D, I, G; L, LF; FT, GT, DT; LT, LFT
    __shared__ R ops[N0 + N1 + N2 + N3];
    const R *const fam = ops + N0, *const adj = fam + N1, *const afam = adj + N2;
    __shared__ R sTu[TT * ESF];      // traces of U; later, across tiles, the partner's U cotangents
    __shared__ R sX[TT * ESX];
    __shared__ double sred[NWV];
    __shared__ R sGeo[TT * 4];
    __shared__ R sEw[TT * 3 * 4];    // as in tri_visc_stage_kernel
    __shared__ R sNs[TT * 3 * 4];    // (the partner's factor 0 across tiles)
    __shared__ int4 sPa[TT * 3];
    __shared__ unsigned char sList[TT * 3];
    __shared__ int sCnt[NWV];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int row = lane >> 4, v = lane & 3;
    const int tile = tile_of_block(a.xcd_groups);
    const int e0 = tile * TT;
    const R g = R(a.gamma), mu = R(a.mu), kappa = R(a.kappa), eta = R(a.eta);
    auto elg = [&](int q) { return (wave * G + q) * 4 + ((lane >> 2) & 3); };
    auto st = [](int elx, int j) { return elx * ESF + j * NV; };
    auto sx_ = [](int elx, int r) { return elx * ESX + r * NV; };
    const PointRows<NP, G> rows(e0, wave, lane, a.E);

    // ---- 0: q, the incoming cotangent, operators and edges
    R ur[G][PB];
    double unb[G][PB], rin[G][PB];
#pragma unroll
    for (int q = 0; q < G; ++q)
#pragma unroll
        for (int b = 0; b < PB; ++b) {
            ur[q][b] = R(*rows.at(a.U_in, q, b));
            unb[q][b] = *rows.at(a.Ub_in, q, b);
            rin[q][b] = MODE != MODE_RESIDUAL && a.dtb_partial ? *rows.at(a.R_in, q, b) : 0.0;
        }
    {
        const R* const src = frag_ops<R>() + tri::frag_offset<R>(P);
        for (int t = 4 * tid; t < N0 + N1 + N2 + N3; t += 4 * NB) {
            const int o = t < N0 ? t
                          : t < N0 + N1 ? t - N0 + FO::COMMON + a.family * N1
                          : t < N0 + N1 + N2 ? t - N0 - N1 + FO::ADJ0
                                             : t - N0 - N1 - N2 + FO::ADJ_FAM0 + a.family * N3;
            R w[4];
            load4(src + o, w);
            store4(ops + t, w);
        }
    }
    static_assert(TT * 3 <= NB, "one lane per edge of the tile");
    bool owned = false;
    if (tid < TT * 3) {
        const int el = tid / 3, k = tid - el * 3, e = min(e0 + el, a.E - 1);
        const R* Ge = a.geo + (int64_t)e * GEO;
        const int2 Lk = a.links[(int64_t)e * 3 + k];
        const int nl = Lk.x - e0, ek = link_edge(Lk.y);
        const bool right = link_role(Lk.y) == ROLE_RIGHT, live = e0 + el < a.E;
        const bool in = !live || (nl >= 0 && nl < TT);
        const R s = a.edge[(int64_t)e * EDG + 2 * k], sn = a.edge[(int64_t)e * EDG + 2 * k + 1], nx = Ge[4 + 2 * k], ny = Ge[5 + 2 * k];
        const R w = right ? -s : s, wn = right ? -eta * sn : eta * sn;
        const R we[4] = {w * nx, w * ny, wn * nx, wn * ny}, ns[4] = {nx, ny, w, in ? (right ? sn : -sn) : R(0)};
        store4(sEw + 4 * tid, we);
        store4(sNs + 4 * tid, ns);
        const bool self = !live || !in;
        sPa[tid] = make_int4(self ? el : nl, (self ? k : ek) * FP + P, in ? 3 : ek,
                             in ? P : (int)((unsigned)Lk.x * NFP + ek * FP + P));
        owned = live && !(right && in);
    }
    if (tid < TT) {
        const R* Ge = a.geo + (int64_t)min(e0 + tid, a.E - 1) * GEO;
        const R w[4] = {Ge[0], Ge[1], Ge[2], Ge[3]};
        store4(sGeo + 4 * tid, w);
    }
    const unsigned long long own_mask = __ballot(owned);
    if (lane == 0) sCnt[wave] = __popcll(own_mask);
#pragma unroll
    for (int q = 0; q < G; ++q)
#pragma unroll
        for (int b = 0; b < PB; ++b) {
            ur[q][b] = 4 * b + row < NP ? ur[q][b] : R(0);
            sX[sx_(elg(q), RU + 4 * b + row) + v] = ur[q][b];
        }
    __syncthreads();
    auto partner = [&](int q, int b) { return sPa[elg(q) * 3 + min(4 * b + row, NFP - 1) / FP]; };
    auto remote = [&](int w, int b) { return ((int64_t)(unsigned)w - min(4 * b + row, NFP - 1) % FP) * TWV + v; };
    R oth[G][FB];
    unsigned edges = 0;  // two bits per slot: the partner's edge, 3 in the tile
#pragma unroll
    for (int q = 0; q < G; ++q)
#pragma unroll
        for (int b = 0; b < FB; ++b) {
            const int4 pa = partner(q, b);
            edges |= (unsigned)pa.z << 2 * (q * FB + b);
            oth[q][b] = a.T_in[remote(pa.w, b)];
        }
    auto edge_of = [&](int q, int b) { return (int)(edges >> 2 * (q * FB + b)) & 3; };
    static_assert(G * FB <= 16, "two bits per slot");
    if (owned) {
        int pos = __popcll(own_mask & ((1ull << lane) - 1));
        for (int w = 0; w < wave; ++w) pos += sCnt[w];
        sList[pos] = (unsigned char)tid;
    }
    R tu[G][FB], gd[G][2 * PB];
    tri::frag_mma<true, R, G, FB, PB>(ops + FO::I, ur, tu);
#pragma unroll
    for (int q = 0; q < G; ++q)
#pragma unroll
        for (int b = 0; b < FB; ++b) sTu[st(elg(q), 4 * b + row) + v] = tu[q][b];
    tri::frag_mma<true, R, G, 2 * PB, PB>(ops + FO::D, ur, gd);

    // ---- R1, R2: cotangents of u_out, of the divergence and of the flux differences; R4: of the point fluxes
    double qb[G][PB], rsum = 0.0;
    R fx[G][2 * PB], db[G][FB];
    {
        if (MODE != MODE_RESIDUAL && a.Tb_in) {
            R f[G][3 * FB], add[G][PB];
#pragma unroll
            for (int q = 0; q < G; ++q) {
                R ge[4];
                load4(sGeo + 4 * elg(q), ge);
#pragma unroll
                for (int b = 0; b < FB; ++b) {
                    // own slots across tiles (the others read the tile's first row in common)
                    const int j = 4 * b + row;
                    const bool on = edge_of(q, b) != 3 && j < NFP;
                    const R* T = a.Tb_in + (on ? (int64_t)(e0 + elg(q)) * NFP + j : (int64_t)0) * TWV + v;
                    const R tb = T[0], xb = T[NV], yb = T[2 * NV];
                    f[q][b] = on ? tb : R(0);
                    f[q][FB + b] = on ? ge[0] * xb + ge[1] * yb : R(0);
                    f[q][2 * FB + b] = on ? ge[2] * xb + ge[3] * yb : R(0);
                }
            }
            tri::frag_mma<true, R, G, PB, 3 * FB>(adj + FO::GT, f, add);
#pragma unroll
            for (int q = 0; q < G; ++q)
#pragma unroll
                for (int b = 0; b < PB; ++b) unb[q][b] += double(add[q][b]);
        }
        const double dt = MODE == MODE_RESIDUAL ? 0.0 : *a.dt_ptr;
        R f[G][PB + FB], dvb[G][PB];
#pragma unroll
        for (int q = 0; q < G; ++q)
#pragma unroll
            for (int b = 0; b < PB; ++b) {
                const bool ok = 4 * b + row < NP && e0 + elg(q) < a.E;
                double rb = unb[q][b];
                qb[q][b] = 0.0;
                if (MODE != MODE_RESIDUAL) {
                    if (MODE == MODE_STAGE3 && ok) *rows.at(a.U0b, q, b) = ca * unb[q][b];
                    if (MODE == MODE_STAGE2 && ok) *rows.at(a.U0b, q, b) += ca * unb[q][b];
                    qb[q][b] = cb * unb[q][b];
                    rb = cc * dt * unb[q][b];
                    rsum += ok ? cc * rin[q][b] * unb[q][b] : 0.0;
                }
                dvb[q][b] = 4 * b + row < NP ? R(-rb) : R(0);  // R = -div
            }
        tri::frag_mma<true, R, G, FB, PB>(afam + FO::LT, dvb, db);
#pragma unroll
        for (int q = 0; q < G; ++q) {
#pragma unroll
            for (int b = 0; b < PB; ++b) f[q][b] = dvb[q][b];
#pragma unroll
            for (int b = 0; b < FB; ++b) f[q][PB + b] = db[q][b];
        }
        tri::frag_mma<true, R, G, 2 * PB, PB + FB>(adj + FO::FT, f, fx);
    }
    if (a.dtb_partial) {
        const double s2 = block_reduce_n<OpSum, NWV>(rsum, sred);
        if (tid == 0) a.dtb_partial[tile] = s2;
    }
    __syncthreads();  // traces of U in place

    // ---- corrected gradient, as the stage forms it; with the flux cotangents to the point lanes
    R jmp[G][FB];
    {
        R jw[2 * G][FB], Q[2 * G][PB], ti[G][FB], fy[G][PB];
#pragma unroll
        for (int q = 0; q < G; ++q)
#pragma unroll
            for (int b = 0; b < FB; ++b) {
                const int4 pa = partner(q, b);
                ti[q][b] = sTu[st(pa.x, pa.y - min(4 * b + row, NFP - 1) % FP) + v];
            }
#pragma unroll
        for (int q = 0; q < G; ++q) {
            R ge[4];
            load4(sGeo + 4 * elg(q), ge);
#pragma unroll
            for (int b = 0; b < PB; ++b) {
                Q[2 * q][b] = ge[0] * gd[q][b] + ge[2] * gd[q][PB + b];
                Q[2 * q + 1][b] = ge[1] * gd[q][b] + ge[3] * gd[q][PB + b];
                fy[q][b] = ge[1] * fx[q][b] + ge[3] * fx[q][PB + b];   // cotangents of F_y, F_x (total fluxes)
                fx[q][b] = ge[0] * fx[q][b] + ge[2] * fx[q][PB + b];
            }
#pragma unroll
            for (int b = 0; b < FB; ++b) {
                const int j = 4 * b + row;
                const R* w = sEw + 4 * (elg(q) * 3 + min(j, NFP - 1) / FP);
                oth[q][b] = edge_of(q, b) == 3 ? ti[q][b] : oth[q][b];
                const R d = R(0.5) * (tu[q][b] + oth[q][b]) - tu[q][b];
                jmp[q][b] = j < NFP ? d : R(0);
                jw[2 * q][b] = w[0] * jmp[q][b];
                jw[2 * q + 1][b] = w[1] * jmp[q][b];
            }
        }
        tri::frag_mma<false, R, 2 * G, PB, FB>(fam + FO::L, jw, Q);
        auto put = [&](int r, auto&& val) {
#pragma unroll
            for (int q = 0; q < G; ++q)
#pragma unroll
                for (int b = 0; b < PB; ++b) sX[sx_(elg(q), r + 4 * b + row) + v] = val(q, b);
            tri::wave_lds_fence();
        };
        put(0, [&](int q, int b) { return Q[2 * q][b]; });
        put(NP, [&](int q, int b) { return Q[2 * q + 1][b]; });
        put(RA, [&](int q, int b) { return fx[q][b]; });
        put(RB, [&](int q, int b) { return fy[q][b]; });
    }
    R ox[G][FB], oy[G][FB];
#pragma unroll
    for (int q = 0; q < G; ++q)
#pragma unroll
        for (int b = 0; b < FB; ++b) {
            const R* T = a.T_in + remote(partner(q, b).w, b);
            ox[q][b] = T[NV];
            oy[q][b] = T[2 * NV];
        }
#pragma unroll 1
    for (int t = lane; t < 4 * G * NP; t += 64) {
        const int el = wave * 4 * G + t / NP, m = t % NP;
        R U4[NV], X4[NV], Y4[NV], A4[NV], B4[NV], Fb[NV], Gb[NV];
        load4(sX + sx_(el, RU + m), U4);
        load4(sX + sx_(el, m), X4);
        load4(sX + sx_(el, NP + m), Y4);
        load4(sX + sx_(el, RA + m), A4);
        load4(sX + sx_(el, RB + m), B4);
        R Ub4[NV] = {R(0), R(0), R(0), R(0)}, Xb4[NV] = {R(0), R(0), R(0), R(0)}, Yb4[NV] = {R(0), R(0), R(0), R(0)};
#pragma unroll
        for (int w = 0; w < NV; ++w) { Fb[w] = -A4[w]; Gb[w] = -B4[w]; }
        euler_flux_vjp(U4, g, A4, B4, Ub4);
        visc_flux_vjp(U4, X4, Y4, g, mu, kappa, Fb, Gb, Ub4, Xb4, Yb4);
        store4(sX + sx_(el, RU + m), Ub4);
        store4(sX + sx_(el, m), Xb4);
        store4(sX + sx_(el, NP + m), Yb4);
    }
    tri::wave_lds_fence();

    // ---- point cotangents back; R5: the lifted jumps backwards, R6: the gradient; the BR2 gradients of both
    // sides of every edge
    R Qb[2 * G][PB], jb[G][FB];
#pragma unroll
    for (int q = 0; q < G; ++q)
#pragma unroll
        for (int b = 0; b < PB; ++b) {
            const R ub = sX[sx_(elg(q), RU + 4 * b + row) + v];
            const R xb = sX[sx_(elg(q), 4 * b + row) + v], yb = sX[sx_(elg(q), NP + 4 * b + row) + v];
            const bool ok = 4 * b + row < NP;
            qb[q][b] += ok ? double(ub) : 0.0;
            Qb[2 * q][b] = ok ? xb : R(0);
            Qb[2 * q + 1][b] = ok ? yb : R(0);
        }
    tri::wave_lds_fence();
    {
        R f2[G][2 * PB], acc[G][PB];
#pragma unroll
        for (int q = 0; q < G; ++q) {
            R ge[4];
            load4(sGeo + 4 * elg(q), ge);
#pragma unroll
            for (int b = 0; b < PB; ++b) {
                f2[q][b] = ge[0] * Qb[2 * q][b] + ge[1] * Qb[2 * q + 1][b];
                f2[q][PB + b] = ge[2] * Qb[2 * q][b] + ge[3] * Qb[2 * q + 1][b];
            }
        }
        tri::frag_mma<true, R, G, PB, 2 * PB>(adj + FO::DT, f2, acc);
#pragma unroll
        for (int q = 0; q < G; ++q)
#pragma unroll
            for (int b = 0; b < PB; ++b) qb[q][b] += double(acc[q][b]);
    }
    {
        R lq[2 * G][FB], tg[G][2 * FB], lo[G][4][FB], gyv[G][FB];
        tri::frag_mma<true, R, 2 * G, FB, PB>(afam + FO::LT, Qb, lq);
        tri::frag_mma<true, R, G, 2 * FB, PB>(ops + FO::G, ur, tg);
        tri::diag_mma<R, P>(fam + FO::LF, jmp, lo);
#pragma unroll
        for (int q = 0; q < G; ++q) {
            R ge[4];
            load4(sGeo + 4 * elg(q), ge);
#pragma unroll
            for (int b = 0; b < FB; ++b) {
                const int j = 4 * b + row, ek = edge_of(q, b);
                R w[4];
                load4(sEw + 4 * (elg(q) * 3 + min(j, NFP - 1) / FP), w);
                jb[q][b] = w[0] * lq[2 * q][b] + w[1] * lq[2 * q + 1][b];
                const R own = eta * lo[q][0][b];
                R gx = ge[0] * tg[q][b] + ge[2] * tg[q][FB + b] + w[0] * own;
                R gy = ge[1] * tg[q][b] + ge[3] * tg[q][FB + b] + w[1] * own;
                const R ln = ek == 0 ? lo[q][1][b] : (ek == 1 ? lo[q][2][b] : lo[q][3][b]);
                gx = ek == 3 ? gx : R(0.5) * (gx + (ox[q][b] + w[2] * ln));
                gy = ek == 3 ? gy : R(0.5) * (gy + (oy[q][b] + w[3] * ln));
                sX[sx_(elg(q), j) + v] = gx;
                gyv[q][b] = gy;
            }
        }
        auto put = [&](int r, const R (&val)[G][FB]) {
            tri::wave_lds_fence();
#pragma unroll
            for (int q = 0; q < G; ++q)
#pragma unroll
                for (int b = 0; b < FB; ++b) sX[sx_(elg(q), r + 4 * b + row) + v] = val[q][b];
        };
        put(RY, gyv);
        put(RO, oth);
        put(RD, db);
    }
    __syncthreads();
    int nsolved = 0;
#pragma unroll
    for (int w = 0; w < NWV; ++w) nsolved += sCnt[w];

    // ---- R3: every solved face point backwards.  Across tiles the partner's
    // slot is the edge's own, written last; each slot is read and written by
    // the lane that solves it alone.
#pragma unroll 1
    for (int t = tid; t < nsolved * FP; t += NB) {
        const int c = sList[t / FP], f = t - (t / FP) * FP;
        const int el = c / 3, j = (c - el * 3) * FP + f;
        const int4 pc = sPa[c];
        const int so = sx_(el, j), sn = pc.z == 3 ? sx_(pc.x, pc.y - f) : so;
        R ns[4], Fcb[NV], ownb[NV], othb[NV], Uc[NV], Ucb[NV] = {R(0), R(0), R(0), R(0)};
        load4(sNs + 4 * c, ns);
        const bool right = ns[2] < R(0);
        {
            R dn[NV];
            load4(sX + so + RD * NV, Fcb);
            load4(sX + sn + RD * NV, dn);
#pragma unroll
            for (int w = 0; w < NV; ++w) Fcb[w] = ns[2] * Fcb[w] + ns[3] * dn[w];
        }
        {
            R own[NV], ot[NV], UL[NV], UR[NV];
            load4(sTu + st(el, j), own);
            load4(sX + so + RO * NV, ot);
            R ULb[NV] = {R(0), R(0), R(0), R(0)}, URb[NV] = {R(0), R(0), R(0), R(0)};
#pragma unroll
            for (int w = 0; w < NV; ++w) {
                Uc[w] = R(0.5) * (own[w] + ot[w]);
                UL[w] = right ? ot[w] : own[w];
                UR[w] = right ? own[w] : ot[w];
            }
            riemann_by_kind_vjp(a.riemann, UL, UR, ns[0], ns[1], g, Fcb, ULb, URb);
#pragma unroll
            for (int w = 0; w < NV; ++w) {
                ownb[w] = right ? URb[w] : ULb[w];
                othb[w] = right ? ULb[w] : URb[w];
            }
        }
        R Qbx[NV], Qby[NV], Qxb[NV] = {R(0), R(0), R(0), R(0)}, Qyb[NV] = {R(0), R(0), R(0), R(0)};
        {
            R gx[NV], gy[NV];
            load4(sX + so, Qbx);
            load4(sX + sn, gx);
            load4(sX + so + RY * NV, Qby);
            load4(sX + sn + RY * NV, gy);
            R Fvb[NV], Gvb[NV];
#pragma unroll
            for (int w = 0; w < NV; ++w) {
                Qbx[w] = R(0.5) * (Qbx[w] + gx[w]);
                Qby[w] = R(0.5) * (Qby[w] + gy[w]);
                Fvb[w] = -Fcb[w] * ns[0];
                Gvb[w] = -Fcb[w] * ns[1];
            }
            visc_flux_vjp(Uc, Qbx, Qby, g, mu, kappa, Fvb, Gvb, Ucb, Qxb, Qyb);
        }
#pragma unroll
        for (int w = 0; w < NV; ++w) {
            ownb[w] += R(0.5) * Ucb[w];
            othb[w] += R(0.5) * Ucb[w];
            Qxb[w] *= R(0.5);
            Qyb[w] *= R(0.5);
        }
        store4(sX + sn, Qxb);
        store4(sX + sn + RY * NV, Qyb);
        store4(sX + sn + RO * NV, othb);
        store4(sTu + st(el, j), othb);
        tri::wave_lds_fence();
        store4(sX + so, Qxb);
        store4(sX + so + RY * NV, Qyb);
        store4(sX + so + RO * NV, ownb);
    }
    __syncthreads();

    // ---- R7: the face liftings backwards; every edge point's jump cotangent, for both sides
    R xh[G][FB], yh[G][FB], jt[G][FB];
    {
        R l[G][4][FB];
#pragma unroll
        for (int q = 0; q < G; ++q)
#pragma unroll
            for (int b = 0; b < FB; ++b) {
                const int j = 4 * b + row, ek = edge_of(q, b);
                const R x = sX[sx_(elg(q), j) + v], y = sX[sx_(elg(q), RY + j) + v];
                R w[4];
                load4(sEw + 4 * (elg(q) * 3 + min(j, NFP - 1) / FP), w);
                xh[q][b] = j < NFP ? x : R(0);
                yh[q][b] = j < NFP ? y : R(0);
                l[q][0][b] = eta * (w[0] * xh[q][b] + w[1] * yh[q][b]);
                const R ln = w[2] * xh[q][b] + w[3] * yh[q][b];
#pragma unroll
                for (int o = 0; o < 3; ++o) l[q][o + 1][b] = ek == o ? ln : R(0);
            }
        tri::diag_mma_t<R, P>(afam + FO::LFT, l, jt);
#pragma unroll
        for (int q = 0; q < G; ++q)
#pragma unroll
            for (int b = 0; b < FB; ++b) {
                jt[q][b] += jb[q][b];
                sX[sx_(elg(q), RD + 4 * b + row) + v] = jt[q][b];
            }
    }
    __syncthreads();

    // ---- R6: traces backwards; cotangent of q
    R f[G][3 * FB], acc[G][PB];
#pragma unroll
    for (int q = 0; q < G; ++q) {
        R ge[4];
        load4(sGeo + 4 * elg(q), ge);
#pragma unroll
        for (int b = 0; b < FB; ++b) {
            const int j = 4 * b + row;
            const int4 pa = partner(q, b);
            const R jn = sX[sx_(pa.x, RD + pa.y - min(j, NFP - 1) % FP) + v];
            const R ub = sX[sx_(elg(q), RO + j) + v], pb = sTu[st(elg(q), j) + v];
            // the partner's own jumps, in the tile; across tiles the other tile adds them there
            const R tub = ub - R(0.5) * jt[q][b] + (pa.z == 3 ? R(0.5) * jn : R(0));
            f[q][b] = j < NFP ? tub : R(0);
            f[q][FB + b] = ge[0] * xh[q][b] + ge[1] * yh[q][b];
            f[q][2 * FB + b] = ge[2] * xh[q][b] + ge[3] * yh[q][b];
            if (pa.z != 3 && j < NFP) {
                R* T = a.Tb_out + remote(pa.w, b);
                T[0] = pb + R(0.5) * jt[q][b];
                T[NV] = xh[q][b];
                T[2 * NV] = yh[q][b];
            }
        }
    }
    tri::frag_mma<true, R, G, PB, 3 * FB>(adj + FO::GT, f, acc);
#pragma unroll
    for (int q = 0; q < G; ++q)
#pragma unroll
        for (int b = 0; b < PB; ++b) {
            if (4 * b + row >= NP || e0 + elg(q) >= a.E) continue;
            double o = qb[q][b] + double(acc[q][b]);
            if (MODE == MODE_STAGE1) o += *rows.at(a.U0b, q, b);
            *rows.at(a.Ub_out, q, b) = o;
        }
}

// The same VJP of large FP32 meshes (TriViscVjpTile): lanes and operators as in
// tri_visc_scalar_kernel, whose reasons hold here too, and the residual formed
// along with the rest, where the matrix-core form takes a launch of its own
// for it.  A step backwards, us, matrix cores / this: P1 without and with
// dJ/d(dt) 500,000 elements 1247 / 966 and 1592 / 1021, 39,200 elements
// 120 / 96 and 171 / 110, 25,088 elements 84 / 80 and 127 / 95; P2 with
// dJ/d(dt) 500,000 elements 2776 / 2161, 32,768 elements 224 / 155, 25,088
// elements 187 / 154 (without, eight waves against four: 2113 / 1909,
// 156 / 130 and 126 / 126).
// Per lane (element, variable) unless stated, after the forward values:
//   R1  cotangent of u_out, the RK combination
//   R2, R4  the lifting, the divergence and the normal fluxes transposed;
//       then one lane per point
//   R5  the corrected gradient's lifted jumps transposed: each edge point's
//       jump cotangent
//   R3  per solved face point; then the face liftings transposed, gathered
//       over the edge's points
//   R6  the traces and the gradient transposed: cotangent of q
template <typename R, int P, int MODE>
__global__ __launch_bounds__(BLOCK) void tri_visc_vjp_scalar_kernel(TriVjpArgs<R> a) {
    using S = TriShape<P>;
    constexpr int NP = S::NP, FP = S::FP, NFP = S::NFP;
    constexpr int TT = TILE, NB = BLOCK, NWV = NB / 64;
    using OP = TriOps<P>;
    constexpr int O0 = ops_offset(P), CA = OP::CA, OI = O0 + OP::C;
    constexpr int XW = 2 * (NP > NFP ? NP : NFP);  // the point fluxes, later the jump cotangents
    constexpr double ca = MODE == MODE_STAGE2 ? 0.75 : (MODE == MODE_STAGE3 ? 1.0 / 3.0 : 0.0);
    constexpr double cb = MODE == MODE_STAGE2 ? 0.25 : (MODE == MODE_STAGE3 ? 2.0 / 3.0 : 1.0);
    constexpr double cc = MODE == MODE_STAGE2 ? 0.25 : (MODE == MODE_STAGE3 ? 2.0 / 3.0 : 1.0);
    const int OLT = O0 + a.lift_off;
    const int LFO = lf_offset(P) + a.lf_off;
    __shared__ R sTu[TT * NFP * NV];   // traces of U
    __shared__ R sTx[TT * NFP * NV];   // traces of the gradient, then their cotangents
    __shared__ R sTy[TT * NFP * NV];
    __shared__ R sD[TT * NFP * NV];    // flux differences, their cotangents, then the U traces' cotangents
    __shared__ R sU[TT * NP * NV];     // q, then the flux VJPs' cotangents of U at the points
    __shared__ R sQx[TT * NP * NV];    // corrected gradient, then its cotangent
    __shared__ R sQy[TT * NP * NV];
    __shared__ R sX[TT * XW * NV];     // contravariant point fluxes, then their x / y cotangents;
                                       // later the jump cotangents and the face liftings' seeds
    __shared__ double sred[NWV];
    __shared__ R sEdge[TT * 3];
    __shared__ int2 sLink[TT * 3];
    __shared__ R sNrm[TT * 3 * 2];
    __shared__ unsigned char sList[TT * 3];
    __shared__ int sCnt[NWV];
    R* const sFR = sX;
    R* const sFS = sX + TT * NP * NV;
    R* const sJ = sX;
    R* const sC = sX + TT * NFP * NV;

    const int tid = threadIdx.x, el = tid >> 2, v = tid & 3;
    const int tile = tile_of_block(a.xcd_groups);
    const int e0 = tile * TT, e = e0 + el;
    const bool live = e < a.E;
    const R g = R(a.gamma), mu = R(a.mu), kappa = R(a.kappa), eta = R(a.eta);
    const int64_t base = blk(e, 0, NP) + v;
    auto sl = [](int elx, int j, int w) { return (elx * NFP + j) * NV + w; };
    auto sp = [](int elx, int m, int w) { return (elx * NP + m) * NV + w; };

    // ---- forward 0: state, gradient, traces of U and of the gradient
    R rx = R(0), ry = R(0), sx = R(0), sy = R(0);
    R jwx[3] = {R(0), R(0), R(0)}, jwy[3] = {R(0), R(0), R(0)};  // each edge's jump weights
    int2 L[3] = {make_int2(0, 0), make_int2(0, 0), make_int2(0, 0)};
    if (live) {
#pragma unroll
        for (int m = 0; m < NP; ++m) sU[sp(el, m, v)] = R(a.U_in[base + (int64_t)m * EB * NV]);
        const R* G = a.geo + (int64_t)e * GEO;
        rx = G[0]; ry = G[1]; sx = G[2]; sy = G[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) L[k] = a.links[(int64_t)e * 3 + k];
        R se[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const R ax = k == 0 ? sx : (k == 1 ? rx + sx : rx), ay = k == 0 ? sy : (k == 1 ? ry + sy : ry);
            se[k] = sqrtR(ax * ax + ay * ay);
            const R sg = link_role(L[k].y) == ROLE_RIGHT ? R(-1) : R(1);
            jwx[k] = sg * se[k] * G[4 + 2 * k];
            jwy[k] = sg * se[k] * G[5 + 2 * k];
        }
        if (v < 3) {
            sEdge[el * 3 + v] = se[v];
            sLink[el * 3 + v] = L[v];
            sNrm[(el * 3 + v) * 2] = G[4 + 2 * v];
            sNrm[(el * 3 + v) * 2 + 1] = G[5 + 2 * v];
        }
        R gr[NP], gs[NP];
#pragma unroll
        for (int i = 0; i < NP; ++i) { gr[i] = R(0); gs[i] = R(0); }
#pragma unroll
        for (int m = 0; m < NP; ++m) {
            const R um = sU[sp(el, m, v)];
#pragma unroll
            for (int i = 0; i < NP; ++i) {
                gr[i] = fmaR(cop<R>(O0 + m * CA + i), um, gr[i]);
                gs[i] = fmaR(cop<R>(O0 + m * CA + NP + i), um, gs[i]);
            }
        }
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            sQx[sp(el, i, v)] = rx * gr[i] + sx * gs[i];
            sQy[sp(el, i, v)] = ry * gr[i] + sy * gs[i];
        }
#pragma unroll 1
        for (int j = 0; j < NFP; ++j) {
            R tu = R(0), tx = R(0), ty = R(0);
#pragma unroll
            for (int m = 0; m < NP; ++m) {
                const R w = cop<R>(OI + j * NP + m);
                tu = fmaR(w, sU[sp(el, m, v)], tu);
                tx = fmaR(w, sQx[sp(el, m, v)], tx);
                ty = fmaR(w, sQy[sp(el, m, v)], ty);
            }
            sTu[sl(el, j, v)] = tu;
            sTx[sl(el, j, v)] = tx;
            sTy[sl(el, j, v)] = ty;
        }
    }
    bool owned = false;
    if (live && v < 3) {
        const int2 Lv = v == 0 ? L[0] : (v == 1 ? L[1] : L[2]);
        const int nl = Lv.x - e0;
        owned = !(link_role(Lv.y) == ROLE_RIGHT && nl >= 0 && nl < TT);
    }
    const unsigned long long own_mask = __ballot(owned);
    const int lane = tid & 63, wave = tid >> 6;
    if (lane == 0) sCnt[wave] = __popcll(own_mask);
    __syncthreads();

    // ---- forward 1: corrected gradient
    if (live) {
        R jx[NFP], jy[NFP];
#pragma unroll
        for (int kk = 0; kk < 3; ++kk) {
            const int2 Lk = L[kk];
            const int nl = Lk.x - e0;
            const bool in = nl >= 0 && nl < TT;
            const int ek = link_edge(Lk.y);
#pragma unroll
            for (int f = 0; f < FP; ++f) {
                const int j = kk * FP + f, oj = ek * FP + (P - f);
                const R own = sTu[sl(el, j, v)];
                R oth;
                if (in) oth = sTu[sl(nl, oj, v)];
                else oth = a.T_in[((int64_t)Lk.x * NFP + oj) * TWV + v];
                const R jmp = R(0.5) * (own + oth) - own;
                jx[j] = jwx[kk] * jmp;
                jy[j] = jwy[kk] * jmp;
            }
        }
#pragma unroll 1
        for (int i = 0; i < NP; ++i) {
            R qx = sQx[sp(el, i, v)], qy = sQy[sp(el, i, v)];
#pragma unroll
            for (int j = 0; j < NFP; ++j) {
                const R l = cop<R>(OLT + j * NP + i);
                qx = fmaR(l, jx[j], qx);
                qy = fmaR(l, jy[j], qy);
            }
            sQx[sp(el, i, v)] = qx;
            sQy[sp(el, i, v)] = qy;
        }
    }
    if (owned) {
        int pos = __popcll(own_mask & ((1ull << lane) - 1));
        for (int w = 0; w < wave; ++w) pos += sCnt[w];
        sList[pos] = (unsigned char)(el * 3 + v);
    }
    __syncthreads();

    // ---- forward 2: contravariant total fluxes at the points (points v, v + 4,
    // ... of the element, four variables each), then this lane's divergence
    // and interpolated normal fluxes
    constexpr int MPL = (NP + NV - 1) / NV;
    if (live) {
#pragma unroll 1
        for (int q = 0; q < MPL; ++q) {
            const int m = v + NV * q;
            if (m >= NP) break;
            R U4[NV], X4[NV], Y4[NV];
#pragma unroll
            for (int w = 0; w < NV; ++w) {
                U4[w] = sU[sp(el, m, w)];
                X4[w] = sQx[sp(el, m, w)];
                Y4[w] = sQy[sp(el, m, w)];
            }
            const R inv = fast_rcp(U4[0]);
            const R ux = U4[1] * inv, uy = U4[2] * inv;
            const R p = (g - R(1)) * (U4[3] - R(0.5) * (U4[1] * ux + U4[2] * uy));
            R Fv[NV], Gv[NV];
            visc_flux(U4, X4, Y4, g, mu, kappa, Fv, Gv);
            const R fx[NV] = {U4[1], U4[1] * ux + p, U4[1] * uy, (U4[3] + p) * ux};
            const R fy[NV] = {U4[2], U4[2] * ux, U4[2] * uy + p, (U4[3] + p) * uy};
#pragma unroll
            for (int w = 0; w < NV; ++w) {
                const R Fx = fx[w] - Fv[w], Fy = fy[w] - Gv[w];
                sFR[sp(el, m, w)] = rx * Fx + ry * Fy;
                sFS[sp(el, m, w)] = sx * Fx + sy * Fy;
            }
        }
    }
    __syncthreads();
    R div[NP];
#pragma unroll
    for (int i = 0; i < NP; ++i) div[i] = R(0);
    if (live) {
        R fn[NFP];
#pragma unroll
        for (int j = 0; j < NFP; ++j) fn[j] = R(0);
#pragma unroll 1
        for (int m = 0; m < NP; ++m) {
            const R fr = sFR[sp(el, m, v)], fs = sFS[sp(el, m, v)], frs = fr + fs;
#pragma unroll
            for (int i = 0; i < NP; ++i)
                div[i] = fmaR(cop<R>(O0 + m * CA + NP + i), fs, fmaR(cop<R>(O0 + m * CA + i), fr, div[i]));
#pragma unroll
            for (int j = 0; j < NFP; ++j)
                fn[j] = fmaR(cop<R>(O0 + m * CA + 2 * NP + j), j < FP ? fs : (j < 2 * FP ? frs : fr), fn[j]);
        }
#pragma unroll
        for (int j = 0; j < NFP; ++j) sD[sl(el, j, v)] = (j >= FP && j < 2 * FP) ? fn[j] : -fn[j];
    }
    __syncthreads();
    int nsolved = 0;
#pragma unroll
    for (int w = 0; w < NWV; ++w) nsolved += sCnt[w];

    // the values of one solved face point (slot j of element elt, edge kk):
    // both sides' traces, edge factors, the face liftings of the jumps and
    // the averaged state and BR2 gradient
    struct Face {
        int elt, kk, j, ek, oj, nl;
        bool in, right;
        int2 Lk;
        R nx, ny, so, sn;
        R own[NV], oth[NV], Uc[NV], Qbx[NV], Qby[NV];
    };
    auto face_at = [&](int t, Face& F) __attribute__((always_inline)) {
        const int c = sList[t / FP], f = t - (t / FP) * FP;
        F.elt = c / 3;
        F.kk = c - F.elt * 3;
        F.j = F.kk * FP + f;
        F.Lk = sLink[F.elt * 3 + F.kk];
        F.right = link_role(F.Lk.y) == ROLE_RIGHT;
        F.nx = sNrm[(F.elt * 3 + F.kk) * 2];
        F.ny = sNrm[(F.elt * 3 + F.kk) * 2 + 1];
        F.ek = link_edge(F.Lk.y);
        F.oj = F.ek * FP + (P - f);
        F.nl = F.Lk.x - e0;
        F.in = F.nl >= 0 && F.nl < TT;
        const R* Tn = a.T_in + (int64_t)F.Lk.x * NFP * TWV;
        R gxo[NV], gyo[NV], gxn[NV], gyn[NV];
#pragma unroll
        for (int w = 0; w < NV; ++w) {
            F.own[w] = sTu[sl(F.elt, F.j, w)];
            gxo[w] = sTx[sl(F.elt, F.j, w)];
            gyo[w] = sTy[sl(F.elt, F.j, w)];
        }
        if (F.in) {
#pragma unroll
            for (int w = 0; w < NV; ++w) {
                F.oth[w] = sTu[sl(F.nl, F.oj, w)];
                gxn[w] = sTx[sl(F.nl, F.oj, w)];
                gyn[w] = sTy[sl(F.nl, F.oj, w)];
            }
            F.sn = sEdge[F.nl * 3 + F.ek];
        } else {
            load4(Tn + (int64_t)F.oj * TWV, F.oth);
            load4(Tn + (int64_t)F.oj * TWV + NV, gxn);
            load4(Tn + (int64_t)F.oj * TWV + 2 * NV, gyn);
            const R* Gn = a.geo + (int64_t)F.Lk.x * GEO;
            const R ax = F.ek == 0 ? Gn[2] : (F.ek == 1 ? Gn[0] + Gn[2] : Gn[0]);
            const R ay = F.ek == 0 ? Gn[3] : (F.ek == 1 ? Gn[1] + Gn[3] : Gn[1]);
            F.sn = sqrtR(ax * ax + ay * ay);
        }
        F.so = sEdge[F.elt * 3 + F.kk];
        R lo[NV] = {R(0), R(0), R(0), R(0)}, ln[NV] = {R(0), R(0), R(0), R(0)};
#pragma unroll 1
        for (int f2 = 0; f2 < FP; ++f2) {
            const int j2 = F.kk * FP + f2, o2 = F.ek * FP + (P - f2);
            R uo[NV], un[NV];
#pragma unroll
            for (int w = 0; w < NV; ++w) uo[w] = sTu[sl(F.elt, j2, w)];
            if (F.in) {
#pragma unroll
                for (int w = 0; w < NV; ++w) un[w] = sTu[sl(F.nl, o2, w)];
            } else {
                load4(Tn + (int64_t)o2 * TWV, un);
            }
            const R wo = clf<R>(LFO + (F.kk * FP + f) * FP + f2);
            const R wn = clf<R>(LFO + (F.ek * FP + (P - f)) * FP + (P - f2));
#pragma unroll
            for (int w = 0; w < NV; ++w) {
                const R jo = R(0.5) * (uo[w] + un[w]) - uo[w];
                lo[w] = fmaR(wo, jo, lo[w]);
                ln[w] = fmaR(wn, jo, ln[w]);
            }
        }
        const R sg = F.right ? R(-1) : R(1);
        const R nox = sg * F.nx, noy = sg * F.ny;
#pragma unroll
        for (int w = 0; w < NV; ++w) {
            F.Uc[w] = R(0.5) * (F.own[w] + F.oth[w]);
            F.Qbx[w] = R(0.5) * ((gxo[w] + eta * F.so * nox * lo[w]) + (gxn[w] + eta * F.sn * nox * ln[w]));
            F.Qby[w] = R(0.5) * ((gyo[w] + eta * F.so * noy * lo[w]) + (gyn[w] + eta * F.sn * noy * ln[w]));
        }
    };

    // ---- forward 3: flux differences of both sides of every solved face point
#pragma unroll 1
    for (int t = tid; t < nsolved * FP; t += NB) {
        Face F;
        face_at(t, F);
        R UL[NV], UR[NV], Fc[NV], Fv[NV], Gv[NV];
#pragma unroll
        for (int w = 0; w < NV; ++w) {
            UL[w] = F.right ? F.oth[w] : F.own[w];
            UR[w] = F.right ? F.own[w] : F.oth[w];
        }
        visc_flux(F.Uc, F.Qbx, F.Qby, g, mu, kappa, Fv, Gv);
        riemann_by_kind(a.riemann, UL, UR, F.nx, F.ny, g, Fc);
        const R sc = F.right ? -F.so : F.so;
#pragma unroll
        for (int w = 0; w < NV; ++w) {
            const R fi = Fc[w] - (Fv[w] * F.nx + Gv[w] * F.ny);
            sD[sl(F.elt, F.j, w)] = sc * fi - sD[sl(F.elt, F.j, w)];
            if (F.in) sD[sl(F.nl, F.oj, w)] = -F.sn * fi - sD[sl(F.nl, F.oj, w)];
        }
    }
    __syncthreads();

    // ---- forward 4 and R1: residual; cotangent of u_out, RK combination
    double rsum = 0.0;
    R divb[NP];
    double qb[NP];
    if (live) {
#pragma unroll 1
        for (int j = 0; j < NFP; ++j) {
            const R d = sD[sl(el, j, v)];
#pragma unroll
            for (int i = 0; i < NP; ++i) div[i] = fmaR(cop<R>(OLT + j * NP + i), d, div[i]);
        }
        double unb[NP];
#pragma unroll
        for (int i = 0; i < NP; ++i) unb[i] = a.Ub_in[base + (int64_t)i * EB * NV];
        if (MODE != MODE_RESIDUAL && a.Tb_in) {
            // edge cotangents of u_out's traces (U, gradient) left on this element's cross-tile edges
            R tu[NFP], tx[NFP], ty[NFP];
            bool any = false;
#pragma unroll
            for (int kk = 0; kk < 3; ++kk) {
                const int nl = L[kk].x - e0;
                const bool cross = !(nl >= 0 && nl < TT);
                any = any || cross;
#pragma unroll
                for (int f = 0; f < FP; ++f) {
                    const int j = kk * FP + f;
                    const R* Tb = a.Tb_in + ((int64_t)e * NFP + j) * TWV;
                    tu[j] = cross ? Tb[v] : R(0);
                    tx[j] = cross ? Tb[NV + v] : R(0);
                    ty[j] = cross ? Tb[2 * NV + v] : R(0);
                }
            }
            if (any) {
                R grb[NP], gsb[NP];
#pragma unroll
                for (int m = 0; m < NP; ++m) {
                    R su = R(0), qx = R(0), qy = R(0);
#pragma unroll
                    for (int j = 0; j < NFP; ++j) {
                        const R w = cop<R>(OI + j * NP + m);
                        su = fmaR(w, tu[j], su);
                        qx = fmaR(w, tx[j], qx);
                        qy = fmaR(w, ty[j], qy);
                    }
                    unb[m] += double(su);
                    grb[m] = rx * qx + ry * qy;
                    gsb[m] = sx * qx + sy * qy;
                }
#pragma unroll
                for (int m = 0; m < NP; ++m) {
                    R acc = R(0);
#pragma unroll
                    for (int i = 0; i < NP; ++i)
                        acc = fmaR(cop<R>(O0 + m * CA + NP + i), gsb[i], fmaR(cop<R>(O0 + m * CA + i), grb[i], acc));
                    unb[m] += double(acc);
                }
            }
        }
        const double dt = MODE == MODE_RESIDUAL ? 0.0 : *a.dt_ptr;
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const int64_t gi = base + (int64_t)i * EB * NV;
            double rb;
            if (MODE == MODE_RESIDUAL) {
                rb = unb[i];
                qb[i] = 0.0;
            } else {
                if (MODE == MODE_STAGE3) a.U0b[gi] = ca * unb[i];
                if (MODE == MODE_STAGE2) a.U0b[gi] += ca * unb[i];
                qb[i] = cb * unb[i];
                rb = cc * dt * unb[i];
                rsum += cc * (-double(div[i])) * unb[i];
            }
            divb[i] = R(-rb);  // R = -div
        }
    } else {
#pragma unroll
        for (int i = 0; i < NP; ++i) { divb[i] = R(0); qb[i] = 0.0; }
    }
    if (a.dtb_partial) {
        const double s2 = block_reduce_n<OpSum, NWV>(rsum, sred);
        if (tid == 0) a.dtb_partial[tile] = s2;
    }
    __syncthreads();

    // ---- R2, R4: the lifting transposed; the divergence and normal fluxes
    // transposed to the x / y flux cotangents at the points
    if (live) {
#pragma unroll 1
        for (int j = 0; j < NFP; ++j) {
            R acc = R(0);
#pragma unroll
            for (int i = 0; i < NP; ++i) acc = fmaR(cop<R>(OLT + j * NP + i), divb[i], acc);
            sD[sl(el, j, v)] = acc;
        }
#pragma unroll 1
        for (int m = 0; m < NP; ++m) {
            R frb = R(0), fsb = R(0);
#pragma unroll
            for (int i = 0; i < NP; ++i) {
                frb = fmaR(cop<R>(O0 + m * CA + i), divb[i], frb);
                fsb = fmaR(cop<R>(O0 + m * CA + NP + i), divb[i], fsb);
            }
#pragma unroll
            for (int j = 0; j < NFP; ++j) {
                // d = sc F^I - Fn with Fn = -fn (edges 0, 2), +fn (edge 1); fn_j
                // interpolates fs, fr + fs, fr on edges 0, 1, 2
                const R im = cop<R>(O0 + m * CA + 2 * NP + j);
                const R db = sD[sl(el, j, v)];
                const R fnb = (j >= FP && j < 2 * FP) ? -db : db;
                if (j >= FP) frb = fmaR(im, fnb, frb);
                if (j < 2 * FP) fsb = fmaR(im, fnb, fsb);
            }
            sFR[sp(el, m, v)] = rx * frb + sx * fsb;  // cotangent of F_x = f_x - F_v
            sFS[sp(el, m, v)] = ry * frb + sy * fsb;  // and of F_y
        }
    }
    __syncthreads();
    if (live) {
#pragma unroll 1
        for (int q = 0; q < MPL; ++q) {
            const int m = v + NV * q;
            if (m >= NP) break;
            R U4[NV], X4[NV], Y4[NV], A4[NV], B4[NV], Fb[NV], Gb[NV];
#pragma unroll
            for (int w = 0; w < NV; ++w) {
                U4[w] = sU[sp(el, m, w)];
                X4[w] = sQx[sp(el, m, w)];
                Y4[w] = sQy[sp(el, m, w)];
                A4[w] = sFR[sp(el, m, w)];
                B4[w] = sFS[sp(el, m, w)];
                Fb[w] = -A4[w];
                Gb[w] = -B4[w];
            }
            R Ub4[NV] = {R(0), R(0), R(0), R(0)}, Xb4[NV] = {R(0), R(0), R(0), R(0)},
              Yb4[NV] = {R(0), R(0), R(0), R(0)};
            euler_flux_vjp(U4, g, A4, B4, Ub4);
            visc_flux_vjp(U4, X4, Y4, g, mu, kappa, Fb, Gb, Ub4, Xb4, Yb4);
#pragma unroll
            for (int w = 0; w < NV; ++w) {
                sU[sp(el, m, w)] = Ub4[w];
                sQx[sp(el, m, w)] = Xb4[w];
                sQy[sp(el, m, w)] = Yb4[w];
            }
        }
    }
    __syncthreads();

    // ---- R5: the corrected gradient's lifted jumps transposed
    if (live) {
#pragma unroll 1
        for (int j = 0; j < NFP; ++j) {
            R bx = R(0), by = R(0);
#pragma unroll
            for (int i = 0; i < NP; ++i) {
                const R l = cop<R>(OLT + j * NP + i);
                bx = fmaR(l, sQx[sp(el, i, v)], bx);
                by = fmaR(l, sQy[sp(el, i, v)], by);
            }
            const int kk = j / FP;
            sJ[sl(el, j, v)] = (kk == 0 ? jwx[0] : (kk == 1 ? jwx[1] : jwx[2])) * bx +
                               (kk == 0 ? jwy[0] : (kk == 1 ? jwy[1] : jwy[2])) * by;
        }
    }
    __syncthreads();

    // ---- R3: every solved face point backwards
#pragma unroll 1
    for (int t = tid; t < nsolved * FP; t += NB) {
        Face F;
        face_at(t, F);
        R UL[NV], UR[NV], Fcb[NV], Fvb[NV], Gvb[NV];
        const R sc = F.right ? -F.so : F.so;
#pragma unroll
        for (int w = 0; w < NV; ++w) {
            UL[w] = F.right ? F.oth[w] : F.own[w];
            UR[w] = F.right ? F.own[w] : F.oth[w];
            R fb = sc * sD[sl(F.elt, F.j, w)];
            if (F.in) fb += -F.sn * sD[sl(F.nl, F.oj, w)];
            Fcb[w] = fb;
            Fvb[w] = -fb * F.nx;
            Gvb[w] = -fb * F.ny;
        }
        R ULb[NV] = {R(0), R(0), R(0), R(0)}, URb[NV] = {R(0), R(0), R(0), R(0)};
        riemann_by_kind_vjp(a.riemann, UL, UR, F.nx, F.ny, g, Fcb, ULb, URb);
        R Ucb[NV] = {R(0), R(0), R(0), R(0)}, Qxb[NV] = {R(0), R(0), R(0), R(0)}, Qyb[NV] = {R(0), R(0), R(0), R(0)};
        visc_flux_vjp(F.Uc, F.Qbx, F.Qby, g, mu, kappa, Fvb, Gvb, Ucb, Qxb, Qyb);
        const R sg = F.right ? R(-1) : R(1);
        const R nox = sg * F.nx, noy = sg * F.ny;
        R ownb[NV], othb[NV];
#pragma unroll
        for (int w = 0; w < NV; ++w) {
            const R jo = sJ[sl(F.elt, F.j, w)], jn = F.in ? sJ[sl(F.nl, F.oj, w)] : R(0);
            ownb[w] = (F.right ? URb[w] : ULb[w]) + R(0.5) * Ucb[w] - R(0.5) * jo + R(0.5) * jn;
            othb[w] = (F.right ? ULb[w] : URb[w]) + R(0.5) * Ucb[w] + R(0.5) * jo - R(0.5) * jn;
            Qxb[w] *= R(0.5);
            Qyb[w] *= R(0.5);
            sC[sl(F.elt, F.j, w)] = eta * (nox * Qxb[w] + noy * Qyb[w]);
            sD[sl(F.elt, F.j, w)] = ownb[w];
            sTx[sl(F.elt, F.j, w)] = Qxb[w];
            sTy[sl(F.elt, F.j, w)] = Qyb[w];
        }
        if (F.in) {
#pragma unroll
            for (int w = 0; w < NV; ++w) {
                sD[sl(F.nl, F.oj, w)] = othb[w];
                sTx[sl(F.nl, F.oj, w)] = Qxb[w];
                sTy[sl(F.nl, F.oj, w)] = Qyb[w];
            }
        } else {
            R* Tb = a.Tb_out + ((int64_t)F.Lk.x * NFP + F.oj) * TWV;
            store4(Tb, othb);
            store4(Tb + NV, Qxb);
            store4(Tb + 2 * NV, Qyb);
        }
    }
    __syncthreads();
    // the face liftings transposed: the jump at this point from every point's
    // lifting cotangents (the seeds c, times each side's edge factor)
#pragma unroll 1
    for (int t = tid; t < nsolved * FP; t += NB) {
        const int c = sList[t / FP], f = t - (t / FP) * FP;
        const int elt = c / 3, kk = c - elt * 3, j = kk * FP + f;
        const int2 Lk = sLink[elt * 3 + kk];
        const int ek = link_edge(Lk.y), oj = ek * FP + (P - f), nl = Lk.x - e0;
        const bool in = nl >= 0 && nl < TT;
        const R so = sEdge[elt * 3 + kk];
        R sn;
        if (in) {
            sn = sEdge[nl * 3 + ek];
        } else {
            const R* Gn = a.geo + (int64_t)Lk.x * GEO;
            const R ax = ek == 0 ? Gn[2] : (ek == 1 ? Gn[0] + Gn[2] : Gn[0]);
            const R ay = ek == 0 ? Gn[3] : (ek == 1 ? Gn[1] + Gn[3] : Gn[1]);
            sn = sqrtR(ax * ax + ay * ay);
        }
        R jb[NV] = {R(0), R(0), R(0), R(0)};
#pragma unroll 1
        for (int f1 = 0; f1 < FP; ++f1) {
            const R w1 = so * clf<R>(LFO + (kk * FP + f1) * FP + f) +
                         sn * clf<R>(LFO + (ek * FP + (P - f1)) * FP + (P - f));
#pragma unroll
            for (int w = 0; w < NV; ++w) jb[w] = fmaR(w1, sC[sl(elt, kk * FP + f1, w)], jb[w]);
        }
        // jump = (u_n - u_o) / 2 at this point
#pragma unroll
        for (int w = 0; w < NV; ++w) sD[sl(elt, j, w)] -= R(0.5) * jb[w];
        if (in) {
#pragma unroll
            for (int w = 0; w < NV; ++w) sD[sl(nl, oj, w)] += R(0.5) * jb[w];
        } else {
            R* Tb = a.Tb_out + ((int64_t)Lk.x * NFP + oj) * TWV;
#pragma unroll
            for (int w = 0; w < NV; ++w) Tb[w] += R(0.5) * jb[w];
        }
    }
    __syncthreads();

    // ---- R6: traces and gradient transposed; cotangent of q
    if (!live) return;
    R grb[NP], gsb[NP];
    double out[NP];
#pragma unroll
    for (int m = 0; m < NP; ++m) {
        R su = R(0), qx = sQx[sp(el, m, v)], qy = sQy[sp(el, m, v)];
#pragma unroll
        for (int j = 0; j < NFP; ++j) {
            const R w = cop<R>(OI + j * NP + m);
            su = fmaR(w, sD[sl(el, j, v)], su);
            qx = fmaR(w, sTx[sl(el, j, v)], qx);
            qy = fmaR(w, sTy[sl(el, j, v)], qy);
        }
        out[m] = qb[m] + double(sU[sp(el, m, v)]) + double(su);
        grb[m] = rx * qx + ry * qy;
        gsb[m] = sx * qx + sy * qy;
    }
#pragma unroll
    for (int m = 0; m < NP; ++m) {
        R acc = R(0);
#pragma unroll
        for (int i = 0; i < NP; ++i)
            acc = fmaR(cop<R>(O0 + m * CA + NP + i), gsb[i], fmaR(cop<R>(O0 + m * CA + i), grb[i], acc));
        const int64_t gi = base + (int64_t)m * EB * NV;
        double o = out[m] + double(acc);
        if (MODE == MODE_STAGE1) o += a.U0b[gi];
        a.Ub_out[gi] = o;
    }
}

// Completion of a cotangent with the Navier-Stokes terms: U_bar plus the
// transposed traces of U and of its gradient for the cross-tile edge
// cotangents (12 words per point) that the last adjoint launch left (tiles of
// TT elements).  Without any (Tb null) a copy.  Every load that does not hang
// on another goes out first, and 32 elements share the tables in LDS: with
// tables and links read where they are used, and for the copy too,
// adjoint_get_device of 500,000 elements at P3 FP64 with cotangents pending
// took 295 us, this 178, one lane per element and variable 183; at P5 FP32
// 348, 298 and 336.  At P1 and P2, where a wave has little to share, the form
// below is the quicker: 500,000 elements FP64, this / that, P1 78 / 67, P2
// 133 / 126, and 33,800 elements P2 FP32 12.8 / 11.9.
template <typename R, int P, int TT>
__global__ __launch_bounds__(BLOCK) void tri_visc_complete_kernel(int E, const int2* __restrict__ links,
                                                                  const R* __restrict__ geo,
                                                                  const double* __restrict__ Ub,
                                                                  const R* __restrict__ Tb,
                                                                  double* __restrict__ out) {
    using FO = tri::FragOps<R, P>;
    constexpr int NP = FO::NP, FP = FO::FP, NFP = FO::NFP, PB = FO::PB, FB = FO::FB, G = TRACE_G;
    __shared__ R ops[FO::DT - FO::GT];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, row = lane >> 4, v = lane & 3;
    const int e0 = blockIdx.x * TRACE_TILE;
    auto elg = [&](int q) { return e0 + (wave * G + q) * 4 + ((lane >> 2) & 3); };
    const PointRows<NP, G> rows(e0, wave, lane, E);
    double o[G][PB];
#pragma unroll
    for (int q = 0; q < G; ++q)
#pragma unroll
        for (int b = 0; b < PB; ++b) o[q][b] = *rows.at(Ub, q, b);
    if (Tb) {
        const R* const src = frag_ops<R>() + tri::frag_offset<R>(P) + FO::ADJ0 + FO::GT;
        for (int t = 4 * threadIdx.x; t < FO::DT - FO::GT; t += 4 * BLOCK) {
            R w[4];
            load4(src + t, w);
            store4(ops + t, w);
        }
        R f[G][3 * FB], acc[G][PB];
        int n[G][3];
#pragma unroll
        for (int q = 0; q < G; ++q)
#pragma unroll
            for (int k = 0; k < 3; ++k) n[q][k] = links[(int64_t)min(elg(q), E - 1) * 3 + k].x;
#pragma unroll
        for (int q = 0; q < G; ++q) {
            const int e = min(elg(q), E - 1);
            const R* Ge = geo + (int64_t)e * GEO;
            const R rx = Ge[0], ry = Ge[1], sx = Ge[2], sy = Ge[3];
#pragma unroll
            for (int b = 0; b < FB; ++b) {
                // slots across tiles (the others read the first row in common)
                const int j = 4 * b + row, k = min(j, NFP - 1) / FP;
                const bool on = j < NFP && (k == 0 ? n[q][0] : (k == 1 ? n[q][1] : n[q][2])) / TT != e / TT;
                const R* T = Tb + (on ? (int64_t)e * NFP + j : (int64_t)0) * TWV + v;
                const R tb = T[0], xb = T[NV], yb = T[2 * NV];
                f[q][b] = on ? tb : R(0);
                f[q][FB + b] = on ? rx * xb + ry * yb : R(0);
                f[q][2 * FB + b] = on ? sx * xb + sy * yb : R(0);
            }
        }
        __syncthreads();
        tri::frag_mma<true, R, G, PB, 3 * FB>(ops, f, acc);
#pragma unroll
        for (int q = 0; q < G; ++q)
#pragma unroll
            for (int b = 0; b < PB; ++b) o[q][b] += double(acc[q][b]);
    }
#pragma unroll
    for (int q = 0; q < G; ++q)
#pragma unroll
        for (int b = 0; b < PB; ++b)
            if (4 * b + row < NP && elg(q) < E) *rows.at(out, q, b) = o[q][b];
}

// The same at P1 and P2, one lane per element and variable.
template <typename R, int P, int TT>
__global__ __launch_bounds__(TT * NV) void tri_visc_complete_scalar_kernel(int E, const int2* __restrict__ links,
                                                                           const R* __restrict__ geo,
                                                                           const double* __restrict__ Ub,
                                                                           const R* __restrict__ Tb,
                                                                           double* __restrict__ out, int xcd_groups) {
    using S = TriShape<P>;
    constexpr int NP = S::NP, FP = S::FP, NFP = S::NFP;
    constexpr int O0 = ops_offset(P), CA = TriOps<P>::CA, OI = O0 + TriOps<P>::C;
    const int tid = threadIdx.x, el = tid >> 2, v = tid & 3;
    const int e0 = tile_of_block(xcd_groups) * TT, e = e0 + el;
    if (e >= E) return;
    const int64_t base = blk(e, 0, NP) + v;
    double acc[NP];
#pragma unroll
    for (int i = 0; i < NP; ++i) acc[i] = Ub[base + (int64_t)i * EB * NV];
    if (Tb) {
        R tu[NFP], tx[NFP], ty[NFP];
#pragma unroll
        for (int kk = 0; kk < 3; ++kk) {
            const int2 Lk = links[(int64_t)e * 3 + kk];
            const int nl = Lk.x - e0;
            const bool cross = !(nl >= 0 && nl < TT);
#pragma unroll
            for (int f = 0; f < FP; ++f) {
                const int j = kk * FP + f;
                const R* T = Tb + ((int64_t)e * NFP + j) * TWV;
                tu[j] = cross ? T[v] : R(0);
                tx[j] = cross ? T[NV + v] : R(0);
                ty[j] = cross ? T[2 * NV + v] : R(0);
            }
        }
        const R* G = geo + (int64_t)e * GEO;
        const R rx = G[0], ry = G[1], sx = G[2], sy = G[3];
        R grb[NP], gsb[NP];
#pragma unroll
        for (int m = 0; m < NP; ++m) {
            R su = R(0), qx = R(0), qy = R(0);
#pragma unroll
            for (int j = 0; j < NFP; ++j) {
                const R w = cop<R>(OI + j * NP + m);
                su = fmaR(w, tu[j], su);
                qx = fmaR(w, tx[j], qx);
                qy = fmaR(w, ty[j], qy);
            }
            acc[m] += double(su);
            grb[m] = rx * qx + ry * qy;
            gsb[m] = sx * qx + sy * qy;
        }
#pragma unroll
        for (int m = 0; m < NP; ++m) {
            R s = R(0);
#pragma unroll
            for (int i = 0; i < NP; ++i)
                s = fmaR(cop<R>(O0 + m * CA + NP + i), gsb[i], fmaR(cop<R>(O0 + m * CA + i), grb[i], s));
            acc[m] += double(s);
        }
    }
#pragma unroll
    for (int i = 0; i < NP; ++i) out[base + (int64_t)i * EB * NV] = acc[i];
}

// Traces of U on every edge (after a new state is set).
template <typename R, int P>
__global__ __launch_bounds__(BLOCK) void tri_trace_kernel(int E, const double* U, R* T_out) {
    using S = TriShape<P>;
    constexpr int NP = S::NP, NFP = S::NFP, OI = ops_offset(P) + TriOps<P>::C;
    const int e = blockIdx.x * TILE + (threadIdx.x >> 2), v = threadIdx.x & 3;
    if (e >= E) return;
    R u[NP];
#pragma unroll
    for (int m = 0; m < NP; ++m) u[m] = R(U[blk(e, m, NP) + v]);
#pragma unroll 1
    for (int j = 0; j < NFP; ++j) {
        R t = R(0);
#pragma unroll
        for (int m = 0; m < NP; ++m) t = fmaR(cop<R>(OI + j * NP + m), u[m], t);
        T_out[trix(e, j, NFP) + v] = t;
    }
}

// Caller AoS [E][Np][4] (caller numbering) <-> blocked device layout.
__global__ void tri_to_blk_kernel(const double* __restrict__ aos, double* __restrict__ out, int E, int NP,
                                  const int* __restrict__ perm) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (int64_t)E * NP) return;
    const int e = (int)(t / NP), i = (int)(t - (int64_t)e * NP);
    const int src = perm ? perm[e] : e;
    double q[NV];
    load4(aos + ((int64_t)src * NP + i) * NV, q);
    store4(out + blk(e, i, NP), q);
}

__global__ void tri_from_blk_kernel(const double* __restrict__ in, double* __restrict__ aos, int E, int NP,
                                    const int* __restrict__ perm) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (int64_t)E * NP) return;
    const int e = (int)(t / NP), i = (int)(t - (int64_t)e * NP);
    const int dst = perm ? perm[e] : e;
    double q[NV];
    load4(in + blk(e, i, NP), q);
    store4(aos + ((int64_t)dst * NP + i) * NV, q);
}

// CFL step per point of the blocked state, minimum per workgroup.  With the
// viscous terms (nu_k = mu max(4/3, gamma/Pr), else 0) the diffusive rate
// (p+1)^4 nu_k / (rho d^2) joins the convective (2p+1)(|u|+c)/d: the
// spectral radius of the BR2 operator on triangles is about 1.3 (p+1)^4
// nu / d^2 (P2-P4; 1.7 at P1), d the inscribed-circle diameter.
__global__ __launch_bounds__(BLOCK) void tri_dt_kernel(const double* __restrict__ U, const double* __restrict__ hcell,
                                                       int E, int NP, double gamma, double cfl, double cf,
                                                       double visc, double* __restrict__ partial) {
    __shared__ double sRed[BLOCK / 64];
    const int64_t n = (int64_t)E * NP;
    double mn = 1e20;
    for (int64_t t = (int64_t)blockIdx.x * BLOCK + threadIdx.x; t < n; t += (int64_t)gridDim.x * BLOCK) {
        const int e = (int)(t / NP), i = (int)(t - (int64_t)e * NP);
        double q[NV];
        load4(U + blk(e, i, NP), q);
        const double u = q[1] / q[0], w = q[2] / q[0];
        const double p = (gamma - 1.0) * q[0] * (q[3] / q[0] - 0.5 * (u * u + w * w));
        const double ws = sqrt(u * u + w * w) + sqrt(gamma * fmax(p, 1e-10) / fmax(q[0], 1e-10));
        const double h = hcell[e];
        const double d = cfl / (cf * ws / h + visc / (fmax(q[0], 1e-10) * h * h));
        mn = d < mn ? d : mn;
    }
    const double r = block_reduce<OpMin>(mn, sRed);
    if (threadIdx.x == 0) partial[blockIdx.x] = r;
}

template <typename R, int P>
hipError_t tri_launch_p(int mode, const TriArgs<R>& a, hipStream_t s) {
    using TV = TriTile<R, P>;
    auto launch = [&](auto m) {
        constexpr int MODE = decltype(m)::value;
        const int TT = MODE == MODE_RESIDUAL ? TV::residual_tile(a.E) : TV::tile(a.E);
        const int grid = (std::max(a.E, 1) + TT - 1) / TT;
        if constexpr ((MODE == MODE_RESIDUAL ? TV::RESIDUAL_FROM : TV::SCALAR_FROM) < INT_MAX)
            if (TT == TILE) {
                klaunch(tri_scalar_kernel<R, P, MODE>, grid, dim3(BLOCK), 0, s, a);
                return;
            }
        klaunch(tri_stage_kernel<R, P, MODE>, grid, dim3(64 * TV::WV), 0, s, a);
    };
    switch (mode) {
    case MODE_RESIDUAL: launch(std::integral_constant<int, MODE_RESIDUAL>{}); break;
    case MODE_STAGE1: launch(std::integral_constant<int, MODE_STAGE1>{}); break;
    case MODE_STAGE2: launch(std::integral_constant<int, MODE_STAGE2>{}); break;
    default: launch(std::integral_constant<int, MODE_STAGE3>{}); break;
    }
    return hipGetLastError();
}

template <typename R>
hipError_t tri_launch(int P, int mode, const TriArgs<R>& a, hipStream_t s) {
    switch (P) {
    case 1: return tri_launch_p<R, 1>(mode, a, s);
    case 2: return tri_launch_p<R, 2>(mode, a, s);
    case 3: return tri_launch_p<R, 3>(mode, a, s);
    case 4: return tri_launch_p<R, 4>(mode, a, s);
    default: return tri_launch_p<R, 5>(mode, a, s);
    }
}

template <typename R, int P>
hipError_t tri_visc_launch_p(int mode, const TriArgs<R>& a, hipStream_t s) {
    if constexpr (std::is_same<R, double>::value && P == 4) {
        return hipErrorInvalidValue;  // refused when the handle is made
    } else {
        using TV = TriViscTile<R, P>;
        const int TT = TV::tile(a.E), grid = (std::max(a.E, 1) + TT - 1) / TT;
        auto launch = [&](auto m) {
            constexpr int MODE = decltype(m)::value;
            if constexpr (TV::SCALAR_FROM < INT_MAX)
                if (a.E >= TV::SCALAR_FROM) {
                    klaunch(tri_visc_scalar_kernel<R, P, MODE>, grid, dim3(BLOCK), 0, s, a);
                    return;
                }
            klaunch(tri_visc_stage_kernel<R, P, MODE>, grid, dim3(64 * TV::WV), 0, s, a);
        };
        switch (mode) {
        case MODE_RESIDUAL: launch(std::integral_constant<int, MODE_RESIDUAL>{}); break;
        case MODE_STAGE1: launch(std::integral_constant<int, MODE_STAGE1>{}); break;
        case MODE_STAGE2: launch(std::integral_constant<int, MODE_STAGE2>{}); break;
        default: launch(std::integral_constant<int, MODE_STAGE3>{}); break;
        }
        return hipGetLastError();
    }
}

template <typename R>
hipError_t tri_visc_launch(int P, int mode, const TriArgs<R>& a, hipStream_t s) {
    switch (P) {
    case 1: return tri_visc_launch_p<R, 1>(mode, a, s);
    case 2: return tri_visc_launch_p<R, 2>(mode, a, s);
    case 3: return tri_visc_launch_p<R, 3>(mode, a, s);
    case 4: return tri_visc_launch_p<R, 4>(mode, a, s);
    default: return tri_visc_launch_p<R, 5>(mode, a, s);
    }
}

template <typename R>
hipError_t tri_visc_trace(int P, int E, const double* U, const R* geo, R* T, hipStream_t s) {
    const int grid = (std::max(E, 1) + TRACE_TILE - 1) / TRACE_TILE;
    switch (P) {
    case 1: tri_visc_trace_kernel<R, 1><<<grid, BLOCK, 0, s>>>(E, U, geo, T); break;
    case 2: tri_visc_trace_kernel<R, 2><<<grid, BLOCK, 0, s>>>(E, U, geo, T); break;
    case 3: tri_visc_trace_kernel<R, 3><<<grid, BLOCK, 0, s>>>(E, U, geo, T); break;
    case 4: tri_visc_trace_kernel<R, 4><<<grid, BLOCK, 0, s>>>(E, U, geo, T); break;
    default: tri_visc_trace_kernel<R, 5><<<grid, BLOCK, 0, s>>>(E, U, geo, T); break;
    }
    return hipGetLastError();
}

int tri_visc_tile(int P, bool fp64, int E) {
    switch (P) {
    case 1: return fp64 ? TriViscTile<double, 1>::tile(E) : TriViscTile<float, 1>::tile(E);
    case 2: return fp64 ? TriViscTile<double, 2>::tile(E) : TriViscTile<float, 2>::tile(E);
    case 3: return fp64 ? TriViscTile<double, 3>::tile(E) : TriViscTile<float, 3>::tile(E);
    case 4: return fp64 ? TriViscTile<double, 4>::tile(E) : TriViscTile<float, 4>::tile(E);
    default: return fp64 ? TriViscTile<double, 5>::tile(E) : TriViscTile<float, 5>::tile(E);
    }
}

int tri_tile(int P, bool fp64, int E) {
    switch (P) {
    case 1: return fp64 ? TriTile<double, 1>::tile(E) : TriTile<float, 1>::tile(E);
    case 2: return fp64 ? TriTile<double, 2>::tile(E) : TriTile<float, 2>::tile(E);
    case 3: return fp64 ? TriTile<double, 3>::tile(E) : TriTile<float, 3>::tile(E);
    case 4: return fp64 ? TriTile<double, 4>::tile(E) : TriTile<float, 4>::tile(E);
    default: return fp64 ? TriTile<double, 5>::tile(E) : TriTile<float, 5>::tile(E);
    }
}

int tri_residual_tile(int P, bool fp64, int E) {
    switch (P) {
    case 1: return fp64 ? TriTile<double, 1>::residual_tile(E) : TriTile<float, 1>::residual_tile(E);
    case 2: return fp64 ? TriTile<double, 2>::residual_tile(E) : TriTile<float, 2>::residual_tile(E);
    case 3: return fp64 ? TriTile<double, 3>::residual_tile(E) : TriTile<float, 3>::residual_tile(E);
    case 4: return fp64 ? TriTile<double, 4>::residual_tile(E) : TriTile<float, 4>::residual_tile(E);
    default: return fp64 ? TriTile<double, 5>::residual_tile(E) : TriTile<float, 5>::residual_tile(E);
    }
}

template <typename R, int P>
hipError_t tri_vjp_p(int mode, const TriVjpArgs<R>& a, hipStream_t s) {
    const int grid = (std::max(a.E, 1) + TILE - 1) / TILE;
    switch (mode) {
    case MODE_RESIDUAL: tri_vjp_kernel<R, P, MODE_RESIDUAL><<<grid, BLOCK, 0, s>>>(a); break;
    case MODE_STAGE1: tri_vjp_kernel<R, P, MODE_STAGE1><<<grid, BLOCK, 0, s>>>(a); break;
    case MODE_STAGE2: tri_vjp_kernel<R, P, MODE_STAGE2><<<grid, BLOCK, 0, s>>>(a); break;
    default: tri_vjp_kernel<R, P, MODE_STAGE3><<<grid, BLOCK, 0, s>>>(a); break;
    }
    return hipGetLastError();
}

template <typename R>
hipError_t tri_vjp(int P, int mode, const TriVjpArgs<R>& a, hipStream_t s) {
    switch (P) {
    case 1: return tri_vjp_p<R, 1>(mode, a, s);
    case 2: return tri_vjp_p<R, 2>(mode, a, s);
    case 3: return tri_vjp_p<R, 3>(mode, a, s);
    case 4: return tri_vjp_p<R, 4>(mode, a, s);
    default: return tri_vjp_p<R, 5>(mode, a, s);
    }
}

template <typename R>
hipError_t tri_complete(int P, int E, const int2* links, const double* Ub, const R* Tb, double* out, int xcd,
                        hipStream_t s) {
    const int grid = (std::max(E, 1) + TILE - 1) / TILE;
    switch (P) {
    case 1: tri_complete_kernel<R, 1><<<grid, BLOCK, 0, s>>>(E, links, Ub, Tb, out, xcd); break;
    case 2: tri_complete_kernel<R, 2><<<grid, BLOCK, 0, s>>>(E, links, Ub, Tb, out, xcd); break;
    case 3: tri_complete_kernel<R, 3><<<grid, BLOCK, 0, s>>>(E, links, Ub, Tb, out, xcd); break;
    case 4: tri_complete_kernel<R, 4><<<grid, BLOCK, 0, s>>>(E, links, Ub, Tb, out, xcd); break;
    default: tri_complete_kernel<R, 5><<<grid, BLOCK, 0, s>>>(E, links, Ub, Tb, out, xcd); break;
    }
    return hipGetLastError();
}

// The BR2 adjoint's elements per workgroup for an order, precision and mesh size.
int tri_visc_vjp_tile(int P, bool fp64, int E) {
    switch (P) {
    case 1: return fp64 ? TriViscVjpTile<double, 1>::tile(E) : TriViscVjpTile<float, 1>::tile(E);
    case 2: return fp64 ? TriViscVjpTile<double, 2>::tile(E) : TriViscVjpTile<float, 2>::tile(E);
    case 3: return fp64 ? TriViscVjpTile<double, 3>::tile(E) : TriViscVjpTile<float, 3>::tile(E);
    case 4: return fp64 ? TriViscVjpTile<double, 4>::tile(E) : TriViscVjpTile<float, 4>::tile(E);
    default: return fp64 ? TriViscVjpTile<double, 5>::tile(E) : TriViscVjpTile<float, 5>::tile(E);
    }
}

// Whether the VJP of a mesh forms the residual itself for dJ/d(dt).
template <typename R> bool tri_visc_vjp_has_residual(int P, int E) {
    return E >= (P == 1 ? TriViscVjpTile<R, 1>::LARGE_FROM : P == 2 ? TriViscVjpTile<R, 2>::LARGE_FROM : INT_MAX);
}

template <typename R, int P>
hipError_t tri_visc_vjp_p(int mode, const TriVjpArgs<R>& a, hipStream_t s) {
    if constexpr (std::is_same<R, double>::value && P == 4) {
        return hipErrorInvalidValue;  // refused when the handle is made
    } else {
        using TV = TriViscVjpTile<R, P>;
        const int TT = TV::tile(a.E), grid = (std::max(a.E, 1) + TT - 1) / TT;
        auto launch = [&](auto m) {
            constexpr int MODE = decltype(m)::value;
            if constexpr (TV::LARGE_FROM < INT_MAX)
                if (a.E >= TV::LARGE_FROM) {
                    if constexpr (P == 2) {
                        if (MODE == MODE_RESIDUAL || !a.dtb_partial) {
                            klaunch(tri_visc_vjp_kernel<R, P, MODE, 2 * TV::WV>, grid, dim3(128 * TV::WV), 0, s, a);
                            return;
                        }
                    }
                    if constexpr (P == 1 || MODE != MODE_RESIDUAL)
                        klaunch(tri_visc_vjp_scalar_kernel<R, P, MODE>, grid, dim3(BLOCK), 0, s, a);
                    return;
                }
            klaunch(tri_visc_vjp_kernel<R, P, MODE, TV::WV>, grid, dim3(64 * TV::WV), 0, s, a);
        };
        switch (mode) {
        case MODE_RESIDUAL: launch(std::integral_constant<int, MODE_RESIDUAL>{}); break;
        case MODE_STAGE1: launch(std::integral_constant<int, MODE_STAGE1>{}); break;
        case MODE_STAGE2: launch(std::integral_constant<int, MODE_STAGE2>{}); break;
        default: launch(std::integral_constant<int, MODE_STAGE3>{}); break;
        }
        return hipGetLastError();
    }
}

template <typename R>
hipError_t tri_visc_vjp(int P, int mode, const TriVjpArgs<R>& a, hipStream_t s) {
    switch (P) {
    case 1: return tri_visc_vjp_p<R, 1>(mode, a, s);
    case 2: return tri_visc_vjp_p<R, 2>(mode, a, s);
    case 3: return tri_visc_vjp_p<R, 3>(mode, a, s);
    case 4: return tri_visc_vjp_p<R, 4>(mode, a, s);
    default: return tri_visc_vjp_p<R, 5>(mode, a, s);
    }
}

template <typename R, int P>
hipError_t tri_visc_complete_p(int E, const int2* links, const R* geo, const double* Ub, const R* Tb, double* out,
                               int xcd, hipStream_t s) {
    using TV = TriViscVjpTile<R, P>;
    if constexpr (P <= 2) {
        auto launch = [&](auto tile) {
            constexpr int TT = decltype(tile)::value;
            tri_visc_complete_scalar_kernel<R, P, TT><<<(std::max(E, 1) + TT - 1) / TT, TT * NV, 0, s>>>(E, links, geo, Ub, Tb, out, xcd);
        };
        if constexpr (TV::LARGE_FROM < INT_MAX)
            if (E >= TV::LARGE_FROM) {
                launch(std::integral_constant<int, TILE>{});
                return hipGetLastError();
            }
        launch(std::integral_constant<int, TV::tile(1)>{});
    } else {
        tri_visc_complete_kernel<R, P, TV::tile(1)><<<(std::max(E, 1) + TRACE_TILE - 1) / TRACE_TILE, BLOCK, 0, s>>>(E, links, geo, Ub, Tb, out);
    }
    return hipGetLastError();
}

template <typename R>
hipError_t tri_visc_complete(int P, int E, const int2* links, const R* geo, const double* Ub, const R* Tb, double* out,
                             int xcd, hipStream_t s) {
    switch (P) {
    case 1: return tri_visc_complete_p<R, 1>(E, links, geo, Ub, Tb, out, xcd, s);
    case 2: return tri_visc_complete_p<R, 2>(E, links, geo, Ub, Tb, out, xcd, s);
    case 3: return tri_visc_complete_p<R, 3>(E, links, geo, Ub, Tb, out, xcd, s);
    case 4: return tri_visc_complete_p<R, 4>(E, links, geo, Ub, Tb, out, xcd, s);
    default: return tri_visc_complete_p<R, 5>(E, links, geo, Ub, Tb, out, xcd, s);
    }
}

template <typename R>
hipError_t tri_trace(int P, int E, const double* U, R* T, hipStream_t s) {
    const int grid = (std::max(E, 1) + TILE - 1) / TILE;
    switch (P) {
    case 1: tri_trace_kernel<R, 1><<<grid, BLOCK, 0, s>>>(E, U, T); break;
    case 2: tri_trace_kernel<R, 2><<<grid, BLOCK, 0, s>>>(E, U, T); break;
    case 3: tri_trace_kernel<R, 3><<<grid, BLOCK, 0, s>>>(E, U, T); break;
    case 4: tri_trace_kernel<R, 4><<<grid, BLOCK, 0, s>>>(E, U, T); break;
    default: tri_trace_kernel<R, 5><<<grid, BLOCK, 0, s>>>(E, U, T); break;
    }
    return hipGetLastError();
}

hipError_t tri_convert(bool to_blk, const double* src, double* dst, int E, int NP, const int* perm, hipStream_t s) {
    const int64_t n = (int64_t)E * NP;
    const int grid = (int)std::max<int64_t>(1, (n + BLOCK - 1) / BLOCK);
    if (to_blk)
        tri_to_blk_kernel<<<grid, BLOCK, 0, s>>>(src, dst, E, NP, perm);
    else
        tri_from_blk_kernel<<<grid, BLOCK, 0, s>>>(src, dst, E, NP, perm);
    return hipGetLastError();
}

// Operator tables of every order into this device's constant memory, once.
std::mutex g_ops_mutex;
uint64_t g_ops_loaded = 0;  // bit d: device d holds the tables

hipError_t load_tri_ops(int device) {
    std::lock_guard<std::mutex> lock(g_ops_mutex);
    if (device >= 0 && device < 64 && (g_ops_loaded >> device) & 1) return hipSuccess;
    std::vector<double> all((size_t)OPS_TOTAL);
    for (int P = 1; P <= 5; ++P) {
        tri::Operators O, Osd, Ohu;
        if (!tri::operators(P, O) || !tri::operators(P, Osd, ZJ_CORR_SD) || !tri::operators(P, Ohu, ZJ_CORR_HU))
            return hipErrorInvalidValue;
        double* d = all.data() + ops_offset(P);
        const int np = O.np, nf = O.nf, ca = 2 * np + nf;   // TriOps<P> layout
        for (int m = 0; m < np; ++m) {
            for (int i = 0; i < np; ++i) {
                d[m * ca + i] = O.Dr[(size_t)i * np + m];
                d[m * ca + np + i] = O.Ds[(size_t)i * np + m];
            }
            for (int jj = 0; jj < nf; ++jj) d[m * ca + 2 * np + jj] = O.interp[(size_t)jj * np + m];
        }
        double* b = d + (size_t)np * ca;
        for (int jj = 0; jj < nf; ++jj)
            for (int i = 0; i < np; ++i) b[(size_t)jj * np + i] = O.lift[(size_t)i * nf + jj];
        std::copy(O.interp.begin(), O.interp.end(), b + (size_t)nf * np);
        for (int k = 0; k < 2; ++k) {
            const tri::Operators& F = k ? Ohu : Osd;
            double* dl = d + lift_offset(P, k ? ZJ_CORR_HU : ZJ_CORR_SD);
            for (int jj = 0; jj < nf; ++jj)
                for (int i = 0; i < np; ++i) dl[(size_t)jj * np + i] = F.lift[(size_t)i * nf + jj];
        }
    }
    std::vector<double> fr64((size_t)tri::frag_offset<double>(6));
    std::vector<float> fr32((size_t)tri::frag_offset<float>(6));
    auto frags = [&](auto order) {
        constexpr int P = decltype(order)::value;
        tri::Operators F[3];
        const int kinds[3] = {ZJ_CORR_DG, ZJ_CORR_SD, ZJ_CORR_HU};
        for (int k = 0; k < 3; ++k)
            if (!tri::operators(P, F[k], kinds[k])) return false;
        tri::frag_build<double, P>(fr64.data() + tri::frag_offset<double>(P), F);
        tri::frag_build<float, P>(fr32.data() + tri::frag_offset<float>(P), F);
        return true;
    };
    if (!frags(std::integral_constant<int, 1>{}) || !frags(std::integral_constant<int, 2>{}) ||
        !frags(std::integral_constant<int, 3>{}) || !frags(std::integral_constant<int, 4>{}) ||
        !frags(std::integral_constant<int, 5>{}))
        return hipErrorInvalidValue;
    std::vector<double> lf((size_t)LF_TOTAL, 0.0);
    for (int P = 1; P <= LF_ORDERS; ++P) {
        for (int fam = 0; fam < 3; ++fam) {
            tri::Operators O;
            if (!tri::operators(P, O, fam == 0 ? ZJ_CORR_DG : (fam == 1 ? ZJ_CORR_SD : ZJ_CORR_HU)))
                return hipErrorInvalidValue;
            const int np = O.np, nf = O.nf, fp = P + 1;
            double* d = lf.data() + lf_offset(P) + (size_t)fam * lf_words(P);
            for (int k = 0; k < 3; ++k)
                for (int a = 0; a < fp; ++a)
                    for (int b = 0; b < fp; ++b) {
                        double acc = 0.0;
                        for (int i = 0; i < np; ++i)
                            acc += O.interp[(size_t)(k * fp + a) * np + i] * O.lift[(size_t)i * nf + k * fp + b];
                        d[(k * fp + a) * fp + b] = acc;
                    }
        }
    }
    std::vector<float> allf(all.begin(), all.end()), lff(lf.begin(), lf.end());
    hipError_t e = hipMemcpyToSymbol(HIP_SYMBOL(c_ops64), all.data(), all.size() * sizeof(double), 0,
                                     hipMemcpyHostToDevice);
    if (e == hipSuccess)
        e = hipMemcpyToSymbol(HIP_SYMBOL(c_ops32), allf.data(), allf.size() * sizeof(float), 0,
                              hipMemcpyHostToDevice);
    if (e == hipSuccess)
        e = hipMemcpyToSymbol(HIP_SYMBOL(c_lf64), lf.data(), lf.size() * sizeof(double), 0, hipMemcpyHostToDevice);
    if (e == hipSuccess)
        e = hipMemcpyToSymbol(HIP_SYMBOL(c_lf32), lff.data(), lff.size() * sizeof(float), 0, hipMemcpyHostToDevice);
    if (e == hipSuccess)
        e = hipMemcpyToSymbol(HIP_SYMBOL(d_frag64), fr64.data(), fr64.size() * sizeof(double), 0, hipMemcpyHostToDevice);
    if (e == hipSuccess)
        e = hipMemcpyToSymbol(HIP_SYMBOL(d_frag32), fr32.data(), fr32.size() * sizeof(float), 0, hipMemcpyHostToDevice);
    if (e == hipSuccess && device >= 0 && device < 64) g_ops_loaded |= 1ull << device;
    return e;
}

}  // namespace

// ------------------------------------------------------------------ host side
struct zj_tri {
    int device = 0;
    hipStream_t stream = nullptr;
    int P = 0, NP = 0, NFP = 0, E = 0, F = 0;
    int prec = ZJ_PREC_FP64;
    double gamma = 1.4;
    int riemann = 0;
    int corr = ZJ_CORR_DG;
    int xcd_groups = 1;
    int epb = 0, nblk = 0, nred = 0;
    int64_t cross_edges = 0;
    double* U = nullptr;
    double* W = nullptr;
    double* Rres = nullptr;
    double* aos = nullptr;
    void* geo = nullptr;
    void* edge = nullptr;
    int2* links = nullptr;
    void* T[3] = {nullptr, nullptr, nullptr};
    double* bc_data = nullptr;
    double* hcell = nullptr;
    double* d_scalars = nullptr;  // [0] dt, [1] l2, [2] dt_cfl
    double* partial = nullptr;
    double* partial_dt = nullptr;
    double* h_pinned = nullptr;
    int* perm = nullptr;
    int l2_blocks = 0;
    double dt_on_device = NAN;
    bool has_state = false;
    hipGraph_t graph = nullptr;
    hipGraphExec_t gexec = nullptr;
    // discrete adjoint, allocated on first use: the cotangent of the state
    // (blocked layout), of U^n within a step, the recomputed stage states and
    // their traces, the cross-tile edge cotangents (ping-pong, A_cur holds the
    // pending ones), per-tile dt partials of the three stages
    double* A_Ub = nullptr;
    double* A_U0b = nullptr;
    double* A_W1 = nullptr;
    double* A_W2 = nullptr;
    double* A_dtb = nullptr;
    void* A_T[3] = {nullptr, nullptr, nullptr};
    void* A_Tb[2] = {nullptr, nullptr};
    int A_cur = 0;
    int A_blk = 0;   // the adjoint kernels' tiles (the BR2 adjoint's tile may be smaller than the stage kernel's)
    bool A_has_tb = false;
    bool A_seeded = false;
    // Navier-Stokes terms (BR2): mu = 1/Re, kappa, penalty; traces of 12 words
    bool viscous = false;
    double mu = 0.0, kappa = 0.0, eta = 2.0;
    std::string err;
};

static thread_local std::string g_tri_error;

#define ZJ_THIP(h, call)                                                                 \
    do {                                                                                 \
        hipError_t e_ = (call);                                                          \
        if (e_ != hipSuccess) {                                                          \
            (h)->err = std::string(#call) + ": " + hipGetErrorString(e_);               \
            return ZJ_ERR_HIP;                                                           \
        }                                                                                \
    } while (0)

static int tfail(zj_tri* h, int code, const std::string& msg) {
    h->err = msg;
    return code;
}

static hipStream_t tpick(zj_tri* h, void* s) { return s ? (hipStream_t)s : h->stream; }

template <typename T>
static int tupload(zj_tri* h, void** dst, const std::vector<T>& v) {
    ZJ_THIP(h, hipMalloc(dst, std::max<size_t>(v.size(), 1) * sizeof(T)));
    if (!v.empty()) ZJ_THIP(h, hipMemcpy(*dst, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice));
    return ZJ_OK;
}

template <typename R>
static int tupload_as(zj_tri* h, void** dst, const std::vector<double>& v) {
    return tupload(h, dst, std::vector<R>(v.begin(), v.end()));
}

static void trelease(zj_tri* h) {
    if (h->gexec) (void)hipGraphExecDestroy(h->gexec);
    if (h->graph) (void)hipGraphDestroy(h->graph);
    void* bufs[] = {h->U, h->W, h->Rres, h->aos, h->geo, h->edge, h->links, h->T[0], h->T[1], h->T[2],
                    h->bc_data, h->hcell, h->d_scalars, h->partial, h->partial_dt, h->perm,
                    h->A_Ub, h->A_U0b, h->A_W1, h->A_W2, h->A_dtb, h->A_T[0], h->A_T[1], h->A_T[2],
                    h->A_Tb[0], h->A_Tb[1]};
    for (void* b : bufs)
        if (b) (void)hipFree(b);
    if (h->h_pinned) (void)hipHostFree(h->h_pinned);
    if (h->stream) (void)hipStreamDestroy(h->stream);
}

static int tbuild(zj_tri* h, const zj_tri_desc* m, const zj_params* p) {
    const int P = m->poly_order;
    if (P < 1 || P > 5) return tfail(h, ZJ_ERR_ARG, "poly_order must be 1..5");
    if (m->n_elem < 1 || m->n_faces < 1 || m->n_nodes < 3) return tfail(h, ZJ_ERR_ARG, "empty mesh");
    if (!m->xy || !m->tri || !m->normals || !m->face_left_elem || !m->face_left_local || !m->face_right_elem ||
        !m->face_right_local)
        return tfail(h, ZJ_ERR_ARG, "mesh tables missing");
    if (p->precision != ZJ_PREC_FP64 && p->precision != ZJ_PREC_FP32BULK)
        return tfail(h, ZJ_ERR_ARG, "unknown precision");
    if (p->compat != ZJ_COMPAT_TEXTBOOK)
        return tfail(h, ZJ_ERR_UNSUPPORTED, "triangles exist in textbook mode only (the reference's triangle "
                                            "operators are zero)");
    if (p->riemann < 0 || p->riemann > 2) return tfail(h, ZJ_ERR_ARG, "unknown Riemann solver");
    if (p->corr < ZJ_CORR_DG || p->corr > ZJ_CORR_GA) return tfail(h, ZJ_ERR_ARG, "unknown correction function");
    if (p->positivity) return tfail(h, ZJ_ERR_UNSUPPORTED, "the positivity limiter is quadrilateral-only");
    if (!(p->gamma > 1.0)) return tfail(h, ZJ_ERR_ARG, "gamma must exceed 1");
    const int NP = tri::n_sp(P), NFP = tri::n_fp(P);
    if ((int64_t)m->n_elem * NP * 4 > (int64_t)INT32_MAX * 4 || (int64_t)m->n_elem * 3 >= (1ll << 31))
        return tfail(h, ZJ_ERR_UNSUPPORTED, "mesh too large for 32-bit element indices");

    h->P = P; h->NP = NP; h->NFP = NFP; h->E = m->n_elem; h->F = m->n_faces;
    h->prec = p->precision; h->gamma = p->gamma; h->riemann = p->riemann; h->corr = p->corr;
    h->device = p->device;
    h->viscous = p->viscous != 0;
    if (h->viscous) {
        if (!(p->Re > 0.0) || !(p->Pr > 0.0)) return tfail(h, ZJ_ERR_ARG, "viscous terms need Re > 0 and Pr > 0");
        if (P == 4 && p->precision == ZJ_PREC_FP64)
            return tfail(h, ZJ_ERR_UNSUPPORTED, "FP64 P4 triangles with the viscous terms are switched off: an earlier "
                                                "build of their kernel faulted on the GPU, with no cause found");
        h->mu = 1.0 / p->Re;
        h->kappa = h->mu * p->gamma / ((p->gamma - 1.0) * p->Pr);
        h->eta = p->br2_eta > 0.0 ? p->br2_eta : 2.0;
    }
    h->epb = h->viscous ? tri_visc_tile(P, h->prec == ZJ_PREC_FP64, h->E) : tri_tile(P, h->prec == ZJ_PREC_FP64, h->E);
    h->nblk = (h->E + h->epb - 1) / h->epb;
    const int E = h->E;

    // affine geometry in the caller's numbering
    std::vector<double> met((size_t)E * 4), hc((size_t)E), cen((size_t)E * 2);
    for (int e = 0; e < E; ++e) {
        int64_t n[3];
        for (int k = 0; k < 3; ++k) {
            n[k] = m->tri[(size_t)e * 3 + k];
            if (n[k] < 0 || n[k] >= m->n_nodes) return tfail(h, ZJ_ERR_ARG, "triangle node index out of range");
        }
        const double ax = m->xy[2 * n[0]], ay = m->xy[2 * n[0] + 1];
        const double bx = m->xy[2 * n[1]], by = m->xy[2 * n[1] + 1];
        const double cx = m->xy[2 * n[2]], cy = m->xy[2 * n[2] + 1];
        const double xr = 0.5 * (bx - ax), yr = 0.5 * (by - ay), xs = 0.5 * (cx - ax), ys = 0.5 * (cy - ay);
        const double J = xr * ys - xs * yr;
        if (!(J > 0.0)) return tfail(h, ZJ_ERR_ARG, "triangle " + std::to_string(e) + " is degenerate or clockwise");
        met[(size_t)e * 4 + 0] = ys / J;
        met[(size_t)e * 4 + 1] = -xs / J;
        met[(size_t)e * 4 + 2] = -yr / J;
        met[(size_t)e * 4 + 3] = xr / J;
        const double per = std::hypot(bx - ax, by - ay) + std::hypot(cx - bx, cy - by) + std::hypot(ax - cx, ay - cy);
        hc[(size_t)e] = 4.0 * (2.0 * J) / per;  // inscribed-circle diameter
        cen[(size_t)e * 2] = (ax + bx + cx) / 3.0;
        cen[(size_t)e * 2 + 1] = (ay + by + cy) / 3.0;
    }
    // device numbering along a Hilbert curve: perm[new] = old, inv[old] = new
    std::vector<int> perm, inv((size_t)E);
    if (m->reorder && E > 1) perm = host::hilbert_order(E, cen.data());
    for (int e = 0; e < E; ++e) inv[(size_t)(perm.empty() ? e : perm[(size_t)e])] = e;
    auto dev = [&](int old) { return inv[(size_t)old]; };

    std::vector<int2> links((size_t)E * 3, make_int2(-1, -1));
    std::vector<double> geo((size_t)E * GEO, 0.0), edge((size_t)E * EDG, 0.0);
    for (int e = 0; e < E; ++e) {
        const int o = perm.empty() ? e : perm[(size_t)e];
        double* ge = &geo[(size_t)e * GEO];
        for (int c = 0; c < 4; ++c) ge[c] = met[(size_t)o * 4 + c];
        double* ed = &edge[(size_t)e * EDG];
        ed[0] = std::sqrt(ge[2] * ge[2] + ge[3] * ge[3]);
        ed[2] = std::sqrt((ge[0] + ge[2]) * (ge[0] + ge[2]) + (ge[1] + ge[3]) * (ge[1] + ge[3]));
        ed[4] = std::sqrt(ge[0] * ge[0] + ge[1] * ge[1]);
    }
    std::vector<double> hcd((size_t)E);
    for (int e = 0; e < E; ++e) hcd[(size_t)e] = hc[(size_t)(perm.empty() ? e : perm[(size_t)e])];
    for (int f = 0; f < h->F; ++f) {
        const int le = m->face_left_elem[f], ll = m->face_left_local[f];
        const int re = m->face_right_elem[f], rl = m->face_right_local[f];
        if (le < 0 || le >= E || ll < 0 || ll > 2) return tfail(h, ZJ_ERR_ARG, "face left side out of range");
        const int dl = dev(le);
        int2& L = links[(size_t)dl * 3 + ll];
        if (L.y != -1) return tfail(h, ZJ_ERR_ARG, "an element edge belongs to two faces");
        const double nx = m->normals[2 * f], ny = m->normals[2 * f + 1];
        geo[(size_t)dl * GEO + 4 + 2 * ll] = nx;
        geo[(size_t)dl * GEO + 5 + 2 * ll] = ny;
        if (re >= 0) {
            if (re >= E || rl < 0 || rl > 2) return tfail(h, ZJ_ERR_ARG, "face right side out of range");
            const int dr = dev(re);
            int2& Rr = links[(size_t)dr * 3 + rl];
            if (Rr.y != -1 || (re == le && rl == ll)) return tfail(h, ZJ_ERR_ARG, "an element edge belongs to two faces");
            L = make_int2(dr, rl | (ROLE_LEFT << 3));
            Rr = make_int2(dl, ll | (ROLE_RIGHT << 3));
            geo[(size_t)dr * GEO + 4 + 2 * rl] = nx;
            geo[(size_t)dr * GEO + 5 + 2 * rl] = ny;
            if (dl / h->epb != dr / h->epb) h->cross_edges += 2;
        } else {
            if (h->viscous)
                return tfail(h, ZJ_ERR_UNSUPPORTED, "the triangle viscous terms are built for meshes without "
                                                    "boundary faces");
            if (!m->bc_type) return tfail(h, ZJ_ERR_ARG, "boundary face without bc_type");
            const int bct = m->bc_type[f];
            if (bct < 0 || bct > 7) return tfail(h, ZJ_ERR_ARG, "unknown BC type");
            int bci = 0;
            if (bct == ZJ_BC_FARFIELD || bct == ZJ_BC_OUTFLOW) {
                bci = m->bc_face_map ? m->bc_face_map[f] : -1;
                if (!m->bc_data || bci < 0 || bci >= m->n_bc_data)
                    return tfail(h, ZJ_ERR_ARG, "boundary face refers to missing bc_data");
            }
            L = make_int2(-1, bct | (ROLE_BOUNDARY << 3) | (bci << 6));
        }
    }
    for (size_t k = 0; k < links.size(); ++k) {
        if (links[k].y == -1) return tfail(h, ZJ_ERR_ARG, "an element edge has no face");
        if (links[k].x >= 0)
            edge[k * 2 + 1] = edge[(size_t)links[k].x * EDG + 2 * (links[k].y & 7)];
    }

    ZJ_THIP(h, hipSetDevice(h->device));
    ZJ_THIP(h, load_tri_ops(h->device));
    ZJ_THIP(h, hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking));
    int nxcc = 1;
    if (hipDeviceGetAttribute(&nxcc, hipDeviceAttributeNumberOfXccs, h->device) != hipSuccess || nxcc < 1) nxcc = 1;
    h->xcd_groups = nxcc;
    const size_t npts = (size_t)E * NP;
    const size_t eb = ((size_t)E + EB - 1) / EB * EB;  // elements rounded up to whole layout blocks
    const size_t rsz = h->prec == ZJ_PREC_FP64 ? sizeof(double) : sizeof(float);
    ZJ_THIP(h, hipMalloc((void**)&h->U, eb * NP * 4 * sizeof(double)));
    ZJ_THIP(h, hipMalloc((void**)&h->W, eb * NP * 4 * sizeof(double)));
    ZJ_THIP(h, hipMalloc((void**)&h->Rres, eb * NP * 4 * sizeof(double)));
    ZJ_THIP(h, hipMalloc((void**)&h->aos, npts * 4 * sizeof(double)));
    for (int k = 0; k < 3; ++k) ZJ_THIP(h, hipMalloc(&h->T[k], eb * NFP * (h->viscous ? TWV : 4) * rsz));
    int rc;
    if (h->prec == ZJ_PREC_FP64) {
        if ((rc = tupload_as<double>(h, &h->geo, geo)) || (rc = tupload_as<double>(h, &h->edge, edge))) return rc;
    } else {
        if ((rc = tupload_as<float>(h, &h->geo, geo)) || (rc = tupload_as<float>(h, &h->edge, edge))) return rc;
    }
    if ((rc = tupload(h, (void**)&h->links, links))) return rc;
    std::vector<double> bcd;
    if (m->bc_data && m->n_bc_data > 0) bcd.assign(m->bc_data, m->bc_data + (size_t)m->n_bc_data * 8);
    if ((rc = tupload(h, (void**)&h->bc_data, bcd))) return rc;
    if ((rc = tupload(h, (void**)&h->hcell, hcd))) return rc;
    if (!perm.empty() && (rc = tupload(h, (void**)&h->perm, perm))) return rc;
    h->nred = (int)std::min<int64_t>(1024, std::max<int64_t>(1, ((int64_t)npts + BLOCK - 1) / BLOCK));
    ZJ_THIP(h, hipMalloc((void**)&h->partial, (size_t)std::max(h->nblk, 1) * sizeof(double)));
    ZJ_THIP(h, hipMalloc((void**)&h->partial_dt, (size_t)h->nred * sizeof(double)));
    ZJ_THIP(h, hipMalloc((void**)&h->d_scalars, 8 * sizeof(double)));
    ZJ_THIP(h, hipHostMalloc((void**)&h->h_pinned, 8 * sizeof(double), hipHostMallocDefault));
    ZJ_THIP(h, hipMemset(h->d_scalars, 0, 8 * sizeof(double)));
    ZJ_THIP(h, hipDeviceSynchronize());
    return ZJ_OK;
}

template <typename R>
static TriArgs<R> tri_args(zj_tri* h, int mode) {
    TriArgs<R> a{};
    a.E = h->E;
    a.geo = (const R*)h->geo;
    a.edge = (const R*)h->edge;
    a.links = h->links;
    a.bc_data = h->bc_data;
    a.dt_ptr = h->d_scalars;
    a.gamma = h->gamma;
    a.riemann = h->riemann;
    a.xcd_groups = h->xcd_groups;
    a.lift_off = lift_offset(h->P, h->corr);
    a.mu = h->mu;
    a.kappa = h->kappa;
    a.eta = h->eta;
    a.lf_off = lf_family(h->corr) * lf_words(h->P);
    a.family = lf_family(h->corr);
    R** T = (R**)h->T;
    switch (mode) {
    case MODE_RESIDUAL:
        a.U_in = h->U; a.R_out = h->Rres; a.T_in = T[0]; a.l2_partial = h->partial;
        break;
    case MODE_STAGE1:
        a.U_in = h->U; a.U_out = h->W; a.T_in = T[0]; a.T_out = T[1];
        break;
    case MODE_STAGE2:
        a.U0 = h->U; a.U_in = h->W; a.U_out = h->W; a.T_in = T[1]; a.T_out = T[2];
        break;
    default:
        a.U0 = h->U; a.U_in = h->W; a.U_out = h->U; a.T_in = T[2]; a.T_out = T[0]; a.l2_partial = h->partial;
        break;
    }
    return a;
}

static hipError_t tenqueue(zj_tri* h, int mode, hipStream_t s) {
    hipError_t e;
    if (h->viscous)
        e = h->prec == ZJ_PREC_FP64 ? tri_visc_launch<double>(h->P, mode, tri_args<double>(h, mode), s)
                                    : tri_visc_launch<float>(h->P, mode, tri_args<float>(h, mode), s);
    else
        e = h->prec == ZJ_PREC_FP64 ? tri_launch<double>(h->P, mode, tri_args<double>(h, mode), s)
                                    : tri_launch<float>(h->P, mode, tri_args<float>(h, mode), s);
    if (e == hipSuccess && mode == MODE_STAGE3) h->l2_blocks = h->nblk;
    if (e == hipSuccess && mode == MODE_RESIDUAL) {
        const int tt = h->viscous ? h->epb : tri_residual_tile(h->P, h->prec == ZJ_PREC_FP64, h->E);
        h->l2_blocks = (h->E + tt - 1) / tt;
    }
    return e;
}

static int trefresh(zj_tri* h, hipStream_t s) {
    hipError_t e;
    if (h->viscous)
        e = h->prec == ZJ_PREC_FP64
                ? tri_visc_trace<double>(h->P, h->E, h->U, (const double*)h->geo, (double*)h->T[0], s)
                : tri_visc_trace<float>(h->P, h->E, h->U, (const float*)h->geo, (float*)h->T[0], s);
    else
        e = h->prec == ZJ_PREC_FP64 ? tri_trace<double>(h->P, h->E, h->U, (double*)h->T[0], s)
                                    : tri_trace<float>(h->P, h->E, h->U, (float*)h->T[0], s);
    ZJ_THIP(h, e);
    return ZJ_OK;
}

static void tdrop_graph(zj_tri* h) {
    if (h->gexec) { (void)hipGraphExecDestroy(h->gexec); h->gexec = nullptr; }
    if (h->graph) { (void)hipGraphDestroy(h->graph); h->graph = nullptr; }
}

extern "C" int zj_tri_create(zj_tri_handle* out, const zj_tri_desc* m, const zj_params* p) {
    if (!out || !m || !p) {
        g_tri_error = "null argument";
        return ZJ_ERR_ARG;
    }
    *out = nullptr;
    zj_tri* h = new (std::nothrow) zj_tri();
    if (!h) {
        g_tri_error = "out of host memory";
        return ZJ_ERR_NOMEM;
    }
    int rc;
    try {
        rc = tbuild(h, m, p);
    } catch (const std::bad_alloc&) {   // host tables of a mesh too large for host memory
        h->err = "out of host memory";
        rc = ZJ_ERR_NOMEM;
    }
    if (rc != ZJ_OK) {
        g_tri_error = h->err;
        trelease(h);
        delete h;
        return rc;
    }
    *out = h;
    return ZJ_OK;
}

extern "C" int zj_tri_destroy(zj_tri_handle h) {
    if (!h) return ZJ_ERR_ARG;
    (void)hipSetDevice(h->device);
    (void)hipStreamSynchronize(h->stream);
    trelease(h);
    delete h;
    return ZJ_OK;
}

extern "C" const char* zj_tri_last_error(zj_tri_handle h) { return h ? h->err.c_str() : g_tri_error.c_str(); }

extern "C" int zj_tri_set_state_device(zj_tri_handle h, const double* d_aos, void* stream) {
    if (!h || !d_aos) return ZJ_ERR_ARG;
    ZJ_THIP(h, hipSetDevice(h->device));
    hipStream_t s = tpick(h, stream);
    ZJ_THIP(h, tri_convert(true, d_aos, h->U, h->E, h->NP, h->perm, s));
    const int rc = trefresh(h, s);
    if (rc) return rc;
    h->has_state = true;
    return ZJ_OK;
}

extern "C" int zj_tri_set_state(zj_tri_handle h, const double* U_aos) {
    if (!h || !U_aos) return ZJ_ERR_ARG;
    ZJ_THIP(h, hipSetDevice(h->device));
    const size_t n = (size_t)h->E * h->NP * 4;
    ZJ_THIP(h, hipMemcpyAsync(h->aos, U_aos, n * sizeof(double), hipMemcpyHostToDevice, h->stream));
    const int rc = zj_tri_set_state_device(h, h->aos, nullptr);
    if (rc) return rc;
    ZJ_THIP(h, hipStreamSynchronize(h->stream));
    return ZJ_OK;
}

extern "C" int zj_tri_get_state_device(zj_tri_handle h, double* d_aos, void* stream) {
    if (!h || !d_aos) return ZJ_ERR_ARG;
    if (!h->has_state) return tfail(h, ZJ_ERR_STATE, "no state set");
    ZJ_THIP(h, hipSetDevice(h->device));
    ZJ_THIP(h, tri_convert(false, h->U, d_aos, h->E, h->NP, h->perm, tpick(h, stream)));
    return ZJ_OK;
}

extern "C" int zj_tri_get_state(zj_tri_handle h, double* U_aos) {
    if (!h || !U_aos) return ZJ_ERR_ARG;
    const int rc = zj_tri_get_state_device(h, h->aos, nullptr);
    if (rc) return rc;
    ZJ_THIP(h, hipMemcpyAsync(U_aos, h->aos, (size_t)h->E * h->NP * 4 * sizeof(double), hipMemcpyDeviceToHost,
                              h->stream));
    ZJ_THIP(h, hipStreamSynchronize(h->stream));
    return ZJ_OK;
}

extern "C" int zj_tri_residual(zj_tri_handle h, double* dUdt_aos, void* stream) {
    if (!h) return ZJ_ERR_ARG;
    if (!h->has_state) return tfail(h, ZJ_ERR_STATE, "no state set");
    ZJ_THIP(h, hipSetDevice(h->device));
    hipStream_t s = tpick(h, stream);
    ZJ_THIP(h, tenqueue(h, MODE_RESIDUAL, s));
    if (dUdt_aos) {
        ZJ_THIP(h, tri_convert(false, h->Rres, h->aos, h->E, h->NP, h->perm, s));
        ZJ_THIP(h, hipMemcpyAsync(dUdt_aos, h->aos, (size_t)h->E * h->NP * 4 * sizeof(double),
                                  hipMemcpyDeviceToHost, s));
        ZJ_THIP(h, hipStreamSynchronize(s));
    }
    return ZJ_OK;
}

extern "C" int zj_tri_residual_device(zj_tri_handle h, double* d_dUdt_aos, void* stream) {
    if (!h || !d_dUdt_aos) return ZJ_ERR_ARG;
    if (!h->has_state) return tfail(h, ZJ_ERR_STATE, "no state set");
    ZJ_THIP(h, hipSetDevice(h->device));
    hipStream_t s = tpick(h, stream);
    ZJ_THIP(h, tenqueue(h, MODE_RESIDUAL, s));
    ZJ_THIP(h, tri_convert(false, h->Rres, d_dUdt_aos, h->E, h->NP, h->perm, s));
    return ZJ_OK;
}

extern "C" int zj_tri_time_stages(zj_tri_handle h, double dt, int steps, double* stage_ms, void* stream) {
    if (!h || steps < 1 || !stage_ms) return ZJ_ERR_ARG;
    if (!h->has_state) return tfail(h, ZJ_ERR_STATE, "no state set");
    ZJ_THIP(h, hipSetDevice(h->device));
    hipStream_t s = tpick(h, stream);
    if (dt != h->dt_on_device) {
        h->dt_on_device = dt;
        ZJ_THIP(h, launch_set_scalar(h->d_scalars, dt, s));
    }
    ZJ_THIP(h, time_stage_kernels([&](int st) { return tenqueue(h, st, s); }, steps, s, stage_ms));
    return ZJ_OK;
}

extern "C" int zj_tri_rk3_step(zj_tri_handle h, double dt, void* stream) {
    if (!h) return ZJ_ERR_ARG;
    if (!h->has_state) return tfail(h, ZJ_ERR_STATE, "no state set");
    ZJ_THIP(h, hipSetDevice(h->device));
    hipStream_t s = tpick(h, stream);
    if (!h->gexec) {
        ZJ_THIP(h, hipStreamBeginCapture(h->stream, hipStreamCaptureModeThreadLocal));
        hipError_t e = hipSuccess;
        for (int st = 1; st <= 3 && e == hipSuccess; ++st) e = tenqueue(h, st, h->stream);
        hipGraph_t g = nullptr;
        const hipError_t e2 = hipStreamEndCapture(h->stream, &g);
        if (e != hipSuccess || e2 != hipSuccess) {
            if (g) (void)hipGraphDestroy(g);
            ZJ_THIP(h, e != hipSuccess ? e : e2);
        }
        h->graph = g;
        ZJ_THIP(h, hipGraphInstantiate(&h->gexec, h->graph, nullptr, nullptr, 0));
    }
    if (dt != h->dt_on_device) {
        h->dt_on_device = dt;
        ZJ_THIP(h, launch_set_scalar(h->d_scalars, dt, s));
    }
    ZJ_THIP(h, hipGraphLaunch(h->gexec, s));
    return ZJ_OK;
}

extern "C" int zj_tri_dt_cfl(zj_tri_handle h, double cfl, double* dt) {
    if (!h || !dt) return ZJ_ERR_ARG;
    if (!h->has_state) return tfail(h, ZJ_ERR_STATE, "no state set");
    ZJ_THIP(h, hipSetDevice(h->device));
    const double p1 = h->P + 1.0;
    const double visc = h->viscous ? p1 * p1 * p1 * p1 * std::max(h->mu * 4.0 / 3.0, h->kappa * (h->gamma - 1.0))
                                   : 0.0;  // kappa (gamma-1) = mu gamma / Pr
    tri_dt_kernel<<<h->nred, BLOCK, 0, h->stream>>>(h->U, h->hcell, h->E, h->NP, h->gamma, cfl, 2.0 * h->P + 1.0,
                                                    visc, h->partial_dt);
    ZJ_THIP(h, hipGetLastError());
    ZJ_THIP(h, launch_finalize(h->partial_dt, h->nred, FIN_MIN, h->d_scalars + 2, h->stream));
    ZJ_THIP(h, hipMemcpyAsync(h->h_pinned, h->d_scalars + 2, sizeof(double), hipMemcpyDeviceToHost, h->stream));
    ZJ_THIP(h, hipStreamSynchronize(h->stream));
    *dt = h->h_pinned[0];
    return ZJ_OK;
}

extern "C" int zj_tri_residual_l2(zj_tri_handle h, double* l2) {
    if (!h || !l2) return ZJ_ERR_ARG;
    if (h->l2_blocks == 0) return tfail(h, ZJ_ERR_STATE, "no residual has been evaluated");
    ZJ_THIP(h, hipSetDevice(h->device));
    ZJ_THIP(h, hipDeviceSynchronize());
    ZJ_THIP(h, launch_finalize(h->partial, h->l2_blocks, FIN_SQRT_SUM, h->d_scalars + 1, h->stream));
    ZJ_THIP(h, hipMemcpyAsync(h->h_pinned, h->d_scalars + 1, sizeof(double), hipMemcpyDeviceToHost, h->stream));
    ZJ_THIP(h, hipStreamSynchronize(h->stream));
    *l2 = h->h_pinned[0];
    return ZJ_OK;
}

extern "C" int zj_tri_synchronize(zj_tri_handle h) {
    if (!h) return ZJ_ERR_ARG;
    ZJ_THIP(h, hipSetDevice(h->device));
    ZJ_THIP(h, hipDeviceSynchronize());
    return ZJ_OK;
}

extern "C" int zj_tri_set_xcd_groups(zj_tri_handle h, int groups) {
    if (!h || groups < 1) return ZJ_ERR_ARG;
    h->xcd_groups = groups;
    tdrop_graph(h);
    return ZJ_OK;
}

extern "C" int zj_tri_get_scheme(zj_tri_handle h, int* poly_order, double* gamma) {
    if (!h) return ZJ_ERR_ARG;
    if (poly_order) *poly_order = h->P;
    if (gamma) *gamma = h->gamma;
    return ZJ_OK;
}

extern "C" int zj_tri_get_info(zj_tri_handle h, int64_t* n_dof, int* elems_per_block, int* n_sp,
                               int64_t* cross_tile_edges) {
    if (!h) return ZJ_ERR_ARG;
    if (n_dof) *n_dof = (int64_t)h->E * h->NP * 4;
    if (elems_per_block) *elems_per_block = h->epb;
    if (n_sp) *n_sp = h->NP;
    if (cross_tile_edges) *cross_tile_edges = h->cross_edges;
    return ZJ_OK;
}

// ------------------------------------------------------------ adjoint (host)
static int tensure_adjoint(zj_tri* h) {
    if (h->A_Ub) return ZJ_OK;
    int tt = TILE;
    if (h->viscous) tt = tri_visc_vjp_tile(h->P, h->prec == ZJ_PREC_FP64, h->E);
    ZJ_THIP(h, hipSetDevice(h->device));
    h->A_blk = (h->E + tt - 1) / tt;
    const size_t eb = ((size_t)h->E + EB - 1) / EB * EB;
    const size_t nst = eb * h->NP * 4 * sizeof(double);
    const size_t ntr = eb * h->NFP * (h->viscous ? TWV : 4) * (h->prec == ZJ_PREC_FP64 ? sizeof(double) : sizeof(float));
    for (double** b : {&h->A_Ub, &h->A_U0b, &h->A_W1, &h->A_W2}) ZJ_THIP(h, hipMalloc((void**)b, nst));
    for (int k = 0; k < 3; ++k) ZJ_THIP(h, hipMalloc(&h->A_T[k], ntr));
    for (int k = 0; k < 2; ++k) ZJ_THIP(h, hipMalloc(&h->A_Tb[k], ntr));
    ZJ_THIP(h, hipMalloc((void**)&h->A_dtb, (size_t)3 * std::max(h->A_blk, 1) * sizeof(double)));
    return ZJ_OK;
}

template <typename R>
static TriVjpArgs<R> tvjp_args(zj_tri* h) {
    TriVjpArgs<R> a{};
    a.E = h->E;
    a.geo = (const R*)h->geo;
    a.edge = (const R*)h->edge;
    a.links = h->links;
    a.bc_data = h->bc_data;
    a.dt_ptr = h->d_scalars;
    a.gamma = h->gamma;
    a.riemann = h->riemann;
    a.xcd_groups = h->xcd_groups;
    a.lift_off = lift_offset(h->P, h->corr);
    a.mu = h->mu;
    a.kappa = h->kappa;
    a.eta = h->eta;
    a.lf_off = lf_family(h->corr) * lf_words(h->P);
    a.family = lf_family(h->corr);
    return a;
}

// One step backwards: stages 1 and 2 recomputed into A_W1 and A_W2 (with their
// cross-tile traces), then the stage VJPs 3, 2, 1, each
// consuming the edge cotangents the previous launch left.
template <typename R>
static hipError_t tri_adjoint_step(zj_tri* h, bool want_dt, hipStream_t s) {
    R** AT = (R**)h->A_T;
    R** Tb = (R**)h->A_Tb;
    const R* geo = (const R*)h->geo;
    // The Navier-Stokes adjoint's tiles are mostly whole tiles of the stage
    // kernel, whose traces (T[0] of the state, then each recomputed stage's)
    // cover the edges across them; else every edge's traces are formed after
    // each stage.
    const bool same = h->viscous && tri_visc_vjp_tile(h->P, h->prec == ZJ_PREC_FP64, h->E) % h->epb == 0;
    const bool retrace = h->viscous && !same;
    const R* T[3] = {same ? (const R*)h->T[0] : AT[0], AT[1], AT[2]};
    hipError_t e = hipSuccess;
    if (!same)
        e = h->viscous ? tri_visc_trace<R>(h->P, h->E, h->U, geo, AT[0], s) : tri_trace<R>(h->P, h->E, h->U, AT[0], s);
    if (e != hipSuccess) return e;
    TriArgs<R> f = tri_args<R>(h, MODE_STAGE1);
    f.U_in = h->U; f.U_out = h->A_W1; f.T_in = T[0]; f.T_out = AT[1]; f.l2_partial = nullptr;
    if ((e = h->viscous ? tri_visc_launch<R>(h->P, MODE_STAGE1, f, s) : tri_launch<R>(h->P, MODE_STAGE1, f, s)) != hipSuccess)
        return e;
    if (retrace && (e = tri_visc_trace<R>(h->P, h->E, h->A_W1, geo, AT[1], s)) != hipSuccess) return e;
    f = tri_args<R>(h, MODE_STAGE2);
    f.U0 = h->U; f.U_in = h->A_W1; f.U_out = h->A_W2; f.T_in = AT[1]; f.T_out = AT[2]; f.l2_partial = nullptr;
    if ((e = h->viscous ? tri_visc_launch<R>(h->P, MODE_STAGE2, f, s) : tri_launch<R>(h->P, MODE_STAGE2, f, s)) != hipSuccess)
        return e;
    if (retrace && (e = tri_visc_trace<R>(h->P, h->E, h->A_W2, geo, AT[2], s)) != hipSuccess) return e;
    for (int st = 3; st >= 1; --st) {
        TriVjpArgs<R> a = tvjp_args<R>(h);
        a.U_in = st == 3 ? h->A_W2 : (st == 2 ? h->A_W1 : h->U);
        a.U0 = h->U;
        a.T_in = T[st - 1];
        a.Ub_in = h->A_Ub;
        a.Ub_out = h->A_Ub;
        a.Tb_in = h->A_has_tb ? Tb[h->A_cur] : nullptr;
        a.Tb_out = Tb[1 - h->A_cur];
        a.U0b = h->A_U0b;
        a.dtb_partial = want_dt ? h->A_dtb + (size_t)(3 - st) * h->A_blk : nullptr;
        if (h->viscous && want_dt && !tri_visc_vjp_has_residual<R>(h->P, h->E)) {
            // the residual at q, of which the time step's cotangent is made
            f = tri_args<R>(h, MODE_RESIDUAL);
            f.U_in = a.U_in; f.T_in = a.T_in; f.l2_partial = nullptr;
            if ((e = tri_visc_launch<R>(h->P, MODE_RESIDUAL, f, s)) != hipSuccess) return e;
            a.R_in = h->Rres;
        }
        if ((e = h->viscous ? tri_visc_vjp<R>(h->P, st, a, s) : tri_vjp<R>(h->P, st, a, s)) != hipSuccess) return e;
        h->A_cur = 1 - h->A_cur;
        h->A_has_tb = true;
    }
    return hipSuccess;
}

extern "C" int zj_tri_adjoint_set_device(zj_tri_handle h, const double* d_ubar_aos, void* stream) {
    if (!h || !d_ubar_aos) return ZJ_ERR_ARG;
    const int rc = tensure_adjoint(h);
    if (rc) return rc;
    ZJ_THIP(h, hipSetDevice(h->device));
    ZJ_THIP(h, tri_convert(true, d_ubar_aos, h->A_Ub, h->E, h->NP, h->perm, tpick(h, stream)));
    h->A_has_tb = false;
    h->A_seeded = true;
    return ZJ_OK;
}

extern "C" int zj_tri_adjoint_set(zj_tri_handle h, const double* ubar_aos) {
    if (!h || !ubar_aos) return ZJ_ERR_ARG;
    ZJ_THIP(h, hipSetDevice(h->device));
    ZJ_THIP(h, hipMemcpyAsync(h->aos, ubar_aos, (size_t)h->E * h->NP * 4 * sizeof(double), hipMemcpyHostToDevice,
                              h->stream));
    const int rc = zj_tri_adjoint_set_device(h, h->aos, nullptr);
    if (rc) return rc;
    ZJ_THIP(h, hipStreamSynchronize(h->stream));
    return ZJ_OK;
}

extern "C" int zj_tri_adjoint_get_device(zj_tri_handle h, double* d_ubar_aos, void* stream) {
    if (!h || !d_ubar_aos) return ZJ_ERR_ARG;
    if (!h->A_seeded) return tfail(h, ZJ_ERR_STATE, "no adjoint seed set");
    ZJ_THIP(h, hipSetDevice(h->device));
    hipStream_t s = tpick(h, stream);
    const void* tb = h->A_has_tb ? h->A_Tb[h->A_cur] : nullptr;
    hipError_t e;
    if (h->viscous)
        e = h->prec == ZJ_PREC_FP64
                ? tri_visc_complete<double>(h->P, h->E, h->links, (const double*)h->geo, h->A_Ub, (const double*)tb,
                                            h->Rres, h->xcd_groups, s)
                : tri_visc_complete<float>(h->P, h->E, h->links, (const float*)h->geo, h->A_Ub, (const float*)tb,
                                           h->Rres, h->xcd_groups, s);
    else
        e = h->prec == ZJ_PREC_FP64
                ? tri_complete<double>(h->P, h->E, h->links, h->A_Ub, (const double*)tb, h->Rres, h->xcd_groups, s)
                : tri_complete<float>(h->P, h->E, h->links, h->A_Ub, (const float*)tb, h->Rres, h->xcd_groups, s);
    ZJ_THIP(h, e);
    ZJ_THIP(h, tri_convert(false, h->Rres, d_ubar_aos, h->E, h->NP, h->perm, s));
    return ZJ_OK;
}

extern "C" int zj_tri_adjoint_get(zj_tri_handle h, double* ubar_aos) {
    if (!h || !ubar_aos) return ZJ_ERR_ARG;
    const int rc = zj_tri_adjoint_get_device(h, h->aos, nullptr);
    if (rc) return rc;
    ZJ_THIP(h, hipMemcpyAsync(ubar_aos, h->aos, (size_t)h->E * h->NP * 4 * sizeof(double), hipMemcpyDeviceToHost,
                              h->stream));
    ZJ_THIP(h, hipStreamSynchronize(h->stream));
    return ZJ_OK;
}

extern "C" int zj_tri_rk3_step_vjp(zj_tri_handle h, double dt, double* dt_bar, void* stream) {
    if (!h) return ZJ_ERR_ARG;
    if (!h->has_state) return tfail(h, ZJ_ERR_STATE, "no state set");
    if (!h->A_seeded) return tfail(h, ZJ_ERR_STATE, "no adjoint seed set");
    ZJ_THIP(h, hipSetDevice(h->device));
    hipStream_t s = tpick(h, stream);
    if (dt != h->dt_on_device) {
        h->dt_on_device = dt;
        ZJ_THIP(h, launch_set_scalar(h->d_scalars, dt, s));
    }
    const bool want = dt_bar != nullptr;
    ZJ_THIP(h, h->prec == ZJ_PREC_FP64 ? tri_adjoint_step<double>(h, want, s) : tri_adjoint_step<float>(h, want, s));
    if (want) {
        ZJ_THIP(h, launch_finalize(h->A_dtb, 3 * h->A_blk, FIN_SUM, h->d_scalars + 3, s));
        ZJ_THIP(h, hipMemcpyAsync(h->h_pinned + 3, h->d_scalars + 3, sizeof(double), hipMemcpyDeviceToHost, s));
        ZJ_THIP(h, hipStreamSynchronize(s));
        *dt_bar = h->h_pinned[3];
    }
    return ZJ_OK;
}

template <typename R>
static hipError_t tri_residual_vjp(zj_tri* h, hipStream_t s) {
    R** AT = (R**)h->A_T;
    R* tb = (R*)h->A_Tb[1 - h->A_cur];  // the pending edge cotangents of the accumulator stay in A_Tb[A_cur]
    const R* geo = (const R*)h->geo;
    hipError_t e = h->viscous ? tri_visc_trace<R>(h->P, h->E, h->U, geo, AT[0], s) : tri_trace<R>(h->P, h->E, h->U, AT[0], s);
    if (e != hipSuccess) return e;
    TriVjpArgs<R> a = tvjp_args<R>(h);
    a.U_in = h->U;
    a.T_in = AT[0];
    a.Ub_in = h->Rres;
    a.Ub_out = h->Rres;
    a.Tb_out = tb;
    if (h->viscous) {
        if ((e = tri_visc_vjp<R>(h->P, MODE_RESIDUAL, a, s)) != hipSuccess) return e;
        return tri_visc_complete<R>(h->P, h->E, h->links, geo, h->Rres, tb, h->W, h->xcd_groups, s);
    }
    if ((e = tri_vjp<R>(h->P, MODE_RESIDUAL, a, s)) != hipSuccess) return e;
    return tri_complete<R>(h->P, h->E, h->links, h->Rres, tb, h->W, h->xcd_groups, s);
}

extern "C" int zj_tri_residual_vjp_device(zj_tri_handle h, const double* d_w_aos, double* d_ubar_aos, void* stream) {
    if (!h || !d_w_aos || !d_ubar_aos) return ZJ_ERR_ARG;
    if (!h->has_state) return tfail(h, ZJ_ERR_STATE, "no state set");
    const int rc = tensure_adjoint(h);
    if (rc) return rc;
    ZJ_THIP(h, hipSetDevice(h->device));
    hipStream_t s = tpick(h, stream);
    ZJ_THIP(h, tri_convert(true, d_w_aos, h->Rres, h->E, h->NP, h->perm, s));
    ZJ_THIP(h, h->prec == ZJ_PREC_FP64 ? tri_residual_vjp<double>(h, s) : tri_residual_vjp<float>(h, s));
    ZJ_THIP(h, tri_convert(false, h->W, d_ubar_aos, h->E, h->NP, h->perm, s));
    return ZJ_OK;
}

extern "C" int zj_tri_residual_vjp(zj_tri_handle h, const double* w_aos, double* ubar_aos) {
    if (!h || !w_aos || !ubar_aos) return ZJ_ERR_ARG;
    ZJ_THIP(h, hipSetDevice(h->device));
    const size_t n = (size_t)h->E * h->NP * 4;
    ZJ_THIP(h, hipMemcpyAsync(h->aos, w_aos, n * sizeof(double), hipMemcpyHostToDevice, h->stream));
    const int rc = zj_tri_residual_vjp_device(h, h->aos, h->aos, nullptr);  // w is consumed before aos is rewritten
    if (rc) return rc;
    ZJ_THIP(h, hipMemcpyAsync(ubar_aos, h->aos, n * sizeof(double), hipMemcpyDeviceToHost, h->stream));
    ZJ_THIP(h, hipStreamSynchronize(h->stream));
    return ZJ_OK;
}

extern "C" int zj_tri_operators(int p, double* sp, double* fp, double* wg, double* Dr, double* Ds, double* interp,
                                double* lift) {
    tri::Operators O;
    if (!tri::operators(p, O)) return ZJ_ERR_ARG;
    auto put = [](double* dst, const std::vector<double>& v) {
        if (dst) std::memcpy(dst, v.data(), v.size() * sizeof(double));
    };
    put(sp, O.sp); put(fp, O.fp); put(wg, O.wg);
    put(Dr, O.Dr); put(Ds, O.Ds); put(interp, O.interp); put(lift, O.lift);
    return ZJ_OK;
}

extern "C" int zj_tri_lift(int p, int corr, double* lift) {
    tri::Operators O;
    if (!lift || corr < ZJ_CORR_DG || corr > ZJ_CORR_GA || !tri::operators(p, O, corr)) return ZJ_ERR_ARG;
    std::memcpy(lift, O.lift.data(), O.lift.size() * sizeof(double));
    return ZJ_OK;
}
