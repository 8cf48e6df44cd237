// device.hpp -- device helpers shared by the stage kernels (kernels.hip) and the adjoint kernels
// (adjoint.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "internal.hpp"

namespace ndg {

// Workgroups are dispatched round-robin over the 8 XCDs; remap so that each XCD walks one
// contiguous stretch of the Hilbert-ordered elements (neighbours share its L2).
__device__ __forceinline__ int64_t xcd_block(int64_t b, int64_t G) {
    const int64_t per = G / 8, rem = G % 8, x = b % 8, i = b / 8;
    return x < rem ? x * (per + 1) + i : rem * (per + 1) + (x - rem) * per + i;
}

// Bilinear metrics (include/functions/quad_metrics.tpp:3-8): x_xi, x_eta, y_xi, y_eta.
__device__ __forceinline__ void metrics(const double *P, double xi, double eta, double &xxi,
                                        double &xeta, double &yxi, double &yeta) {
    xxi = ((1 - eta) * (P[2] - P[0]) + (1 + eta) * (P[4] - P[6])) / 4;
    xeta = ((1 - xi) * (P[6] - P[0]) + (1 + xi) * (P[4] - P[2])) / 4;
    yxi = ((1 - eta) * (P[3] - P[1]) + (1 + eta) * (P[5] - P[7])) / 4;
    yeta = ((1 - xi) * (P[7] - P[1]) + (1 + xi) * (P[5] - P[3])) / 4;
}

// Edge Jacobian of side s (src/entities/Element2D_t.cpp:756-769): constant along a side of a
// bilinear element, so it is evaluated once at the side's first node.
__device__ __forceinline__ double side_scale(const double *P, int s, double x0) {
    double xxi, xeta, yxi, yeta;
    if (s == 0) { metrics(P, x0, -1.0, xxi, xeta, yxi, yeta); return sqrt(xxi * xxi + yxi * yxi); }
    if (s == 1) { metrics(P, 1.0, x0, xxi, xeta, yxi, yeta); return sqrt(xeta * xeta + yeta * yeta); }
    if (s == 2) { metrics(P, x0, 1.0, xxi, xeta, yxi, yeta); return sqrt(xxi * xxi + yxi * yxi); }
    metrics(P, -1.0, x0, xxi, xeta, yxi, yeta);
    return sqrt(xeta * xeta + yeta * yeta);
}

// Thread layout of the line-per-lane kernels: a workgroup is three waves, one per field (p, u, v);
// lane (element e, line l) of the wave for field f handles one (N+1)-point line of that field for
// EPB = floor(64/(N+1)) elements.
template <int N>
struct LineShape {
    static constexpr int NF = N + 1;
    static constexpr int NE = NF * NF;
    static constexpr int T = 192;                            // one wave per field
    static constexpr int EPB = 64 / NF;                       // elements per workgroup
    static constexpr int FPT = (EPB * 4 * NF + T - 1) / T;    // flux points per thread
    static constexpr int QPT = (EPB * 3 * NE + T - 1) / T;    // state values per thread (tile load)
    static constexpr int VPT = (EPB * 8 + T - 1) / T;         // vertex coordinates per thread
};

// Outward normal of the edge P_s -> P_s+1 of vertices V; returns its Jacobian (src/entities/
// Element2D_t.cpp:756-769), constant along a side of a bilinear element and half its length.
__device__ __forceinline__ double side_geometry(const double *V, int s, double &nx, double &ny) {
    const int s1 = (s + 1) & 3;
    const double ex = V[2 * s1] - V[2 * s], ey = V[2 * s1 + 1] - V[2 * s + 1];
    const double len = sqrt(ex * ex + ey * ey);
    nx = ey / len;
    ny = -(ex / len);
    return len / 2;
}

// A table of L values held across the lanes of each row of 16 (value e in lane e mod 16 of register
// e / 16), so that a wave-uniform entry is a DPP operand (row broadcast) of its multiply-add: the stage
// kernel's D^ entries as scalar loads came a few at a time (81 doubles are more than the scalar
// registers hold), each batch a wait of some 300 cycles that the contraction of the line could
// not hide: 3,650 cycles for the 81 multiply-adds of a line at N = 8.
template <int L>
struct LaneTable {
    double v[(L + 15) / 16];
    __device__ __forceinline__ void load(const double *t) {
        const int m = threadIdx.x & 15;
#pragma unroll
        for (int p = 0; p < (L + 15) / 16; ++p) v[p] = t[min(p * 16 + m, L - 1)];
    }
};

// a[i S] += D(entry E + i Step) F for the R rows i: the entry is a DPP operand of the multiply-add (the
// compiler moves it to a register pair first, with a wait: three issues instead of one). A block first
// waits out the two cycles that a register written just before it takes to reach a DPP
// instruction, and within one every row is another register.
template <int E, int Step, int R, int S, int L>
__device__ __forceinline__ void rows(const LaneTable<L> &D, double F, double *a) {
#define NDG_MAC(o, d, f, e) "v_fmac_f64_dpp %" #o ", %" #d ", %" #f " row_newbcast:%" #e " row_mask:0xf bank_mask:0xf\n\t"
#define NDG_ENTRY(i) D.v[(E + (i) * Step) / 16]
#define NDG_LANE(i) (E + (i) * Step) % 16
    if constexpr (R > 4) {
        rows<E, Step, 4, S>(D, F, a);
        rows<E + 4 * Step, Step, R - 4, S>(D, F, a + 4 * S);
    } else if constexpr (R == 4) {
        asm volatile("s_nop 1\n\t" NDG_MAC(0, 4, 8, 9) NDG_MAC(1, 5, 8, 10) NDG_MAC(2, 6, 8, 11) NDG_MAC(3, 7, 8, 12)
                     : "+&v"(a[0]), "+&v"(a[S]), "+&v"(a[2 * S]), "+&v"(a[3 * S])
                     : "v"(NDG_ENTRY(0)), "v"(NDG_ENTRY(1)), "v"(NDG_ENTRY(2)), "v"(NDG_ENTRY(3)), "v"(F),
                       "n"(NDG_LANE(0)), "n"(NDG_LANE(1)), "n"(NDG_LANE(2)), "n"(NDG_LANE(3)));
    } else if constexpr (R == 3) {
        asm volatile("s_nop 1\n\t" NDG_MAC(0, 3, 6, 7) NDG_MAC(1, 4, 6, 8) NDG_MAC(2, 5, 6, 9)
                     : "+&v"(a[0]), "+&v"(a[S]), "+&v"(a[2 * S])
                     : "v"(NDG_ENTRY(0)), "v"(NDG_ENTRY(1)), "v"(NDG_ENTRY(2)), "v"(F), "n"(NDG_LANE(0)),
                       "n"(NDG_LANE(1)), "n"(NDG_LANE(2)));
    } else if constexpr (R == 2) {
        asm volatile("s_nop 1\n\t" NDG_MAC(0, 2, 4, 5) NDG_MAC(1, 3, 4, 6)
                     : "+&v"(a[0]), "+&v"(a[S])
                     : "v"(NDG_ENTRY(0)), "v"(NDG_ENTRY(1)), "v"(F), "n"(NDG_LANE(0)), "n"(NDG_LANE(1)));
    } else if constexpr (R == 1) {
        asm volatile("s_nop 1\n\t" NDG_MAC(0, 1, 2, 3) : "+&v"(a[0]) : "v"(NDG_ENTRY(0)), "v"(F), "n"(NDG_LANE(0)));
    }
#undef NDG_MAC
#undef NDG_ENTRY
#undef NDG_LANE
}

// D^ F of a line by even and odd parts: the Gauss nodes are symmetric, so D^[N-i][N-k] = -D^[i][k], and with
// s_k = F[k] + F[N-k], d_k = F[k] - F[N-k] (k < h = (N+1)/2) and the middle node m of an even order
//   Q_i = sum_k A[i][k] s_k + D^[i][m] F[m],  P_i = sum_k B[i][k] d_k,  A, B = (D^[i][k] +- D^[i][N-k])/2,
//   (D^ F)[i] = P_i + Q_i,  (D^ F)[N-i] = P_i - Q_i,  (D^ F)[m] = P_m,
// about half the multiply-adds and entries of D^. The table holds row by row A[i][.], D^[i][m], B[i][.],
// then B[m][.].

// Q_i (summed in place N - i) and P_i (in place i) of the rows i < h, and P_m, a column at a time:
// entry c of a row multiplies F[c], s in [0, h), F[m] at h, then d.
template <int NF, int c = 0>
__device__ __forceinline__ void even_odd_columns(const LaneTable<even_odd_len(NF)> &D, const double *F, double *a) {
    constexpr int h = NF / 2, odd = NF & 1, per = 2 * h + odd;
    if constexpr (c < h + odd) rows<c, per, h, -1>(D, F[c], a + NF - 1);
    else rows<c, per, h, 1>(D, F[c], a);
    if constexpr (odd && c >= h + 1) rows<h * per + c - h - 1, 1, 1, 1>(D, F[c], a + h);
    if constexpr (c + 1 < per) even_odd_columns<NF, c + 1>(D, F, a);
}

// a = D^ F.
template <int NF>
__device__ __forceinline__ void contract(const LaneTable<even_odd_len(NF)> &D, const double *F, double *a) {
    constexpr int h = NF / 2, odd = NF & 1;
    double t[NF];
#pragma unroll
    for (int k = 0; k < h; ++k) {
        t[k] = F[k] + F[NF - 1 - k];
        t[h + odd + k] = F[k] - F[NF - 1 - k];
    }
    if (odd) t[h] = F[h];
#pragma unroll
    for (int i = 0; i < NF; ++i) a[i] = 0.0;
    even_odd_columns<NF>(D, t, a);
#pragma unroll
    for (int i = 0; i < h; ++i) {
        const double P = a[i], Q = a[NF - 1 - i];
        a[i] = P + Q;
        a[NF - 1 - i] = P - Q;
    }
}

// 1/x from the hardware reciprocal estimate and two Newton steps (quadratic convergence from its
// ~2^-29 relative error to the rounding error of the last step).
__device__ __forceinline__ double recip(double x) {
    double r = __builtin_amdgcn_rcp(x);
    r = fma(r, fma(-x, r, 1.0), r);
    r = fma(r, fma(-x, r, 1.0), r);
    return r;
}

// Element2D_t::almost_equal with 2 ulp (src/meshes/Mesh2D_t.cpp:3785-3792).
__device__ __forceinline__ bool almost_equal2(double a, double b) {
    return fabs(a - b) <= 2.220446049250313e-16 * fabs(a + b) * 2 || fabs(a - b) < 2.2250738585072014e-308;
}

// Element2D_t::interpolate_from (src/entities/Element2D_t.cpp:345-579) at reference point (X, Y) of
// the old element of order No, from one field sf[(No+1)^2] of it: the old element's node when
// both coordinates match a node (almost_equal, the last matching index wins), a 1D barycentric
// interpolation along the other coordinate when one matches, else the tensor barycentric
// interpolation. xo, lo: nodes and barycentric weights of order No.
__device__ inline double interpolate_at(const double *sf, int No, double X, double Y, const double *xo,
                                        const double *lo) {
    const int nfo = No + 1;
    int col = -1, row = -1;
    for (int m = 0; m <= No; ++m) {
        if (almost_equal2(X, xo[m])) col = m;
        if (almost_equal2(Y, xo[m])) row = m;
    }
    if (row >= 0 && col >= 0) return sf[col * nfo + row];
    if (row >= 0) {
        double num = 0.0, den = 0.0;
        for (int m = 0; m <= No; ++m) {
            const double t = lo[m] / (X - xo[m]);
            num += t * sf[m * nfo + row];
            den += t;
        }
        return num / den;
    }
    if (col >= 0) {
        double num = 0.0, den = 0.0;
        for (int n = 0; n <= No; ++n) {
            const double t = lo[n] / (Y - xo[n]);
            num += t * sf[col * nfo + n];
            den += t;
        }
        return num / den;
    }
    double dx = 0.0, dy = 0.0;
    for (int k = 0; k <= No; ++k) {
        dx += lo[k] / (X - xo[k]);
        dy += lo[k] / (Y - xo[k]);
    }
    double v = 0.0;
    for (int m = 0; m <= No; ++m) {
        const double tx = lo[m] / ((X - xo[m]) * dx);
        for (int n = 0; n <= No; ++n) v += sf[m * nfo + n] * tx * (lo[n] / ((Y - xo[n]) * dy));
    }
    return v;
}

}  // namespace ndg
