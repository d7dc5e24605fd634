// geom_body.hpp -- the Jacobian of the element map at a quadrature column, by
// sum factorization; shared by the PA set-up, the geometric factors, the
// domain right-hand side (geometry.hip) and the physical derivatives of the
// quadrature interpolator (qinterp.hip).
//
// A thread owns the quadrature column (qx, qy) of one element and ends up
// with the Jacobian (and the physical point) at its Q points in registers.
// Evaluating the Dg^3 nodes at every point separately cost 12 Dg^3
// multiply-adds and 3 Dg^3 loads a point: 2171 us of PA set-up at Dg = 5, Q = 6,
// 32^3 elements, 120 us so (340 MB of PA data written; 66 us at the rate of a
// large copy).  What bounds it now is latency: the Jacobian of a column takes
// 18 Q registers, which leaves 2-3 waves per SIMD for the barrier-separated
// stages (curved), and the write stream (straight: 1.52 ms for the 5.1 GB of
// 79^3 elements at Q = 6, 3.24 ms before).
//   straight-sided elements (Dg = 2): the 24 corner coordinates are the same
//     addresses for the element's Q^2 threads, so they are read straight from
//     memory and contracted along x and y in registers: no LDS, no barrier,
//     any number of elements per block;
//   curved elements: one coordinate at a time, nodes -> LDS, x-contraction
//     (B and G) -> LDS, y in registers at the thread's own (qx, qy), and the z
//     sums of all Q points accumulated in registers with wave-uniform rows of
//     the table.  LDS holds Dg^3 + 2 Dg^2 Q doubles per element.
#pragma once

#include "internal.hpp"

namespace h1pa {
namespace kern {

struct GeomBasis {          // geometry basis at the Q Gauss-Legendre points
    int Q, Dg;
    double B[10 * 10];      // B[q + Q*d]
    double G[10 * 10];
    double w[10];           // 1D Gauss-Legendre weights
};

GeomBasis make_geom_basis(int Q, int pg);

// Doubles of LDS of the curved evaluation: per element, and per block for the
// tables.
inline __host__ __device__ int geom_lds(int Q, int Dg) {
    return Dg > 2 ? Dg * Dg * Dg + 2 * Dg * Dg * Q : 0;
}
inline __host__ __device__ int geom_tab_lds(int Q, int Dg) { return Dg > 2 ? 2 * Q * Dg : 0; }
__device__ __forceinline__ void load_geom_tables(const GeomBasis &gb, int Q, double *tab) {
    const int n = Q * gb.Dg;
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        tab[i] = gb.B[i];
        tab[n + i] = gb.G[i];
    }
}
// Elements per block of `per` LDS doubles each: at most 256 threads (one
// element's Q^2 at least) and 40 KiB, so that four blocks stay on a CU.
inline int geom_nb(int Q, int per) {
    int nb = 256 / (Q * Q);
    if (nb < 1) nb = 1;
    while (nb > 1 && nb * per * 8 > 40 * 1024) --nb;
    return nb;
}

// Jacobian columns of one thread: at(qz, J, P) gives J[r + 3 c] = dx_r / dxi_c
// and the point P at (qx, qy, qz).  WP: points wanted.  DG: nodes per
// direction -- 2 straight-sided; above 2 known when the kernel is compiled (the
// thread's table rows then stay in registers and the next coordinate's nodes
// are requested a coordinate ahead: 239 -> 120 us for the set-up above); 0 read
// from the table at run time.
template <int Q, bool WP, int DG>
struct GeomColumn;

template <int Q, bool WP>
struct GeomColumn<Q, WP, 2> {
    double c0[3][2], c1[3][2], c2[3][2];  // [coordinate][dz]: G_x B_y, B_x G_y, B_x B_y

    // X: the element's nodes [8][3]; a, b = qx, qy.
    __device__ __forceinline__ void eval(const GeomBasis &gb, const double *__restrict__ X, int a,
                                         int b, int, bool valid, double *, const double *) {
        if (!valid) return;
        const double bx0 = gb.B[a], bx1 = gb.B[a + Q], gx0 = gb.G[a], gx1 = gb.G[a + Q];
        const double by0 = gb.B[b], by1 = gb.B[b + Q], gy0 = gb.G[b], gy1 = gb.G[b + Q];
#pragma unroll
        for (int r = 0; r < 3; ++r) {
            double x[8];
#pragma unroll
            for (int l = 0; l < 8; ++l) x[l] = X[l + 8 * r];
#pragma unroll
            for (int dz = 0; dz < 2; ++dz) {
                const double u0 = fma(bx1, x[4 * dz + 1], bx0 * x[4 * dz]);
                const double u1 = fma(bx1, x[4 * dz + 3], bx0 * x[4 * dz + 2]);
                const double v0 = fma(gx1, x[4 * dz + 1], gx0 * x[4 * dz]);
                const double v1 = fma(gx1, x[4 * dz + 3], gx0 * x[4 * dz + 2]);
                c0[r][dz] = fma(by1, v1, by0 * v0);
                c1[r][dz] = fma(gy1, u1, gy0 * u0);
                c2[r][dz] = fma(by1, u1, by0 * u0);
            }
        }
    }
    __device__ __forceinline__ void at(const GeomBasis &gb, int qz, double (&J)[9],
                                       double (&P)[3]) const {
        const double b0 = gb.B[qz], b1 = gb.B[qz + Q], g0 = gb.G[qz], g1 = gb.G[qz + Q];
#pragma unroll
        for (int r = 0; r < 3; ++r) {
            J[r] = fma(b1, c0[r][1], b0 * c0[r][0]);
            J[r + 3] = fma(b1, c1[r][1], b0 * c1[r][0]);
            J[r + 6] = fma(g1, c2[r][1], g0 * c2[r][0]);
            if constexpr (WP) P[r] = fma(b1, c2[r][1], b0 * c2[r][0]);
        }
    }
};

template <int Q, bool WP, int DG>
struct GeomColumn {
    double j0[3][Q], j1[3][Q], j2[3][Q];
    double p[WP ? 3 : 1][WP ? Q : 1];

    // Every thread of the block must call this (barriers); s: the element's
    // geom_lds(Q, Dg) doubles; t: thread of the element's Q^2; tab: the
    // block's copy of B and G (load_geom_tables).
    __device__ __forceinline__ void eval(const GeomBasis &gb, const double *__restrict__ X, int a,
                                         int b, int t, bool valid, double *s, const double *tab) {
        constexpr int QQ = Q * Q;
        const int Dg = DG ? DG : gb.Dg, nd = Dg * Dg * Dg, dd = Dg * Dg;
        double *sx = s, *A0 = s + nd, *A1 = A0 + dd * Q;
        const double *tB = tab, *tG = tab + Q * Dg;
        // the thread's rows of the tables: at its qx for x, at its qy for y
        double xb[DG ? DG : 1], xg[DG ? DG : 1], yb[DG ? DG : 1], yg[DG ? DG : 1];
        if constexpr (DG > 0) {
#pragma unroll
            for (int i = 0; i < DG; ++i) {
                xb[i] = tB[a + Q * i];
                xg[i] = tG[a + Q * i];
                yb[i] = tB[b + Q * i];
                yg[i] = tG[b + Q * i];
            }
        }
        // the nodes of the next coordinate are requested before this one's stages
        constexpr int NL = DG ? (DG * DG * DG + QQ - 1) / QQ : 1;
        double nx[NL];
        auto request = [&](int r) {
#pragma unroll
            for (int k = 0; k < NL; ++k) {
                const int i = t + QQ * k;
                nx[k] = X[(i < nd ? i : nd - 1) + nd * r];
            }
        };
        if constexpr (DG > 0) {
            if (valid) request(0);
        }
#pragma unroll
        for (int r = 0; r < 3; ++r) {
            if constexpr (DG > 0) {
                if (valid) {
#pragma unroll
                    for (int k = 0; k < NL; ++k)
                        if (t + QQ * k < nd) sx[t + QQ * k] = nx[k];
                    if (r < 2) request(r + 1);
                }
            } else if (valid) {
                for (int i = t; i < nd; i += QQ) sx[i] = X[i + nd * r];
            }
            __syncthreads();
            if (valid)
#pragma unroll 1
                for (int row = b; row < dd; row += Q) {
                    double u = 0.0, v = 0.0;
                    if constexpr (DG > 0) {
#pragma unroll
                        for (int i = 0; i < DG; ++i) {
                            const double in = sx[i + DG * row];
                            u = fma(in, xb[i], u);
                            v = fma(in, xg[i], v);
                        }
                    } else {
                        for (int i = 0; i < Dg; ++i) {
                            const double in = sx[i + Dg * row];
                            u = fma(in, tB[a + Q * i], u);
                            v = fma(in, tG[a + Q * i], v);
                        }
                    }
                    A0[a + Q * row] = u;
                    A1[a + Q * row] = v;
                }
            __syncthreads();
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                j0[r][q] = j1[r][q] = j2[r][q] = 0.0;
                if constexpr (WP) p[r][q] = 0.0;
            }
            if (valid)
#pragma unroll 1
                for (int dz = 0; dz < Dg; ++dz) {
                    double c0 = 0.0, c1 = 0.0, c2 = 0.0;
                    const double *r0 = A0 + a + Q * Dg * dz, *r1 = A1 + a + Q * Dg * dz;
                    if constexpr (DG > 0) {
#pragma unroll
                        for (int dy = 0; dy < DG; ++dy) {
                            const double a0 = r0[Q * dy], a1 = r1[Q * dy];
                            c0 = fma(a1, yb[dy], c0);
                            c1 = fma(a0, yg[dy], c1);
                            c2 = fma(a0, yb[dy], c2);
                        }
                    } else {
                        for (int dy = 0; dy < Dg; ++dy) {
                            const double by = tB[b + Q * dy], gy = tG[b + Q * dy];
                            const double a0 = r0[Q * dy], a1 = r1[Q * dy];
                            c0 = fma(a1, by, c0);
                            c1 = fma(a0, gy, c1);
                            c2 = fma(a0, by, c2);
                        }
                    }
                    const double *zb = gb.B + Q * dz, *zg = gb.G + Q * dz;
#pragma unroll
                    for (int q = 0; q < Q; ++q) {
                        j0[r][q] = fma(c0, zb[q], j0[r][q]);
                        j1[r][q] = fma(c1, zb[q], j1[r][q]);
                        j2[r][q] = fma(c2, zg[q], j2[r][q]);
                        if constexpr (WP) p[r][q] = fma(c2, zb[q], p[r][q]);
                    }
                }
        }
    }
    __device__ __forceinline__ void at(const GeomBasis &, int qz, double (&J)[9],
                                       double (&P)[3]) const {
#pragma unroll
        for (int r = 0; r < 3; ++r) {
            J[r] = j0[r][qz];
            J[r + 3] = j1[r][qz];
            J[r + 6] = j2[r][qz];
            if constexpr (WP) P[r] = p[r][qz];
        }
    }
};

// det J with J[r + 3 c]
__device__ __forceinline__ double det3(const double (&J)[9]) {
    return J[0] * (J[4] * J[8] - J[5] * J[7]) - J[1] * (J[3] * J[8] - J[5] * J[6]) +
           J[2] * (J[3] * J[7] - J[4] * J[6]);
}

}  // namespace kern
}  // namespace h1pa
