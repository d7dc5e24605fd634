// qinterp.hip -- QuadratureInterpolator::Mult for H1 E-vectors on hexahedra
// (fem/quadinterpolator.cpp:226-341, tensor kernels fem/qinterp/eval.hpp and
// fem/qinterp/grad.hpp:233-375; determinants as fem/qinterp/det.hpp).
//
// A Q x Q thread plane per element, several elements per work-group: each
// component of the element's lexicographic E-vector block (D^3 values) is
// staged in LDS and contracted along x into LDS (B and G), then along y and z in
// registers at the thread's own (qx, qy).  Physical derivatives apply J^-T: on
// straight-sided meshes the Jacobian comes from the element's corners in the
// same kernel, on curved ones from the geometric factors (a pass of its own:
// the 18 Q registers of a curved column beside the field's would leave one wave
// per SIMD).  Determinants (vdim = 3) are taken of the 3 x 3 reference
// derivative matrix in a second, per-point pass.
//
// Values and physical derivatives at p = 3, Q = 5, 40 x 39 x 38 straight
// elements (237 MB written): 71 us; with one element's 25 threads per
// work-group and the Jacobians through memory it was 247 + 237 us.
#include <hip/hip_runtime.h>

#include "geom_body.hpp"
#include "internal.hpp"

namespace h1pa {
namespace kern {
namespace {

// Q-vector offsets of value (c) and derivative (c, d) at point q of element e.
__device__ __forceinline__ int64_t val_at(int by_vdim, int64_t q, int c, int64_t e, int64_t nq,
                                          int vdim) {
    return by_vdim ? c + vdim * (q + nq * e) : q + nq * (c + vdim * e);
}
__device__ __forceinline__ int64_t der_at(int by_vdim, int64_t q, int c, int d, int64_t e,
                                          int64_t nq, int vdim) {
    return by_vdim ? c + vdim * (d + 3 * (q + nq * e)) : q + nq * (c + vdim * (d + 3 * e));
}

struct FieldBasis {  // the field's basis at the Q Gauss-Legendre points
    double B[90], G[90];  // B[d + D q]
};

template <int D, int Q>
constexpr int qi_lds() { return D * D * D + 2 * D * D * Q; }

// STRAIGHT: physical derivatives with the Jacobian of the corners X; else J
// holds the geometric factors, or is null for reference derivatives.
template <int D, int Q, bool STRAIGHT>
__global__ void __launch_bounds__(256)
k_qinterp(int64_t ne, int nb, int vdim, int want_val, int want_der, int by_vdim, FieldBasis fb,
          GeomBasis gb, const double *__restrict__ X, const double *__restrict__ J,
          const double *__restrict__ x, double *__restrict__ val, double *__restrict__ der) {
    constexpr int QQ = Q * Q, NQ = Q * Q * Q, DDD = D * D * D, DD = D * D;
    constexpr int NL = (DDD + QQ - 1) / QQ;
    extern __shared__ double smem[];
    const int le = threadIdx.x / QQ, t = threadIdx.x - le * QQ;
    const int a = t % Q, b = t / Q;
    const int64_t e = (int64_t)blockIdx.x * nb + le;
    const bool valid = e < ne;
    // the tables of the rows that differ between threads; the z rows are uniform
    double *const sB = smem, *const sG = smem + Q * D;
    double *const sx = smem + 2 * Q * D + le * qi_lds<D, Q>();
    double *const A0 = sx + DDD, *const A1 = A0 + DD * Q;
    for (int i = threadIdx.x; i < Q * D; i += blockDim.x) {
        sB[i] = fb.B[i];
        sG[i] = fb.G[i];
    }
    GeomColumn<Q, false, 2> geo;
    if constexpr (STRAIGHT) geo.eval(gb, X + 24 * e, a, b, t, valid, nullptr, nullptr);
    // the nodes of the next component are requested before this one's stages
    double nx[NL];
    auto request = [&](int c) {
        const double *xe = x + (int64_t)DDD * (c + (int64_t)vdim * e);
#pragma unroll
        for (int k = 0; k < NL; ++k) {
            const int i = t + QQ * k;
            nx[k] = xe[i < DDD ? i : DDD - 1];
        }
    };
    if (valid) request(0);
    for (int c = 0; c < vdim; ++c) {
        if (valid) {
#pragma unroll
            for (int k = 0; k < NL; ++k)
                if (t + QQ * k < DDD) sx[t + QQ * k] = nx[k];
            if (c + 1 < vdim) request(c + 1);
        }
        __syncthreads();
        // x: u = sum_dx X B(qx, dx), v = sum_dx X G(qx, dx) for rows (dy, dz)
        if (valid) {
            double xb[D], xg[D];
#pragma unroll
            for (int d = 0; d < D; ++d) {
                xb[d] = sB[d + D * a];
                xg[d] = sG[d + D * a];
            }
#pragma unroll 1
            for (int r = b; r < DD; r += Q) {
                double u = 0.0, v = 0.0;
#pragma unroll
                for (int dx = 0; dx < D; ++dx) {
                    const double in = sx[dx + D * r];
                    u = fma(in, xb[dx], u);
                    v = fma(in, xg[dx], v);
                }
                A0[a + Q * r] = u;
                A1[a + Q * r] = v;
            }
        }
        __syncthreads();
        if (!valid) continue;
        // y at the thread's (qx, qy) for each dz
        double u[D], v[D], w[D];
        {
            double yb[D], yg[D];
#pragma unroll
            for (int d = 0; d < D; ++d) {
                yb[d] = sB[d + D * b];
                yg[d] = sG[d + D * b];
            }
#pragma unroll
            for (int dz = 0; dz < D; ++dz) {
                u[dz] = v[dz] = w[dz] = 0.0;
#pragma unroll
                for (int dy = 0; dy < D; ++dy) {
                    const double a0 = A0[a + Q * (dy + D * dz)], a1 = A1[a + Q * (dy + D * dz)];
                    u[dz] = fma(a1, yb[dy], u[dz]);  // d/dx
                    v[dz] = fma(a0, yg[dy], v[dz]);  // d/dy
                    w[dz] = fma(a0, yb[dy], w[dz]);  // value, d/dz
                }
            }
        }
        // z: all points of the column
#pragma unroll 1
        for (int qz = 0; qz < Q; ++qz) {
            const double *zb = fb.B + D * qz, *zg = fb.G + D * qz;
            double d0 = 0.0, d1 = 0.0, d2 = 0.0, vv = 0.0;
#pragma unroll
            for (int dz = 0; dz < D; ++dz) {
                d0 = fma(u[dz], zb[dz], d0);
                d1 = fma(v[dz], zb[dz], d1);
                d2 = fma(w[dz], zg[dz], d2);
                vv = fma(w[dz], zb[dz], vv);
            }
            const int64_t q = a + Q * (b + Q * qz);
            if (want_val) val[val_at(by_vdim, q, c, e, NQ, vdim)] = vv;
            if (want_der) {
                if (STRAIGHT || J) {
                    // grad_x = J^-T grad_xi with J(r, c) = dx_r / dxi_c = j[r + 3 c]:
                    // (J^-T)(r, c) = C(r, c) / det J, C the cofactor matrix
                    double j[9], P[3];
                    if constexpr (STRAIGHT) {
                        geo.at(gb, qz, j, P);
                    } else {
#pragma unroll
                        for (int k = 0; k < 9; ++k) j[k] = J[q + NQ * (k + 9 * e)];
                    }
                    const double c00 = j[4] * j[8] - j[7] * j[5];
                    const double c01 = j[7] * j[2] - j[1] * j[8];
                    const double c02 = j[1] * j[5] - j[4] * j[2];
                    const double c10 = j[6] * j[5] - j[3] * j[8];
                    const double c11 = j[0] * j[8] - j[6] * j[2];
                    const double c12 = j[3] * j[2] - j[0] * j[5];
                    const double c20 = j[3] * j[7] - j[6] * j[4];
                    const double c21 = j[6] * j[1] - j[0] * j[7];
                    const double c22 = j[0] * j[4] - j[3] * j[1];
                    const double s = 1.0 / (j[0] * c00 + j[3] * c01 + j[6] * c02);
                    const double U = (c00 * d0 + c01 * d1 + c02 * d2) * s;
                    const double V = (c10 * d0 + c11 * d1 + c12 * d2) * s;
                    const double W = (c20 * d0 + c21 * d1 + c22 * d2) * s;
                    d0 = U;
                    d1 = V;
                    d2 = W;
                }
                der[der_at(by_vdim, q, c, 0, e, NQ, vdim)] = d0;
                der[der_at(by_vdim, q, c, 1, e, NQ, vdim)] = d1;
                der[der_at(by_vdim, q, c, 2, e, NQ, vdim)] = d2;
            }
        }
        // the next component's first barrier keeps A0, A1 until every column is done
    }
}

// det of the 3 x 3 reference derivative matrix M(c, d) (byNODES derivatives)
__global__ void k_qi_det(int64_t nq, int64_t ne, const double *__restrict__ der,
                         double *__restrict__ det) {
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= nq * ne) return;
    const int64_t q = i % nq, e = i / nq;
    double m[9];  // m[c + 3 d]
#pragma unroll
    for (int k = 0; k < 9; ++k) m[k] = der[q + nq * (k + 9 * e)];
    det[i] = m[0] * (m[4] * m[8] - m[5] * m[7]) - m[3] * (m[1] * m[8] - m[2] * m[7]) +
             m[6] * (m[1] * m[5] - m[2] * m[4]);
}

template <int D, int Q>
void launch_qi(int64_t ne, int vdim, int want_val, int want_der, int by_vdim,
               const FieldBasis &fb, const GeomBasis &gb, const double *X, const double *J,
               const double *x, double *val, double *der, hipStream_t s) {
    const int nb = geom_nb(Q, qi_lds<D, Q>());
    const dim3 grid((unsigned)((ne + nb - 1) / nb)), block(nb * Q * Q);
    const unsigned lds = 8 * (2 * Q * D + nb * qi_lds<D, Q>());
    if (X)
        hipLaunchKernelGGL((k_qinterp<D, Q, true>), grid, block, lds, s, ne, nb, vdim, want_val,
                           want_der, by_vdim, fb, gb, X, J, x, val, der);
    else
        hipLaunchKernelGGL((k_qinterp<D, Q, false>), grid, block, lds, s, ne, nb, vdim, want_val,
                           want_der, by_vdim, fb, gb, X, J, x, val, der);
}

}  // namespace

bool qinterp_supported(int p, int q1d) {
    return p >= 1 && p <= 8 && q1d >= p + 1 && q1d <= p + 3 && q1d <= 10;
}

void qinterp(Space &sp, int q1d, int vdim, unsigned flags, int by_vdim, const double *x,
             double *val, double *der, double *det, hipStream_t s) {
    const int p = sp.p, D = p + 1, Q = q1d;
    const int64_t ne = sp.ne, nq = (int64_t)Q * Q * Q;
    const bool want_val = flags & H1PA_QI_VALUES;
    const bool phys = flags & H1PA_QI_PHYSICAL_DERIVATIVES;
    const bool want_der = (flags & H1PA_QI_DERIVATIVES) || phys;
    const bool want_det = flags & H1PA_QI_DETERMINANTS;
    if (ne == 0) return;
    // basis at the Gauss-Legendre points
    double xq[16], wq[16], B[128], G[128];
    gauss_legendre(Q, xq, wq);
    lagrange_basis(p, Q, xq, B, G);  // B[q + Q d]
    FieldBasis fb;
    for (int q = 0; q < Q; ++q)
        for (int d = 0; d < D; ++d) {
            fb.B[d + D * q] = B[q + Q * d];
            fb.G[d + D * q] = G[q + Q * d];
        }
    GeomBasis gb{};
    const double *X = nullptr;  // corners of a straight-sided mesh
    StreamBuf<double> J;
    if (phys) {
        sp.mesh->ensure_nodes(s);
        if (sp.mesh->node_order == 1) {
            gb = make_geom_basis(Q, 1);
            X = sp.mesh->d_nodes.p;
        } else {
            J.alloc(nq * 9 * ne, s);
            geometric_factors(*sp.mesh, q1d, nullptr, J.p, nullptr, s);
        }
    }
    // determinants need byNODES reference derivatives
    StreamBuf<double> dtmp;
    const double *dref = nullptr;
    if (want_det) {
        if ((flags & H1PA_QI_DERIVATIVES) && !by_vdim) {
            dref = der;
        } else {
            dtmp.alloc(nq * 9 * ne, s);
            dref = dtmp.p;
        }
    }
    auto run = [&](int wv, int wd, bool ph, int bv, double *dv) {
#define X(DD, QQ)                                                                         \
    if (D == DD && Q == QQ) {                                                             \
        launch_qi<DD, QQ>(ne, vdim, wv, wd, bv, fb, gb, ph ? X : nullptr,                 \
                          ph ? J.p : nullptr, x, val, dv, s);                             \
        H1PA_HIP(hipGetLastError());                                                      \
        return;                                                                           \
    }
        X(2, 2) X(2, 3) X(2, 4) X(3, 3) X(3, 4) X(3, 5) X(4, 4) X(4, 5) X(4, 6) X(5, 5)
        X(5, 6) X(5, 7) X(6, 6) X(6, 7) X(6, 8) X(7, 7) X(7, 8) X(7, 9) X(8, 8) X(8, 9)
        X(8, 10) X(9, 9) X(9, 10)
#undef X
        throw Error{H1PA_EUNSUP, "qinterp: unsupported (p, q1d)"};
    };
    if (want_val || want_der) run(want_val, want_der, phys, by_vdim, der);
    if (want_det) {
        if (dref != der) run(0, 1, false, 0, dtmp.p);
        hipLaunchKernelGGL(k_qi_det, dim3((unsigned)((nq * ne + 255) / 256)), dim3(256), 0, s, nq,
                           ne, dref, det);
        H1PA_HIP(hipGetLastError());
    }
    // the temporaries are freed at return, in stream order
}

}  // namespace kern
}  // namespace h1pa
