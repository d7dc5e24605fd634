// geometry.hip -- mesh nodes, geometric factors and PA setup on the device.
//
// The setup is one fused pass per (quadrature point, element): Jacobian from
// the element nodes (QuadratureInterpolator derivatives, fem/qinterp/grad.hpp:
// 233-375), adj(J) and det(J), the coefficient at the physical point, and the
// PA data (PADiffusionSetup3D, fem/integ/bilininteg_diffusion_kernels.cpp:
// 262-386; MassIntegrator::AssemblePA, fem/integ/bilininteg_mass_pa.cpp:76-88).
// J is never stored: at 32M DOFs and p = 1 it alone would be 61 GB.
#include <algorithm>
#include <cmath>

#include "apply_body.hpp"
#include "geom_body.hpp"
#include "internal.hpp"

namespace h1pa {
namespace kern {

GeomBasis make_geom_basis(int Q, int pg) {
    GeomBasis gb{};
    gb.Q = Q;
    gb.Dg = pg + 1;
    double x[16], w[16];
    gauss_legendre(Q, x, w);
    lagrange_basis(pg, Q, x, gb.B, gb.G);
    for (int i = 0; i < Q; ++i) gb.w[i] = w[i];
    return gb;
}

namespace {

constexpr int kBlock = 256;
inline unsigned nblocks(int64_t n) { return (unsigned)((n + kBlock - 1) / kBlock); }

struct Fourier8 {           // g(x) = sum_m a cos(2 pi k_m . x + phi_m)
    double k[8][3];
    double phi[8];
    double a;
};

__host__ __device__ inline uint64_t splitmix64(uint64_t x) {
    x += 0x9E3779B97F4A7C15ULL;
    x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ULL;
    x = (x ^ (x >> 27)) * 0x94D049BB133111EBULL;
    return x ^ (x >> 31);
}

Fourier8 make_fourier(uint64_t seed) {
    // 8 modes; integer wave vectors in [-3,3]^3 \ {0}, phases U[0, 2 pi),
    // amplitude 0.5 / sqrt(8) each (root sum of squares 0.5; RMS of g
    // 0.5 / sqrt(2) for distinct modes).
    Fourier8 f{};
    uint64_t ctr = 0;
    auto draw = [&]() { return (double)(splitmix64(seed ^ splitmix64(ctr++)) >> 11) * (1.0 / 9007199254740992.0); };
    for (int m = 0; m < 8; ++m) {
        int kk[3];
        do {
            for (int c = 0; c < 3; ++c) kk[c] = (int)std::floor(draw() * 7.0) - 3;
        } while (kk[0] == 0 && kk[1] == 0 && kk[2] == 0);
        for (int c = 0; c < 3; ++c) f.k[m][c] = kk[c];
        f.phi[m] = 6.283185307179586 * draw();
    }
    f.a = 0.5 / std::sqrt(8.0);
    return f;
}

// x[i] = lo + (hi - lo) u_i, u_i = (splitmix64(seed ^ splitmix64(i)) >> 11) 2^-53.
__global__ void k_randomize(int64_t n, double *__restrict__ x, uint64_t seed, double lo,
                            double hi) {
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double u = (double)(splitmix64(seed ^ splitmix64((uint64_t)i)) >> 11) *
                     (1.0 / 9007199254740992.0);
    x[i] = lo + (hi - lo) * u;
}

// ---- nodes -------------------------------------------------------------------
__global__ void k_nodes_trilinear(int64_t ne, const int *__restrict__ topo,
                                  const double *__restrict__ xyz, double *__restrict__ X) {
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= ne * 8) return;
    const int64_t e = i / 8;
    const int l = (int)(i % 8);
    // lex (a,b,c) -> MFEM hex vertex (p = 1 dof_map)
    const int lex2v[8] = {0, 1, 3, 2, 4, 5, 7, 6};
    const int v = topo[29 * e + lex2v[l]];
    for (int c = 0; c < 3; ++c) X[l + 8 * (c + 3 * e)] = xyz[3 * (int64_t)v + c];
}

__global__ void k_nodes_curved(int64_t ne, int Dg, const int *__restrict__ topo,
                               const double *__restrict__ xyz, const double *__restrict__ gll,
                               double amp, double *__restrict__ X) {
    const int nd = Dg * Dg * Dg;
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= ne * nd) return;
    const int64_t e = i / nd;
    const int l = (int)(i - e * nd);
    const double s[3] = {gll[l % Dg], gll[(l / Dg) % Dg], gll[l / (Dg * Dg)]};
    const int lex2v[8] = {0, 1, 3, 2, 4, 5, 7, 6};
    double P[3] = {0.0, 0.0, 0.0};
    for (int c8 = 0; c8 < 8; ++c8) {
        const double N = ((c8 & 1) ? s[0] : 1.0 - s[0]) * ((c8 & 2) ? s[1] : 1.0 - s[1]) *
                         ((c8 & 4) ? s[2] : 1.0 - s[2]);
        const int v = topo[29 * e + lex2v[c8]];
        for (int c = 0; c < 3; ++c) P[c] += N * xyz[3 * (int64_t)v + c];
    }
    const double tp = 6.283185307179586476925286766559;
    const double xp = P[0] + amp * sin(tp * P[1]) * sin(tp * P[2]);
    const double yp = P[1] + amp * sin(tp * P[2]) * sin(tp * P[0]);
    const double zp = P[2] + amp * sin(tp * P[0]) * sin(tp * P[1]);
    X[l + nd * (0 + 3 * e)] = xp;
    X[l + nd * (1 + 3 * e)] = yp;
    X[l + nd * (2 + 3 * e)] = zp;
}

__device__ inline double coeff_value(int kind, double cval, const double *__restrict__ cdata,
                                     const Fourier8 &fm, int64_t e, int q, int nq,
                                     const double (&P)[3]) {
    const double tp = 6.283185307179586476925286766559;
    switch (kind) {
        case H1PA_COEFF_SINCOS:
            return 1.0 + 0.5 * sin(tp * P[0]) * cos(tp * P[1]) * sin(tp * P[2]);
        case H1PA_COEFF_PER_ELEMENT: return cdata[e];
        case H1PA_COEFF_QUADRATURE: return cdata[q + (int64_t)nq * e];
        case H1PA_COEFF_FOURIER: {
            double g = 0.0;
            for (int m = 0; m < 8; ++m)
                g += fm.a * cos(tp * (fm.k[m][0] * P[0] + fm.k[m][1] * P[1] + fm.k[m][2] * P[2]) +
                                fm.phi[m]);
            return exp(g);
        }
        default: return cval;
    }
}

// What the element, the quadrature column (a, b) and the LDS of this thread
// are.  Straight-sided elements need no barrier and no LDS, so their threads
// run over (element, column) without a gap; the curved evaluation keeps the
// Q^2 threads of nb whole elements in a block.
template <int Q, int DG>
struct ColumnOf {
    int64_t e;
    int a, b, t;
    bool valid;
    double *s;
    __device__ __forceinline__ ColumnOf(int64_t ne, int nb, int Dg, double *smem) {
        constexpr int QQ = Q * Q;
        if constexpr (DG != 2) {
            const int le = threadIdx.x / QQ;
            t = threadIdx.x - le * QQ;
            e = (int64_t)blockIdx.x * nb + le;
            valid = e < ne;
            s = smem + geom_tab_lds(Q, Dg) + le * geom_lds(Q, Dg);
        } else {
            const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
            e = i / QQ;
            t = (int)(i - e * QQ);
            valid = e < ne;
            s = nullptr;
        }
        a = t % Q;
        b = t / Q;
    }
};

template <int Q, bool WP, int DG>
__global__ void __launch_bounds__(kBlock)
k_geometric_factors(int64_t ne, int nb, GeomBasis gb, const double *__restrict__ X,
                    double *__restrict__ Xq, double *__restrict__ Jq, double *__restrict__ detJ) {
    extern __shared__ double smem[];
    constexpr int nq = Q * Q * Q;
    if constexpr (DG != 2) load_geom_tables(gb, Q, smem);
    const ColumnOf<Q, DG> k(ne, nb, gb.Dg, smem);
    const int nd = gb.Dg * gb.Dg * gb.Dg;
    if constexpr (DG != 2) __syncthreads();
    GeomColumn<Q, WP, DG> g;
    g.eval(gb, X + (int64_t)nd * 3 * k.e, k.a, k.b, k.t, k.valid, k.s, smem);
    if (!k.valid) return;
#pragma unroll
    for (int qz = 0; qz < Q; ++qz) {
        double J[9], P[3];
        g.at(gb, qz, J, P);
        const int q = k.a + Q * (k.b + Q * qz);
        if constexpr (WP)
#pragma unroll
            for (int r = 0; r < 3; ++r) Xq[q + (int64_t)nq * (r + 3 * k.e)] = P[r];
        if (Jq)
#pragma unroll
            for (int c = 0; c < 9; ++c) Jq[q + (int64_t)nq * (c + 9 * k.e)] = J[c];
        if (detJ) detJ[q + (int64_t)nq * k.e] = det3(J);
    }
}

// D = W k adj(J) adj(J)^T / det J and / or W k det J at the Q points of a
// column.  WP: the coefficient needs the physical point.
template <int Q, bool WP, int DG>
__global__ void __launch_bounds__(kBlock)
k_pa_setup(int64_t ne, int nb, GeomBasis gb, const double *__restrict__ X, int kind,
           double cval, const double *__restrict__ cdata, Fourier8 fm, double *__restrict__ Dd,
           double *__restrict__ Mv) {
    extern __shared__ double smem[];
    constexpr int nq = Q * Q * Q;
    if constexpr (DG != 2) load_geom_tables(gb, Q, smem);
    const ColumnOf<Q, DG> c(ne, nb, gb.Dg, smem);
    const int nd = gb.Dg * gb.Dg * gb.Dg;
    if constexpr (DG != 2) __syncthreads();
    GeomColumn<Q, WP, DG> g;
    g.eval(gb, X + (int64_t)nd * 3 * c.e, c.a, c.b, c.t, c.valid, c.s, smem);
    if (!c.valid) return;
    const double wxy = gb.w[c.a] * gb.w[c.b];
    double *const dcol = Dd ? Dd + (int64_t)nq * 6 * c.e + c.a + Q * c.b : nullptr;
    double *const mcol = Mv ? Mv + (int64_t)nq * c.e + c.a + Q * c.b : nullptr;
    // the curved evaluation holds its Q points in registers: fully unrolled
    constexpr int UZ = DG != 2 ? Q : 1;
#pragma unroll UZ
    for (int qz = 0; qz < Q; ++qz) {
        double J[9], P[3] = {0.0, 0.0, 0.0};
        g.at(gb, qz, J, P);
        const double W = wxy * gb.w[qz];
        const double k = coeff_value(kind, cval, cdata, fm, c.e, c.a + Q * (c.b + Q * qz), nq, P);
        const double J11 = J[0], J21 = J[1], J31 = J[2];
        const double J12 = J[3], J22 = J[4], J32 = J[5];
        const double J13 = J[6], J23 = J[7], J33 = J[8];
        const double detJ = det3(J);
        if (mcol) mcol[Q * Q * qz] = W * k * detJ;
        if (dcol) {
            // (1/detJ) adj(J) adj(J)^T, symmetric storage 11,21,31,22,32,33
            const double A11 = J22 * J33 - J23 * J32, A12 = J32 * J13 - J12 * J33,
                         A13 = J12 * J23 - J22 * J13;
            const double A21 = J31 * J23 - J21 * J33, A22 = J11 * J33 - J13 * J31,
                         A23 = J21 * J13 - J11 * J23;
            const double A31 = J21 * J32 - J31 * J22, A32 = J31 * J12 - J11 * J32,
                         A33 = J11 * J22 - J12 * J21;
            const double s = W / detJ * k;
            double *d = dcol + Q * Q * qz;
            d[0 * nq] = s * (A11 * A11 + A12 * A12 + A13 * A13);
            d[1 * nq] = s * (A11 * A21 + A12 * A22 + A13 * A23);
            d[2 * nq] = s * (A11 * A31 + A12 * A32 + A13 * A33);
            d[3 * nq] = s * (A21 * A21 + A22 * A22 + A23 * A23);
            d[4 * nq] = s * (A21 * A31 + A22 * A32 + A23 * A33);
            d[5 * nq] = s * (A31 * A31 + A32 * A32 + A33 * A33);
        }
    }
}

// Launch shape of a geometry kernel: blocks, threads and LDS bytes.
struct GeomLaunch {
    dim3 grid, block;
    unsigned lds;
    int nb;  // elements per block
};
GeomLaunch geom_launch(int64_t ne, int Q, int Dg) {
    GeomLaunch l;
    if (Dg == 2) {
        l.nb = 0;
        l.grid = dim3(nblocks(ne * Q * Q));
        l.block = dim3(kBlock);
        l.lds = 0;
    } else {
        l.nb = geom_nb(Q, geom_lds(Q, Dg));
        l.grid = dim3((unsigned)((ne + l.nb - 1) / l.nb));
        l.block = dim3(l.nb * Q * Q);
        l.lds = 8 * (geom_tab_lds(Q, Dg) + l.nb * geom_lds(Q, Dg));
    }
    return l;
}

// DomainLFIntegrator (fem/lininteg.cpp:51-79) at Q = D points per direction:
// b_e = (B^T x B^T x B^T) [w det J f], f at quadrature point q of element e:
// fq[q + nq e] when fq is given (a QuadratureFunction, points x fastest), else
// the constant f.  The sum over the D^3 points of each of the D^3 rows taken
// directly cost 2 D^6 operations an element and was all of the time (933 us at
// p = 5, 23^3 elements); contracted along z, y, x it is 6 D^4 and the kernel
// takes 19 us: latency, 7 blocks per CU at that size; its 37 MB take 7 us at the
// rate of a large copy.
struct LfBasis {
    double B[81];  // B[q + Q d]
};

template <int D, int DG>
__global__ void __launch_bounds__(kBlock)
k_domain_lf(int64_t ne, int nb, int per, GeomBasis gb, LfBasis lb, const double *__restrict__ X,
            double f, const double *__restrict__ fq, const EOut out) {
    extern __shared__ double smem[];
    constexpr int Q = D, QQ = Q * Q, nq = Q * Q * Q;
    if constexpr (DG != 2) load_geom_tables(gb, Q, smem);
    const int le = threadIdx.x / QQ, t = threadIdx.x - le * QQ;
    const int a = t % Q, b = t / Q;
    const int64_t e = (int64_t)blockIdx.x * nb + le;
    const bool valid = e < ne;
    double *const s = smem + geom_tab_lds(Q, gb.Dg) + le * per;
    const int nd = gb.Dg * gb.Dg * gb.Dg;
    double v[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) v[q] = (valid && fq) ? fq[a + Q * b + QQ * q + nq * e] : f;
    if constexpr (DG != 2) __syncthreads();
    {
        GeomColumn<Q, false, DG> g;
        g.eval(gb, X + (int64_t)nd * 3 * e, a, b, t, valid, s, smem);
        const double wxy = gb.w[a] * gb.w[b];
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            double J[9], P[3];
            g.at(gb, q, J, P);
            v[q] *= wxy * gb.w[q] * det3(J);
        }
    }
    if constexpr (DG != 2) __syncthreads();  // the geometry's LDS is free
    if (valid) {   // z: thread (qx, qy)
#pragma unroll
        for (int dz = 0; dz < D; ++dz) {
            double z = 0.0;
#pragma unroll
            for (int q = 0; q < Q; ++q) z = fma(lb.B[q + Q * dz], v[q], z);
            s[a + Q * (b + Q * dz)] = z;
        }
    }
    __syncthreads();
    if (valid)   // y: thread (qx, dz)
#pragma unroll
        for (int q = 0; q < Q; ++q) v[q] = s[a + Q * (q + Q * b)];
    __syncthreads();
    if (valid)
#pragma unroll
        for (int dy = 0; dy < D; ++dy) {
            double y = 0.0;
#pragma unroll
            for (int q = 0; q < Q; ++q) y = fma(lb.B[q + Q * dy], v[q], y);
            s[a + Q * (dy + D * b)] = y;
        }
    __syncthreads();
    if (valid) {   // x: thread (dy, dz)
#pragma unroll
        for (int q = 0; q < Q; ++q) v[q] = s[q + Q * (a + D * b)];
        double yv[D];
#pragma unroll
        for (int dx = 0; dx < D; ++dx) {
            double x = 0.0;
#pragma unroll
            for (int q = 0; q < Q; ++q) x = fma(lb.B[q + Q * dx], v[q], x);
            yv[dx] = x;
        }
        store_line<D, double>(out, e, a, b, yv, 0);
    }
}

}  // namespace

void nodes_trilinear(const Mesh &m, double *d_nodes, hipStream_t s) {
    StreamBuf<double> xyz;
    xyz.upload(m.xyz.data(), m.xyz.size(), s);
    hipLaunchKernelGGL(k_nodes_trilinear, dim3(nblocks(m.ne * 8)), dim3(kBlock), 0, s, m.ne,
                       m.d_topo.p, xyz.p, d_nodes);
    H1PA_HIP(hipGetLastError());
    H1PA_HIP(hipStreamSynchronize(s));
}

void nodes_curved(const Mesh &m, int pg, double amp, double *d_nodes, hipStream_t s) {
    const int Dg = pg + 1;
    double z[16], w[16];
    gauss_lobatto(Dg, z, w);
    StreamBuf<double> xyz, gll;
    xyz.upload(m.xyz.data(), m.xyz.size(), s);
    gll.upload(z, Dg, s);
    hipLaunchKernelGGL(k_nodes_curved, dim3(nblocks(m.ne * Dg * Dg * Dg)), dim3(kBlock), 0, s, m.ne,
                       Dg, m.d_topo.p, xyz.p, gll.p, amp, d_nodes);
    H1PA_HIP(hipGetLastError());
    H1PA_HIP(hipStreamSynchronize(s));
}

// Launches K_(Q, WP, DG) for the number of points and the node count: the field's
// own order (isoparametric, Q = Dg, Dg + 1 and, for the interpolator, Dg + 2) and
// quadratic geometry under any field have their node count compiled in; other
// curved orders read it at run time.  Quadratic geometry, run time -> compiled, us
// of Assemble (of the geometric factors): p = 4, 30^3 elements 128 -> 109 (180 ->
// 162), p = 6, 20^3 77 -> 63 (109 -> 100), p = 8, 16^3 80 -> 67 (142 -> 118); 2^3
// elements at p = 8 38 -> 34 (34 -> 30, as long as one thread a point took).  A mesh
// of a few elements is all latency, and a column's points one after another cost
// more than a thread each where the coefficient is long (8 cosines a point: 48 us
// then, 56 now at p = 8, 2^3; 94 and 59 at 7^3).
#define W_(Q, DG)                                                                             \
    do {                                                                                      \
        if (wp) K_(Q, true, DG);                                                              \
        else K_(Q, false, DG);                                                                \
    } while (0)
#define X_(Q)                                                                                 \
    if (q1d == Q) {                                                                           \
        if (gb.Dg == 2) W_(Q, 2);                                                             \
        else if (gb.Dg == 3 && Q > 3) W_(Q, (Q > 3 ? 3 : 0));                                 \
        else if (gb.Dg == Q && Q > 2 && Q < 10) W_(Q, (Q > 2 && Q < 10 ? Q : 0));             \
        else if (gb.Dg == Q - 1 && Q > 3) W_(Q, (Q > 3 ? Q - 1 : 0));                         \
        else if (gb.Dg == Q - 2 && Q > 4 && ISO2) W_(Q, (Q > 4 && ISO2 ? Q - 2 : 0));         \
        else W_(Q, 0);                                                                        \
    }

void geometric_factors(const Mesh &m, int q1d, double *X, double *J, double *detJ,
                       hipStream_t s) {
    H1PA_CHECK(q1d >= 1 && q1d <= 10, H1PA_EUNSUP, "q1d must be in [1,10]");
    const GeomBasis gb = make_geom_basis(q1d, m.node_order);
    const GeomLaunch l = geom_launch(m.ne, q1d, gb.Dg);
    const bool wp = X != nullptr;
    constexpr bool ISO2 = true;
#define K_(Q, WP, DG)                                                                         \
    hipLaunchKernelGGL((k_geometric_factors<Q, WP, DG>), l.grid, l.block, l.lds, s, m.ne,     \
                       l.nb, gb, m.d_nodes.p, X, J, detJ)
    X_(1) X_(2) X_(3) X_(4) X_(5) X_(6) X_(7) X_(8) X_(9) X_(10)
#undef K_
    H1PA_HIP(hipGetLastError());
}

void pa_setup(const Mesh &m, const Form &f, hipStream_t s) {
    const int q1d = f.q1d;
    H1PA_CHECK(q1d >= 2 && q1d <= 10, H1PA_EUNSUP, "q1d must be in [2,10]");
    const GeomBasis gb = make_geom_basis(q1d, m.node_order);
    const Fourier8 fm = make_fourier(f.desc.coeff_seed);
    const bool wp = f.desc.coeff_kind == H1PA_COEFF_SINCOS ||
                    f.desc.coeff_kind == H1PA_COEFF_FOURIER;
    const GeomLaunch l = geom_launch(m.ne, q1d, gb.Dg);
    constexpr bool ISO2 = false;
#define K_(Q, WP, DG)                                                                         \
    hipLaunchKernelGGL((k_pa_setup<Q, WP, DG>), l.grid, l.block, l.lds, s, m.ne, l.nb,    \
                       gb, m.d_nodes.p, f.desc.coeff_kind, f.desc.coeff_value,          \
                       f.desc.d_coeff, fm, f.pa_diff.p, f.pa_mass.p)
    X_(2) X_(3) X_(4) X_(5) X_(6) X_(7) X_(8) X_(9) X_(10)
#undef X_
#undef W_
#undef K_
    H1PA_HIP(hipGetLastError());
}

void randomize(int64_t n, double *x, uint64_t seed, double lo, double hi, hipStream_t s) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_randomize, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, n, x, seed,
                       lo, hi);
    H1PA_HIP(hipGetLastError());
}

void domain_lf(const Mesh &m, int p, double f, const double *fq, const EOut &out,
               hipStream_t s) {
    const int D = p + 1;
    const GeomBasis gb = make_geom_basis(D, m.node_order);
    double x[16], w[16], G[256];
    LfBasis lb;
    gauss_legendre(D, x, w);
    lagrange_basis(p, D, x, lb.B, G);
    const int per = std::max(geom_lds(D, gb.Dg), D * D * D);
    const int nb = geom_nb(D, per);
    const dim3 grid((unsigned)((m.ne + nb - 1) / nb)), block(nb * D * D);
    const unsigned lds = 8 * (geom_tab_lds(D, gb.Dg) + nb * per);
#define K_(D_, DG)                                                                            \
    hipLaunchKernelGGL((k_domain_lf<D_, DG>), grid, block, lds, s, m.ne, nb, per, gb, lb,     \
                       m.d_nodes.p, f, fq, out)
#define X_(D_)                                                                                \
    if (D == D_) {                                                                            \
        if (gb.Dg == 2) K_(D_, 2);                                                            \
        else if (gb.Dg == D_) K_(D_, D_);                                                     \
        else if (gb.Dg == 3) K_(D_, 3);                                                       \
        else K_(D_, 0);                                                                       \
    }
    X_(2) X_(3) X_(4) X_(5) X_(6) X_(7) X_(8) X_(9)
#undef X_
#undef K_
    H1PA_HIP(hipGetLastError());
}

}  // namespace kern
}  // namespace h1pa
