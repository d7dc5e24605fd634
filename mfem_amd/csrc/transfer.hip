// transfer.hip -- p-refinement transfer between two H1 spaces on one mesh
// (TensorProductPRefinementTransferOperator, fem/transfer.cpp:2619-2990).
//
// MFEM gathers the low-order L-vector into an E-vector, interpolates each
// element's values to the high-order nodes (B = low-order basis at the
// high-order GLL nodes, three 1D contractions), multiplies by the high
// restriction's BooleanMask (1 at the first E-entry of each L-DOF) and sums
// the E-vector into the high L-vector; the transpose runs the same steps
// backwards.  Here the mask is a byte per E-entry, and since exactly one
// masked entry of each high L-DOF is nonzero, the prolongation writes that
// entry's value straight to the L-vector (no high E-vector, no sum: the sum
// of one value and zeros is that value), or adds it there (a cycle's
// correction).  The restriction gathers the masked high values, contracts them
// with B^T into the low E-vector (native layout, interior DOFs straight to the
// result) and the low space's deterministic E->L sum finishes it.
//
// Each contraction is an ascending sum; the prolongation contracts x, y, z as
// MFEM does, the restriction z, y, x, so results differ from MFEM's by rounding.
#include "apply_body.hpp"
#include "internal.hpp"

namespace h1pa {
namespace kern {

namespace {

// emask[E] = 1 when E-index E is the first entry (indices order) of its
// L-DOF's row: ElementRestriction::BooleanMask (fem/restriction.cpp:255-290)
// as one byte per entry.
__global__ void k_first_entry_mask(int64_t nE, const int *__restrict__ gmap,
                                   const int *__restrict__ offsets,
                                   const int *__restrict__ indices, uint8_t *__restrict__ emask) {
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= nE) return;
    const int g = gmap[i];
    const int row = g >= 0 ? g : -1 - g;
    const int first = indices[offsets[row]];
    emask[i] = (first >= 0 ? first : -1 - first) == i ? 1 : 0;
}

// Several elements per work-group, a Dh x Dh thread plane each, the orders
// compiled in: x through LDS, y and z in registers of the thread's own column.
// What bounds them is latency at the sizes of a cycle: 4913 elements, the three
// transfers between orders 1, 2, 3 and 6 on average, prolongation 13.1 -> 6.3 us,
// restriction 11.8 -> 4.8 us against one element of 128 threads per work-group
// with run-time orders.
template <int DL, int DH>
constexpr int tr_nb() { return 256 / (DH * DH); }

template <int DL, int DH>
__global__ void __launch_bounds__(256)
k_prolong(int64_t ne, const double *__restrict__ B, const int *__restrict__ gmap_l,
          const int *__restrict__ gmap_h, const uint8_t *__restrict__ emask_h,
          const double *__restrict__ xl, double *__restrict__ yh, int add) {
    constexpr int NB = tr_nb<DL, DH>(), PL = DH * DH, NL = DL * DL * DL, NH = DH * DH * DH;
    __shared__ double sB[DH * DL];                 // B[qh + Dh dl]
    __shared__ double su[NB][NL], st[NB][DH * DL * DL];  // low values, x contracted
    const int le = threadIdx.x / PL, t = threadIdx.x - le * PL;
    const int a = t % DH, b = t / DH;
    const int64_t e = (int64_t)blockIdx.x * NB + le;
    const bool valid = le < NB && e < ne;
    for (int i = threadIdx.x; i < DH * DL; i += blockDim.x) sB[i] = B[i];
    int g[DH];
    uint8_t m[DH];
    if (valid) {
#pragma unroll
        for (int q = 0; q < DH; ++q) {
            const int64_t E = e * NH + t + PL * q;
            g[q] = gmap_h[E];
            m[q] = emask_h[E];
        }
        for (int i = t; i < NL; i += PL) su[le][i] = xl[gmap_l[e * NL + i]];
    }
    __syncthreads();
    if (valid)
        for (int r = b; r < DL * DL; r += DH) {  // r = dy + Dl dz
            double v = 0.0;
#pragma unroll
            for (int d = 0; d < DL; ++d) v = fma(sB[a + DH * d], su[le][d + DL * r], v);
            st[le][a + DH * r] = v;
        }
    __syncthreads();
    if (!valid) return;
    double v[DH];
#pragma unroll
    for (int q = 0; q < DH; ++q) v[q] = 0.0;
#pragma unroll
    for (int dz = 0; dz < DL; ++dz) {
        double c = 0.0;
#pragma unroll
        for (int dy = 0; dy < DL; ++dy)
            c = fma(sB[b + DH * dy], st[le][a + DH * (dy + DL * dz)], c);
#pragma unroll
        for (int q = 0; q < DH; ++q) v[q] = fma(B[q + DH * dz], c, v[q]);
    }
    if (add) {
        double o[DH];
#pragma unroll
        for (int q = 0; q < DH; ++q) o[q] = m[q] ? yh[g[q]] : 0.0;
#pragma unroll
        for (int q = 0; q < DH; ++q)
            if (m[q]) yh[g[q]] = o[q] + v[q];
    } else {
#pragma unroll
        for (int q = 0; q < DH; ++q)
            if (m[q]) yh[g[q]] = v[q];
    }
}

template <int DL, int DH>
__global__ void __launch_bounds__(256)
k_restrict(int64_t ne, const double *__restrict__ B, const int *__restrict__ gmap_h,
           const uint8_t *__restrict__ emask_h, const double *__restrict__ xh, const EOut out) {
    constexpr int NB = tr_nb<DL, DH>(), PL = DH * DH, NH = DH * DH * DH;
    __shared__ double ss[NB][DH * DH * DL];
    const int le = threadIdx.x / PL, t = threadIdx.x - le * PL;
    const int a = t % DH, b = t / DH;
    const int64_t e = (int64_t)blockIdx.x * NB + le;
    const bool valid = le < NB && e < ne;
    if (valid) {  // z: thread (qx, qy)
        int g[DH];
        uint8_t m[DH];
#pragma unroll
        for (int q = 0; q < DH; ++q) {
            const int64_t E = e * NH + t + PL * q;
            g[q] = gmap_h[E];
            m[q] = emask_h[E];
        }
        double u[DH];
#pragma unroll
        for (int q = 0; q < DH; ++q) u[q] = m[q] ? xh[g[q]] : 0.0;
#pragma unroll
        for (int dz = 0; dz < DL; ++dz) {
            double c = 0.0;
#pragma unroll
            for (int q = 0; q < DH; ++q) c = fma(B[q + DH * dz], u[q], c);
            ss[le][a + DH * (b + DH * dz)] = c;
        }
    }
    __syncthreads();
    const bool acty = valid && b < DL;  // y: thread (qx, dz)
    double u[DH];
    if (acty)
#pragma unroll
        for (int q = 0; q < DH; ++q) u[q] = ss[le][a + DH * (q + DH * b)];
    __syncthreads();
    if (acty)
#pragma unroll
        for (int dy = 0; dy < DL; ++dy) {
            double c = 0.0;
#pragma unroll
            for (int q = 0; q < DH; ++q) c = fma(B[q + DH * dy], u[q], c);
            ss[le][a + DH * (dy + DL * b)] = c;
        }
    __syncthreads();
    if (acty && a < DL) {  // x: thread (dy, dz)
#pragma unroll
        for (int q = 0; q < DH; ++q) u[q] = ss[le][q + DH * (a + DL * b)];
        double yv[DL];
#pragma unroll
        for (int dx = 0; dx < DL; ++dx) {
            double c = 0.0;
#pragma unroll
            for (int q = 0; q < DH; ++q) c = fma(B[q + DH * dx], u[q], c);
            yv[dx] = c;
        }
        store_line<DL, double>(out, e, a, b, yv, 0);
    }
}

}  // namespace

void first_entry_mask(int64_t nE, const int *gmap, const int *offsets, const int *indices,
                      uint8_t *emask, hipStream_t s) {
    if (nE <= 0) return;
    hipLaunchKernelGGL(k_first_entry_mask, dim3((unsigned)((nE + 255) / 256)), dim3(256), 0, s, nE,
                       gmap, offsets, indices, emask);
    H1PA_HIP(hipGetLastError());
}

// (pl + 1, ph + 1) pairs, pl < ph <= 8
#define H1PA_TR_ALL(X)                                                                 \
    X(2, 3) X(2, 4) X(2, 5) X(2, 6) X(2, 7) X(2, 8) X(2, 9) X(3, 4) X(3, 5) X(3, 6)    \
    X(3, 7) X(3, 8) X(3, 9) X(4, 5) X(4, 6) X(4, 7) X(4, 8) X(4, 9) X(5, 6) X(5, 7)    \
    X(5, 8) X(5, 9) X(6, 7) X(6, 8) X(6, 9) X(7, 8) X(7, 9) X(8, 9)

void transfer_prolong(int64_t ne, int pl, int ph, const double *B, const int *gmap_l,
                      const int *gmap_h, const uint8_t *emask_h, const double *xl, double *yh,
                      bool add, hipStream_t s) {
    H1PA_CHECK(pl >= 1 && ph <= 8 && pl < ph, H1PA_EUNSUP, "transfer: orders");
    if (ne <= 0) return;
#define X(L, H)                                                                              \
    if (pl + 1 == L && ph + 1 == H) {                                                        \
        constexpr int NB = tr_nb<L, H>();                                                    \
        hipLaunchKernelGGL((k_prolong<L, H>), dim3((unsigned)((ne + NB - 1) / NB)),          \
                           dim3(NB * H * H), 0, s, ne, B, gmap_l, gmap_h, emask_h, xl, yh,   \
                           add ? 1 : 0);                                                     \
        H1PA_HIP(hipGetLastError());                                                         \
        return;                                                                              \
    }
    H1PA_TR_ALL(X)
#undef X
}

void transfer_restrict_e(int64_t ne, int pl, int ph, const double *B, const int *gmap_h,
                         const uint8_t *emask_h, const double *xh, const EOut &out,
                         hipStream_t s) {
    H1PA_CHECK(pl >= 1 && ph <= 8 && pl < ph, H1PA_EUNSUP, "transfer: orders");
    if (ne <= 0) return;
#define X(L, H)                                                                              \
    if (pl + 1 == L && ph + 1 == H) {                                                        \
        constexpr int NB = tr_nb<L, H>();                                                    \
        hipLaunchKernelGGL((k_restrict<L, H>), dim3((unsigned)((ne + NB - 1) / NB)),         \
                           dim3(NB * H * H), 0, s, ne, B, gmap_h, emask_h, xh, out);         \
        H1PA_HIP(hipGetLastError());                                                         \
        return;                                                                              \
    }
    H1PA_TR_ALL(X)
#undef X
}

}  // namespace kern
}  // namespace h1pa
