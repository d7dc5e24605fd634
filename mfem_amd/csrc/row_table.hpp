// row_table.hpp -- the E -> L reduction of the fused operators, from a table of
// fixed-width rows: shared by the scatter (restriction.hip) and the solver
// kernels (pcg.hip, batch.hip).
//
// The native E-vector's transpose table in CSR form costs a row four dependent
// loads (row -> offsets -> indices -> values) and 8 bytes of offsets.  A
// conforming hexahedral mesh gives almost every vertex at most 8 entries, every
// edge DOF 4 and every face DOF 2, so the indices are stored padded to those
// widths in the order in which the rows are summed: a row's indices are one or
// two 16-byte loads (8 bytes for a face) at an address known from the thread,
// and a row costs two dependent loads.  A row with more entries than its width
// (vertices and edges of unstructured meshes) is marked and read from the CSR
// table, which is kept only for meshes that have one.  Sums run over a row's
// entries in MFEM's order, as before.
//
// E -> L of p = 4, 79^3 elements: 199 -> 181 us with the table, 174 with the
// E-vector's interior gaps closed, 165 with four rows a thread (scatter_rows);
// p = 6, 48^3: 93 -> 76; p = 3, 16^3: 5.2 -> 3.9.  At the large sizes it moves
// 0.73 GB of table, E-vector and result at 4.4 TB/s; what is left is E-lines
// fetched again by the rows of a face that a far element numbered.
#pragma once

#include "internal.hpp"

namespace h1pa {
namespace kern {

constexpr int kRowOver = -2147483647 - 1;  // first entry of a row left to the CSR table
typedef int rt2i __attribute__((ext_vector_type(2)));
typedef int rt4i __attribute__((ext_vector_type(4)));

// L-DOF of row position t.
__device__ __forceinline__ int row_dof(const RowTab &tb, int t) {
    return t < tb.ebeg ? tb.perm[t] : t;
}

// Sum of a row that does not fit the table (rare).
template <typename T>
__device__ __forceinline__ T row_overflow(const RowTab &tb, int t, const T *__restrict__ xe) {
    const int i = row_dof(tb, t);
    T s = T(0);
    for (int j = tb.offsets[i]; j < tb.offsets[i + 1]; ++j) s += xe[tb.indices[j]];
    return s;
}

template <int W, typename T>
__device__ __forceinline__ T row_add(const int (&ix)[W], const T (&v)[W]) {
    T s = T(0);
#pragma unroll
    for (int k = 0; k < W; ++k) s = ix[k] >= 0 ? s + v[k] : s;
    return s;
}

// The W indices of the row at p (aligned to its width).
template <int W, bool NT>
__device__ __forceinline__ void row_load(const int *__restrict__ p, int (&ix)[W]) {
    if constexpr (W == 2) {
        const rt2i *q = reinterpret_cast<const rt2i *>(p);
        const rt2i a = NT ? __builtin_nontemporal_load(q) : *q;
        ix[0] = a.x;
        ix[1] = a.y;
    } else {
#pragma unroll
        for (int k = 0; k < W; k += 4) {
            const rt4i *q = reinterpret_cast<const rt4i *>(p + k);
            const rt4i a = NT ? __builtin_nontemporal_load(q) : *q;
            ix[k] = a.x;
            ix[k + 1] = a.y;
            ix[k + 2] = a.z;
            ix[k + 3] = a.w;
        }
    }
}

// R rows of one width: every index load, then every value load, then the sums.
// p0: table entry of the row at position t0.
template <int R, int W, bool NT, typename T>
__device__ __forceinline__ void rows_of_width(const RowTab &tb, const int *__restrict__ p0,
                                              int t0, const int *t,
                                              const T *__restrict__ xe, T *s) {
    int ix[R][W];
#pragma unroll
    for (int r = 0; r < R; ++r) row_load<W, NT>(p0 + W * (int64_t)(t[r] - t0), ix[r]);
    T v[R][W];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int k = 0; k < W; ++k) v[r][k] = xe[ix[r][k] >= 0 ? ix[r][k] : 0];
#pragma unroll
    for (int r = 0; r < R; ++r) s[r] = row_add<W>(ix[r], v[r]);
    if (tb.over)
#pragma unroll
        for (int r = 0; r < R; ++r)
            if (ix[r][0] == kRowOver) s[r] = row_overflow(tb, t[r], xe);
}

// A row of any kind, for the few waves that hold several kinds: eight entries, of
// which a row narrower than that leaves the rest out.  Interior-DOF rows
// (position bbeg on) have one entry, in the same order after the surface ones.
template <bool NT, typename T>
__device__ __forceinline__ T row_any(const RowTab &tb, int t, const T *__restrict__ xe) {
    const bool in = t >= tb.bbeg;
    if (!__ballot(!in)) return T(0) + xe[tb.ebub + (t - tb.bbeg)];
    const int q = in ? tb.bbeg - 1 : t;
    const int w = q < tb.ebeg ? 8 : q < tb.fbeg ? 4 : 2;
    const int nv = min(q, tb.ebeg), ne = min(max(q - tb.ebeg, 0), tb.fbeg - tb.ebeg),
              nf = max(q - tb.fbeg, 0);
    const int *const p = tb.tab + (8 * (int64_t)nv + 4 * (int64_t)ne + 2 * (int64_t)nf);
    int ix[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const int *const pk = p + (k < w ? k : w - 1);
        ix[k] = NT ? __builtin_nontemporal_load(pk) : *pk;
    }
#pragma unroll
    for (int k = 0; k < 8; ++k)
        if (in || k >= w) ix[k] = -1;
    if (in) ix[0] = (int)(tb.ebub + (t - tb.bbeg));
    T v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = xe[ix[k] >= 0 ? ix[k] : 0];
    T s = row_add<8>(ix, v);
    if (tb.over && ix[0] == kRowOver) s = row_overflow(tb, t, xe);
    return s;
}

// s[r] = sum of the E-entries of the row at position t[r], t[0] <= ... <= t[R-1]
// (rows of any kind; a wave whose rows are all vertices, edges or faces --
// nearly every wave -- takes the loop of that width).
// NT: the table is streamed past the caches.
template <int R, bool NT = false, typename T>
__device__ __forceinline__ void rows_sum(const RowTab &tb, const int (&t)[R],
                                         const T *__restrict__ xe, T (&s)[R]) {
    const int lo = t[0], hi = t[R - 1];
    const int *const ev = tb.tab, *const ee = ev + 8 * (int64_t)tb.ebeg,
                     *const ef = ee + 4 * (int64_t)(tb.fbeg - tb.ebeg);
    if (!__ballot(!(lo >= tb.fbeg && hi < tb.bbeg))) {
        rows_of_width<R, 2, NT>(tb, ef, tb.fbeg, t, xe, s);
    } else if (!__ballot(!(lo >= tb.ebeg && hi < tb.fbeg))) {
        rows_of_width<R, 4, NT>(tb, ee, tb.ebeg, t, xe, s);
    } else if (!__ballot(!(hi < tb.ebeg))) {
        constexpr int P = R > 2 ? 2 : R;  // two rows of eight at a time
#pragma unroll
        for (int r = 0; r < R; r += P) {
            rows_of_width<P, 8, NT>(tb, ev, 0, t + r, xe, s + r);
            __builtin_amdgcn_sched_barrier(0);
        }
    } else {
#pragma unroll
        for (int r = 0; r < R; ++r) s[r] = row_any<NT>(tb, t[r], xe);
    }
}

}  // namespace kern
}  // namespace h1pa
