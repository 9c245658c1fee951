// Panel leaf of the blocked LU: column-by-column elimination of an m x w
// block (w <= 32) held in registers across P co-resident workgroups.
//
// Restates the leaf of _lu_panel! (src/lapack/factorizations.jl:116-140) with
// the pivot choice of _lu_pivot (:89-107): the pivot is the first row of
// largest |value| (strict '>' scan semantics: NaN never beats a number except
// in the diagonal position), rows are swapped across the whole leaf, the
// column is divided by the pivot (a division, as the reference) and the
// leaf's remaining columns get fma(-l, u, a); a zero pivot records info (the
// first one, 1-based) and skips the column.
//
// Operands live in the transposed working layout W = A^T (see getrf.hip):
// the w leaf values of one row of A are contiguous.  Each workgroup owns a
// contiguous block of rows (one or two per thread, in registers).  Per column
// every workgroup publishes its candidate (key, position and the whole row)
// as a record of tagged words (panel_kernel.hpp) and reads all the others;
// every workgroup picks the same winner.  The wait is bounded: on timeout a
// flag is raised and every wave leaves, so the grid always drains.  With
// P == 1 the exchange stays in LDS.
//
// Rows never move between threads: an interchange changes the positions that
// the threads hold, and every row, multipliers included, is stored once at
// its final position, which gives the same rows as swapping whole rows at
// each step.  A second, small kernel applies the leaf's interchanges to the
// other columns of the enclosing panel (the sibling swaps of the getrf2
// recursion, done once per leaf).
#include "panel_kernel.hpp"

int oxi_launch_lu_leaf(oxi_handle_t h, hipStream_t s, const LeafArgs& a, int kind) {
    if (a.P == 1 && kind == 0) OXI_TRY(launch_leaf(h, s, a, lu_leaf_kernel<double, 256, 1, 1>));
    else if (a.P == 1 && kind == 1) OXI_TRY(launch_leaf(h, s, a, lu_leaf_kernel<double, 256, 2, 1>));
    else if (a.P <= 64 && kind == 0) OXI_TRY(launch_leaf(h, s, a, lu_leaf_kernel<double, 256, 1, 64>));
    else if (a.P <= 64 && kind == 1) OXI_TRY(launch_leaf(h, s, a, lu_leaf_kernel<double, 256, 2, 64>));
    else OXI_TRY(launch_leaf(h, s, a, lu_leaf_kernel<double, 256, 2, OXI_LEAF_MAX_P>));
    // the leaf's interchanges on the rest of its panel (its own columns are final)
    const unsigned nblk = unsigned(cdiv(a.c0 - a.xlo, 64) + cdiv(a.xhi - a.c0 - a.w, 64));
    if (nblk > 0) {
        hipLaunchKernelGGL(leaf_swaps_kernel<double>, dim3(nblk), dim3(128), 0, s, (double*)a.Wm, a.ldw, a.c0, a.w,
                           (const i64*)a.ipiv, (const int*)a.flags, a.xlo, a.xhi);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return oxi_set_error(h, OXI_ERR_HIP, "leaf_swaps launch: %s", hipGetErrorString(e));
    }
    return OXI_OK;
}
