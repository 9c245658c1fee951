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
// each step.  At its end the leaf applies its interchanges to the other
// columns of the enclosing panel (the sibling swaps of the getrf2 recursion,
// done once per leaf).
#include "panel_kernel.hpp"

int oxi_launch_lu_leaf(oxi_handle_t h, hipStream_t s, const LeafArgs& a, int kind) {
    if (a.P == 1 && kind == 0) return launch_leaf(h, s, a, lu_leaf_kernel<double, 1, 1>);
    if (kind == 0) return launch_leaf(h, s, a, lu_leaf_kernel<double, 1, 64>);
    if (a.P == 1) return launch_leaf(h, s, a, lu_leaf_kernel<double, 2, 1>);
    if (a.P <= 64) return launch_leaf(h, s, a, lu_leaf_kernel<double, 2, 64>);
    return launch_leaf(h, s, a, lu_leaf_kernel<double, 2, OXI_LEAF_MAX_P>);
}
