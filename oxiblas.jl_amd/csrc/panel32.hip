// FP32 instances of the panel leaf (the working precision of the
// mixed-precision LU, as the reference's mixed_solve factors in Float32:
// src/lapack/extended_lapack.jl:183,195-198).  FP32 rows take half the
// registers, so up to four rows per thread stay in registers.
#include "panel_kernel.hpp"

int oxi_launch_lu_leaf32(oxi_handle_t h, hipStream_t s, const LeafArgs& a, int kind) {
    if (a.P == 1 && kind == 0) return launch_leaf(h, s, a, lu_leaf_kernel<float, 1, 1>);
    if (kind == 0) return launch_leaf(h, s, a, lu_leaf_kernel<float, 1, 64>);
    if (a.P == 1 && kind == 1) return launch_leaf(h, s, a, lu_leaf_kernel<float, 2, 1>);
    if (kind == 1) return launch_leaf(h, s, a, lu_leaf_kernel<float, 2, 64>);
    return launch_leaf(h, s, a, lu_leaf_kernel<float, 4, OXI_LEAF_MAX_P>);
}
