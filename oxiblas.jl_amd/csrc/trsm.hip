// Triangular solves (trsm!, src/blas/level3.jl:309-544) on gfx950: the
// reference's recursive halving (_trsm_blocks_left! / _trsm_blocks_right!,
// level3.jl:338-376) with FP64 MFMA GEMM updates, down to blocks of 256 rows in
// one launch (trsm_block_kernel), or to leaves of at most 64 rows solved in
// registers, one wave per right-hand side.
#include "tri_inv.hpp"

#include <algorithm>

namespace {
__device__ __forceinline__ double fma_t(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ __forceinline__ float fma_t(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

constexpr int TRL = 64;
constexpr int SB = 256;   // rows of a block of the blocked solves
// A 64-row diagonal block M is solved through its inverse V only while the row
// sums of |V| |M| stay below this (and are numbers).  Up to there one refinement leaves
// a backward error no larger than substitution's (emulated for random, row- and
// column-scaled triangles and the blocks of LU factors, sums of 1 to 10^10: at
// most 3.2e-16 componentwise, 4.8e-16 by substitution, 6e-15 without the
// refinement); far beyond, 64 eps times the sum passes 1 and it need not contract.
constexpr double MAX_COND = 0x1p40;

// Right side: X (rows x n) <- X * op(T)^-1, n <= 64.  Element order matches
// the reference's right leaf (src/blas/level3.jl:319-333):
// op(T) upper: x_c = (b_c - sum_{p<c} x_p U[p][c]) / U[c][c], c ascending;
// op(T) lower: x_c = (b_c - sum_{p>c} x_p L[p][c]) / L[c][c], c descending.
// One wave per row, lane q = column q: lane q keeps column q of op(T) in
// registers, and the solve is a column sweep (step c: lane c finishes x_c,
// the wave reads it with readlane, every later lane applies one FMA), so each
// element sees exactly the operations above, in that order.  A wave takes
// `rpw` consecutive rows in turn.
__device__ __forceinline__ double rlane(double v, int l) {
    const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = __builtin_amdgcn_readlane(unsigned(u), l);
    const unsigned hi = __builtin_amdgcn_readlane(unsigned(u >> 32), l);
    return __builtin_bit_cast(double, (static_cast<unsigned long long>(hi) << 32) | lo);
}
__device__ __forceinline__ float rlane(float v, int l) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(unsigned, v), l));
}

template <typename TY, bool LOWER, bool UNIT, bool TRANS, int NW>
__global__ __launch_bounds__(256) void trsm_right_leaf(TY* __restrict__ X, i64 ldx, i64 rows, int rpw,
                                                       const TY* __restrict__ T, i64 ldt) {
    const int lane = threadIdx.x & 63;
    const i64 wave = i64(blockIdx.x) * (blockDim.x / 64) + (threadIdx.x >> 6);
    const i64 r0 = wave * rpw;
    if (r0 >= rows) return;
    const int q = lane < NW ? lane : NW - 1;          // lanes beyond the width mirror the last column
    TY u[NW];                                         // u[c] = op(T)[c][q]
#pragma unroll
    for (int c = 0; c < NW; ++c) u[c] = TRANS ? T[q + i64(c) * ldt] : T[c + i64(q) * ldt];
    const i64 r1 = min(rows, r0 + rpw);
    for (i64 r = r0; r < r1; ++r) {
        TY x = X[r + i64(q) * ldx];
        if (!LOWER) {
#pragma unroll
            for (int c = 0; c < NW; ++c) {
                if (!UNIT && lane == c) x = x / u[c];
                const TY xc = rlane(x, c);
                if (lane > c) x = fma_t(-xc, u[c], x);
            }
        } else {
#pragma unroll
            for (int c = NW - 1; c >= 0; --c) {
                if (!UNIT && lane == c) x = x / u[c];
                const TY xc = rlane(x, c);
                if (lane < c) x = fma_t(-xc, u[c], x);
            }
        }
        if (lane < NW) X[r + i64(q) * ldx] = x;
    }
}

// Any width n <= 64: the width-64 layout with the steps past n skipped.
template <typename TY, bool LOWER, bool UNIT, bool TRANS>
__global__ __launch_bounds__(256) void trsm_right_leaf_any(TY* __restrict__ X, i64 ldx, i64 rows, int rpw, int n,
                                                           const TY* __restrict__ T, i64 ldt) {
    const int lane = threadIdx.x & 63;
    const i64 wave = i64(blockIdx.x) * (blockDim.x / 64) + (threadIdx.x >> 6);
    const i64 r0 = wave * rpw;
    if (r0 >= rows) return;
    const int q = lane < n ? lane : n - 1;
    TY u[TRL];
#pragma unroll
    for (int c = 0; c < TRL; ++c) u[c] = c < n ? (TRANS ? T[q + i64(c) * ldt] : T[c + i64(q) * ldt]) : TY(0);
    const i64 r1 = min(rows, r0 + rpw);
    for (i64 r = r0; r < r1; ++r) {
        TY x = X[r + i64(q) * ldx];
        if (!LOWER) {
#pragma unroll
            for (int c = 0; c < TRL; ++c) {
                if (c < n) {
                    if (!UNIT && lane == c) x = x / u[c];
                    const TY xc = rlane(x, c);
                    if (lane > c) x = fma_t(-xc, u[c], x);
                }
            }
        } else {
#pragma unroll
            for (int c = TRL - 1; c >= 0; --c) {
                if (c < n) {
                    if (!UNIT && lane == c) x = x / u[c];
                    const TY xc = rlane(x, c);
                    if (lane < c) x = fma_t(-xc, u[c], x);
                }
            }
        }
        if (lane < n) X[r + i64(q) * ldx] = x;
    }
}

template <typename TY, bool LOWER, bool UNIT, bool TRANS>
void launch_right_leaf_w(hipStream_t s, i64 rows, int n, const TY* T, i64 ldt, TY* X, i64 ldx) {
    // about 1024 waves in flight; consecutive rows per wave share cache lines
    const int rpw = int(std::max<i64>(1, cdiv(rows, 1024)));
    const i64 waves = cdiv(rows, rpw);
    const dim3 grid(unsigned(cdiv(waves, 4))), block(256);
    if (n == 64) hipLaunchKernelGGL((trsm_right_leaf<TY, LOWER, UNIT, TRANS, 64>), grid, block, 0, s, X, ldx, rows, rpw, T, ldt);
    else if (n == 32) hipLaunchKernelGGL((trsm_right_leaf<TY, LOWER, UNIT, TRANS, 32>), grid, block, 0, s, X, ldx, rows, rpw, T, ldt);
    else if (n == 16) hipLaunchKernelGGL((trsm_right_leaf<TY, LOWER, UNIT, TRANS, 16>), grid, block, 0, s, X, ldx, rows, rpw, T, ldt);
    else if (n == 8) hipLaunchKernelGGL((trsm_right_leaf<TY, LOWER, UNIT, TRANS, 8>), grid, block, 0, s, X, ldx, rows, rpw, T, ldt);
    else hipLaunchKernelGGL((trsm_right_leaf_any<TY, LOWER, UNIT, TRANS>), grid, block, 0, s, X, ldx, rows, rpw, n, T, ldt);
}

template <typename TY, bool LOWER>
void launch_right_leaf(hipStream_t s, int unit, int trans, i64 rows, int n, const TY* T, i64 ldt, TY* X, i64 ldx) {
    if (unit) {
        if (trans) launch_right_leaf_w<TY, LOWER, true, true>(s, rows, n, T, ldt, X, ldx);
        else launch_right_leaf_w<TY, LOWER, true, false>(s, rows, n, T, ldt, X, ldx);
    } else {
        if (trans) launch_right_leaf_w<TY, LOWER, false, true>(s, rows, n, T, ldt, X, ldx);
        else launch_right_leaf_w<TY, LOWER, false, false>(s, rows, n, T, ldt, X, ldx);
    }
}

// Inverses of the 64 x 64 diagonal blocks of a triangle M of n rows, M(i, k) =
// T(i, k) (TRANS: T(k, i)), UPPER or lower: block b's goes to inv + 4096 b,
// column-major (ld 64, zeros in the other triangle, the identity beyond n);
// with strip > 0, to its place in a column-major strip of ld `ldv` whose rows
// z*strip .. (z+1)*strip - 1 hold the strip x strip block z (inv + 64 b +
// ((64 b) % strip) * ldv); CLEAN: to inv + 8192 b, and the block itself,
// completed in the same way, 4096 elements behind it, where an inverse that
// trsm_block_kernel must not use is NaN throughout.  The block in
// LDS (UPPER: both indices reversed, so that it is lower triangular), inverted
// on the matrix cores (tri::invert); bound by the latency of its loads and
// barriers: 8 us, against 27 for a column a lane swept over 64 steps.
template <bool UNIT, bool TRANS, bool UPPER, bool CLEAN>
__global__ __launch_bounds__(256) void trsm_inv64_kernel(const double* __restrict__ T, i64 ldt, i64 n,
                                                         double* __restrict__ inv, i64 ldv = 64, int strip = 0) {
    constexpr int L = tri::LD<64>;
    __shared__ double D[tri::SPACE<64>];   // D(i, k) = M(i, k), or M(63 - i, 63 - k)
    __shared__ double part[CLEAN ? 256 : 1], sums[CLEAN ? 64 : 1];   // of each row of |D|
    __shared__ int avoid;                                            // the inverse as it is
    const int t = threadIdx.x;
    const i64 o = i64(blockIdx.x) * 64;
    double* out = strip > 0 ? inv + o + (o % strip) * ldv : inv + 64 * (CLEAN ? 2 : 1) * o;
    auto load = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            const int e = t + u * 256;
            const int x = e % 64, y = e / 64;        // T(o + x, o + y), the thread index along its columns
            const int r = TRANS ? y : x, c = TRANS ? x : y, i = UPPER ? 63 - r : r, k = UPPER ? 63 - c : c;
            const double v = T[min(o + x, n - 1) + min(o + y, n - 1) * ldt];
            const bool in = o + x < n && o + y < n;
            D[k * L + i] = i == k ? (UNIT || !in ? 1.0 : v) : in && i > k ? v : 0.0;
        }
    };
    load();
    if (t == 0) avoid = 0;
    __syncthreads();
    // this thread's elements of the result: row r, columns t / 64 + 4 u
    const int r = t % 64, i = UPPER ? 63 - r : r;
    auto column = [&](int u) __attribute__((always_inline)) { return t / 64 + 4 * u; };
    auto lower = [&](int u) __attribute__((always_inline)) {
        const int k = UPPER ? 63 - column(u) : column(u);
        return i >= k ? D[k * L + i] : 0.0;
    };
    if (CLEAN) {
        double sum = 0.0;
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            const double v = lower(u);
            out[4096 + r + column(u) * 64] = v;
            sum += __builtin_fabs(v);
        }
        part[t / 64 * 64 + i] = sum;
        __syncthreads();
        if (t < 64) sums[t] = (part[t] + part[t + 64]) + (part[t + 128] + part[t + 192]);
    }
    tri::invert<double, 64, 4, UNIT>(D, t);
    double v[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) v[u] = lower(u);
    if (CLEAN) {
        // row i of |D^-1| |D| e, a quarter of its columns
        double c = 0.0;
#pragma unroll
        for (int u = 0; u < 16; ++u) c += __builtin_fabs(v[u]) * sums[UPPER ? 63 - column(u) : column(u)];
        if (!(c < MAX_COND)) avoid = 1;
        __syncthreads();
        if (avoid)
#pragma unroll
            for (int u = 0; u < 16; ++u) v[u] = __builtin_nan("");
    } else {
        bool finite = true;
#pragma unroll
        for (int u = 0; u < 16; ++u) finite = finite && __builtin_isfinite(v[u]);
        if (!finite) avoid = 1;
        __syncthreads();
        if (__builtin_expect(avoid, 0)) {
            load();
            __syncthreads();
            tri::invert_by_substitution<double, 64, UNIT>(D, t, out, ldv);
#pragma unroll
            for (int u = 0; u < 16; ++u) v[u] = lower(u);
            __syncthreads();   // out has been read
        }
    }
#pragma unroll
    for (int u = 0; u < 16; ++u) out[r + column(u) * ldv] = v[u];
}

// One block of up to SB = 256 rows of a triangular solve M x = b in place, M
// lower (BWD: upper) triangular, M(i, k) = T(i, k) (TM: T(k, i)); LEFT: right-
// hand sides are columns of B, element (i, j) at B[i + j * ldb], else rows, at
// B[j + i * ldb] (X op(T) = B is op(T)^T X^T = B^T).  V: for each of the block's
// 64-row diagonal blocks, M_pp^-1 and M_pp (trsm_inv64_kernel).  FULL: rows is
// SB (no masks; a load behind one is waited for at once).
//
// A workgroup owns 16 right-hand sides and goes through the 64-row blocks in
// solve order: r = b_p - sum M_pq x_q over the blocks before, x = M_pp^-1 r, and
// one refinement x += M_pp^-1 (r - M_pp x), so that x is no further off than by
// substitution; a wave has 16 of the 64 rows, x in LDS, the operands of M and
// V straight from memory, the next product's loaded while one runs.  The
// products take their k in solve order (the diagonal's large term last).
// Where an element of x is not finite, the right-hand sides are solved again
// with the 64-row blocks by substitution: the products multiply the zeros of
// the other triangle too, so an infinity of r reaches the rows before it, an
// inverse may overflow where x does not, and an inverse not to be used is NaN
// (trsm_inv64_kernel).
// 256 rows cost one launch.  Bound by the
// 18 products a wave has one after the other (16 matrix instructions of 64
// cycles each, 9 us) and the 16 turns through LDS and a barrier: 22 us.
template <bool LEFT, bool TM, bool BWD, bool FULL>
__global__ __launch_bounds__(256, 1) void trsm_block_kernel(const double* __restrict__ T, i64 ldt,
                                                            const double* __restrict__ V, double* __restrict__ B,
                                                            i64 ldb, int nrows, i64 nrhs) {
    typedef tri::Mfma<double> Mf;
    constexpr int C = 16, LX = C + 1;
    __shared__ double xs[SB * LX], rs[64 * LX];
    __shared__ int again;                          // an element of x is not finite
    const int t = threadIdx.x, lane = t & 63, w = t >> 6, lk = lane >> 4, li = lane & 15;
    const int rows = FULL ? SB : nrows, nsb = (rows + 63) / 64;
    const i64 j0 = i64(blockIdx.x) * C;
    const int nc = int(min(i64(C), nrhs - j0));
    // the k of a product, four at a time, in solve order
    auto in_order = [](int e) __attribute__((always_inline)) { return BWD ? 15 - e : e; };
    // this lane's operands of M_pq, and of M_pp^-1 (at 0) or M_pp (at 4096) of block p
    auto load_m = [&](int p, int q, double (&a)[16]) __attribute__((always_inline)) {
        const int i = p * 64 + w * 16 + li, ic = FULL ? i : min(i, rows - 1);
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int k = q * 64 + 4 * in_order(e) + lk, kc = FULL ? k : min(k, rows - 1);
            const double m = TM ? T[kc + i64(ic) * ldt] : T[ic + i64(kc) * ldt];
            a[e] = FULL || (i < rows && k < rows) ? m : 0.0;
        }
    };
    auto load_v = [&](int p, int off, double (&a)[16]) __attribute__((always_inline)) {
        const double* vp = V + p * 8192 + off + w * 16 + li + 64 * lk;
#pragma unroll
        for (int e = 0; e < 16; ++e) a[e] = vp[256 * in_order(e)];
    };
    auto product = [&](const double (&a)[16], const double* x, Mf::acc c) __attribute__((always_inline)) {
        double y[16];
#pragma unroll
        for (int e = 0; e < 16; ++e) y[e] = x[(4 * in_order(e) + lk) * LX + li];
        __builtin_amdgcn_sched_barrier(0);   // all of x on its way before the first product
#pragma unroll
        for (int e = 0; e < 16; ++e) c = Mf::mul(a[e], y[e], c);
        return c;
    };
    auto copy = [&](const double (&from)[16], double (&to)[16]) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < 16; ++e) to[e] = from[e];
    };
    // barrier of the LDS traffic alone: loads stay in flight
    auto barrier_lds = [&]() __attribute__((always_inline)) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    };
    const int j = LEFT ? 0 : t % C, i0 = LEFT ? t : t / C;   // this thread's elements of B: rows i0 + 16 u, or column u
    auto element = [&](int u) __attribute__((always_inline)) {
        return LEFT ? min(i0, rows - 1) + (j0 + min(u, nc - 1)) * ldb : j0 + min(j, nc - 1) + min(i0 + 16 * u, rows - 1) * ldb;
    };
    double b[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) b[u] = B[element(u)];
    double cur[16], nxt[16];
    load_v(BWD ? nsb - 1 : 0, 0, cur);
    auto b_to_x = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            const int i = LEFT ? i0 : i0 + 16 * u;
            xs[i * LX + (LEFT ? u : j)] = FULL || i < rows ? b[u] : 0.0;
        }
    };
    b_to_x();
    if (t == 0) again = 0;
    __syncthreads();
    const int own = (w * 16 + lk) * LX + li;                 // this lane's element of a block's rows, + 4 LX r
    const Mf::acc zero = {0, 0, 0, 0};
    // Rolled (unrolled, the code of the 18 products took longer to fetch than
    // to run: 25 us), the operands of the next product in flight
#pragma unroll 1
    for (int s = 0; s < nsb; ++s) {
        const int p = BWD ? nsb - 1 - s : s;
        double* xp = xs + p * 64 * LX;
        Mf::acc r = zero;
#pragma unroll 1
        for (int u = 0; u < s; ++u) {
            const int q = BWD ? nsb - 1 - u : u;
            if (u + 1 < s) load_m(p, BWD ? q - 1 : q + 1, nxt);
            else load_v(p, 0, nxt);
            r = product(cur, xs + q * 64 * LX, r);
            copy(nxt, cur);
        }
        load_v(p, 4096, nxt);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            r[k] = xp[own + 4 * LX * k] - r[k];
            rs[own + 4 * LX * k] = r[k];
        }
        barrier_lds();
        Mf::acc x = product(cur, rs, zero);
#pragma unroll
        for (int k = 0; k < 4; ++k) xp[own + 4 * LX * k] = x[k];
        barrier_lds();
        const Mf::acc m = product(nxt, xp, zero);
        if (s + 1 < nsb) load_m(BWD ? p - 1 : p + 1, BWD ? nsb - 1 : 0, nxt);
#pragma unroll
        for (int k = 0; k < 4; ++k) rs[own + 4 * LX * k] = r[k] - m[k];
        barrier_lds();
        const Mf::acc d = product(cur, rs, zero);
#pragma unroll
        for (int k = 0; k < 4; ++k) xp[own + 4 * LX * k] = x[k] + d[k];
        copy(nxt, cur);
        barrier_lds();
    }
    bool finite = true;
    double xo[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) {
        const int i = LEFT ? i0 : i0 + 16 * u;
        xo[u] = xs[i * LX + (LEFT ? u : j)];
        finite = finite && (__builtin_isfinite(xo[u]) || !(FULL || i < rows));
    }
    if (!finite) again = 1;
    __syncthreads();
    if (__builtin_expect(again, 0)) {
#pragma unroll
        for (int u = 0; u < 16; ++u) b[u] = B[element(u)];
        b_to_x();
        __syncthreads();
#pragma unroll 1
        for (int s = 0; s < nsb; ++s) {
            const int p = BWD ? nsb - 1 - s : s;
            double* xp = xs + p * 64 * LX;
            Mf::acc r = zero;
#pragma unroll 1
            for (int u = 0; u < s; ++u) {
                const int q = BWD ? nsb - 1 - u : u;
                load_m(p, q, cur);
                r = product(cur, xs + q * 64 * LX, r);
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) xp[own + 4 * LX * k] -= r[k];
            __syncthreads();
            // a lane per row, a wave for four right-hand sides
            const double* mp = V + p * 8192 + 4096 + lane;
            double y[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) y[c] = xp[lane * LX + 4 * w + c];
#pragma unroll 1
            for (int g = 0; g < 64; g += 8) {
                double m[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) m[u] = mp[64 * (BWD ? 63 - g - u : g + u)];
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const int k = BWD ? 63 - g - u : g + u;
                    double yk = rlane(y[3], k);              // lane c: of right-hand side c
#pragma unroll
                    for (int c = 0; c < 3; ++c) yk = lane == c ? rlane(y[c], k) : yk;
                    yk /= rlane(m[u], k);
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        const double v = rlane(yk, c);
                        y[c] = lane == k ? v : (BWD ? lane < k : lane > k) ? fma_t(-m[u], v, y[c]) : y[c];
                    }
                }
            }
#pragma unroll
            for (int c = 0; c < 4; ++c) xp[lane * LX + 4 * w + c] = y[c];
            __syncthreads();
        }
#pragma unroll
        for (int u = 0; u < 16; ++u) xo[u] = xs[(LEFT ? i0 : i0 + 16 * u) * LX + (LEFT ? u : j)];
    }
#pragma unroll
    for (int u = 0; u < 16; ++u) {
        const int i = LEFT ? i0 : i0 + 16 * u, c = LEFT ? u : j;
        if ((FULL || i < rows) && c < nc) B[element(u)] = xo[u];
    }
}

// Left side: X (n x nrhs) <- op(T)^-1 X, one wave per right-hand side, lane =
// row.  LOWER refers to op(T).  Per element: s = b_i; s = fma(-T[i][p], x_p, s)
// in order of p; s / T[i][i] when not unit (src/blas/level3.jl:309-318,
// src/blas/triangular_microkernels.jl:31-59).
template <typename TY, bool LOWER, bool UNIT>
__global__ __launch_bounds__(256) void trsm_left_leaf(TY* __restrict__ X, i64 ldx, i64 nrhs, int n,
                                                      const TY* __restrict__ T, i64 ldt, int trans) {
    __shared__ TY S[TRL * (TRL + 1)];  // S[p*(TRL+1) + i] = op(T)[i][p]
    for (int e = threadIdx.x; e < TRL * TRL; e += blockDim.x) {
        const int pp = e / TRL, i = e % TRL;
        TY val = TY(0);
        if (pp < n && i < n) val = trans ? T[pp + i64(i) * ldt] : T[i + i64(pp) * ldt];
        S[pp * (TRL + 1) + i] = val;
    }
    __syncthreads();
    const int lane = threadIdx.x & 63;
    const i64 col = i64(blockIdx.x) * (blockDim.x / 64) + (threadIdx.x >> 6);
    if (col >= nrhs) return;
    TY* xc = X + col * ldx;
    TY x = lane < n ? xc[lane] : TY(0);
    if (LOWER) {
        for (int pp = 0; pp < n; ++pp) {
            if (!UNIT && lane == pp) x = x / S[pp * (TRL + 1) + pp];
            const TY xp = __shfl(x, pp);
            if (lane > pp) x = fma_t(-S[pp * (TRL + 1) + lane], xp, x);
        }
    } else {
        for (int pp = n - 1; pp >= 0; --pp) {
            if (!UNIT && lane == pp) x = x / S[pp * (TRL + 1) + pp];
            const TY xp = __shfl(x, pp);
            if (lane < pp) x = fma_t(-S[pp * (TRL + 1) + lane], xp, x);
        }
    }
    if (lane < n) xc[lane] = x;
}

// Diagonal check for the non-unit solves: first zero on the diagonal of T (1-based) or 0.
__global__ void diag_zero_kernel(const double* __restrict__ T, i64 ldt, i64 n, i64* __restrict__ out) {
    for (i64 i = i64(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += i64(gridDim.x) * blockDim.x)
        if (T[i + i * ldt] == 0.0) atomicMin((unsigned long long*)out, (unsigned long long)(i + 1));
}
__global__ void set_i64_kernel(i64* p, i64 v) { *p = v; }


int launch_check(oxi_handle_t h, const char* what) {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return oxi_set_error(h, OXI_ERR_HIP, "%s launch: %s", what, hipGetErrorString(e));
    return OXI_OK;
}
}  // namespace

template <typename TY>
int gemm_t(oxi_handle_t h, hipStream_t s, int ta, int tb, i64 m, i64 n, i64 k, TY alpha, const TY* A, i64 lda,
           const TY* B, i64 ldb, TY beta, TY* C, i64 ldc);
template <>
int gemm_t<double>(oxi_handle_t h, hipStream_t s, int ta, int tb, i64 m, i64 n, i64 k, double alpha, const double* A,
                   i64 lda, const double* B, i64 ldb, double beta, double* C, i64 ldc) {
    return oxi_launch_dgemm(h, s, ta, tb, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
}
template <>
int gemm_t<float>(oxi_handle_t h, hipStream_t s, int ta, int tb, i64 m, i64 n, i64 k, float alpha, const float* A,
                  i64 lda, const float* B, i64 ldb, float beta, float* C, i64 ldc) {
    return oxi_launch_sgemm(h, s, ta, tb, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
}

// Right-side triangular solve X <- X * op(T)^-1 where op(T) is upper
// triangular (T upper and trans == 0, or T lower and trans == 1), recursive
// halving with GEMM updates (src/blas/level3.jl:358-376).
// inv: when not null (FP64 only), the inverses of op(T)'s 64 x 64 diagonal
// blocks (n a multiple of 64), and each 64-column leaf is the in-place
// product X_b <- X_b V_b on the matrix cores instead of a column sweep.
template <typename TY>
static int trsm_right_upper(oxi_handle_t h, hipStream_t s, int trans, int unit, i64 rows, i64 n, const TY* T,
                            i64 ldt, TY* X, i64 ldx, const double* inv = nullptr) {
    if (rows <= 0 || n <= 0) return OXI_OK;
    if (n <= TRL) {
        if constexpr (sizeof(TY) == 8) {
            if (inv) {
                if (oxi_dgemm_right64_inplace(s, rows, inv, (double*)X, ldx) != OXI_OK)
                    return oxi_set_error(h, OXI_ERR_HIP, "trsm in-place block product launch failed");
                return OXI_OK;
            }
        }
        launch_right_leaf<TY, false>(s, unit, trans, rows, int(n), T, ldt, X, ldx);
        return launch_check(h, "trsm_right_leaf");
    }
    i64 hh = n / 2;
    if (hh > TRL) hh = (hh / TRL) * TRL;
    // X1 = X[:, :hh], X2 = X[:, hh:]; op(T) = [U11 U12; 0 U22]
    OXI_TRY(trsm_right_upper(h, s, trans, unit, rows, hh, T, ldt, X, ldx, inv));
    // X2 -= X1 * U12, U12 = op(T)[0:hh, hh:n]
    const TY* U12 = trans ? T + hh : T + hh * ldt;  // op(T)[0][hh]: trans -> T[hh][0]
    OXI_TRY(gemm_t<TY>(h, s, 0, trans, rows, n - hh, hh, TY(-1), X, ldx, U12, ldt, TY(1), X + hh * ldx, ldx));
    return trsm_right_upper(h, s, trans, unit, rows, n - hh, T + hh + hh * ldt, ldt, X + hh * ldx, ldx,
                            inv ? inv + (hh / TRL) * 4096 : nullptr);
}

template <bool UPPER, bool CLEAN>
static void launch_inv64(hipStream_t s, int trans, int unit, i64 n, const double* T, i64 ldt, double* inv, i64 ldv = 64,
                         int strip = 0) {
    const dim3 grid(unsigned(cdiv(n, TRL))), block(256);
    if (unit) {
        if (trans) hipLaunchKernelGGL((trsm_inv64_kernel<true, true, UPPER, CLEAN>), grid, block, 0, s, T, ldt, n, inv, ldv, strip);
        else hipLaunchKernelGGL((trsm_inv64_kernel<true, false, UPPER, CLEAN>), grid, block, 0, s, T, ldt, n, inv, ldv, strip);
    } else {
        if (trans) hipLaunchKernelGGL((trsm_inv64_kernel<false, true, UPPER, CLEAN>), grid, block, 0, s, T, ldt, n, inv, ldv, strip);
        else hipLaunchKernelGGL((trsm_inv64_kernel<false, false, UPPER, CLEAN>), grid, block, 0, s, T, ldt, n, inv, ldv, strip);
    }
}

// Tall right-side solves (FP64, rows >= 1024, n a multiple of 64): the
// diagonal blocks' inverses first, then the recursion with in-place products
// for the leaves (a leaf's column sweep is a chain of 64 dependent steps per
// row; the product runs on the matrix cores).
static const double* right_upper_inverses(oxi_handle_t h, hipStream_t s, int trans, int unit, i64 rows, i64 n,
                                          const double* T, i64 ldt) {
    if (rows < 1024 || n < TRL || n % TRL || n / TRL > TRSM_INV_BLOCKS || !h->trsm_inv) return nullptr;
    launch_inv64<true, false>(s, trans, unit, n, T, ldt, h->trsm_inv);
    return hipGetLastError() == hipSuccess ? h->trsm_inv : nullptr;
}

// Right-side solve with op(T) lower: X <- X * op(T)^-1 (backward over columns).
template <typename TY>
static int trsm_right_lower(oxi_handle_t h, hipStream_t s, int trans, int unit, i64 rows, i64 n, const TY* T,
                            i64 ldt, TY* X, i64 ldx);

// Solves with FP64 triangles of n >= 128 rows, `other` (>= 16) right-hand
// sides (columns of B on the left side, rows on the right), in place: by
// halves down to blocks of SB rows, which are one launch of trsm_block_kernel
// each, the updates one product each.  (Right-looking over the blocks took the
// same time, but rounds an element once per block before it instead of once
// per level: error against 64 bits 3.4e-16 instead of 2.8e-16 at 2048 x 2048.)
// 2048 x 2048: 437 us by a recursion down to in-place products with 64 x 64
// inverses, 392 so; 2001 x 1999, whose 64-row leaves were column sweeps: 897
// and 405.  Against extended precision the error of x is 2.4e-16 at 2048 x 2048
// either way, 2.4e-16 instead of 3.6e-16 at 2001 x 1999.  Bound by the chain of blocks and the smaller updates.
static int trsm_blocked(oxi_handle_t h, hipStream_t s, bool left, int upper, int trans, int unit, i64 n, i64 other,
                        const double* A, i64 lda, double* B, i64 ldb) {
    const bool lower_op = (!upper) != (trans != 0);   // op(A) lower?
    const bool ascending = left == lower_op;
    // M of the block kernel: op(A) on the left side, op(A)^T on the right
    const bool mt = left == (trans != 0), bwd = !ascending;
    // rows (left) or columns (right) of B from i on
    auto at = [&](i64 i) { return left ? B + i : B + i * ldb; };
    const i64 most = i64(TRSM_INV_BLOCKS) / 2 * TRL;  // rows whose blocks and inverses fit the handle's buffer
    i64 inv0 = -1;                                    // first row of those in it
    auto block = [&](i64 b0, i64 nb) -> int {
        const dim3 grid(unsigned(cdiv(other, 16))), bl(256);
        const double* Ab = A + b0 * (lda + 1);
        const double* Vb = h->trsm_inv + (b0 - inv0) / TRL * 8192;
#define OXI_BLOCK(L, M, W)                                                                                           \
    if (left == L && mt == M && bwd == W) {                                                                          \
        if (nb == SB) hipLaunchKernelGGL((trsm_block_kernel<L, M, W, true>), grid, bl, 0, s, Ab, lda, Vb, at(b0), ldb, int(nb), other); \
        else hipLaunchKernelGGL((trsm_block_kernel<L, M, W, false>), grid, bl, 0, s, Ab, lda, Vb, at(b0), ldb, int(nb), other); \
    }
        OXI_BLOCK(true, false, false) OXI_BLOCK(true, false, true) OXI_BLOCK(true, true, false) OXI_BLOCK(true, true, true)
        OXI_BLOCK(false, false, false) OXI_BLOCK(false, false, true) OXI_BLOCK(false, true, false) OXI_BLOCK(false, true, true)
#undef OXI_BLOCK
        return launch_check(h, "trsm block");
    };
    // rows [i, i + ni) of B -= op(A)[i.., k..] X, X rows [k, k + nk) (columns on the right side)
    auto update = [&](i64 i, i64 ni, i64 k, i64 nk) -> int {
        const i64 r = left ? i : k, c = left ? k : i;   // op(A) from element (r, c) on
        const double* Ar = trans ? A + c + r * lda : A + r + c * lda;
        if (left) return oxi_launch_dgemm(h, s, trans ? 1 : 0, 0, ni, other, nk, -1.0, Ar, lda, at(k), ldb, 1.0, at(i), ldb);
        return oxi_launch_dgemm(h, s, 0, trans ? 1 : 0, other, ni, nk, -1.0, at(k), ldb, Ar, lda, 1.0, at(i), ldb);
    };
    auto solve = [&](auto& self, i64 i, i64 ni) -> int {
        const bool fill = inv0 < 0 && ni <= most;
        if (fill) {
            inv0 = i;
            if (bwd) launch_inv64<true, true>(s, mt, unit, ni, A + i * (lda + 1), lda, h->trsm_inv);
            else launch_inv64<false, true>(s, mt, unit, ni, A + i * (lda + 1), lda, h->trsm_inv);
        }
        if (ni <= SB) {
            OXI_TRY(block(i, ni));
        } else {
            const i64 hh = cdiv(ni / 2, SB) * SB, i1 = i + hh, n1 = ni - hh;
            OXI_TRY(ascending ? self(self, i, hh) : self(self, i1, n1));
            OXI_TRY(ascending ? update(i1, n1, i, hh) : update(i, hh, i1, n1));
            OXI_TRY(ascending ? self(self, i1, n1) : self(self, i, hh));
        }
        if (fill) inv0 = -1;
        return OXI_OK;
    };
    return solve(solve, 0, n);
}

// Left solves with a moderate number of right-hand sides on large triangles
// (FP64, m a multiple of TRB and at least 2 TRB, 16 .. TRB_MAX_RHS
// right-hand sides).  The recursion's updates are skinny (m/2 x nrhs x m/2 at
// the top, and every level costs about as much, one product after the
// other, each on a few workgroups); here op(A) is swept in blocks of TRB
// rows: X_b = op(A)_bb^-1 B_b, one product with the block's explicit
// inverse, then B_rest -= op(A)[rest, b] X_b, whose rows spread over the
// chip.  The TRB x TRB inverses come from the 64 x 64 ones by doubling: for
// U = [U11 U12; 0 U22], U^-1 = [V11, -V11 U12 V22; 0, V22], two batched
// products per doubling and position.  (trsm_block_kernel's 22 us a block
// are hidden only by updates of more right-hand sides: 4096 x 100 486 us so
// and 610 with it, 8192 x 128 901 and 1008, 4096 x 512 587 and 615.)
constexpr int TRB = 256, TRB_MAX_RHS = 512;

static bool left_strip_applies(i64 m, i64 nrhs) {
    return m >= 2 * TRB && m % TRB == 0 && nrhs >= 16 && nrhs <= TRB_MAX_RHS;
}

static int trsm_left_strip(oxi_handle_t h, hipStream_t s, int upper, int trans, int unit, i64 m, i64 nrhs,
                             const double* A, i64 lda, double* B, i64 ldb) {
    const bool lower_op = (!upper) != (trans != 0);   // op(A) lower?
    // the upper matrix U' whose inverse the kernels build: U' = op(A) for an
    // upper op(A), op(A)^T for a lower one; U'(i, j) = ktrans ? A(j, i) : A(i, j)
    const bool ktrans = lower_op ? !trans : (trans != 0);
    // S: m x TRB strip (ld m), rows z*TRB.. hold block z's inverse; T: the
    // doubling's temporaries; X: the solution until the final copy
    const size_t sS = size_t(m) * TRB, sT = size_t(m) * TRB / 2, sX = size_t(m) * size_t(nrhs);
    void* ws;
    OXI_TRY(oxi_workspace3(h, (sS + sT + sX) * sizeof(double), &ws));
    double* S = (double*)ws;
    double* T = S + sS;
    double* X = T + sT;
    if (oxi_launch_dscale(s, m, TRB, 0.0, S, m) != OXI_OK) return oxi_set_error(h, OXI_ERR_HIP, "trsm strip clear");
    launch_inv64<true, false>(s, ktrans, unit, m, A, lda, S, m, int(TRB));
    OXI_TRY(launch_check(h, "trsm block inverses"));
    const i64 nz = m / TRB;
    for (i64 w = TRL; w < TRB; w *= 2) {
        for (i64 l = 0; l < TRB; l += 2 * w) {
            // in every block z: p = local rows/columns [l, l+w), q = [l+w, l+2w)
            const double* Upq = ktrans ? A + (l + w) + l * lda : A + l + (l + w) * lda;
            const double* Vp = S + l + l * m;
            const double* Vq = S + (l + w) + (l + w) * m;
            double* Xpq = S + l + (l + w) * m;
            OXI_TRY(oxi_launch_dgemm_strided(h, s, ktrans ? 1 : 0, 0, w, w, w, 1.0, Upq, lda, TRB * (lda + 1), Vq, m,
                                             TRB, 0.0, T, w, w * w, nz));
            OXI_TRY(oxi_launch_dgemm_strided(h, s, 0, 0, w, w, w, -1.0, Vp, m, TRB, T, w, w * w, 0.0, Xpq, m, TRB,
                                             nz));
        }
    }
    if (lower_op) {
        // op(A)_bb^-1 = (U'_bb^-1)^T
        for (i64 b0 = 0; b0 < m; b0 += TRB) {
            OXI_TRY(oxi_launch_dgemm(h, s, 1, 0, TRB, nrhs, TRB, 1.0, S + b0, m, B + b0, ldb, 0.0, X + b0, m));
            const i64 r0 = b0 + TRB;
            if (r0 < m) {
                const double* Ar = trans ? A + b0 + r0 * lda : A + r0 + b0 * lda;   // op(A)[r0][b0]
                OXI_TRY(oxi_launch_dgemm(h, s, trans ? 1 : 0, 0, m - r0, nrhs, TRB, -1.0, Ar, lda, X + b0, m, 1.0,
                                         B + r0, ldb));
            }
        }
    } else {
        for (i64 b0 = m - TRB; b0 >= 0; b0 -= TRB) {
            OXI_TRY(oxi_launch_dgemm(h, s, 0, 0, TRB, nrhs, TRB, 1.0, S + b0, m, B + b0, ldb, 0.0, X + b0, m));
            if (b0 > 0) {
                const double* Ar = trans ? A + b0 : A + b0 * lda;                   // op(A)[0][b0]
                OXI_TRY(oxi_launch_dgemm(h, s, trans ? 1 : 0, 0, b0, nrhs, TRB, -1.0, Ar, lda, X + b0, m, 1.0, B,
                                         ldb));
            }
        }
    }
    OXI_HIP(h, hipMemcpy2DAsync(B, size_t(ldb) * 8, X, size_t(m) * 8, size_t(m) * 8, size_t(nrhs),
                                hipMemcpyDeviceToDevice, s));
    return OXI_OK;
}

template <typename TY>
static int trsm_left_t(oxi_handle_t h, hipStream_t s, int upper, int trans, int unit, i64 m, i64 nrhs, const TY* A,
                       i64 lda, TY* B, i64 ldb) {
    if (m <= 0 || nrhs <= 0) return OXI_OK;
    const bool lower_op = (!upper) != (trans != 0);  // op(A) lower?
    if (m <= TRL) {
        dim3 grid(unsigned(cdiv(nrhs, 4)));
        if (lower_op) {
            if (unit) hipLaunchKernelGGL((trsm_left_leaf<TY, true, true>), grid, dim3(256), 0, s, B, ldb, nrhs, int(m), A, lda, trans);
            else hipLaunchKernelGGL((trsm_left_leaf<TY, true, false>), grid, dim3(256), 0, s, B, ldb, nrhs, int(m), A, lda, trans);
        } else {
            if (unit) hipLaunchKernelGGL((trsm_left_leaf<TY, false, true>), grid, dim3(256), 0, s, B, ldb, nrhs, int(m), A, lda, trans);
            else hipLaunchKernelGGL((trsm_left_leaf<TY, false, false>), grid, dim3(256), 0, s, B, ldb, nrhs, int(m), A, lda, trans);
        }
        return launch_check(h, "trsm_left_leaf");
    }
    i64 hh = m / 2;
    if (hh > TRL) hh = (hh / TRL) * TRL;
    // op(A) = [A11 A12; A21 A22] in op coordinates; op(A)[i][j] = trans ? A[j][i] : A[i][j]
    const TY* A11 = A;
    const TY* A22 = A + hh + hh * lda;
    if (lower_op) {
        OXI_TRY(trsm_left_t(h, s, upper, trans, unit, hh, nrhs, A11, lda, B, ldb));
        // B2 -= op(A)[hh:, :hh] * B1 ; op(A)[hh][0] = trans ? A[0][hh] : A[hh][0]
        const TY* A21 = trans ? A + hh * lda : A + hh;
        OXI_TRY(gemm_t<TY>(h, s, trans, 0, m - hh, nrhs, hh, TY(-1), A21, lda, B, ldb, TY(1), B + hh, ldb));
        return trsm_left_t(h, s, upper, trans, unit, m - hh, nrhs, A22, lda, B + hh, ldb);
    }
    OXI_TRY(trsm_left_t(h, s, upper, trans, unit, m - hh, nrhs, A22, lda, B + hh, ldb));
    // B1 -= op(A)[:hh, hh:] * B2 ; op(A)[0][hh] = trans ? A[hh][0] : A[0][hh]
    const TY* A12 = trans ? A + hh : A + hh * lda;
    OXI_TRY(gemm_t<TY>(h, s, trans, 0, hh, nrhs, m - hh, TY(-1), A12, lda, B + hh, ldb, TY(1), B, ldb));
    return trsm_left_t(h, s, upper, trans, unit, hh, nrhs, A11, lda, B, ldb);
}

// Right-side solve with op(T) lower: X <- X * op(T)^-1.  op(T) = [L11 0; L21 L22]:
// X2 = B2 * L22^-1 first, then B1 -= X2 * L21, then X1 = B1 * L11^-1.
template <typename TY>
static int trsm_right_lower(oxi_handle_t h, hipStream_t s, int trans, int unit, i64 rows, i64 n, const TY* T,
                            i64 ldt, TY* X, i64 ldx) {
    if (rows <= 0 || n <= 0) return OXI_OK;
    if (n <= TRL) {
        launch_right_leaf<TY, true>(s, unit, trans, rows, int(n), T, ldt, X, ldx);
        return launch_check(h, "trsm_right_leaf");
    }
    i64 hh = n / 2;
    if (hh > TRL) hh = (hh / TRL) * TRL;
    OXI_TRY(trsm_right_lower(h, s, trans, unit, rows, n - hh, T + hh + hh * ldt, ldt, X + hh * ldx, ldx));
    const TY* L21 = trans ? T + hh * ldt : T + hh;  // op(T)[hh][0]
    OXI_TRY(gemm_t<TY>(h, s, 0, trans, rows, hh, n - hh, TY(-1), X + hh * ldx, ldx, L21, ldt, TY(1), X, ldx));
    return trsm_right_lower(h, s, trans, unit, rows, hh, T, ldt, X, ldx);
}

template <typename TY>
static int trsm_right_t(oxi_handle_t h, hipStream_t s, int upper, int trans, int unit, i64 m, i64 n, const TY* A,
                        i64 lda, TY* B, i64 ldb) {
    const bool upper_op = (upper != 0) != (trans != 0);
    if (upper_op) {
        const double* inv = nullptr;
        if constexpr (sizeof(TY) == 8) inv = right_upper_inverses(h, s, trans, unit, m, n, (const double*)A, lda);
        return trsm_right_upper(h, s, trans, unit, m, n, A, lda, B, ldb, inv);
    }
    return trsm_right_lower(h, s, trans, unit, m, n, A, lda, B, ldb);
}


// From 128 rows and 16 right-hand sides: below, the sweeps' launches are as few.
static bool blocked_applies(oxi_handle_t h, i64 n, i64 other) { return n >= 2 * TRL && other >= 16 && h->trsm_inv; }

int oxi_dtrsm_left(oxi_handle_t h, hipStream_t s, int upper, int trans, int unit, i64 m, i64 nrhs, const double* A,
                   i64 lda, double* B, i64 ldb) {
    if (left_strip_applies(m, nrhs)) return trsm_left_strip(h, s, upper, trans, unit, m, nrhs, A, lda, B, ldb);
    if (blocked_applies(h, m, nrhs)) {
        OXI_TRY(oxi_inv_acquire(h, s));
        OXI_TRY(trsm_blocked(h, s, true, upper, trans, unit, m, nrhs, A, lda, B, ldb));
        return oxi_inv_release(h, s);
    }
    return trsm_left_t<double>(h, s, upper, trans, unit, m, nrhs, A, lda, B, ldb);
}
// Inside a factorization (rows of B below its panel), on either of its streams.
int oxi_dtrsm_right(oxi_handle_t h, hipStream_t s, int upper, int trans, int unit, i64 m, i64 n, const double* A,
                    i64 lda, double* B, i64 ldb) {
    return trsm_right_t<double>(h, s, upper, trans, unit, m, n, A, lda, B, ldb);
}
int oxi_dtrsm_right_alone(oxi_handle_t h, hipStream_t s, int upper, int trans, int unit, i64 m, i64 n, const double* A,
                          i64 lda, double* B, i64 ldb) {
    if (blocked_applies(h, n, m)) return trsm_blocked(h, s, false, upper, trans, unit, n, m, A, lda, B, ldb);
    return oxi_dtrsm_right(h, s, upper, trans, unit, m, n, A, lda, B, ldb);
}
int oxi_strsm_left(oxi_handle_t h, hipStream_t s, int upper, int trans, int unit, i64 m, i64 nrhs, const float* A,
                   i64 lda, float* B, i64 ldb) {
    return trsm_left_t<float>(h, s, upper, trans, unit, m, nrhs, A, lda, B, ldb);
}
int oxi_strsm_right(oxi_handle_t h, hipStream_t s, int upper, int trans, int unit, i64 m, i64 n, const float* A,
                    i64 lda, float* B, i64 ldb) {
    return trsm_right_t<float>(h, s, upper, trans, unit, m, n, A, lda, B, ldb);
}

static int trans_kind(char t) {
    if (t == 'N' || t == 'n') return 0;
    if (t == 'T' || t == 't' || t == 'C' || t == 'c') return 1;
    return -1;
}

// First zero on the diagonal of an n x n triangle (1-based), synchronising.
int oxi_first_zero_diag(oxi_handle_t h, hipStream_t s, const double* T, i64 ldt, i64 n, i64* where) {
    void* ws;
    OXI_TRY(oxi_workspace(h, 256, &ws));
    i64* d = (i64*)ws;
    hipLaunchKernelGGL(set_i64_kernel, dim3(1), dim3(1), 0, s, d, i64(0x7fffffffffffffffLL));
    hipLaunchKernelGGL(diag_zero_kernel, dim3(unsigned(std::min<i64>(cdiv(n, 256), 1024))), dim3(256), 0, s, T, ldt, n, d);
    OXI_TRY(launch_check(h, "diag check"));
    i64 v = 0;
    OXI_HIP(h, hipMemcpyAsync(&v, d, sizeof(i64), hipMemcpyDeviceToHost, s));
    OXI_HIP(h, hipStreamSynchronize(s));
    *where = (v == i64(0x7fffffffffffffffLL)) ? 0 : v;
    return OXI_OK;
}

extern "C" int oxi_dtrsm(oxi_handle_t h, char side, char uplo, char trans, char diag, int64_t m, int64_t n,
                         double alpha, const double* A, int64_t lda, double* B, int64_t ldb, int64_t* singular_index) {
    if (!h) return -1;
    const bool left = side == 'L' || side == 'l';
    if (!left && !(side == 'R' || side == 'r')) return -2;
    const bool upper = uplo == 'U' || uplo == 'u';
    if (!upper && !(uplo == 'L' || uplo == 'l')) return -3;
    const int tk = trans_kind(trans);
    if (tk < 0) return -4;
    const bool unit = diag == 'U' || diag == 'u';
    if (!unit && !(diag == 'N' || diag == 'n')) return -5;
    if (m < 0) return -6;
    if (n < 0) return -7;
    const i64 na = left ? m : n;
    if (lda < std::max<i64>(1, na)) return -10;
    if (ldb < std::max<i64>(1, m)) return -12;
    if (singular_index) *singular_index = 0;
    std::lock_guard<std::recursive_mutex> lk(h->guard);
    if (m == 0 || n == 0) return OXI_OK;
    (void)hipSetDevice(h->device);
    hipStream_t s = h->stream;
    if (alpha == 0.0) return oxi_launch_dscale(s, m, n, 0.0, B, ldb);
    if (!unit) {
        i64 z = 0;
        OXI_TRY(oxi_first_zero_diag(h, s, A, lda, na, &z));
        if (z) {
            if (singular_index) *singular_index = z;
            return oxi_set_error(h, OXI_ERR_SINGULAR, "trsm: zero diagonal at %lld", (long long)z);
        }
    }
    if (alpha != 1.0) OXI_TRY(oxi_launch_dscale(s, m, n, alpha, B, ldb));
    if (left) return oxi_dtrsm_left(h, s, upper, tk, unit, m, n, A, lda, B, ldb);
    OXI_TRY(oxi_inv_acquire(h, s));
    OXI_TRY(oxi_dtrsm_right_alone(h, s, upper, tk, unit, m, n, A, lda, B, ldb));
    return oxi_inv_release(h, s);
}

