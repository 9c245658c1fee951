// Inverse of a triangular block in LDS on the matrix cores, shared by the
// preparations of the triangular solves (trsv.hip, trsm_chain.hip, trsm.hip),
// and by substitution for blocks whose inverse is not finite.
#pragma once
#include "oxi_internal.hpp"

namespace tri {

// v_mfma_f64_16x16x4 / v_mfma_f32_16x16x4: A[i][k] at lane 16k + i, B[k][j] at
// lane 16k + j, row(lk, r) of column j in accumulator r of lane 16 lk + j.
template <typename T> struct Mfma;
template <> struct Mfma<double> {
    typedef double acc __attribute__((ext_vector_type(4)));
    __device__ static __forceinline__ acc mul(double a, double b, acc c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    __device__ static __forceinline__ int row(int lk, int r) { return 4 * r + lk; }
};
template <> struct Mfma<float> {
    typedef float acc __attribute__((ext_vector_type(4)));
    __device__ static __forceinline__ acc mul(float a, float b, acc c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    __device__ static __forceinline__ int row(int lk, int r) { return 4 * lk + r; }
};

// The block in LDS: N columns of LD = N + 1; SPACE elements, the last 16 only read.
template <int N> constexpr int LD = N + 1;
template <int N> constexpr int SPACE = N * LD<N> + 16;

__device__ __forceinline__ double nfma(double a, double b, double c) { return __builtin_fma(-a, b, c); }
__device__ __forceinline__ float nfma(float a, float b, float c) { return __builtin_fmaf(-a, b, c); }

// D (lower triangular, its diagonal in place, N a power of two >= 32) <- its
// inverse, by NW waves (thread t of them).  Above the diagonal only the 16 x 16
// blocks on it hold zeros afterwards: readers skip the others (tile row <
// tile column).
//
// A serial sweep over N columns, as long as the block itself, is what bounds
// such an inverse.  Here only the 16 x 16 blocks are swept, 16 lanes each with
// a column in registers; then pairs of inverted blocks A, B are joined with
// the block C below A, -B^-1 (C A^-1), 16 -> 32 -> .. -> N: two products a
// level on the matrix cores, the first parked in the unused half above the
// diagonal.  A 64 x 64 block with its loads and stores: 8 us, swept by a column
// a lane 27.  Loops stay rolled: unrolled throughout, 128 x 128 with its
// coupling took 44 us instead of 38, fetching code that runs once.
template <typename T, int N, int NW, bool UNIT>
__device__ __forceinline__ void invert(T* D, int t) {
    typedef Mfma<T> M;
    constexpr int L = LD<N>;
    const int lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int lk = lane >> 4, li = lane & 15;
    for (int b = 4 * wave + lk; b < N / 16; b += 4 * NW) {
        // column li by right-looking substitution, x[i] for row k + i: rows
        // move down one register a step.  Row k of the inverse goes to its
        // place at once: the elements there have been used.
        T* B = D + b * 16 * (L + 1);
        T x[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) x[i] = i == li ? T(1) : T(0);
#pragma unroll 1
        for (int k = 0; k < 16; ++k) {
            T c[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) c[i] = B[k * (L + 1) + i];
            const T xk = UNIT ? x[0] : x[0] / c[0];
#pragma unroll
            for (int i = 1; i < 16; ++i) x[i - 1] = nfma(c[i], xk, x[i]);
            B[li * L + k] = k < li ? T(0) : xk;
        }
    }
    __syncthreads();
#pragma unroll 1
    for (int lt = 0; (16 << lt) < N; ++lt) {               // blocks of 2^lt tiles of 16
        const int h = 16 << lt, tt = 1 << lt, tiles = (N / 32) << lt;
#pragma unroll 1
        for (int e = wave; e < tiles; e += NW) {           // W = C A^-1
            const int p = (e >> 2 * lt) * 2 * h, it = e & (tt - 1), jt = (e >> lt) & (tt - 1);
            const T* c = D + (p + lk) * L + p + h + it * 16 + li;
            const T* a = D + (p + jt * 16 + li) * L + p + lk;
            typename M::acc w = {0, 0, 0, 0};
#pragma unroll 1
            for (int k = jt * 16; k < h; k += 16)
#pragma unroll
                for (int s = 0; s < 16; s += 4) w = M::mul(c[(k + s) * L], a[k + s], w);
#pragma unroll
            for (int r = 0; r < 4; ++r) D[(p + h + jt * 16 + li) * L + p + it * 16 + M::row(lk, r)] = w[r];
        }
        __syncthreads();
#pragma unroll 1
        for (int e = wave; e < tiles; e += NW) {           // C <- -B^-1 W
            const int p = (e >> 2 * lt) * 2 * h, it = e & (tt - 1), jt = (e >> lt) & (tt - 1);
            const T* b = D + (p + h + lk) * L + p + h + it * 16 + li;
            const T* w = D + (p + h + jt * 16 + li) * L + p + lk;
            typename M::acc x = {0, 0, 0, 0};
#pragma unroll 1
            for (int k = 0; k <= it * 16; k += 16)
#pragma unroll
                for (int s = 0; s < 16; s += 4) x = M::mul(b[(k + s) * L], w[k + s], x);
#pragma unroll
            for (int r = 0; r < 4; ++r) D[(p + jt * 16 + li) * L + p + h + it * 16 + M::row(lk, r)] = -x[r];
        }
        __syncthreads();
    }
}

// The same by substitution, a thread (t < N) per column, for the rare block
// whose inverse holds an infinity or NaN (N^2 / 2 dependent loads).  Such an
// element of D at (i, k) then reaches rows i on of the columns up to k and
// nothing else; the products above, which multiply the zeros of a tile too,
// carry it to all rows and columns of its 16 x 16 tile.  Column t goes through
// tmp (N columns of memory, leading dimension ld, this workgroup's alone).
template <typename T, int N, bool UNIT>
__device__ __forceinline__ void invert_by_substitution(T* D, int t, T* tmp, i64 ld) {
    constexpr int L = LD<N>;
    T* x = tmp + t * ld;
    if (t < N) {
#pragma unroll 1
        for (int i = t; i < N; ++i) {
            T s = i == t ? T(1) : T(0);
#pragma unroll 1
            for (int k = t; k < i; ++k) s = nfma(D[k * L + i], x[k], s);
            x[i] = UNIT ? s : s / D[i * L + i];
        }
    }
    __syncthreads();
    if (t < N)
#pragma unroll 1
        for (int i = 0; i < N; ++i) D[t * L + i] = i < t ? T(0) : x[i];
    __syncthreads();
}

// G (rows i of the block, 16 columns q of this wave, value(i, q) given to
// `put`) = the inverse in D times the N x 16 block whose element (k, q) is
// tv[k / 4] of lane 16 (k % 4) + q.
template <typename T, int N, typename Put>
__device__ __forceinline__ void times(const T* D, const T (&tv)[N / 4], int lane, Put put) {
    typedef Mfma<T> M;
    constexpr int L = LD<N>;
    const int lk = lane >> 4, li = lane & 15;
#pragma unroll 1
    for (int it = 0; it < N / 16; ++it) {
        const T* d = D + lk * L + it * 16 + li;
        typename M::acc g = {0, 0, 0, 0};
#pragma unroll
        for (int kt = 0; kt < N / 16; ++kt)
            if (kt <= it) {
#pragma unroll
                for (int s = 4 * kt; s < 4 * kt + 4; ++s) g = M::mul(d[4 * s * L], tv[s], g);
            }
#pragma unroll
        for (int r = 0; r < 4; ++r) put(it * 16 + M::row(lk, r), li, g[r]);
    }
}

}  // namespace tri
