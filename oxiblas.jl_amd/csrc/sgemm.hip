// FP32 GEMM on CDNA4 matrix cores (v_mfma_f32_16x16x4f32):
// C <- alpha*op(A)*op(B) + beta*C.  Used by the FP32 working precision of the
// mixed-precision LU (the panel's recursive updates and the FP32 solves), the
// Float32 path of gemm! (src/blas/gemm.jl:625-703; GemmConfig kc=896 for
// 4-byte types, :14).
//
// A 256-thread workgroup owns a 128 x 128, 64 x 64 or 32 x 32 tile (chosen
// per product so that the grid fills the CUs), each wave a quarter of it in
// blocks of 16 x 16.  sgemm_direct_kernel takes nearly all products,
// sgemm_mfma_kernel those whose operands have columns of fewer than four.
// Measured lane layout of v_mfma_f32_16x16x4f32 on gfx950: A[l%16][l/16] at
// lane l, B[l/16][l%16], D item r of lane l = row 4*(l/16)+r, column l%16.
#include "oxi_internal.hpp"

#include <algorithm>
#include <cstdlib>
#include <type_traits>

typedef float f4v __attribute__((ext_vector_type(4)));

namespace {

constexpr int BK = 16, NT = 256;

template <bool OUTER_CONTIG, int O>
__device__ __forceinline__ void load_slab(float (&r)[O * BK / NT], const float* __restrict__ X, i64 ldx, i64 o0,
                                          i64 k0, i64 outer, i64 K, int t) {
#pragma unroll
    for (int i = 0; i < O * BK / NT; ++i) {
        int o, kk;
        if (OUTER_CONTIG) { o = t % O; kk = t / O + i * (NT / O); }
        else { kk = t % BK; o = t / BK + i * (NT / BK); }
        const i64 go = o0 + o, gk = k0 + kk;
        r[i] = (go < outer && gk < K) ? (OUTER_CONTIG ? X[go + gk * ldx] : X[gk + go * ldx]) : 0.0f;
    }
}

template <bool OUTER_CONTIG, int O>
__device__ __forceinline__ void store_slab(float* __restrict__ S, const float (&r)[O * BK / NT], int t) {
#pragma unroll
    for (int i = 0; i < O * BK / NT; ++i) {
        int o, kk;
        if (OUTER_CONTIG) { o = t % O; kk = t / O + i * (NT / O); }
        else { kk = t % BK; o = t / BK + i * (NT / BK); }
        S[kk * (O + 1) + o] = r[i];
    }
}

__device__ __forceinline__ void tile_of(int bid, int tiles_m, int tiles_n, int& tm, int& tn) {
    const int total = tiles_m * tiles_n, nx = 8;
    int logical = bid;
    if (total >= nx) {
        const int xcd = bid % nx, local = bid / nx, per = total / nx, rem = total % nx;
        logical = xcd < rem ? xcd * (per + 1) + local : rem * (per + 1) + (xcd - rem) * per + local;
    }
    const int G = 8, group_size = G * tiles_n, group = logical / group_size, first_m = group * G;
    const int gm = min(tiles_m - first_m, G), in = logical % group_size;
    tm = first_m + in % gm;
    tn = in / gm;
}

// A BM x BN tile (BM, BN in {32, 64, 128}); the four waves split it 2 x 2,
// each wave (BM/2) x (BN/2) as QI x QJ blocks of 16 x 16.
template <int BM, int BN, bool TA, bool TB, bool BETA0>
__global__ __launch_bounds__(NT) void sgemm_mfma_kernel(i64 M, i64 N, i64 K, float alpha, const float* __restrict__ A,
                                                        i64 lda, const float* __restrict__ B, i64 ldb, float beta,
                                                        float* __restrict__ C, i64 ldc, int tiles_m, int tiles_n) {
    constexpr int LDS_A = BM + 1, LDS_B = BN + 1, QI = BM / 32, QJ = BN / 32;
    __shared__ float As[2][BK * LDS_A];
    __shared__ float Bs[2][BK * LDS_B];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int wm = wave & 1, wn = wave >> 1;
    int tm, tn;
    tile_of(blockIdx.x, tiles_m, tiles_n, tm, tn);
    const i64 m0 = i64(tm) * BM, n0 = i64(tn) * BN;
    constexpr bool A_OC = !TA, B_OC = TB;

    f4v acc[QI][QJ];
#pragma unroll
    for (int i = 0; i < QI; ++i)
#pragma unroll
        for (int j = 0; j < QJ; ++j) acc[i][j] = f4v{0.f, 0.f, 0.f, 0.f};

    float ra[BM * BK / NT], rb[BN * BK / NT];
    const int nslab = int((K + BK - 1) / BK);
    load_slab<A_OC, BM>(ra, A, lda, m0, 0, M, K, t);
    load_slab<B_OC, BN>(rb, B, ldb, n0, 0, N, K, t);
    store_slab<A_OC, BM>(As[0], ra, t);
    store_slab<B_OC, BN>(Bs[0], rb, t);
    __syncthreads();
    const int lrow = lane >> 4, lcol = lane & 15;
    for (int s = 0; s < nslab; ++s) {
        const int cur = s & 1;
        if (s + 1 < nslab) {
            load_slab<A_OC, BM>(ra, A, lda, m0, i64(s + 1) * BK, M, K, t);
            load_slab<B_OC, BN>(rb, B, ldb, n0, i64(s + 1) * BK, N, K, t);
        }
        const float* as = As[cur];
        const float* bs = Bs[cur];
#pragma unroll
        for (int ks = 0; ks < BK / 4; ++ks) {
            const int kr = ks * 4 + lrow;
            float a[QI], b[QJ];
#pragma unroll
            for (int i = 0; i < QI; ++i) a[i] = as[kr * LDS_A + wm * (BM / 2) + i * 16 + lcol];
#pragma unroll
            for (int j = 0; j < QJ; ++j) b[j] = bs[kr * LDS_B + wn * (BN / 2) + j * 16 + lcol];
#pragma unroll
            for (int i = 0; i < QI; ++i)
#pragma unroll
                for (int j = 0; j < QJ; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[j], acc[i][j], 0, 0, 0);
        }
        if (s + 1 < nslab) {
            store_slab<A_OC, BM>(As[cur ^ 1], ra, t);
            store_slab<B_OC, BN>(Bs[cur ^ 1], rb, t);
        }
        __syncthreads();
    }
    // All loads of C are issued before the first store, without branches (an
    // element outside C reads the nearest element inside it and is not
    // stored): a load behind a bounds branch is waited for before the next
    // one is issued, one memory round trip per element.
    float cv[QI][QJ][4];
    if (!BETA0) {
#pragma unroll
        for (int i = 0; i < QI; ++i)
#pragma unroll
            for (int j = 0; j < QJ; ++j) {
                const i64 col = min(n0 + wn * (BN / 2) + j * 16 + lcol, N - 1);
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    cv[i][j][r] = C[col * ldc + min(m0 + wm * (BM / 2) + i * 16 + lrow * 4 + r, M - 1)];
            }
    }
#pragma unroll
    for (int i = 0; i < QI; ++i)
#pragma unroll
        for (int j = 0; j < QJ; ++j) {
            const i64 col = n0 + wn * (BN / 2) + j * 16 + lcol;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const i64 row = m0 + wm * (BM / 2) + i * 16 + lrow * 4 + r;
                const float v = alpha * acc[i][j][r];
                if (row < M && col < N) C[col * ldc + row] = BETA0 ? v : __builtin_fmaf(beta, cv[i][j][r], v);
            }
        }
}

// 64 lanes x 16 bytes from base + off (per lane) to LDS at lds .. lds + 1023,
// without registers; counted in vmcnt until the bytes are in LDS.
__device__ __forceinline__ void load_to_lds(const char* base, unsigned off, unsigned lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(lds)
                 : "memory");
}
// a workgroup's operand, the same in every lane, as an address in scalar registers
__device__ __forceinline__ const char* in_sgprs(const float* p) {
    const unsigned long long a = (unsigned long long)p;
    const unsigned lo = __builtin_amdgcn_readfirstlane(unsigned(a)), hi = __builtin_amdgcn_readfirstlane(unsigned(a >> 32));
    return (const char*)((unsigned long long)hi << 32 | lo);
}

// One operand's slab of O outer elements x KB of k in LDS.
//   OUTER_CONTIG: rows of k, element (o, k) at k * O + (o ^ turn(k));
//   else rows of o, the four from k on (k % 4 == 0) in slot (k / 4) ^ ((o / 2) % 8).
// Either way the 64 lanes of an LDS read (16 o, four k) touch every bank once.
// A lane fetches the fours of its places; where the contiguous direction ends
// inside one, the last four there are take its place (found()).
template <bool OUTER_CONTIG, int O, int KB>
struct Slab {
    static_assert(KB == 32, "slots");
    static constexpr int LOADS = O * KB / 256;             // wave loads of a slab
    __device__ static __forceinline__ int turn(int k) { return O >= 64 ? 16 * (k & 3) : 16 * ((k >> 1) & 1); }
    // byte offset, from the slab's first element, of what the lane fetches in
    // load q; o_last, k_last: the last elements there are, the contiguous
    // one's at least 3
    __device__ static __forceinline__ unsigned source(int q, int lane, i64 ldx, i64 o_last, int k_last) {
        const int e = q * 256 + lane * 4;                  // first of the lane's four places
        if (OUTER_CONTIG) {
            const int k = e / O, o = (e % O) ^ turn(k);
            return unsigned((min(i64(o), o_last - 3) + i64(min(k, k_last)) * ldx) * 4);
        }
        const int o = e / KB, k = 4 * (((e % KB) / 4) ^ ((o >> 1) & 7));
        return unsigned((i64(min(k, k_last - 3)) + min(i64(o), o_last) * ldx) * 4);
    }
    // place of element (o, k)
    __device__ static __forceinline__ int at(int o, int k) {
        if (OUTER_CONTIG) return k * O + (o ^ turn(k));
        return o * KB + 4 * ((k / 4) ^ ((o >> 1) & 7)) + (k & 3);
    }
};
// where element x of the contiguous direction is found when `last` is the last one there is
__device__ __forceinline__ int found(int x, i64 last) {
    const int four = x & ~3;
    return x <= last && four > last - 3 ? x + int(four - (last - 3)) : x;
}

// The kernel of nearly all products: slabs straight to LDS, as
// dgemm_direct_kernel (dgemm.hip): no registers hold loads in flight, slab
// s + 1 is under way during the whole of slab s, one barrier a slab, operands of
// any size and alignment.  Bound by the matrix cores where K is long, by C's
// traffic where it is short.  Through registers, a 16-deep slab and the
// padded LDS rows it took 12.9 ms (85 TF/s) at 8192^3 and takes 7.5 (147; a
// library's product reaches 151), 51.5 -> 35.3 us at 1500 x 1111 x 777 TN,
// 28.6 -> 15.1 at 2048 x 2048 x 128, 934 -> 725 at 16384 x 16384 x 128.
// Products are summed in the same order of k, so the results have the same
// errors against 64 bits.
template <int BM, int BN, int OCC, bool TA, bool TB, bool BETA0>
__global__ __launch_bounds__(NT, OCC) void sgemm_direct_kernel(i64 M, i64 N, i64 K, float alpha,
                                                               const float* __restrict__ A, i64 lda,
                                                               const float* __restrict__ B, i64 ldb, float beta,
                                                               float* __restrict__ C, i64 ldc, int tiles_m, int tiles_n) {
    constexpr int KB = 32, NW = 4, MI = BM / 32, NJ = BN / 32;
    using SA = Slab<!TA, BM, KB>;
    using SB = Slab<TB, BN, KB>;
    constexpr int STAGE = (BM + BN) * KB, LA = SA::LOADS / NW, LB = SB::LOADS / NW;
    static_assert(SA::LOADS % NW == 0 && SB::LOADS % NW == 0, "loads");
    constexpr int EC = BN / 2 > 32 ? 32 : BN / 2, LDE = BM + 1;   // epilogue: EC columns at a time
    constexpr int SPACE = 2 * STAGE > LDE * EC ? 2 * STAGE : LDE * EC;
    __shared__ __align__(1024) float lds[SPACE];
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int wm = wave & 1, wn = wave >> 1;
    int tm, tn;
    tile_of(blockIdx.x, tiles_m, tiles_n, tm, tn);
    const i64 m0 = i64(tm) * BM, n0 = i64(tn) * BN;

    // this wave's loads of a slab: LA of A's, LB of B's
    const int nst = int((K + KB - 1) / KB), ktail = int(K - i64(nst - 1) * KB);
    const i64 mlast = M - 1 - m0, nlast = N - 1 - n0;
    // fewer than four rows (columns) are fetched as the last of four
    const char* abase = in_sgprs(TA ? A + m0 * lda : A + m0 - max(3 - mlast, i64(0)));
    const char* bbase = in_sgprs(TB ? B + n0 - max(3 - nlast, i64(0)) : B + n0 * ldb);
    const i64 astep = (TA ? i64(KB) : KB * lda) * 4, bstep = (TB ? KB * ldb : i64(KB)) * 4;
    const unsigned lds0 = unsigned((unsigned long long)(__attribute__((address_space(3))) float*)lds);
    const int nfull = ktail < KB ? nst - 1 : nst;          // slabs of KB
    unsigned offa[LA], offb[LB];
    auto offsets = [&](int klast) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < LA; ++q)
            offa[q] = SA::source(wave * LA + q, lane, lda, TA ? mlast : max(mlast, i64(3)), TA ? max(klast, 3) : klast);
#pragma unroll
        for (int q = 0; q < LB; ++q)
            offb[q] = SB::source(wave * LB + q, lane, ldb, TB ? max(nlast, i64(3)) : nlast, TB ? klast : max(klast, 3));
    };
    offsets(nst > 1 ? KB - 1 : ktail - 1);
    auto issue = [&](int s) __attribute__((always_inline)) {
        i64 back = 0;
        if (s == nfull && nst > 1) {                       // the last ktail of k; fewer than four as the last of four
            offsets(ktail - 1);
            back = 4 * max(4 - ktail, 0);
        }
        const unsigned to = lds0 + unsigned(s & 1) * (STAGE * 4);
        const char* a = abase + s * astep - (TA ? back : 0);
        const char* b = bbase + s * bstep - (TB ? 0 : back);
#pragma unroll
        for (int q = 0; q < LA; ++q) load_to_lds(a, offa[q], to + (wave * LA + q) * 1024);
#pragma unroll
        for (int q = 0; q < LB; ++q) load_to_lds(b, offb[q], to + (SA::LOADS + wave * LB + q) * 1024);
    };

    f4v acc[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = f4v{0.f, 0.f, 0.f, 0.f};
    const int lk = lane >> 4, li = lane & 15;
    // this lane's rows and columns in the slabs: places at k = lk where they
    // are contiguous, else the first row or column (the others 16, 32, .. on)
    const int ar = wm * (BM / 2) + li, bc = wn * (BN / 2) + li;
    int pa[MI], pb[NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i) pa[i] = SA::at(TA ? ar + i * 16 : found(ar + i * 16, mlast), lk);
#pragma unroll
    for (int j = 0; j < NJ; ++j) pb[j] = SB::at(TB ? found(bc + j * 16, nlast) : bc + j * 16, lk);
    issue(0);
    auto arrive = [&]() __attribute__((always_inline)) {
        // the slab has arrived (this wave's loads, then everyone's)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    };
    auto products = [&](int s, auto tail) __attribute__((always_inline)) {
        constexpr bool TAIL = decltype(tail)::value;
        const float* as = lds + (s & 1) * STAGE;
        const float* bs = as + BM * KB;
#pragma unroll
        for (int ks = 0; ks < KB / 4; ++ks) {
            const int k = ks * 4 + lk;
            const int ka = TAIL && TA ? found(k, ktail - 1) : k;
            const int kb = TAIL && !TB ? found(k, ktail - 1) : k;
            float a[MI], b[NJ];
#pragma unroll
            for (int i = 0; i < MI; ++i) a[i] = as[TA ? SA::at(ar, ka) + i * 16 * KB : pa[i] + ks * 4 * BM];
#pragma unroll
            for (int j = 0; j < NJ; ++j) b[j] = bs[TB ? pb[j] + ks * 4 * BN : SB::at(bc, kb) + j * 16 * KB];
            if (TAIL) {   // past K: zeros
#pragma unroll
                for (int i = 0; i < MI; ++i) a[i] = k < ktail ? a[i] : 0.f;
#pragma unroll
                for (int j = 0; j < NJ; ++j) b[j] = k < ktail ? b[j] : 0.f;
            }
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int j = 0; j < NJ; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[j], acc[i][j], 0, 0, 0);
        }
    };
    for (int s = 0; s < nfull; ++s) {
        arrive();
        // everyone is past slab s - 1: its space takes slab s + 1
        if (s + 1 < nst) issue(s + 1);
        products(s, std::false_type{});
    }
    if (nfull < nst) {
        arrive();
        products(nfull, std::true_type{});
    }

    if (m0 + BM <= M && n0 + BN <= N) {
        // C, EC columns at a time, through LDS: every wave then covers
        // consecutive rows of a column, and every thread issues its loads of
        // a piece before its first store
        constexpr int CPT = BM * EC / NT, CPP = NT / BM, WC = BN / 2;
        const int er = t % BM, ec0 = t / BM;
#pragma unroll
        for (int h = 0; h < BN / EC; ++h) {
            float* cc = C + (n0 + h * EC + ec0) * ldc + m0 + er;
            float cv[CPT];
            if (!BETA0) {
#pragma unroll
                for (int k = 0; k < CPT; ++k) cv[k] = cc[i64(CPP * k) * ldc];
            }
            __syncthreads();
            if (wn == h * EC / WC) {
#pragma unroll
                for (int j = 0; j < EC / 16; ++j)
#pragma unroll
                    for (int i = 0; i < MI; ++i)
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            lds[(j * 16 + li) * LDE + wm * (BM / 2) + i * 16 + 4 * lk + r] = acc[i][h * EC % WC / 16 + j][r];
            }
            __syncthreads();
#pragma unroll
            for (int k = 0; k < CPT; ++k) {
                const float v = alpha * lds[(ec0 + CPP * k) * LDE + er];
                cc[i64(CPP * k) * ldc] = BETA0 ? v : __builtin_fmaf(beta, cv[k], v);
            }
        }
        return;
    }
    // edge tile: one block column at a time, its C loads (an element outside C
    // reads the nearest one inside and is not stored) before its stores
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const i64 col = n0 + wn * (BN / 2) + j * 16 + li, colc = min(col, N - 1);
        float cv[MI][4];
        if (!BETA0) {
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) cv[i][r] = C[colc * ldc + min(m0 + wm * (BM / 2) + i * 16 + 4 * lk + r, M - 1)];
        }
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const i64 row = m0 + wm * (BM / 2) + i * 16 + 4 * lk + r;
                const float v = alpha * acc[i][j][r];
                if (row < M && col < N) C[col * ldc + row] = BETA0 ? v : __builtin_fmaf(beta, cv[i][r], v);
            }
    }
}

__global__ void sscale_kernel(i64 m, i64 n, float beta, float* __restrict__ C, i64 ldc) {
    const i64 total = m * n;
    for (i64 idx = i64(blockIdx.x) * blockDim.x + threadIdx.x; idx < total; idx += i64(gridDim.x) * blockDim.x) {
        const i64 j = idx / m, i = idx - j * m;
        float& c = C[i + j * ldc];
        c = (beta == 0.0f) ? 0.0f : c * beta;
    }
}

template <int BM, int BN, bool TA, bool TB>
void launch_tiles(hipStream_t s, i64 m, i64 n, i64 k, float alpha, const float* A, i64 lda, const float* B, i64 ldb,
                  float beta, float* C, i64 ldc) {
    const int tiles_m = int(cdiv(m, BM)), tiles_n = int(cdiv(n, BN));
    dim3 grid(tiles_m * tiles_n), block(NT);
    if (beta == 0.0f)
        hipLaunchKernelGGL((sgemm_mfma_kernel<BM, BN, TA, TB, true>), grid, block, 0, s, m, n, k, alpha, A, lda, B,
                           ldb, beta, C, ldc, tiles_m, tiles_n);
    else
        hipLaunchKernelGGL((sgemm_mfma_kernel<BM, BN, TA, TB, false>), grid, block, 0, s, m, n, k, alpha, A, lda, B,
                           ldb, beta, C, ldc, tiles_m, tiles_n);
}

// false (nothing launched) where sgemm_direct_kernel cannot read the operands:
// it loads fours along their columns, at 32-bit offsets inside a tile
template <int BM, int BN, int OCC, bool TA, bool TB>
bool launch_direct(hipStream_t s, i64 m, i64 n, i64 k, float alpha, const float* A, i64 lda, const float* B, i64 ldb,
                   float beta, float* C, i64 ldc) {
    const i64 far = std::max((TA ? BM : 32) * lda, (TB ? 32 : BN) * ldb);
    if ((TA ? k : m) < 4 || (TB ? n : k) < 4 || far > (i64(1) << 28)) return false;
    const int tiles_m = int(cdiv(m, BM)), tiles_n = int(cdiv(n, BN));
    dim3 grid(tiles_m * tiles_n), block(NT);
    if (beta == 0.0f)
        hipLaunchKernelGGL((sgemm_direct_kernel<BM, BN, OCC, TA, TB, true>), grid, block, 0, s, m, n, k, alpha, A, lda, B,
                           ldb, beta, C, ldc, tiles_m, tiles_n);
    else
        hipLaunchKernelGGL((sgemm_direct_kernel<BM, BN, OCC, TA, TB, false>), grid, block, 0, s, m, n, k, alpha, A, lda, B,
                           ldb, beta, C, ldc, tiles_m, tiles_n);
    return true;
}

template <bool TA, bool TB>
void launch_variant(hipStream_t s, i64 m, i64 n, i64 k, float alpha, const float* A, i64 lda, const float* B, i64 ldb,
                    float beta, float* C, i64 ldc) {
    constexpr i64 NCU = 256;
    const i64 t128 = cdiv(m, 128) * cdiv(n, 128), t64 = cdiv(m, 64) * cdiv(n, 64);
    // 128 wide from 1.75 workgroups a CU on: two share a CU (8192^3: 7.5 ms, 64
    // wide 8.0; 16384 x 16384 x 128: 725 us, 762; 4096 x 4096 x 128: 49.6, 47.3);
    // 64 from 1.5 (2048^3: 142 us, 32 wide 165; 1500 x 1111 x 777: 34.2, 34.8),
    // below it 32 (1000^3: 29.4 us, 64 wide 30.8; 512^3: 8.5, 14.4).
    const int tile = t128 >= NCU * 7 / 4 ? 128 : t64 >= NCU * 3 / 2 ? 64 : 32;
    if (tile == 128 && launch_direct<128, 128, 2, TA, TB>(s, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc)) return;
    if (tile >= 64 && launch_direct<64, 64, 4, TA, TB>(s, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc)) return;
    if (launch_direct<32, 32, 4, TA, TB>(s, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc)) return;
    // fewer than four along an operand's columns, or columns at least 32 MiB apart
    if (t64 >= NCU * 3 / 2) return launch_tiles<64, 64, TA, TB>(s, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
    return launch_tiles<32, 32, TA, TB>(s, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
}

}  // namespace

int oxi_launch_sgemm(oxi_handle_t h, hipStream_t s, int ta, int tb, i64 m, i64 n, i64 k, float alpha, const float* A,
                     i64 lda, const float* B, i64 ldb, float beta, float* C, i64 ldc) {
    if (m <= 0 || n <= 0) return OXI_OK;
    if (alpha == 0.0f || k <= 0) {
        if (beta == 1.0f) return OXI_OK;
        const int blocks = int(std::min<i64>(cdiv(m * n, 256), 4096));
        hipLaunchKernelGGL(sscale_kernel, dim3(blocks), dim3(256), 0, s, m, n, beta, C, ldc);
    } else if (cdiv(m, 64) * cdiv(n, 64) >= OXI_MAX_WG) {
        // more tiles than a launch takes: the longer side in two
        const i64 hm = m >= n ? cdiv(m / 2, 128) * 128 : 0, hn = m >= n ? 0 : cdiv(n / 2, 128) * 128;
        OXI_TRY(oxi_launch_sgemm(h, s, ta, tb, hm ? hm : m, hn ? hn : n, k, alpha, A, lda, B, ldb, beta, C, ldc));
        return oxi_launch_sgemm(h, s, ta, tb, m - hm, n - hn, k, alpha, A + (ta ? hm * lda : hm), lda,
                                B + (tb ? hn : hn * ldb), ldb, beta, C + hm + hn * ldc, ldc);
    } else if (!ta && !tb) launch_variant<false, false>(s, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
    else if (!ta && tb) launch_variant<false, true>(s, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
    else if (ta && !tb) launch_variant<true, false>(s, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
    else launch_variant<true, true>(s, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return oxi_set_error(h, OXI_ERR_HIP, "sgemm launch: %s", hipGetErrorString(e));
    return OXI_OK;
}

extern "C" int oxi_sgemm(oxi_handle_t h, char transA, char transB, int64_t m, int64_t n, int64_t k, float alpha,
                         const float* A, int64_t lda, const float* B, int64_t ldb, float beta, float* C,
                         int64_t ldc) {
    if (!h) return -1;
    auto kind = [](char t) { return (t == 'N' || t == 'n') ? 0 : (t == 'T' || t == 't' || t == 'C' || t == 'c') ? 1 : -1; };
    const int ka = kind(transA), kb = kind(transB);
    if (ka < 0) return -2;
    if (kb < 0) return -3;
    if (m < 0) return -4;
    if (n < 0) return -5;
    if (k < 0) return -6;
    if (lda < std::max<i64>(1, ka ? k : m)) return -9;
    if (ldb < std::max<i64>(1, kb ? n : k)) return -11;
    if (ldc < std::max<i64>(1, m)) return -14;
    std::lock_guard<std::recursive_mutex> lk(h->guard);
    if (m == 0 || n == 0) return OXI_OK;
    (void)hipSetDevice(h->device);
    return oxi_launch_sgemm(h, h->stream, ka, kb, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
}
