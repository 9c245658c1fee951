// Float16 gemm! (src/blas/extended_blas.jl:39-88): Float16 operands and
// output, Float32 accumulation of each element over all of K, one rounding to
// Float16 at the end: C = Float16(a * acc + b * Float32(C)) with a, b the
// Float32 values of alpha and beta rounded to Float16 (beta == 0 never reads C).
//
// The product kernel reads both operands with k contiguous: rows of op(A) and
// columns of op(B).  A transposed A and an untransposed B are that already and
// are read in place when their rows are 16-byte aligned and K is a multiple of
// the slab depth; otherwise (and when the operand overlaps C) a packing pass
// writes them so, zero padded, to the workspace.
#include "oxi_internal.hpp"

#include <algorithm>

namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef float f4v __attribute__((ext_vector_type(4)));

constexpr int HBK = 32;                    // slab depth: one v_mfma_f32_16x16x32_f16
constexpr int HROW = HBK * 2;              // bytes of a slab row
constexpr int HSTAGES = 4;                 // slabs in LDS

// Tiles of one XCD are contiguous in an order that walks groups of 8 tile
// rows column by column, so that they share operand panels in its L2.
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

// 64 lanes x 16 bytes from global memory to LDS at m0 .. m0 + 1023, without
// registers; counted in vmcnt until the bytes are in LDS.
__device__ __forceinline__ void load_to_lds(const char* g, unsigned lds) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(g), "s"(lds) : "memory");
}
template <int N>
__device__ __forceinline__ void wait_loads() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// C (M x N, column-major) = Float16(aw * A B + bw * C); A as M rows, B as N
// rows of K contiguous values (ldka, ldkb bytes a row), K a multiple of HBK.
//
// A workgroup of WM x WN waves owns a BM x BN tile, a wave BM/WM x BN/WN of it
// as 16 x 16 blocks.  The operands' slabs go straight to LDS
// (global_load_lds_dwordx4), HSTAGES deep: the loads of slab s + 3 are issued
// when slab s is started, so a load has three slabs' products (about 1.3 us
// for the 256 x 256 tile) to arrive, and there is one barrier a slab.  A lane's
// place in LDS follows from its number, so the bank conflicts of the 64-byte
// rows are avoided by the order in which the lanes fetch: the 16-byte chunk c
// of row r sits in slot c ^ ((r / 4) % 4), and the 16 lanes that read chunk c
// of 16 rows touch every bank once.
// Bound by the matrix cores (1024 cycles of products per 768 of LDS reads a
// slab and CU for the 256 x 256 tile).  Measured: 4096^3 131 us = 1050 TF/s with
// nothing to pack (A transposed), 140 us with A packed, 8192^3 1063 us = 1034 TF/s
// with its packing pass; before, packing both operands, clearing and updating
// an FP32 C, and a conversion pass around a register-staged 128 x 128 kernel took
// 271 us at 4096^3.
// vec: C 8-byte aligned with ldc a multiple of 4.
template <int BM, int BN, int WM, int WN>
__global__ __launch_bounds__(64 * WM * WN) void hgemm_kernel(i64 M, i64 N, i64 K, float aw, float bw, int beta0,
                                                             const char* __restrict__ A, i64 ldka,
                                                             const char* __restrict__ B, i64 ldkb,
                                                             _Float16* __restrict__ C, i64 ldc, int tiles_m,
                                                             int tiles_n, int vec) {
    constexpr int NW = WM * WN, MI = BM / WM / 16, NJ = BN / WN / 16;
    constexpr int STAGE = (BM + BN) * HROW, LOADS = (BM + BN) / 16 / NW;   // bytes a slab; loads a wave and slab
    static_assert((BM + BN) / 16 % NW == 0 && BM % 16 == 0, "loads");
    __shared__ __attribute__((aligned(1024))) char lds[HSTAGES * STAGE];
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int wm = wave % WM, wn = wave / WM;
    int tm, tn;
    tile_of(blockIdx.x, tiles_m, tiles_n, tm, tn);
    const i64 m0 = i64(tm) * BM, n0 = i64(tn) * BN;
    const int nst = int(K / HBK);

    // this lane's source of each of the wave's loads (16 rows of 64 bytes
    // each); rows past the operand read its last one (their results are not
    // stored)
    const char* src[LOADS];
    const unsigned lds0 = unsigned((unsigned long long)(__attribute__((address_space(3))) char*)lds);
#pragma unroll
    for (int q = 0; q < LOADS; ++q) {
        const int r = (wave * LOADS + q) * 16 + lane / 4;      // row of the slab: A's BM rows, then B's
        const int c = (lane & 3) ^ ((r >> 2) & 3);
        src[q] = (r < BM ? A + min(m0 + r, M - 1) * ldka : B + min(n0 + r - BM, N - 1) * ldkb) + c * 16;
    }
    auto issue = [&](int s) __attribute__((always_inline)) {
        const unsigned to = lds0 + unsigned(s % HSTAGES) * STAGE + unsigned(wave) * (LOADS * 1024);
#pragma unroll
        for (int q = 0; q < LOADS; ++q) {
            load_to_lds(src[q], to + q * 1024);
            src[q] += HROW;
        }
    };

    f4v acc[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = f4v{0.f, 0.f, 0.f, 0.f};

    const int li = lane & 15, lg = lane >> 4;
    const int slot = (lg ^ ((li >> 2) & 3)) * 16;
    const int offa = (wm * (BM / WM) + li) * HROW + slot, offb = (BM + wn * (BN / WN) + li) * HROW + slot;
#pragma unroll
    for (int s = 0; s < HSTAGES - 1; ++s)
        if (s < nst) issue(s);
    for (int s = 0; s < nst; ++s) {
        // slab s has arrived (this wave's loads, then everyone's)
        if (s + 2 < nst) wait_loads<2 * LOADS>();
        else if (s + 1 < nst) wait_loads<LOADS>();
        else wait_loads<0>();
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
        // everyone is past slab s - 1: its space takes slab s + 3
        if (s + HSTAGES - 1 < nst) issue(s + HSTAGES - 1);
        const char* st = lds + (s % HSTAGES) * STAGE;
        f16x8 a[MI], b[NJ];
#pragma unroll
        for (int j = 0; j < NJ; ++j) b[j] = *(const f16x8*)(st + offb + j * 16 * HROW);
#pragma unroll
        for (int i = 0; i < MI; ++i) a[i] = *(const f16x8*)(st + offa + i * 16 * HROW);
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[i], b[j], acc[i][j], 0, 0, 0);
    }

    // D item r of a lane is row 4 * (lane / 16) + r, column lane % 16 of its block
    const bool full = vec && m0 + BM <= M && n0 + BN <= N;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const i64 col = n0 + wn * (BN / WN) + j * 16 + li, row0 = m0 + wm * (BM / WM) + 4 * lg;
        if (full) {
            f16x4* c = (f16x4*)(C + col * ldc + row0);
            f16x4 old[MI];
            if (!beta0)
#pragma unroll
                for (int i = 0; i < MI; ++i) old[i] = c[4 * i];
#pragma unroll
            for (int i = 0; i < MI; ++i) {
                f16x4 o;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    float v = aw * acc[i][j][r];
                    if (!beta0) v += bw * float(old[i][r]);
                    o[r] = _Float16(v);
                }
                c[4 * i] = o;
            }
        } else {
            // all loads of C (an element outside reads the nearest one inside)
            // before the first store
            _Float16 old[MI][4];
            const i64 cc = min(col, N - 1);
            if (!beta0)
#pragma unroll
                for (int i = 0; i < MI; ++i)
#pragma unroll
                    for (int r = 0; r < 4; ++r) old[i][r] = C[cc * ldc + min(row0 + 16 * i + r, M - 1)];
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const i64 row = row0 + 16 * i + r;
                    float v = aw * acc[i][j][r];
                    if (!beta0) v += bw * float(old[i][r]);
                    if (row < M && col < N) C[col * ldc + row] = _Float16(v);
                }
        }
    }
}

// out[o][p] (Kp halves a row) = op(X)(o, p) for o < O, p < K, zero up to Kp;
// element (o, p) at X[o * so + p * sp].  P_CONTIG: sp == 1, a thread writes
// eight values; otherwise so == 1: a 64 x 64 tile through LDS, read and
// written 16 bytes a thread where X allows it (vec: X 16-byte aligned, sp a
// multiple of 8).
template <bool P_CONTIG>
__global__ __launch_bounds__(256) void pack_half_kernel(const _Float16* __restrict__ X, i64 so, i64 sp, i64 O, i64 K,
                                                        i64 Kp, _Float16* __restrict__ out, int vec) {
    const int t = threadIdx.x;
    const i64 o0 = i64(blockIdx.x) * 64, p0 = i64(blockIdx.y) * 64;
    const int pc = (t & 7) * 8;                       // this thread's eight columns of a 64-column row
    if (P_CONTIG) {
        for (int y = t >> 3; y < 64; y += 32) {
            const i64 o = o0 + y, p = p0 + pc;
            if (o >= O || p >= Kp) continue;
            f16x8 v;
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = p + e < K ? X[o * so + p + e] : _Float16(0);
            *(f16x8*)(out + o * Kp + p) = v;
        }
        return;
    }
    __shared__ _Float16 tile[64][64 + 2];             // tile[p][o]
    if (vec && o0 + 64 <= O && p0 + 64 <= K) {
#pragma unroll
        for (int y = t >> 3; y < 64; y += 32) {
            const f16x8 v = *(const f16x8*)(X + o0 + pc + (p0 + y) * sp);
#pragma unroll
            for (int e = 0; e < 8; ++e) tile[y][pc + e] = v[e];
        }
    } else {
        for (int y = t >> 6; y < 64; y += 4) {
            const i64 o = o0 + (t & 63), p = p0 + y;
            tile[y][t & 63] = (o < O && p < K) ? X[o + p * sp] : _Float16(0);
        }
    }
    __syncthreads();
    for (int y = t >> 3; y < 64; y += 32) {
        const i64 o = o0 + y, p = p0 + pc;
        if (o >= O || p >= Kp) continue;
        f16x8 v;
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = tile[pc + e][y];
        *(f16x8*)(out + o * Kp + p) = v;
    }
}

__global__ void hscale_kernel(i64 M, i64 N, _Float16 beta, _Float16* __restrict__ C, i64 ldc) {
    const i64 total = M * N;
    for (i64 idx = i64(blockIdx.x) * blockDim.x + threadIdx.x; idx < total; idx += i64(gridDim.x) * blockDim.x) {
        const i64 j = idx / M, i = idx - j * M;
        C[i + j * ldc] = beta == _Float16(0) ? _Float16(0) : _Float16(float(beta) * float(C[i + j * ldc]));
    }
}

bool overlap(const void* a, size_t ab, const void* b, size_t bb) {
    const char* x = (const char*)a; const char* y = (const char*)b;
    return x < y + bb && y < x + ab;
}
size_t span(i64 rows, i64 cols, i64 ld) { return size_t((cols - 1) * ld + rows) * 2; }

}  // namespace

extern "C" int oxi_hgemm(oxi_handle_t h, char transA, char transB, int64_t m, int64_t n, int64_t k, float alpha,
                         const void* Av, int64_t lda, const void* Bv, int64_t ldb, float beta, void* Cv, int64_t ldc) {
    if (!h) return -1;
    const int ta = (transA == 'N' || transA == 'n') ? 0 : (transA == 'T' || transA == 't' || transA == 'C' || transA == 'c') ? 1 : -1;
    const int tb = (transB == 'N' || transB == 'n') ? 0 : (transB == 'T' || transB == 't' || transB == 'C' || transB == 'c') ? 1 : -1;
    if (ta < 0) return -2;
    if (tb < 0) return -3;
    if (m < 0) return -4;
    if (n < 0) return -5;
    if (k < 0) return -6;
    if (lda < std::max<i64>(1, ta ? k : m)) return -9;
    if (ldb < std::max<i64>(1, tb ? n : k)) return -11;
    if (ldc < std::max<i64>(1, m)) return -14;
    std::lock_guard<std::recursive_mutex> lk(h->guard);
    if (m == 0 || n == 0) return OXI_OK;
    if (!Cv) return -13;
    (void)hipSetDevice(h->device);
    hipStream_t s = h->stream;
    const _Float16* A = (const _Float16*)Av;
    const _Float16* B = (const _Float16*)Bv;
    _Float16* C = (_Float16*)Cv;
    // alpha and beta are converted to Float16 first (extended_blas.jl:43)
    const _Float16 ah = _Float16(alpha), bh = _Float16(beta);
    if (ah == _Float16(0) || k == 0) {
        const unsigned eg = unsigned(std::min<i64>(cdiv(m * n, 256), 8192));
        hipLaunchKernelGGL(hscale_kernel, dim3(eg), dim3(256), 0, s, m, n, bh, C, ldc);
        hipError_t e = hipGetLastError();
        return e == hipSuccess ? OXI_OK : oxi_set_error(h, OXI_ERR_HIP, "hgemm launch: %s", hipGetErrorString(e));
    }
    if (!A) return -8;
    if (!B) return -10;
    const i64 Kp = cdiv(k, HBK) * HBK;
    if (cdiv(m, 128) * cdiv(n, 128) >= OXI_MAX_WG || std::max(cdiv(m, 64), cdiv(n, 64)) >= OXI_MAX_WG || cdiv(Kp, 64) > 65535)
        return oxi_set_error(h, OXI_ERR_UNSUPPORTED, "hgemm: %lld x %lld x %lld is too large", (long long)m, (long long)n,
                             (long long)k);
    // read in place: k contiguous, aligned, no padding, apart from C
    const size_t cspan = span(m, n, ldc);
    const auto in_place = [&](const _Float16* X, i64 ld, i64 rows, i64 cols) {
        return k % HBK == 0 && ld % 8 == 0 && (reinterpret_cast<uintptr_t>(X) & 15) == 0 &&
               !overlap(C, cspan, X, span(rows, cols, ld));
    };
    const bool a_in = ta && in_place(A, lda, k, m), b_in = !tb && in_place(B, ldb, k, n);
    const size_t abytes = a_in ? 0 : (size_t(m) * Kp * 2 + 255) & ~size_t(255);
    const size_t bbytes = b_in ? 0 : (size_t(n) * Kp * 2 + 255) & ~size_t(255);
    void* ws = nullptr;
    if (abytes + bbytes) OXI_TRY(oxi_workspace(h, abytes + bbytes, &ws));
    _Float16* Ap = (_Float16*)ws;
    _Float16* Bp = (_Float16*)((char*)ws + abytes);
    // op(A)(i, p): A[i + p*lda] ('N', i contiguous) or A[p + i*lda] ('T', p contiguous);
    // op(B)(p, j) as rows j: B[p + j*ldb] ('N') or B[j + p*ldb] ('T')
    const auto pack = [&](bool p_contig, const _Float16* X, i64 ld, i64 rows, _Float16* out) {
        const dim3 grid(unsigned(cdiv(rows, 64)), unsigned(cdiv(Kp, 64)));
        const int vec = int(ld % 8 == 0 && (reinterpret_cast<uintptr_t>(X) & 15) == 0);
        if (p_contig) hipLaunchKernelGGL(pack_half_kernel<true>, grid, dim3(256), 0, s, X, ld, i64(1), rows, k, Kp, out, vec);
        else hipLaunchKernelGGL(pack_half_kernel<false>, grid, dim3(256), 0, s, X, i64(1), ld, rows, k, Kp, out, vec);
    };
    if (!a_in) pack(ta, A, lda, m, Ap);
    if (!b_in) pack(!tb, B, ldb, n, Bp);
    const char* Ak = (const char*)(a_in ? A : Ap);
    const char* Bk = (const char*)(b_in ? B : Bp);
    const i64 ldka = 2 * (a_in ? lda : Kp), ldkb = 2 * (b_in ? ldb : Kp);
    const int vec = int(ldc % 4 == 0 && (reinterpret_cast<uintptr_t>(C) & 7) == 0);
    const float aw = float(ah), bw = float(bh);
    const int beta0 = int(bh == _Float16(0));
#define OXI_HGEMM(BM, BN, WM, WN)                                                                                     \
    do {                                                                                                              \
        const int tm = int(cdiv(m, BM)), tn = int(cdiv(n, BN));                                                       \
        hipLaunchKernelGGL((hgemm_kernel<BM, BN, WM, WN>), dim3(unsigned(tm) * unsigned(tn)), dim3(64 * WM * WN), 0,  \
                           s, m, n, Kp, aw, bw, beta0, Ak, ldka, Bk, ldkb, C, ldc, tm, tn, vec);                      \
    } while (0)
    // Rounds over the chip (one 256 x 256 tile a CU, two 128 x 128): a round of
    // the large tile takes 1.56 times one of the other (K = 4096: 131 and
    // 84 us), so it is taken where it needs that many fewer rounds (5000^3
    // 333 us against 393, 4096^3 140 against 177; but 2500^3 96 against 69).
    // Products of fewer than 192 128 x 128 tiles take 64 x 64 ones (1000^3:
    // 18.5 us against 27; 512 x 512 x 8192: 54 against 95).
    const i64 t256 = cdiv(m, 256) * cdiv(n, 256), t128 = cdiv(m, 128) * cdiv(n, 128);
    if (t128 < 192) OXI_HGEMM(64, 64, 2, 2);
    else if (156 * cdiv(t256, 256) <= 100 * cdiv(t128, 512)) OXI_HGEMM(256, 256, 2, 4);
    else OXI_HGEMM(128, 128, 2, 2);
#undef OXI_HGEMM
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return oxi_set_error(h, OXI_ERR_HIP, "hgemm launch: %s", hipGetErrorString(e));
    return OXI_OK;
}
