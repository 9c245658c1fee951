// Panel leaf kernel template (the algorithm is described in panel.hip);
// included by panel.hip (FP64) and panel32.hip (FP32, the working precision
// of the mixed-precision LU).
#pragma once
#include "oxi_internal.hpp"

#include <utility>
#include <type_traits>

namespace {

typedef unsigned long long u64;

__device__ __forceinline__ double fma_t(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ __forceinline__ float fma_t(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

__device__ __forceinline__ void put_agent(double* p, double v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ double get_agent(const double* p) {
    return __hip_atomic_load(const_cast<double*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ u64 bits(double v) { return __builtin_bit_cast(u64, v); }
__device__ __forceinline__ double from_bits(u64 v) { return __builtin_bit_cast(double, v); }
// field f's share of a record's checksum, keyed by the tag (tournament leaf)
__device__ __forceinline__ u64 rec_term(u64 b, u64 tag, int f) {
    return (b ^ (tag * 0x9E3779B97F4A7C15ull + u64(f + 1) * 0xD1B54A32D192ED03ull)) * 0x94D049BB133111EBull;
}
__device__ __forceinline__ u64 readlane64(u64 x, int l) {
    const unsigned lo = __builtin_amdgcn_readlane(unsigned(x), l), hi = __builtin_amdgcn_readlane(unsigned(x >> 32), l);
    return (u64(hi) << 32) | lo;
}
__device__ __forceinline__ int first_lane(u64 m) { return int(__builtin_ctzll(m)); }

// ---------------------------------------------------------------------------
// Pivot keys.  The search compares the high words of |value| (for FP32 the
// whole |value|) as integers, which order like the values; equal high words
// (rare) are settled by the low word and then by the position.  Semantics of
// the reference's strict '>' scan from the diagonal down: NaN in the diagonal
// position wins (nothing compares greater), NaN elsewhere never wins.
// ---------------------------------------------------------------------------
constexpr int KEY_NONE = -2;             // no candidate
__device__ __forceinline__ unsigned word_hi(double v) { return unsigned(bits(v) >> 32); }
__device__ __forceinline__ unsigned word_lo(double v) { return unsigned(bits(v)); }
__device__ __forceinline__ unsigned word_hi(float v) { return __builtin_bit_cast(unsigned, v); }
__device__ __forceinline__ unsigned word_lo(float) { return 0u; }
template <typename T> __device__ __forceinline__ T from_words(unsigned lo, unsigned hi);
template <> __device__ __forceinline__ double from_words<double>(unsigned lo, unsigned hi) {
    return from_bits((u64(hi) << 32) | lo);
}
template <> __device__ __forceinline__ float from_words<float>(unsigned, unsigned hi) {
    return __builtin_bit_cast(float, hi);
}
template <typename T> constexpr int KEY_INF = sizeof(T) == 8 ? 0x7ff00000 : 0x7f800000;
template <typename T>
__device__ __forceinline__ int pivot_key(T v, bool diag) {
    const int k = int(word_hi(v) & 0x7fffffffu);
    return v != v ? (diag ? KEY_INF<T> : -1) : k;
}
template <typename T>
__device__ __forceinline__ unsigned pivot_key_lo(T v) { return v != v ? 0u : word_lo(v); }
// exponent all ones (infinity or NaN)
template <typename T>
__device__ __forceinline__ bool non_finite(T v) { return (word_hi(v) & unsigned(KEY_INF<T>)) == unsigned(KEY_INF<T>); }

template <int CTRL, int ROWM = 0xf>
__device__ __forceinline__ int dpp_imax(int x) {
    // lanes whose source is outside the row (or masked off) keep their own
    // value; with the maximum's identity as the old value it is one instruction
    return max(x, __builtin_amdgcn_update_dpp(-0x7fffffff - 1, x, CTRL, ROWM, 0xf, false));
}
// maximum over the 64 lanes of a wave, in every lane: inclusive prefix maxima
// inside each row of 16, then across rows to lane 63
__device__ __forceinline__ int wave_imax(int x) {
    x = dpp_imax<0x111>(x);         // row_shr:1
    x = dpp_imax<0x112>(x);         // row_shr:2
    x = dpp_imax<0x114>(x);         // row_shr:4
    x = dpp_imax<0x118>(x);         // row_shr:8
    x = dpp_imax<0x142, 0xa>(x);    // row_bcast:15 into rows 1, 3
    x = dpp_imax<0x143, 0xc>(x);    // row_bcast:31 into rows 2, 3
    return __builtin_amdgcn_readlane(x, 63);
}
// The lane, among those with `tie` set, whose (low word, position) wins: the
// largest low word, then the lowest position (uniform; tie != 0).
__device__ __forceinline__ int settle_tie(u64 tie, unsigned lo, int pos) {
    int best = first_lane(tie);
    unsigned blo = __builtin_amdgcn_readlane(lo, best);
    int bpos = __builtin_amdgcn_readlane(pos, best);
    for (tie &= tie - 1; tie; tie &= tie - 1) {
        const int l = first_lane(tie);
        const unsigned l_lo = __builtin_amdgcn_readlane(lo, l);
        const int l_pos = __builtin_amdgcn_readlane(pos, l);
        if (l_lo > blo || (l_lo == blo && l_pos < bpos)) { best = l; blo = l_lo; bpos = l_pos; }
    }
    return best;
}
template <typename T>
__device__ __forceinline__ T readlane_t(T v, int l) {
    if constexpr (sizeof(T) == 8) return from_bits(readlane64(bits(v), l));
    else return __builtin_bit_cast(T, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), l));
}

// x of lane N of each row of 16 lanes, in every lane of the row
template <int N> __device__ __forceinline__ double row_bcast(double x) {
    return __builtin_amdgcn_update_dpp(0.0, x, 0x150 + N, 0xf, 0xf, true);   // row_newbcast:N
}
template <int N> __device__ __forceinline__ float row_bcast(float x) {
    return __builtin_amdgcn_update_dpp(0.0f, x, 0x150 + N, 0xf, 0xf, true);
}
// lane i + 1's x in lane i of each row of 16 lanes (lane 15: zero)
__device__ __forceinline__ float row_shl1(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x101, 0xf, 0xf, true));
}
__device__ __forceinline__ double row_shl1(double x) {
    const u64 b = bits(x);
    const unsigned lo = unsigned(__builtin_amdgcn_update_dpp(0, int(unsigned(b)), 0x101, 0xf, 0xf, true));
    const unsigned hi = unsigned(__builtin_amdgcn_update_dpp(0, int(unsigned(b >> 32)), 0x101, 0xf, 0xf, true));
    return from_bits((u64(hi) << 32) | lo);
}
// d = c - a * b with a destination of its own: the rotated update would else
// become the two-operand form and a move per register
__device__ __forceinline__ double nfma_to(double a, double b, double c) {
    double d;
    asm("v_fma_f64 %0, -%1, %2, %3" : "=v"(d) : "v"(a), "v"(b), "v"(c));
    return d;
}
__device__ __forceinline__ float nfma_to(float a, float b, float c) {
    float d;
    asm("v_fma_f32 %0, -%1, %2, %3" : "=v"(d) : "v"(a), "v"(b), "v"(c));
    return d;
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (N > 0) {
        static_for<N - 1>(f);
        f(std::integral_constant<int, N - 1>{});
    }
}

// ---------------------------------------------------------------------------
// Cross-workgroup exchange of one pivot column: tagged words.
//
// Every workgroup publishes one record per column: its best candidate row, as
// eight-byte words { 32 data bits, 32-bit tag }, word 2c the low half of
// value c and word 2c + 1 the high half, stored by the 64 lanes of one wave
// in one instruction, and a header of six words in a 128-byte line of its
// own: values 0 and 1 again and the row's position.  (Headers that share a
// line cost up to 0.35 us an exchange at 32 workgroups: the writes of
// different XCDs to one line follow one another.)  Everyone polls the headers
// only; the winner's row is fetched while the multipliers and the next
// candidates are computed.  An eight-byte store is seen whole, so a word
// whose tag is the column's carries the column's data whatever the order in
// which the stores land: no checksum and no fence.  Tags are unique over
// everything that the exchange buffer has held since it was last cleared
// (getrf.hip).  The data goes through device-scope (agent) relaxed stores and
// loads, which are coherent across XCDs without the L2 write-back /
// invalidate that an agent-scope release / acquire pair costs.
// ---------------------------------------------------------------------------
typedef unsigned uint4v __attribute__((ext_vector_type(4)));
constexpr int NO_POS = 0x7fffffff;       // a header's position when the workgroup has no candidate
// Three device-scope 16-byte loads (two words each), issued back to back and
// waited for once.  Relaxed atomic loads written in C++ are issued one at a
// time, each waited for before the next.
__device__ __forceinline__ void load_words3(const u64* p0, const u64* p1, const u64* p2, uint4v& r0, uint4v& r1,
                                            uint4v& r2) {
    asm volatile(
        "global_load_dwordx4 %0, %3, off sc1\n\t"
        "global_load_dwordx4 %1, %4, off sc1\n\t"
        "global_load_dwordx4 %2, %5, off sc1\n\t"
        "s_waitcnt vmcnt(0)"
        : "=&v"(r0), "=&v"(r1), "=&v"(r2) : "v"(p0), "v"(p1), "v"(p2) : "memory");
}
// The same load for one that the compiler waits for where it is used.
__device__ __forceinline__ uint4v load_words_ahead(__amdgpu_buffer_rsrc_t r, unsigned off_bytes) {
    return __builtin_bit_cast(uint4v, __builtin_amdgcn_raw_buffer_load_b128(r, int(off_bytes), 0, 16));   // sc1
}
// A workgroup barrier that orders LDS only: __syncthreads would also wait for
// the record's stores to be acknowledged.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// ---------------------------------------------------------------------------
// A leaf's interchanges on the other columns of the enclosing panel,
// [x_lo, c0) and [c0+w, x_hi), by the nwg workgroups of 256 threads of a grid
// (this one: wg).  Applying a leaf's interchanges to the rest of its panel at
// once gives the same columns as the getrf2 recursion, which applies them
// level by level: a left subtree's multipliers are not read again once its
// right sibling has started, and the right sibling's columns receive them
// before any update reads them.
//
// pi: lane i < w holds step i's pivot position relative to c0, -1 beyond, in
// every wave.  The interchanges move the contents of 2W slots: slot i < w is
// position i, slot W + i the pivot position of step i when it lies below the
// leaf's w rows and i is its first step.  Every lane follows its slots
// backwards through the transpositions (step i exchanges slot i with slot
// sb_i), so the steps carry no dependence between lanes: one readlane and two
// selects per slot and step.  A wave moves 32 slots of 64 columns (a lane per
// column): the two waves of a group of columns load everything before any
// of them stores (a wait and a barrier).  Loads are issued without branches: a
// slot that does not move reads position 0, a lane outside the columns reads
// column c0 (both in bounds), and only moving slots are stored.  Lane s
// computes its slots' row offsets once; the loops only read them back.
// ---------------------------------------------------------------------------
template <typename T>
__device__ __forceinline__ void other_columns(T* Wm, i64 ldw, i64 c0, int w, int pi, i64 x_lo, i64 x_hi, int wg,
                                              int nwg) {
    constexpr int W = OXI_LEAF_W;
    const int groups_l = int((c0 - x_lo + 63) / 64), groups = groups_l + int((x_hi - c0 - w + 63) / 64);
    static_assert(2 * W == 64, "a slot per lane");
    constexpr int GW = 2, GPW = 2;                 // waves per group of columns, groups per workgroup
    if (wg * GPW >= groups) return;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
    int first = lane;
#pragma unroll 8
    for (int i = 0; i < W; ++i) {
        const int q = __builtin_amdgcn_readlane(pi, i);
        if (i < first && q == pi) first = i;
    }
    const int sbv = lane >= w ? lane : pi < w ? pi : W + first;   // the slot that step `lane` exchanges with its own
    const int outp = lane < w && pi >= w && first == lane ? pi : -1;
    int x = lane;
#pragma unroll 8
    for (int i = W - 1; i >= 0; --i) {
        const int sb = __builtin_amdgcn_readlane(sbv, i);
        x = x == i ? sb : x == sb ? i : x;
    }
    const int out_of = __shfl(outp, lane & (W - 1)), pi_of = __shfl(pi, x & (W - 1));   // of slots W + i
    const int to = lane >= W ? out_of : lane < w ? lane : -1, from = x < W ? x : pi_of;
    const bool moves = to >= 0 && x != lane;
    const u64 os = u64((c0 + (moves ? from : 0)) * ldw), od = u64((c0 + (moves ? to : 0)) * ldw);
    const int s0 = 32 * (wave % GW);               // this wave's slots s0 .. s0 + 31
    const u64 moving = __ballot(moves) >> s0;
#pragma unroll 1
    for (int g0 = wg * GPW; g0 < groups; g0 += nwg * GPW) {
        const int g = g0 + wave / GW;
        const bool left = g < groups_l;
        const i64 xc = left ? x_lo + i64(g) * 64 + lane : c0 + w + i64(g - groups_l) * 64 + lane;
        const bool ok = g < groups && (left ? xc < c0 : xc < x_hi);
        const i64 xr = ok ? xc : c0;
        T v[32];
#pragma unroll
        for (int k = 0; k < 32; ++k) v[k] = Wm[i64(readlane64(os, s0 + k)) + xr];
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
#pragma unroll
        for (int k = 0; k < 32; ++k)
            if ((moving >> k) & 1) {
                const i64 to_row = i64(readlane64(od, s0 + k));
                if (ok) Wm[to_row + xc] = v[k];
            }
    }
}

// ---------------------------------------------------------------------------
// The leaf kernel (up to W = 32 columns).  Thread t of workgroup p holds the rows
// that start at positions p*R + s*256 + t (s < RPT) in registers, and they stay there: an
// interchange only changes positions (pos[s]; a row that became the pivot of
// step j is retired to position j, pos[s] = ~j).  The registers of a row
// rotate by one per column: at column j register c holds column j + c, so the
// pivot column is always register 0, the rank-1 update is the same W - 1 FMAs at
// every step (v[c] <- v[c+1] - l u[c+1]), and every register index is a
// compile-time constant in a rolled loop; the multiplier enters at register
// W - 1.  After W rotations register c holds column c again, multipliers and U values
// alike, and every row is stored once, at its final position: no store and no
// interchange inside the column loop.  (u is zero past the row's live
// columns, so the multipliers of earlier columns pass through the update
// unchanged; from the first step that meets an infinity or NaN, or a zero
// pivot, the update takes a select per value.)
//
// The exchange of column j+1 is overlapped with the update of column j: once
// the multipliers of column j are known, every row computes only its next
// column, the candidates for column j+1 are chosen from those values, the
// chosen row is updated on its own (one column per lane) and published, and
// only then do all rows take the full update while the records travel.  One
// barrier per column, for the comparison of the waves' candidates: every wave
// reads all the headers itself and picks the winner in registers.
//
// WGS 1: one workgroup holds all the rows; the chosen row goes to the other
// waves through LDS.
//
// At the end the leaf applies its interchanges to the other columns of the
// panel (as a kernel of its own that took 5 to 9 us a leaf: n = 2000 5.30 ->
// 5.11 ms, 16384 84.7 -> 83.7 ms).
//
// A column is a chain of dependent steps in one wave per SIMD, bound by
// instruction and LDS latency plus one exchange between workgroups (1.1 us
// alone for 32 of them).  Measured per FP64 column, 32 columns, launch
// included: 1.23 us at 256 rows, 1.62 at 512 (one workgroup), 1.91 at 2048, 2.2
// at 8192, 2.4 at 16384 rows.  Rows that move between threads at every
// interchange, 64-bit keys, checksummed records and multipliers stored column
// by column took 1.9, 3.4 (2048), 4.1 (8192) and 4.6 us (16384) inside an LU.
// At 16384 rows a column's critical path is 0.1 us to the winner, 0.1 to the
// multipliers, 0.2-0.3 to the wave's candidate, 0.2 across the barrier, 0.2 to
// the header, then the exchange; the row's trip through LDS and the update
// run in the exchange's shadow.
// ---------------------------------------------------------------------------
template <typename T, int RPT, int WGS>
__global__ __launch_bounds__(256) void lu_leaf_kernel(LeafArgs a) {
    constexpr int W = OXI_LEAF_W, LT = 256, NWV = LT / 64, NB = W / 16;   // NB: values of a row per lane of its spread form
    static_assert(W == 32, "record layout");
    constexpr bool MULTI = WGS != 1;                  // WGS: 1, 64 or OXI_LEAF_MAX_P workgroups at most
    const unsigned spin_limit = a.spins;              // bound of every wait
    __shared__ __align__(16) int4 wcand[2][NWV];                   // each wave's candidate: key, low word, position; failed
    __shared__ __align__(16) T raw[W];                             // the chosen row before the pending update
    __shared__ T raw_l;                                            // !MULTI: its multiplier
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int p = blockIdx.x, P = a.P;
    const int w = a.w;
    const int R = LT * RPT;

    T v[RPT][W];
    T* Wm = (T*)a.Wm;
    int pos[RPT];
#pragma unroll
    for (int s = 0; s < RPT; ++s) {
        const int lr = p * R + s * LT + t;
        const bool ok = lr < a.mrows;
        pos[s] = ok ? lr : -0x40000000;               // no row: never a candidate, never stored
        const T* row = Wm + a.c0 + (a.c0 + (ok ? lr : 0)) * a.ldw;
        if (w == W) {   // a full leaf: wide loads (a thread without a row reads the first one)
#pragma unroll
            for (int c = 0; c < W; ++c) v[s][c] = row[c];
        } else {
#pragma unroll
            for (int c = 0; c < W; ++c) v[s][c] = c < w ? row[c] : T(0);
        }
    }
    // a wait of an earlier leaf timed out: the factorization is already
    // reported as failed, leave at once.  The flag is read with the rows (one
    // memory round trip for both; the rows lie inside the panel either way)
    // and nothing has been stored before the test.
    const int failed = __hip_atomic_load(a.flags, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    // the rows have arrived before the loop (otherwise the first use inside a
    // conditional block leaves a wait on vector memory at the top of every column)
    __builtin_amdgcn_s_waitcnt(0);
    if (failed != 0) return;

    // the winner of the current column, as every wave knows it
    T d = T(0), u1 = T(0);                  // values 0 and 1 of the pivot row
    int piv = 0;                            // its position
    T rv[NB] = {};                          // its values 16 b + (lane & 15) in every row of 16 lanes
    T uu = T(0);                            // MULTI: its value that the lane publishing value c needs, c + 1
    unsigned row_off = 0, row_tag = 0;      // MULTI: the row's place in the exchange buffer, its tag
    // the lane's column of a published row: two lanes per column (low and high half)
    const int pc = lane >> 1;
    const unsigned oa = (lane & 15) * 16, ou = min(pc + 1, W - 1) * 16;
    const __amdgpu_buffer_rsrc_t pub_rsrc =
        __builtin_amdgcn_make_buffer_rsrc((void*)a.pub, 0, int(OXI_LEAF_PUB * 8), 0x00027000);
    bool timed_out = false;                 // this wave's last wait failed

    // ---- MULTI: the winner's row from the words fetched ahead; fetched again
    // (bounded) while a word is not the column's yet
    struct Ahead { uint4v b[NB], u; };
    auto row_ahead = [&]() __attribute__((always_inline)) -> Ahead {
        Ahead x;
#pragma unroll
        for (int b = 0; b < NB; ++b) x.b[b] = load_words_ahead(pub_rsrc, row_off + oa + 256 * b);
        x.u = load_words_ahead(pub_rsrc, row_off + ou);
        return x;
    };
    auto row_arrives = [&](Ahead x) __attribute__((always_inline)) {
        const unsigned tag = row_tag;
        unsigned spins = 0;
#pragma unroll 1
        while (true) {
            unsigned diff = (x.u.y ^ tag) | (x.u.w ^ tag);
#pragma unroll
            for (int b = 0; b < NB; ++b) diff |= (x.b[b].y ^ tag) | (x.b[b].w ^ tag);
            asm("" : "+v"(diff));   // one compare, not six and a chain of scalar ors
            if (__builtin_expect(__ballot(diff != 0) == 0, 1)) break;
            if (++spins > spin_limit) { timed_out = true; break; }   // uniform per wave
            const char* row = (const char*)a.pub + row_off;
            load_words3((const u64*)(row + oa), (const u64*)(row + oa + 256), (const u64*)(row + ou), x.b[0], x.b[1], x.u);
        }
#pragma unroll
        for (int b = 0; b < NB; ++b) rv[b] = from_words<T>(x.b[b].x, x.b[b].z);
        uu = from_words<T>(x.u.x, x.u.z);
    };

    // ---- the candidate of column jn and its publication.  x[s]: row s's
    // value in column jn (register REG).  PEND: the registers still await the
    // update of column jn - 1 (multipliers l, the row in ahead); only
    // the chosen row is then updated here.  False when a wave of the
    // workgroup timed out.  Straight-line code but for ties: a taken branch
    // costs about as much as ten dependent instructions.
    auto select_publish = [&](int jn, const T (&x)[RPT], auto pend_c, const T (&l)[RPT], bool upd,
                              Ahead ahead) __attribute__((always_inline)) -> bool {
        constexpr bool PEND = decltype(pend_c)::value;
        constexpr int REG = PEND ? 1 : 0;
        const int parn = jn & 1;
        // this lane's best row
        int k[RPT], kb = KEY_NONE - 1, sb = 0;
        bool tie = false;
#pragma unroll
        for (int s = 0; s < RPT; ++s) {
            k[s] = pos[s] >= 0 ? pivot_key(x[s], pos[s] == jn) : KEY_NONE;
            tie = k[s] > kb ? false : tie || k[s] == kb;
            sb = k[s] > kb ? s : sb;
            kb = max(kb, k[s]);
        }
        const int m = wave_imax(kb);
        u64 b = __ballot(kb == m);
        int wl = first_lane(b);
        const bool none = m == KEY_NONE;
        if (__builtin_expect(!none && ((b & (b - 1)) != 0 || (RPT > 1 && (__ballot(tie) & b) != 0)), 0)) {
            // equal high words: low word, then position
            unsigned lob = 0;
            int pb = NO_POS;
#pragma unroll
            for (int s = 0; s < RPT; ++s) {
                const unsigned lo_s = pivot_key_lo(x[s]);
                const bool win = k[s] == m && (pb == NO_POS || lo_s > lob || (lo_s == lob && pos[s] < pb));
                sb = win ? s : sb; lob = win ? lo_s : lob; pb = win ? pos[s] : pb;
            }
            wl = settle_tie(b, lob, pb);
        }
        T xs = x[0], ls = l[0], ys = REG + 1 < W ? v[0][REG + 1] : T(0);
        int ps = pos[0];
#pragma unroll
        for (int s = 1; s < RPT; ++s) {
            xs = sb == s ? x[s] : xs;
            ls = sb == s ? l[s] : ls;
            ps = sb == s ? pos[s] : ps;
            if (REG + 1 < W) ys = sb == s ? v[s][REG + 1] : ys;
        }
        const int pos_w = none ? NO_POS : __builtin_amdgcn_readlane(ps, wl);
        if (lane == wl) wcand[parn][wave] = int4{m, int(pivot_key_lo(xs)), none ? NO_POS : ps, int(timed_out)};
        const int ws = RPT > 1 ? __builtin_amdgcn_readlane(sb, wl) : 0;
        const T lw = readlane_t(ls, wl);
        // the chosen row from its lane's registers to LDS, eight values at a
        // time while any of them is live (a 16-byte LDS store takes about as
        // long for one lane as for 64)
        auto row_out = [&](T* dst) __attribute__((always_inline)) {
#pragma unroll
            for (int s = 0; s < RPT; ++s)
                if (ws == s && lane == wl) {
                    T* o = (T*)__builtin_assume_aligned(dst, 16);
#pragma unroll
                    for (int g = 0; g < W; g += 8)
                        if (g < W - jn) {
#pragma unroll
                            for (int c = g; c < g + 8; ++c) o[c] = REG + c < W ? v[s][REG + c] : T(0);
                        }
                    // keeps the slots' stores apart: merged into stores of a
                    // chosen row they would put the rows in scratch memory
                    asm volatile("; slot %0" ::"n"(s));
                }
        };
        lds_barrier();
        const int4 e = wcand[parn][lane & (NWV - 1)];
        int em = dpp_imax<0xB1>(e.x);                   // quad_perm [1,0,3,2]
        em = dpp_imax<0x4E>(em);                        // quad_perm [2,3,0,1]
        const u64 eb = __ballot(e.x == em) & ((1ull << NWV) - 1);
        int ww = first_lane(eb);
        if (__builtin_expect((eb & (eb - 1)) != 0, 0)) ww = settle_tie(eb, unsigned(e.y), e.z);
        if constexpr (!MULTI) {
            // the chosen row goes to every wave, which updates it itself: the
            // new row's spread values from the old one's, one value further
            // (every wave's candidate in LDS before the first barrier, and no
            // second one, takes longer: the stores of the four waves share
            // the LDS)
            piv = __builtin_amdgcn_readlane(e.z, ww);
            if (wave == ww) {
                row_out(raw);
                if (lane == 0) raw_l = lw;
            }
            lds_barrier();
            const int i = lane & 15;
            T nv[NB];
#pragma unroll
            for (int b = 0; b < NB; ++b) nv[b] = raw[16 * b + i];
            if (PEND && upd) {
                const T wl_ = raw_l;
                T sh[NB];
#pragma unroll
                for (int b = 0; b < NB; ++b) {
                    const T next = b + 1 < NB ? row_bcast<0>(rv[b + 1 < NB ? b + 1 : 0]) : T(0);
                    const T sl = row_shl1(rv[b]);
                    sh[b] = i == 15 ? next : sl;
                }
#pragma unroll
                for (int b = 0; b < NB; ++b) nv[b] = fma_t(-wl_, sh[b], nv[b]);
            }
#pragma unroll
            for (int b = 0; b < NB; ++b) rv[b] = 16 * b + i < W - jn ? nv[b] : T(0);
            d = readlane_t(rv[0], 0);
            u1 = readlane_t(rv[0], 1);
            return true;
        } else {
            if (PEND) row_arrives(ahead);
            if (wave == ww && jn < w) {
                // this wave holds the workgroup's candidate: the header first,
                // from its lane's registers (value 1 is column jn + 1 updated)
                const u64 tag = u64(a.tag + unsigned(jn)) << 32;
                if (PEND && upd) ys = fma_t(-ls, row_bcast<2>(rv[0]), ys);
                const T h0 = none ? T(0) : readlane_t(xs, wl), h1 = none || jn + 1 >= W ? T(0) : readlane_t(ys, wl);
                const unsigned hd = lane == 0 ? word_lo(h0) : lane == 1 ? word_hi(h0) : lane == 2 ? word_lo(h1)
                                  : lane == 3 ? word_hi(h1) : unsigned(pos_w);
                if (lane < 6)
                    __hip_atomic_store(a.pub + size_t(w) * P * OXI_PUB_STRIDE + (size_t(jn) * P + p) * OXI_PUB_HDR + lane,
                                       tag | hd, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                // then the whole row
                row_out(raw);
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");   // the lane's LDS writes before the reads below
                __builtin_amdgcn_wave_barrier();
                T r = raw[pc];
                if (PEND && upd) r = fma_t(-lw, uu, r);
                if (none || pc >= W - jn) r = T(0);
                u64* row = a.pub + (size_t(jn) * P + p) * OXI_PUB_STRIDE;
                __hip_atomic_store(row + lane, tag | ((lane & 1) ? word_hi(r) : word_lo(r)), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
            }
            if (__builtin_expect(__ballot(e.w != 0) != 0, 0)) {   // a wave's wait timed out (the same in every wave)
                if (t == 0) __hip_atomic_store(a.flags, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                return false;
            }
            return true;
        }
    };

    // ---- MULTI: the headers of column jn (lane q: workgroup q), polled by
    // every wave until all are there; the winner is found in registers
    auto poll = [&](int jn) __attribute__((always_inline)) {
        const unsigned tag = a.tag + unsigned(jn);
        const u64* heads = a.pub + size_t(w) * P * OXI_PUB_STRIDE + size_t(jn) * P * OXI_PUB_HDR;
        unsigned spins = 0;
        auto header = [&](int q, T& v0, T& v1, int& hpos) __attribute__((always_inline)) {
            const u64* hq = heads + q * OXI_PUB_HDR;
            uint4v x0, x1, x2;
#pragma unroll 1
            while (true) {
                load_words3(hq, hq + 2, hq + 4, x0, x1, x2);
                unsigned diff = (x0.y ^ tag) | (x0.w ^ tag) | (x1.y ^ tag) | (x1.w ^ tag) | (x2.y ^ tag) | (x2.w ^ tag);
                asm("" : "+v"(diff));
                if (__builtin_expect(__ballot(diff != 0) == 0, 1)) break;
                if (++spins > spin_limit) break;   // uniform per wave
            }
            v0 = from_words<T>(x0.x, x0.z);
            v1 = from_words<T>(x1.x, x1.z);
            hpos = int(x2.x);
        };
        int q = min(lane, P - 1), hp;
        T dl, ul;
        header(q, dl, ul, hp);
        int key = lane < P && hp != NO_POS ? pivot_key(dl, hp == jn) : KEY_NONE;
        if constexpr (WGS > 64) {   // two records a lane
            const int q2 = min(lane + 64, P - 1);
            T d2, u2;
            int p2;
            header(q2, d2, u2, p2);
            const int k2 = lane + 64 < P && p2 != NO_POS ? pivot_key(d2, p2 == jn) : KEY_NONE;
            const unsigned la = pivot_key_lo(dl), lb = pivot_key_lo(d2);
            if (k2 > key || (k2 == key && (lb > la || (lb == la && p2 < hp)))) {
                key = k2; hp = p2; q = q2; dl = d2; ul = u2;
            }
        }
        const int m = wave_imax(key);
        const u64 b = __ballot(key == m);
        int gl = first_lane(b);
        if (__builtin_expect((b & (b - 1)) != 0, 0)) gl = settle_tie(b, pivot_key_lo(dl), hp);
        row_off = unsigned(jn * P + __builtin_amdgcn_readlane(q, gl)) * (OXI_PUB_STRIDE * 8);
        row_tag = tag;
        d = readlane_t(dl, gl);
        u1 = readlane_t(ul, gl);
        piv = __builtin_amdgcn_readlane(hp, gl);
        if (spins > spin_limit) {   // what came is not this column's: keep positions in range until the leaf ends
            timed_out = true;
            piv = jn;
        }
    };

    // column 0: the registers as loaded
    {
        T x0[RPT], l0[RPT];
#pragma unroll
        for (int s = 0; s < RPT; ++s) { x0[s] = v[s][0]; l0[s] = T(0); }
        if (!select_publish(0, x0, std::false_type{}, l0, false, {})) return;
        if constexpr (MULTI) poll(0);
    }

    int my_piv = -1, first_zero = -1;   // lane j holds step j's pivot position
    // state of column j between its record's publication and its update
    T l[RPT], lin[RPT];   // the multiplier for the update (0: row not updated), the value entering register W - 1
    T ru[NB] = {};            // the pivot row's values
    bool updates = false;     // column j has a pivot
    bool odd = false;         // the update needs its selects: an infinity, a NaN or a zero pivot

    // The multipliers of column j, then column j+1's values, candidate and
    // record (past the last column nothing is published).  False on timeout.
    auto head = [&](int j) __attribute__((always_inline)) -> bool {
        // the winner's row starts on its way
        Ahead ahead = {};
        if constexpr (MULTI) ahead = row_ahead();
        const bool upd = d != T(0);
        my_piv = lane == j ? piv : my_piv;
        first_zero = !upd && first_zero < 0 ? j : first_zero;
        updates = upd;
        bool strange = !upd || non_finite(d);
        T x[RPT];
#pragma unroll
        for (int s = 0; s < RPT; ++s) {
            // interchange: positions only
            pos[s] = pos[s] == piv ? ~j : pos[s] == j ? piv : pos[s];
            const T qv = v[s][0] / d;
            const bool act = pos[s] >= 0 && upd;   // a zero pivot leaves the column as it is
            l[s] = act ? qv : T(0);
            lin[s] = act ? qv : v[s][0];
            x[s] = upd ? fma_t(-l[s], u1, v[s][1]) : v[s][1];
            strange |= non_finite(l[s]);
        }
        // !MULTI: select_publish makes the next column's row
#pragma unroll
        for (int b = 0; b < NB; ++b) ru[b] = rv[b];
        if (!select_publish(j + 1, x, std::true_type{}, l, upd, ahead)) return false;
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            if constexpr (MULTI) ru[b] = rv[b];   // it arrived in select_publish
            strange |= non_finite(ru[b]);
        }
        odd = __ballot(strange) != 0;
        return true;
    };
    if (!head(0)) return;

    // Per turn: the rank-1 update of column j with the rotation, while the
    // records of column j + 1 travel, then those records and the head of
    // column j + 1.
    int j = 0;
#pragma unroll 1
    for (; j < w && !odd; ++j) {
        static_for<W / 4>([&](auto g_c) __attribute__((always_inline)) {
            // four broadcast values at a time (all of them ahead would not fit
            // in the registers)
            constexpr int G = 4 * decltype(g_c)::value;
            T u[4];
            static_for<4>([&](auto c_c) __attribute__((always_inline)) {
                constexpr int C = G + decltype(c_c)::value;
                if constexpr (C > 0) u[C - G] = row_bcast<C & 15>(ru[C / 16]);
            });
            __builtin_amdgcn_sched_barrier(0);
            static_for<4>([&](auto c_c) __attribute__((always_inline)) {
                constexpr int C = G + decltype(c_c)::value;
                if constexpr (C > 0) {
#pragma unroll
                    for (int s = 0; s < RPT; ++s) v[s][C - 1] = nfma_to(l[s], u[C - G], v[s][C]);
                }
            });
            __builtin_amdgcn_sched_barrier(0);
        });
#pragma unroll
        for (int s = 0; s < RPT; ++s) v[s][W - 1] = lin[s];
        if (j + 1 < w) {
            if constexpr (MULTI) poll(j + 1);
            if (!head(j + 1)) return;
        }
    }
    // the same from the first odd column on, the update with a select per value
#pragma unroll 1
    for (; j < w; ++j) {
        static_for<W - 1>([&](auto c_c) __attribute__((always_inline)) {
            constexpr int C = decltype(c_c)::value + 1;
            const T uc = row_bcast<C & 15>(ru[C / 16]);
#pragma unroll
            for (int s = 0; s < RPT; ++s) {
                const bool live = updates && pos[s] >= 0 && C < W - j;
                v[s][C - 1] = live ? fma_t(-l[s], uc, v[s][C]) : v[s][C];
            }
            if constexpr (C % 4 == 0) __builtin_amdgcn_sched_barrier(0);
        });
#pragma unroll
        for (int s = 0; s < RPT; ++s) v[s][W - 1] = lin[s];
        if (j + 1 < w) {
            if constexpr (MULTI) poll(j + 1);
            if (!head(j + 1)) return;
        }
    }
    // a narrower leaf completes the rotation
#pragma unroll 1
    for (int k = w; k < W; ++k) {
#pragma unroll
        for (int s = 0; s < RPT; ++s) {
            const T x = v[s][0];
#pragma unroll
            for (int c = 0; c + 1 < W; ++c) v[s][c] = v[s][c + 1];
            v[s][W - 1] = x;
        }
    }
    // every workgroup has its rows in registers once the first column's
    // records are complete: the rows go to their final positions
#pragma unroll
    for (int s = 0; s < RPT; ++s) {
        if (pos[s] < -W) continue;
        const int to = pos[s] >= 0 ? pos[s] : ~pos[s];
        T* row = Wm + a.c0 + (a.c0 + to) * a.ldw;
        if (w == W) {
#pragma unroll
            for (int c = 0; c < W; ++c) row[c] = v[s][c];
        } else {
#pragma unroll
            for (int c = 0; c < W; ++c)
                if (c < w) row[c] = v[s][c];
        }
    }
    if (timed_out && lane == 0) __hip_atomic_store(a.flags, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (p == 0 && wave == 0) {
        if (lane < w) a.ipiv[a.c0 + lane] = a.c0 + my_piv + 1;
        if (lane == 0 && first_zero >= 0 && *a.info == 0) *a.info = a.c0 + first_zero + 1;
    }
    // the interchanges on the rest of the panel: columns that no workgroup
    // has touched
    other_columns(Wm, a.ldw, a.c0, w, lane < w ? my_piv : -1, a.xlo, a.xhi, p, P);
}

// One leaf launch.  Up to as many workgroups as getrf keeps CUs free of the
// trailing update ask for LEAF_LDS bytes of LDS each, far more than they use, so
// that each gets one of those CUs to itself: beside a workgroup of the update
// (66 KB of LDS), whose waves compete for its SIMDs, a column took 3.9 us at 16384
// rows instead of 2.4.  More workgroups than that (above 16384 FP64 rows, 32768
// FP32 rows) have to share CUs with the update, which the LDS would not let
// them: the last would wait until both tiles of some CU end at once, and the
// rest for them (n = 20000 132 ms with it, 124 without, 24576 230 and 206,
// 33000 525 and 469; 17000 84.5 and 84.8).
constexpr unsigned LEAF_LDS = 96 * 1024;
template <typename K>
int launch_leaf(oxi_handle_t h, hipStream_t s, const LeafArgs& a, K kernel) {
    const hipError_t se = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, LEAF_LDS);
    if (se != hipSuccess) return oxi_set_error(h, OXI_ERR_HIP, "lu_leaf attribute: %s", hipGetErrorString(se));
    hipLaunchKernelGGL(kernel, dim3(unsigned(a.P)), dim3(256), a.P <= h->panel_cus ? LEAF_LDS : 0, s, a);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return oxi_set_error(h, OXI_ERR_HIP, "lu_leaf launch: %s", hipGetErrorString(e));
    return OXI_OK;
}

}  // namespace
