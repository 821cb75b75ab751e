// Band LDL^T factorization and solves on the device: the reference's skyline
// solver (skyfact/skysolve, solve.c:539-698) recast for the GPU.
//
// The matrix is taken in the reference's equation order, so the pivots D are
// those of the reference's active-column factorization (same matrix, same
// order, no pivoting) up to rounding; they drive the arc-length predictor sign
// and the psi switch exactly as ssd does (solve.c:612-621, main.c:2636-2642).
//
// Storage: the lower band (half-bandwidth b = max column height) in dense T x T
// tiles; tile row I holds tiles J = I-w .. I (w = ceil(b/T)), column-major.
// Factorization by tile tasks of column K (left-looking in one launch, or
// right-looking with a launch per kind of task):
//   diag : D_K and Linv_K = L_KK^{-1} of A_KK = L_KK D_K L_KK^T, in LDS
//   panel: L_IK = A_IK Linv_K^T D_K^{-1},            K < I <= K+w
//   update: A_IJ -= (L_IK D_K) L_JK^T,               K < J <= I <= K+w
// Solves: pipelined forward and backward sweeps, one workgroup per tile row or
// several per block of four, with Linv_I for the diagonal blocks and pivot
// scaling folded into the backward sweep.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "band.h"

namespace cb {
namespace {

constexpr int T = 64;
constexpr int TT = T * T;

template <class R, class KS = double>
__global__ void k_band_from_bsr(R* __restrict__ tiles, const KS* __restrict__ K,
                                const int32_t* __restrict__ rowptr, const int32_t* __restrict__ colidx,
                                const int32_t* __restrict__ eq, long nj, int bs, int w, int* __restrict__ bad) {
    long r = blockIdx.x * (long)blockDim.x + threadIdx.x;   // slot row
    if (r >= nj * bs) return;
    long A = r / bs;
    int p = int(r % bs);
    int32_t i = eq[r];
    if (i < 0) return;
    for (int32_t k = rowptr[A]; k < rowptr[A + 1]; ++k) {
        long B = colidx[k];
        for (int q = 0; q < bs; ++q) {
            int32_t j = eq[B * bs + q];
            if (j < 0 || j > i) continue;
            long I = i / T, J = j / T;
            if (I - J > w) { *bad = 2; continue; }
            tiles[(I * (w + 1) + (J - I + w)) * (long)TT + (j % T) * T + (i % T)] =
                R(K[(long)k * bs * bs + p * bs + q]);
        }
    }
}

template <class R>
__global__ void k_band_pad(R* __restrict__ tiles, long n, long nt, int w) {
    long i = n + blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i >= nt * T) return;
    long I = i / T;
    tiles[(I * (w + 1) + w) * (long)TT + (i % T) * T + (i % T)] = R(1);
}

// ---- factorization --------------------------------------------------------
// Tile tasks of column K:
//   D_K          D_K and Linv_K of tile (K,K)
//   P_{I,K}      L_IK = A_IK Linv_K^T D_K^{-1},            K < I <= K+m
//   U_{I,J,K}    A_IJ -= (L_IK D_K) L_JK^T,               K < J <= I <= K+m
// (m = min(w, nt-1-K)).  Two schedules run the same tile arithmetic:
//  - fused (default): one launch, k_band_factor, whose workgroups hand tiles
//    to each other through progress counters;
//  - split: three launches per column (diag, panels, updates), for timing
//    the tile tasks one by one.
// Tiles handed between workgroups of one launch are stored and loaded with
// system-scope coherent accesses (written through to memory, read past the
// XCD caches): a producer waits for its stores to complete (vmcnt 0) before
// it raises the counter, a consumer reads the data after it has seen it.
// Everything else crosses a launch boundary.
constexpr int NTH = 512;   // threads of every factorization workgroup (8 wavefronts)
constexpr int NWAVE = NTH / 64;

__device__ inline long tile_index(long I, long J, int w) { return I * (w + 1) + (J - I + w); }

template <bool CO, class R> __device__ __forceinline__ R cld(const R* p) {
    if constexpr (CO) return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    else return *p;
}
template <bool CO, class R> __device__ __forceinline__ void cst(R* p, R v) {
    if constexpr (CO) __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    else *p = v;
}

// Progress counters of a batch's models sit one per 256-byte line so that
// pollers of different counters do not share a memory channel.
constexpr long FLAG_STRIDE = 64;

__device__ __forceinline__ int peek(const int* c) {
    return __hip_atomic_load(c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// one thread: polls *c until it is at least target (or an error is raised
// anywhere); returns the value seen, below target on failure
__device__ inline int poll_count(const int* c, int target, long spin_limit, int* err) {
    for (long n = 0;; ++n) {
        const int v = peek(c);
        if (v >= target) return v;
        if (n >= spin_limit || ((n & 63) == 63 && (peek(err) & 1))) {
            atomicOr(err, 1);
            return v;
        }
        __builtin_amdgcn_s_sleep(1);
    }
}

// *c = value once every thread's stores have completed
__device__ inline void publish(int* c, int value) {
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (threadIdx.x == 0) __hip_atomic_store(c, value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// ---- workgroups that wait for each other ------------------------------------
// Kernels whose workgroups wait for each other give every workgroup a number
// when it starts, and it waits on lower numbers only.  blockIdx.x would do for
// a launch that has the GPU to itself.  Beside another one it would not: each
// XCD starts its eighth of a launch's workgroups in order, and the waiting
// workgroups of two launches could each fill the XCD that the other's next
// one needs.

// By count: all numbers below a workgroup's belong to workgroups that have
// started, so the lowest unfinished one can always go on, whatever else has
// the GPU.  counter[0] is zero before the launch.
__device__ __forceinline__ long start_by_count(int* counter) {
    __shared__ int number;
    if (threadIdx.x == 0) number = atomicAdd(counter, 1);
    __syncthreads();
    return __builtin_amdgcn_readfirstlane(number);
}

// blockIdx.x where that is safe: it spreads consecutive numbers over the XCDs
// and CUs, which counts do not (the atomics of one XCD land together).  A
// workgroup takes its own number once that is less than AHEAD past the count
// of the numbers taken.  While one XCD cannot start its workgroups, the other
// seven so take at most 7 AHEAD numbers past the lowest free one.  The rest
// of the workgroups hold back, and after PATIENCE polls (about 8 ms) take the
// lowest free number, as does one whose own number was taken like that.  A
// launch that has the GPU to itself holds back too, for some ten us at its
// start and while one XCD is behind the others: with a patience of 1024 polls
// a full matrix of 390 and 608 tile rows took 1.12 and 1.4 times as long to
// factor, from 4096 on no longer than by blockIdx.x.
// So some workgroup can go on as long as the GPU has room for 7 AHEAD
// workgroups of every such launch at once.
// Not for launches of many short workgroups: the block sweeps, whose helpers
// live for some ten us, take seven times as long (388 tiles below the
// diagonal).
// counter[0] is the count, counter[1 ..] the numbers taken, a bit each, zero
// before the launch.
constexpr int AHEAD = 8, PATIENCE = 1 << 13;
__device__ __forceinline__ long start_by_index(int* counter) {
    __shared__ int number;
    if (threadIdx.x == 0) {
        const int own = blockIdx.x, n = gridDim.x;
        auto take = [&](int i) { return !(atomicOr(&counter[1 + i / 32], 1 << i % 32) >> i % 32 & 1); };
        int got = -1;
        bool mine = true;
        for (int k = 0; got < 0; ++k) {
            if (mine && own < peek(counter) + AHEAD) {
                if (take(own)) got = own;
                mine = false;
            } else if (!mine || k >= PATIENCE) {
                // every other pass from a little below the count, where the lowest free number is
                for (int i = k & 1 ? 0 : max(0, (peek(counter) & ~31) - 256); got < 0 && i < n; ++i) {
                    if (i % 32 == 0 && peek(&counter[1 + i / 32]) == -1) i += 31;
                    else if (take(i)) got = i;
                }
            } else {
                __builtin_amdgcn_s_sleep(8);
            }
        }
        atomicAdd(counter, 1);
        number = got;
    }
    __syncthreads();
    return __builtin_amdgcn_readfirstlane(number);
}

__device__ __forceinline__ long start_number(int* counter, bool by_count) {
    return by_count ? start_by_count(counter) : start_by_index(counter);
}

__device__ __forceinline__ double lane_value(double x, int lane) {
    const unsigned long long u = __builtin_bit_cast(unsigned long long, x);
    const unsigned lo = __builtin_amdgcn_readlane(unsigned(u), lane);
    const unsigned hi = __builtin_amdgcn_readlane(unsigned(u >> 32), lane);
    return __builtin_bit_cast(double, (unsigned long long)hi << 32 | lo);
}

// threadIdx.x, opaque to the compiler: addresses formed from it are formed
// where they are used.  In a loop over columns they would all be hoisted out,
// and spilled.
__device__ __forceinline__ int thread_index() {
    int t = threadIdx.x;
    __asm__ volatile("" : "+v"(t));
    return t;
}

// ---- tile product C = X Y^T -------------------------------------------------
// Operands staged in LDS column-major: xs[k][row] = X[row][k], ys[k][col] =
// Y[col][k]; the result stays in registers and is handed out entry by entry.
template <class R> struct TileAcc;

typedef double d4 __attribute__((ext_vector_type(4)));

// FP64: FP64 MFMA 16x16x4, two 16x16 output blocks per wavefront.  The MFMA
// is fed Y as its A operand and X as its B operand (lane l: Y[16bj + l%16][k]
// and X[16bi + l%16][k], k = k0 + l/16), so element e of lane l is
// C[16bi + l%16][16bj + l/16 + 4e]: sixteen consecutive rows per column, which
// makes the column-major tile stores coalesced.  Both blocks of a wavefront lie
// in one block column, and the two wavefronts of a SIMD (wv and wv + 4) take
// columns 3 and 0 or 2 and 1, which evens out product_ylower.
template <> struct TileAcc<double> {
    d4 acc[2];
    static __device__ __forceinline__ int block_col(int wv) { return (wv >> 1) ^ (wv < 4 ? 3 : 2); }
    static __device__ __forceinline__ int block_row(int wv, int b) { return (2 * wv + b) & 3; }
    __device__ __forceinline__ void product(const double (*xs)[T], const double (*ys)[T]) {
        const int t0 = thread_index(), l = t0 & 63, wv = t0 >> 6, bj = block_col(wv);
        acc[0] = d4{0.0, 0.0, 0.0, 0.0};
        acc[1] = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll 8
        for (int k0 = 0; k0 < T; k0 += 4) {
            const int k = k0 + (l >> 4);
#pragma unroll
            for (int b = 0; b < 2; ++b)
                acc[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(ys[k][16 * bj + (l & 15)],
                                                             xs[k][16 * block_row(wv, b) + (l & 15)], acc[b], 0, 0, 0);
        }
    }
    // The same product for a lower-triangular Y (Y[col][k] = 0 for k > col):
    // the k-steps past the last column of the output block column add exact
    // zeros and are skipped.
    __device__ __forceinline__ void product_ylower(const double (*xs)[T], const double (*ys)[T]) {
        const int t0 = thread_index(), l = t0 & 63, wv = __builtin_amdgcn_readfirstlane(t0 >> 6), bj = block_col(wv);
        acc[0] = d4{0.0, 0.0, 0.0, 0.0};
        acc[1] = d4{0.0, 0.0, 0.0, 0.0};
        // 16-wide k blocks, the next one's operands read beside the products
        double y[4], x[4][2];
        auto read = [&](int kb) {
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const int k = 16 * kb + 4 * t + (l >> 4);
                y[t] = ys[k][16 * bj + (l & 15)];
#pragma unroll
                for (int b = 0; b < 2; ++b) x[t][b] = xs[k][16 * block_row(wv, b) + (l & 15)];
            }
        };
        read(0);
        for (int kb = 0; kb <= bj; ++kb) {
            double yc[4], xc[4][2];
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                yc[t] = y[t];
                xc[t][0] = x[t][0];
                xc[t][1] = x[t][1];
            }
            if (kb < bj) read(kb + 1);
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int b = 0; b < 2; ++b)
                    acc[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(yc[t], xc[t][b], acc[b], 0, 0, 0);
        }
    }
    static constexpr int N = 8;   // entries per thread
    template <class F> __device__ __forceinline__ void each_i(F&& f) const {
        const int t0 = thread_index(), l = t0 & 63, wv = t0 >> 6;
#pragma unroll
        for (int b = 0; b < 2; ++b) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                f(16 * block_row(wv, b) + (l & 15), 16 * block_col(wv) + (l >> 4) + 4 * e, acc[b][e], 4 * b + e);
        }
    }
    template <class F> __device__ __forceinline__ void each(F&& f) const {
        each_i([&](int row, int col, double v, int) { f(row, col, v); });
    }
};

// FP32: vector FMA, thread (tr, tc) owns rows tr + 16u and columns tc + 32v.
template <> struct TileAcc<float> {
    float acc[4][2];
    __device__ __forceinline__ void product(const float (*xs)[T], const float (*ys)[T]) {
        const int tr = threadIdx.x & 15, tc = threadIdx.x >> 4;
#pragma unroll
        for (int u = 0; u < 4; ++u) acc[u][0] = acc[u][1] = 0.0f;
        for (int k = 0; k < T; ++k) {
            float av[4], bv[2];
#pragma unroll
            for (int u = 0; u < 4; ++u) av[u] = xs[k][tr + 16 * u];
#pragma unroll
            for (int v = 0; v < 2; ++v) bv[v] = ys[k][tc + 32 * v];
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int v = 0; v < 2; ++v) acc[u][v] += av[u] * bv[v];
        }
    }
    __device__ __forceinline__ void product_ylower(const float (*xs)[T], const float (*ys)[T]) { product(xs, ys); }
    static constexpr int N = 8;   // entries per thread
    template <class F> __device__ __forceinline__ void each_i(F&& f) const {
        const int tr = threadIdx.x & 15, tc = threadIdx.x >> 4;
#pragma unroll
        for (int v = 0; v < 2; ++v)
#pragma unroll
            for (int u = 0; u < 4; ++u) f(tr + 16 * u, tc + 32 * v, acc[u][v], 4 * v + u);
    }
    template <class F> __device__ __forceinline__ void each(F&& f) const {
        each_i([&](int row, int col, float v, int) { f(row, col, v); });
    }
};

// The tile entries at the positions TileAcc<R>::each_i hands out, in its order.
template <class R>
__device__ __forceinline__ void gather_tile(const R* __restrict__ tile, R* buf) {
    TileAcc<R> pos;
    pos.each_i([&](int row, int col, R, int i) { buf[i] = tile[col * T + row]; });
}

// C = X Y^T (operands as for TileAcc) for a symmetric C of which only the ten
// 16x16 blocks on and below the diagonal are wanted: one or two blocks per
// wavefront, three blocks' work on two of the four SIMDs and two on the
// others (wavefronts wv and wv + 4 share a SIMD), so the product takes 48
// MFMA steps per SIMD instead of 64.  Element e of slot s of lane l is
// C[16 bi_s + l % 16][16 bj_s + l / 16 + 4e], as in TileAcc<double>.
struct LowerAcc {
    d4 acc[2];
    int bi[2], bj[2], n;
    __device__ __forceinline__ LowerAcc() {
        const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        // per wavefront: (bi, bj) of slot 0, then of slot 1 (-1: none)
        constexpr signed char tab[8][4] = {{0, 0, 3, 3}, {1, 1, 2, 2}, {2, 1, -1, -1}, {3, 1, -1, -1},
                                           {1, 0, -1, -1}, {2, 0, -1, -1}, {3, 0, -1, -1}, {3, 2, -1, -1}};
        bi[0] = tab[wv][0];
        bj[0] = tab[wv][1];
        bi[1] = tab[wv][2];
        bj[1] = tab[wv][3];
        n = bi[1] >= 0 ? 2 : 1;
    }
    __device__ __forceinline__ void product(const double (*xs)[T], const double (*ys)[T]) {
        const int l = thread_index() & 63;
        acc[0] = d4{0.0, 0.0, 0.0, 0.0};
        acc[1] = d4{0.0, 0.0, 0.0, 0.0};
        auto run = [&](auto two) {
#pragma unroll 8
            for (int k0 = 0; k0 < T; k0 += 4) {
                const int k = k0 + (l >> 4);
                acc[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(ys[k][16 * bj[0] + (l & 15)],
                                                             xs[k][16 * bi[0] + (l & 15)], acc[0], 0, 0, 0);
                if constexpr (decltype(two)::value)
                    acc[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(ys[k][16 * bj[1] + (l & 15)],
                                                                 xs[k][16 * bi[1] + (l & 15)], acc[1], 0, 0, 0);
            }
        };
        if (n == 2) run(std::true_type());
        else run(std::false_type());
    }
    // f(row, col, value, i), i = 4 s + e
    template <class F> __device__ __forceinline__ void each_i(F&& f) const {
        const int l = thread_index() & 63;
#pragma unroll
        for (int s = 0; s < 2; ++s)
            if (s < n) {
#pragma unroll
                for (int e = 0; e < 4; ++e) f(16 * bi[s] + (l & 15), 16 * bj[s] + (l >> 4) + 4 * e, acc[s][e], 4 * s + e);
            }
    }
};

// the symmetric product's accumulator at each precision
template <class R> struct SymAcc : TileAcc<R> {};
template <> struct SymAcc<double> : LowerAcc { static constexpr int N = 8; };

// ---- D_K --------------------------------------------------------------------
// The task takes the 64x64 tile S (lower part; the part above the diagonal is
// never read) in LDS as xs[col][row], writes D to piv and Linv = L^{-1} (zeros
// above the diagonal) to lout, and overwrites xs.  L_KK itself is read by
// neither the panels and updates nor the solves and is not stored.  FP32
// tiles go through the FP64 task (below).
template <class R> struct DiagScratch;
template <> struct DiagScratch<double> { double tsc[5][256]; double ub[16]; };
// FP64: blocked by 16.  For each column block k:
//  - wavefront 0 factorizes the 64x16 panel (rows 16k..63, lane = row):
//    16 pivot steps, each broadcasting column c of the block through LDS; the
//    pivot and the next step's critical entry travel by readlane, and the
//    reciprocal of the next pivot is formed while the rest of the step's
//    updates are issued.  The block lanes also form column p of Linv_kk by
//    the same elimination applied to the identity.  Multipliers are
//    l = a * (1/d) with the reciprocal refined by two Newton steps.
//  - the other wavefronts meanwhile form the off-diagonal blocks of Linv
//    that are ready, Linv_ij = -Linv_ii sum_{k=j}^{i-1} L_ik Linv_kj, as
//    16x16x16 FP64 MFMA products, avoiding wavefront 4 (which shares a SIMD
//    with wavefront 0);
//  - after a barrier, up to six wavefronts update the trailing blocks
//    A_ij -= L_ik D_k L_jk^T (16x16x16 FP64 MFMA).
// Linv is kept in ys column-major with the row index swizzled by the column
// (ysw), which makes both row and column accesses free of bank conflicts.

__device__ __forceinline__ int ysw(int col, int row) { return col * T + (row ^ (col & 15)); }

__device__ __forceinline__ double recip(double d) {
    double r = __builtin_amdgcn_rcp(d);
    double e = __builtin_fma(-d, r, 1.0);
    r = __builtin_fma(r, e, r);
    e = __builtin_fma(-d, r, 1.0);
    return __builtin_fma(r, e, r);
}

// D[m][n] = sum_t A(m, t) B(t, n) over 16x16 blocks on one wavefront (FP64
// MFMA 16x16x4: lane l supplies A(l%16, t) and B(t, l%16), t = t0 + l/16);
// element e of lane l is D[l/16 + 4e][l%16].
template <class FA, class FB>
__device__ __forceinline__ d4 mm16(FA A, FB B, d4 acc) {
    const int l = threadIdx.x & 63, rr = l & 15, lg = l >> 4;
#pragma unroll
    for (int t0 = 0; t0 < 16; t0 += 4) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(A(rr, t0 + lg), B(t0 + lg, rr), acc, 0, 0, 0);
    return acc;
}

struct NoSide {
    __device__ void operator()(int, int) const {}
};

// side(k, wv) runs on every wavefront in each block column's phase, on
// wavefront 0 before the pivot steps and on the others beside them (after
// their own products), and on all of them once more, with k = 4, before the
// last products.  LDS_ONLY: Linv goes to lds_out alone and D stays in
// dd; the caller stores them.
template <bool LDS_ONLY = false, class O = double, class Side = NoSide>
__device__ __forceinline__ void diag_task(double (*xs)[T], double* ys, double* dd, DiagScratch<double>& sm,
                                          O* __restrict__ lout, double* __restrict__ piv, long Kt,
                                          O* lds_out = nullptr, Side side = Side()) {
    const int wv = threadIdx.x >> 6, l = threadIdx.x & 63, rr = l & 15, lg = l >> 4;
    double(*tsc)[256] = sm.tsc;
    // operand views: L_ik (rows r, cols t), Linv_ij as (t, c) and as (r, t), T slot s as (t, c)
    auto Lb = [&](int i, int k) { return [&, i, k](int r, int t) { return xs[16 * k + t][16 * i + r]; }; };
    auto Vb = [&](int i, int j) { return [&, i, j](int t, int c) { return ys[ysw(16 * j + c, 16 * i + t)]; }; };
    auto Vr = [&](int i, int j) { return [&, i, j](int r, int t) { return ys[ysw(16 * j + t, 16 * i + r)]; }; };
    auto Tb = [&](int s) { return [&, s](int t, int c) { return tsc[s][t * 16 + c]; }; };
    auto getT = [&](int s) {
        d4 acc;
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] = tsc[s][(lg + 4 * e) * 16 + rr];
        return acc;
    };
    auto putT = [&](int s, d4 acc) {
#pragma unroll
        for (int e = 0; e < 4; ++e) tsc[s][(lg + 4 * e) * 16 + rr] = acc[e];
        __builtin_amdgcn_wave_barrier();
    };
    auto putV = [&](int i, int j, d4 acc) {   // Linv_ij = -acc
#pragma unroll
        for (int e = 0; e < 4; ++e) ys[ysw(16 * j + rr, 16 * i + lg + 4 * e)] = -acc[e];
        __builtin_amdgcn_wave_barrier();
    };
    const d4 z = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 1
    for (int k = 0; k < 4; ++k) {
        if (wv == 0) {
            side(k, 0);
            const int r = l, base = 16 * k, p = r - base;
            double v[16], bcol[16];
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                v[q] = xs[base + q][r];
                bcol[q] = (q == p) ? 1.0 : 0.0;
            }
            if (p >= 0 && p < 16) sm.ub[p] = v[0];
            __builtin_amdgcn_wave_barrier();
            double d = lane_value(v[0], base);
            double rd = recip(d);
            double dr = 0.0;
            double U[16];
#pragma unroll
            for (int q = 0; q < 16; ++q) U[q] = sm.ub[q];
#pragma unroll
            for (int c = 0; c < 16; ++c) {
                int po = p;
                __asm__ volatile("" : "+v"(po));   // keeps the per-step lane tests in the step
                const bool below = po > c;
                dr = (po == c) ? d : dr;
                const double le = below ? v[c] * rd : 0.0;
                const double fb = below ? 0.0 : bcol[c] * rd;
                double dn = 0.0, rdn = 0.0, un = 0.0;
                if (c + 1 < 16) {
                    v[c + 1] = __builtin_fma(-le, U[c + 1], v[c + 1]);
                    __builtin_amdgcn_wave_barrier();
                    if (po >= 0 && po < 16) sm.ub[po] = v[c + 1];
                    __builtin_amdgcn_wave_barrier();
                    dn = lane_value(v[c + 1], base + c + 1);
                    if (c + 2 < 16) un = lane_value(v[c + 1], base + c + 2);
                    rdn = recip(dn);
                }
#pragma unroll
                for (int q = c + 2; q < 16; ++q) v[q] = __builtin_fma(-le, U[q], v[q]);
#pragma unroll
                for (int q = c + 1; q < 16; ++q) bcol[q] = __builtin_fma(-fb, U[q], bcol[q]);
                v[c] = below ? le : v[c];
                if (c + 1 < 16) {
#pragma unroll
                    for (int q = 0; q < 16; ++q) U[q] = (q == c + 2) ? un : sm.ub[q];
                    d = dn;
                    rd = rdn;
                }
                // keep every update in its own step (no deferred chains)
#pragma unroll
                for (int q = 0; q < 16; ++q) {
                    __asm__ volatile("" : "+v"(v[q]));
                    __asm__ volatile("" : "+v"(bcol[q]));
                }
            }
            if (p >= 0) {
#pragma unroll
                for (int q = 0; q < 16; ++q) xs[base + q][r] = v[q];
            }
            if (p >= 0 && p < 16) {
                dd[r] = dr;
                if (!LDS_ONLY) piv[Kt * T + r] = dr;
#pragma unroll
                for (int q = 0; q < 16; ++q) ys[ysw(base + p, base + q)] = (q >= p) ? bcol[q] : 0.0;
            }
        } else if (k == 1) {
            if (wv == 1) putT(0, mm16(Lb(1, 0), Vb(0, 0), z));                      // T_10
        } else if (k == 2) {
            if (wv == 1) {
                putV(1, 0, mm16(Vr(1, 1), Tb(0), z));                                // Linv_10
                putT(1, mm16(Lb(2, 1), Vb(1, 0), mm16(Lb(2, 0), Vb(0, 0), z)));      // T_20
            } else if (wv == 2) {
                putT(2, mm16(Lb(2, 1), Vb(1, 1), z));                                // T_21
            } else if (wv == 3) {
                putT(3, mm16(Lb(3, 0), Vb(0, 0), z));                                // T_30, first term
            } else if (wv == 5) {
                putT(4, mm16(Lb(3, 1), Vb(1, 1), z));                                // T_31, first term
            }
        } else if (k == 3) {
            if (wv == 1) putV(2, 0, mm16(Vr(2, 2), Tb(1), z));                       // Linv_20
            else if (wv == 2) putV(2, 1, mm16(Vr(2, 2), Tb(2), z));                  // Linv_21
            else if (wv == 3) putT(3, mm16(Lb(3, 1), Vb(1, 0), getT(3)));            // T_30, second term
            else if (wv == 5) putT(0, mm16(Lb(3, 2), Vb(2, 2), z));                  // T_32
        }
        if (wv != 0) side(k, wv);
        __syncthreads();
        if (k == 3) break;
        // trailing update of the blocks k < j <= i <= 3, one per wavefront
        {
            const int nb = 3 - k;
            int pp = wv, i = -1, j = -1;
            for (int a = 0; a < nb && i < 0; ++a)
                for (int b = 0; b <= a; ++b) {
                    if (pp == 0) { i = k + 1 + a; j = k + 1 + b; break; }
                    --pp;
                }
            if (i >= 0) {
                // D[m = c][n = r] = sum_t L_jk[c][t] (L_ik[r][t] d_t)
                const d4 acc = mm16([&](int c, int t) { return xs[16 * k + t][16 * j + c]; },
                                    [&](int t, int r) { return xs[16 * k + t][16 * i + r] * dd[16 * k + t]; }, z);
#pragma unroll
                for (int e = 0; e < 4; ++e) xs[16 * j + lg + 4 * e][16 * i + rr] -= acc[e];
            }
        }
        __syncthreads();
    }
    side(4, wv);
    // the last row of blocks: T_3j completed, Linv_3j = -Linv_33 T_3j
    if (wv == 0) {
        putT(1, mm16(Lb(3, 2), Vb(2, 0), getT(3)));
        putV(3, 0, mm16(Vr(3, 3), Tb(1), z));
    } else if (wv == 1) {
        putT(2, mm16(Lb(3, 2), Vb(2, 1), getT(4)));
        putV(3, 1, mm16(Vr(3, 3), Tb(2), z));
    } else if (wv == 2) {
        putV(3, 2, mm16(Vr(3, 3), Tb(0), z));
    }
    __syncthreads();
    for (int idx = threadIdx.x; idx < TT; idx += NTH) {
        const int col = idx / T, row = idx % T;
        const double v = (row >= col) ? ys[ysw(col, row)] : 0.0;
        if (!LDS_ONLY) lout[idx] = O(v);
        if (LDS_ONLY || lds_out) lds_out[idx] = O(v);
    }
}

// FP32 tiles: the FP64 task on the tile widened in LDS, with Linv rounded once
// to FP32 and the pivots kept in FP64.  The FP64 task is blocked by 16 and
// carries each panel on one wavefront; a 64-step FP32 chain with a workgroup
// barrier per pivot made the FP32 column launch slower than the FP64 one.
template <> struct DiagScratch<float> { double xd[T][T]; double yd[TT]; DiagScratch<double> in; };

template <bool LDS_ONLY = false, class Side = NoSide>
__device__ __forceinline__ void diag_task(float (*xs)[T], float* /*ys*/, double* dd, DiagScratch<float>& sm,
                                          float* __restrict__ lout, double* __restrict__ piv, long Kt,
                                          float* lds_out = nullptr, Side side = Side()) {
    for (int idx = threadIdx.x; idx < TT; idx += NTH) (&sm.xd[0][0])[idx] = double((&xs[0][0])[idx]);
    __syncthreads();
    diag_task<LDS_ONLY>(sm.xd, sm.yd, dd, sm.in, lout, piv, Kt, lds_out, side);
}

// ---- staging ----------------------------------------------------------------
template <bool CO, class D, class R>
__device__ __forceinline__ void stage(D (*dst)[T], const R* __restrict__ src) {
    R buf[TT / NTH];   // all loads in flight before the first is used
#pragma unroll
    for (int i = 0; i < TT / NTH; ++i) buf[i] = cld<CO>(&src[threadIdx.x + NTH * i]);
#pragma unroll
    for (int i = 0; i < TT / NTH; ++i) (&dst[0][0])[threadIdx.x + NTH * i] = D(buf[i]);
}

// dst[k][row] = src[row][k], src column-major, by 8x8 blocks: a wavefront's
// loads touch whole 64-byte segments and its LDS writes eight rows
template <class D, class R>
__device__ __forceinline__ void stage_t(D (*dst)[T], const R* __restrict__ src) {
    const int r = threadIdx.x & 7, c = threadIdx.x >> 3 & 7, wv = threadIdx.x >> 6;
    R buf[64 / NWAVE];
#pragma unroll
    for (int i = 0; i < 64 / NWAVE; ++i) {
        const int b = wv + NWAVE * i;
        buf[i] = src[(8 * (b >> 3) + c) * T + 8 * (b & 7) + r];
    }
#pragma unroll
    for (int i = 0; i < 64 / NWAVE; ++i) {
        const int b = wv + NWAVE * i;
        dst[8 * (b & 7) + r][8 * (b >> 3) + c] = D(buf[i]);
    }
}
// A tile from LDS to memory by nthr threads, coherently, 16 bytes a store
template <class R>
__device__ __forceinline__ void put_tile(R* dst, const R (*src)[T], int i0, int nthr) {
    typedef int i4 __attribute__((ext_vector_type(4)));
    const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(dst, 0, TT * sizeof(R), 0x00020000);
#pragma unroll 4
    for (int i = i0; i < int(TT * sizeof(R) / 16); i += nthr)
        __builtin_amdgcn_raw_buffer_store_b128(reinterpret_cast<const i4*>(src)[i], rsrc, 16 * i, 0, 17);   // sc0 sc1
}
// dst[k][row] = src[k][row] * d[k]
template <bool CO, class R>
__device__ __forceinline__ void stage_scaled(R (*dst)[T], const R* __restrict__ src, const double* __restrict__ d) {
    for (int idx = threadIdx.x; idx < TT; idx += NTH) dst[idx / T][idx % T] = cld<CO>(&src[idx]) * R(d[idx / T]);
}

// P_{I,K}: out = A_IK Linv_K^T D_K^{-1} (out may alias a); tout receives the
// transposed tile (row-major), which the backward sweep reads
template <bool CO, class R>
__device__ __forceinline__ void panel_task(R* __restrict__ out, const R* __restrict__ a, const R* __restrict__ lv,
                                           const double* __restrict__ dk, R (*xs)[T], R (*ys)[T],
                                           R* __restrict__ tout) {
    stage<false>(xs, a);
    stage<false>(ys, lv);
    __syncthreads();
    TileAcc<R> acc;
    acc.product(xs, ys);
    acc.each([&](int row, int col, R v) {
        const R p = v * (R(1) / R(dk[col]));
        cst<CO>(&out[col * T + row], p);
        tout[row * T + col] = p;
    });
}

// U_{I,J,K}: out -= (L_IK D_K) L_JK^T
template <bool CO, class R>
__device__ __forceinline__ void update_task(R* __restrict__ out, const R* __restrict__ lik, const R* __restrict__ ljk,
                                            const double* __restrict__ dk, R (*xs)[T], R (*ys)[T]) {
    stage_scaled<CO>(xs, lik, dk);
    stage<CO>(ys, ljk);
    __syncthreads();
    TileAcc<R> acc;
    acc.product(xs, ys);
    acc.each([&](int row, int col, R v) { out[col * T + row] -= v; });
}

// ---- split schedule ----------------------------------------------------------
template <class R>
__global__ void __launch_bounds__(NTH) k_tile_diag(const R* __restrict__ tiles, R* __restrict__ linv,
                                                   double* __restrict__ piv, long Kt, int w) {
    __shared__ R xs[T][T];
    __shared__ R ys[TT];
    __shared__ double dd[T];
    __shared__ DiagScratch<R> sm;
    stage<false>(xs, tiles + tile_index(Kt, Kt, w) * TT);
    __syncthreads();
    diag_task(xs, ys, dd, sm, linv + Kt * (long)TT, piv, Kt);
}

// P_{I,K} for I = Kt+1+blockIdx.x
template <class R>
__global__ void __launch_bounds__(NTH) k_tile_panel(R* __restrict__ tiles, R* __restrict__ tiles_t,
                                                    const R* __restrict__ linv, const double* __restrict__ piv,
                                                    long Kt, int w) {
    __shared__ R xs[T][T];
    __shared__ R ys[T][T];
    const long ti = tile_index(Kt + 1 + blockIdx.x, Kt, w) * TT;
    panel_task<false, R>(tiles + ti, tiles + ti, linv + Kt * (long)TT, piv + Kt * T, xs, ys, tiles_t + ti);
}

// (r, s), s <= r, of entry t of the triangle enumerated row by row
__device__ inline void tri_pair(long t, long& r, long& s) {
    r = long((sqrt(8.0 * double(t) + 1.0) - 1.0) / 2.0);
    while ((r + 1) * (r + 2) / 2 <= t) ++r;
    while (r * (r + 1) / 2 > t) --r;
    s = t - r * (r + 1) / 2;
}

// U_{I,J,K} for the pairs K < J <= I <= K+m, blockIdx.x -> (I, J) row by row
template <class R>
__global__ void __launch_bounds__(NTH) k_tile_update(R* __restrict__ tiles, const double* __restrict__ piv,
                                                     long Kt, int w) {
    __shared__ R xs[T][T];
    __shared__ R ys[T][T];
    long r, s;
    tri_pair(blockIdx.x, r, s);
    const long I = Kt + 1 + r, J = Kt + 1 + s;
    update_task<false, R>(tiles + tile_index(I, J, w) * TT, tiles + tile_index(I, Kt, w) * TT,
                          tiles + tile_index(J, Kt, w) * TT, piv + Kt * T, xs, ys);
}

// ---- fused schedule -----------------------------------------------------------
// One launch factors the band.  A tile keeps its entries in the registers of
// the workgroup that owns it from the first update to the last (left-looking),
// so it is read once and written once, and no launch boundary or flush lies
// between the columns:
//   chain      the first workgroup, column after column: P_{J,J-1} and U_{J,J,J-1} in
//              LDS, D_J; Linv_J stays in LDS for the next panel
//   tile(I, J) I - J >= 2: all updates, then P_{I,J}; (I, I-2) is handed to
//              near(I) and corner(I) before its panel product
//   near(I)    (I, I-1): all updates but the chain's, then handed to the chain.  For
//              the last of them it forms P_{I,I-2} and P_{I-1,I-2} itself
//   corner(I)  (I, I) likewise, with P_{I,I-2}
// One column's critical path is then the chain's own P, U, D or half the loop
// Linv_{J-2} -> near(J) -> chain -> Linv_J, whichever is longer.  The chain is:
// 17.6 us a column (256 x 256 panel, 12.1 of it the diagonal task), against
// 21.2 us for a launch per column whose workgroups loaded and stored every
// tile they updated.  The other workgroups of a band of 25 tiles need about 3 us
// a column of the whole chip's matrix units, so they keep up; from about 31 tiles
// on the updates' reads of two tiles each set the pace, 20.2 us a column with 38
// tiles, 32 with 98 and 134 with 219 (a launch per column: 33, 56 and 264).
// Counters (zero
// before the launch): P_ROW the columns of a tile row that its tile() tasks have
// finished, P_LAST L_{J,J-1} stored, P_DIAG D_J and Linv_J stored, P_NEAR and
// P_NEAR2 a row's two last tiles handed over, P_PART tile (I, I-2) handed over (in
// slot (I, I) of tiles, which holds nothing else).
// Workgroups take their tasks as they start (start_number) and wait only on
// earlier tasks and on the chain.  The chain, the first task, waits on near and
// corner of the column it has reached, whose own waits are on earlier columns,
// so the earliest unfinished task beside it can always go on; every wait ends
// as long as there is room beside the chains, which keep a CU each for a whole
// factorization.  Waits are bounded anyway.  Order: the chain, then by column J = 0, 1, ..: tile(J+2, J),
// near(J+2), corner(J+2), tile(J+3, J) .. tile(J+m, J), m = min(w, nt-1-J)
// (m + 1 workgroups, none for m < 2).
// The band is assembled in tiles_t and the factor goes to tiles: no line of
// tiles is read before it is written for good, and a tile's slot in tiles_t
// receives the transposed factor tile when its owner has finished.
constexpr long PSTRIDE = 16;   // a counter per 64 bytes
// BandLDLT::flag: the error bits, then the start counters of the forward and
// backward sweeps; the factorization's follow its progress counters
// (cleared before each factorization and solve)
inline long start_counters(long workgroups) { return (1 + (workgroups + 31) / 32 + PSTRIDE - 1) / PSTRIDE * PSTRIDE; }
enum { P_ROW = 0, P_LAST = 1, P_DIAG = 2, P_NEAR = 3, P_NEAR2 = 4, P_PART = 5, P_N = 6 };

inline long factor_workgroups(long nt, int w) {
    if (w < 2) return 1;
    long g = 1 + std::max(0L, nt - w) * (w + 1);
    for (long m = std::min<long>(w - 1, nt - 1); m >= 2; --m) g += m + 1;
    return g;
}

template <class R>
__global__ void __launch_bounds__(NTH) k_band_factor(R* __restrict__ tiles, R* __restrict__ tiles_t,
                                                     R* __restrict__ linv, double* __restrict__ piv, int w, long nt,
                                                     int* prog, int* started, bool by_count, long spin_limit,
                                                     int* err) {
    constexpr int N = TileAcc<R>::N, NS = TT / NTH;
    __shared__ R xs[T][T];
    __shared__ R ys[T][T];
    __shared__ R zs[T][T];
    __shared__ R lk[T][T];    // the chain's Linv_K
    __shared__ double dk[T];
    __shared__ R rdk[T];      // 1 / D_K
    __shared__ DiagScratch<R> sm;
    __shared__ int seen_s[2][2];
    __shared__ R zd[std::is_same<R, double>::value ? 10 : 1][256];   // the chain's next A_JJ, by 16x16 blocks
    __shared__ int got_s[4], drained_s[2];
    // 4 * block row + block column of lower 16x16 block b, by columns
    auto dblk = [](int b) { return int(0xFEAD95C840ull >> 4 * b & 15); };
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    auto cnt = [&](int kind, long i) { return prog + (kind * nt + i) * PSTRIDE; };
    auto tile = [&](R* base, long I, long J) { return base + tile_index(I, J, w) * TT; };
    // Waits until both counters have reached the target; returns the smaller
    // value, below the target after an error.  seen_s alternates, so that a
    // wait's values are not overwritten before every thread has read them.
    int par = 0;
    auto wait2 = [&](const int* c0, const int* c1, int target) {
        if (tid == 0) seen_s[par][0] = poll_count(c0, target, spin_limit, err);
        if (tid == 64) seen_s[par][1] = poll_count(c1, target, spin_limit, err);
        __syncthreads();
        const int v = min(seen_s[par][0], seen_s[par][1]);
        par ^= 1;
        return v;
    };
    auto wait1 = [&](const int* c, int target) {
        if (tid == 0) seen_s[par][0] = poll_count(c, target, spin_limit, err);
        __syncthreads();
        const int v = seen_s[par][0];
        par ^= 1;
        return v >= target;
    };
    auto load_co = [&](R* buf, const R* src) {
#pragma unroll
        for (int i = 0; i < NS; ++i) buf[i] = cld<true>(&src[tid + NTH * i]);
    };
    auto to_lds = [&](R (*dst)[T], const R* buf) {
#pragma unroll
        for (int i = 0; i < NS; ++i) dst[wv + NWAVE * i][lane] = buf[i];
    };
    // dst = buf scaled by column with D_K, of which this lane holds entry `lane`
    auto to_lds_scaled = [&](R (*dst)[T], const R* buf, double d) {
#pragma unroll
        for (int i = 0; i < NS; ++i) dst[wv + NWAVE * i][lane] = buf[i] * R(lane_value(d, wv + NWAVE * i));
    };
    // ys = Linv_K and dk, rdk = D_K, 1 / D_K, in the coherent copies
    auto stage_linv = [&](long K) {
        if (tid < T) {
            const double d = cld<true>(&piv[K * T + tid]);
            dk[tid] = d;
            rdk[tid] = R(1) / R(d);
        }
        stage<true>(ys, linv + K * (long)TT);
    };

    const long number = gridDim.x > 1 ? start_number(started, by_count) : 0;
    if (number == 0) {
        if (tid < 2) drained_s[tid] = 0;
        // A column's tiles sit in the pair (a0, a1): A_{J,J-1} and Linv_{J-1},
        // then, once the panel product has read them, the diagonal task's
        // tile and rows.  The other pair holds the panel (L D, L) until the
        // diagonal update is done, in the first phase of the task, and
        // receives A_{J+1,J} (as soon as near(J+1) has handed it over) and
        // Linv_J for the next column.
        R (*a0)[T] = xs, (*a1)[T] = ys, (*b0)[T] = zs, (*b1)[T] = lk;
        constexpr bool D64 = std::is_same<R, double>::value;
        for (long J = 0; J < nt; ++J) {
            const bool handed = J >= 2 && w >= 2;              // near(J) exists
            const bool hands = J + 1 >= 2 && w >= 2;           // near(J+1) exists, if row J+1 does
            const R* dt = tile(tiles_t, J, J);
            bool got2 = false;
            if (J == 0) {
                stage<false>(a0, dt);
                __syncthreads();
            } else {
                if (wv >= 4) {   // the last of these sees D_{J-1} and Linv_{J-1} complete in memory
                    put_tile(linv + (J - 1) * (long)TT, a1, tid - NTH / 2, NTH / 2);
                    if (wv == 4) cst<true>(&piv[(J - 1) * T + lane], dk[lane]);
                    __builtin_amdgcn_s_waitcnt(0);
                    if (lane == 0 && atomicAdd(&drained_s[0], 1) == 4 * int(J) - 1)
                        __hip_atomic_store(cnt(P_DIAG, J - 1), 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                }
                const int got = got_s[0] & got_s[1] & got_s[2] & got_s[3];
                got2 = got & 2;
                if (!(got & 1)) {
                    if (handed) {
                        if (!wait1(cnt(P_NEAR, J), 1)) return;
                        stage<true>(a0, tile(tiles_t, J, J - 1));
                    } else {
                        stage<false>(a0, tile(tiles_t, J, J - 1));
                    }
                    __syncthreads();
                }
                TileAcc<R> acc;
                acc.product_ylower(a0, a1);
                R* tout = tile(tiles_t, J, J - 1);
                const bool own_t = !hands || J + 1 >= nt;      // else near(J+1) stores the transposed tile
                acc.each([&](int row, int col, R v) {
                    const R p = v * rdk[col];
                    b0[col][row] = p * R(dk[col]);
                    b1[col][row] = p;
                    if (own_t) tout[row * T + col] = p;
                });
                __syncthreads();
                if (handed && !got2 && !wait1(cnt(P_NEAR2, J), 1)) return;
            }
            // block b of the ten lower 16x16 blocks of A_JJ - U_{J,J,J-1}, one wavefront
            auto diag_block = [&](int b) {
                const int lane = thread_index() & 63;
                const int bi = dblk(b) >> 2, bj = dblk(b) & 3;
                R pre[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int row = 16 * bi + (lane & 15), col = 16 * bj + (lane >> 4) + 4 * e;
                    pre[e] = got2 ? zd[b][64 * e + lane] : handed ? cld<true>(&dt[col * T + row]) : dt[col * T + row];
                }
                d4 u = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
                for (int k0 = 0; k0 < T; k0 += 4) {
                    const int k = k0 + (lane >> 4);
                    u = __builtin_amdgcn_mfma_f64_16x16x4f64(b1[k][16 * bj + (lane & 15)], b0[k][16 * bi + (lane & 15)], u,
                                                            0, 0, 0);
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) a0[16 * bj + (lane >> 4) + 4 * e][16 * bi + (lane & 15)] = pre[e] - u[e];
            };
            if (J > 0) {
                if constexpr (D64) {
                    if (wv < 4) diag_block(wv);   // the first block column; the rest beside its pivots
                    else put_tile(tile(tiles, J, J - 1), b1, tid - NTH / 2, NTH / 2);
                } else {
                    TileAcc<R> u;
                    u.product(b0, b1);
                    u.each([&](int row, int col, R v) {
                        const R p = handed ? cld<true>(&dt[col * T + row]) : dt[col * T + row];
                        a0[col][row] = p - v;
                    });
                    if (wv >= 4) put_tile(tile(tiles, J, J - 1), b1, tid - NTH / 2, NTH / 2);
                }
                __syncthreads();
            }
            // Beside the pivots: the rest of the diagonal update, then
            // wavefronts 3, 5, 6 and 7 fetch the next column's tiles as they
            // are handed over (loaded in one phase, written to LDS in a later
            // one; got: 1, 2 loaded, 4, 8 written).
            int got = 0;
            const int part = wv == 3 ? 0 : wv - 4;
            const bool fetcher = J + 1 < nt && (wv == 3 || wv > 4);
            R buf1[16], buf2[10];
            auto settle = [&](int ln) {
                if ((got & 5) == 1) {
#pragma unroll
                    for (int i = 0; i < 16; ++i) b0[16 * part + i][ln] = buf1[i];
                    got |= 4;
                }
                if (D64 && (got & 10) == 2) {
#pragma unroll
                    for (int i = 0; i < 10; ++i) zd[0][(10 * part + i) * 64 + ln] = buf2[i];
                    got |= 8;
                }
            };
            diag_task<true>(a0, &a1[0][0], dk, sm, (R*)nullptr, piv, J, &b1[0][0], [&](int k, int v) {
                if (v == 0) return;
                const int ln = thread_index() & 63;
                if (k == 0) {
                    if (J > 0 && v >= 4) {   // the panel is complete in memory
                        __builtin_amdgcn_s_waitcnt(0);
                        if (ln == 0 && atomicAdd(&drained_s[1], 1) == 4 * int(J) - 1)
                            __hip_atomic_store(cnt(P_LAST, J), int(J), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                    }
                    if constexpr (D64)
                        if (J > 0 && v != 4) diag_block(v < 4 ? 3 + v : 2 + v);
                    return;
                }
                if (!fetcher) return;
                settle(ln);
                auto there = [&](int kind) { return !hands || __builtin_amdgcn_readfirstlane(peek(cnt(kind, J + 1))) != 0; };
                if (!(got & 1) && there(P_NEAR)) {
                    const R* src = tile(tiles_t, J + 1, J);
#pragma unroll
                    for (int i = 0; i < 16; ++i) {
                        const R* q = &src[(16 * part + i) * T + ln];
                        buf1[i] = hands ? cld<true>(q) : *q;
                    }
                    got |= 1;
                }
                if (D64 && !(got & 2) && there(P_NEAR2)) {
                    const R* src = tile(tiles_t, J + 1, J + 1);
#pragma unroll
                    for (int i = 0; i < 10; ++i) {
                        const int f = 10 * part + i, b = f >> 2, e = f & 3;
                        const R* q = &src[(16 * (dblk(b) & 3) + (ln >> 4) + 4 * e) * T + 16 * (dblk(b) >> 2) + (ln & 15)];
                        buf2[i] = hands ? cld<true>(q) : *q;
                    }
                    got |= 2;
                }
            });
            if (fetcher) settle(lane);
            if (tid < T) rdk[tid] = R(1) / R(dk[tid]);
            if (lane == 0 && (wv == 3 || wv > 4)) got_s[part] = got >> 2;
            __syncthreads();
            R (*p0)[T] = a0, (*p1)[T] = a1;
            a0 = b0;
            a1 = b1;
            b0 = p0;
            b1 = p1;
        }
        put_tile(linv + (nt - 1) * (long)TT, a1, tid, NTH);
        if (tid < T) cst<true>(&piv[(nt - 1) * T + tid], dk[tid]);
        return;
    }

    // column and place in it
    long t = number - 1, J, m = w;
    const long nfull = nt > w ? nt - w : 0;
    if (t < nfull * (w + 1)) {
        J = t / (w + 1);
        t -= J * (w + 1);
    } else {
        t -= nfull * (w + 1);
        J = nfull;
        m = nt - 1 - J;
        while (t >= m + 1) {
            t -= m + 1;
            ++J;
            --m;
        }
    }
    R xr[NS], yr[NS];
    double dr = 0.0;
    if (t == 2) {
        const long I = J + 2;
        SymAcc<R> sym;
        R c[SymAcc<R>::N];
        R* t2 = tile(tiles_t, I, I);
        sym.each_i([&](int row, int col, R, int i) { c[i] = t2[col * T + row]; });
        long K = I - w > 0 ? I - w : 0;
        int ready = 0;
        auto fetch = [&] {
            load_co(xr, tile(tiles, I, K));
            dr = cld<true>(&piv[K * T + lane]);
        };
        if (K < J) {
            ready = wait2(cnt(P_ROW, I), cnt(P_ROW, I), int(K + 1));
            if (ready < K + 1) return;
            fetch();
        }
        while (K < J) {
            to_lds_scaled(xs, xr, dr);
            to_lds(ys, xr);
            __syncthreads();
            ++K;
            const bool next = K < J && K < ready;
            if (next) fetch();
            sym.product(xs, ys);
            sym.each_i([&](int, int, R v, int i) { c[i] -= v; });
            if (next || K >= J) {
                __syncthreads();
            } else {
                ready = wait2(cnt(P_ROW, I), cnt(P_ROW, I), int(K + 1));
                if (ready < K + 1) return;
                fetch();
            }
        }
        if (!wait1(cnt(P_PART, I), 1)) return;
        stage<true>(xs, tile(tiles, I, I));
        if (!wait1(cnt(P_DIAG, J), 1)) return;
        stage_linv(J);
        __syncthreads();
        TileAcc<R> acc;
        acc.product_ylower(xs, ys);
        __syncthreads();
        acc.each([&](int row, int col, R v) {
            const R p = v * rdk[col];
            xs[col][row] = p * R(dk[col]);
            ys[col][row] = p;
        });
        __syncthreads();
        sym.product(xs, ys);
        sym.each_i([&](int row, int col, R v, int i) { cst<true>(&t2[col * T + row], c[i] - v); });
        publish(cnt(P_NEAR2, I), 1);
        return;
    }

    // tile(I, J), and near(I) up to its last update
    const bool near = t == 1;
    const long I = J + (t < 2 ? 2 : t), C = near ? I - 1 : J;   // the workgroup's tile is (I, C)
    R* tt = tile(tiles_t, I, C);
    R c[N];
    gather_tile(tt, c);
    long K = I - w > 0 ? I - w : 0;
    int ready = 0;
    auto fetch = [&] {
        load_co(xr, tile(tiles, I, K));
        load_co(yr, tile(tiles, C, K));
        dr = cld<true>(&piv[K * T + lane]);
    };
    // L_{C,C-1} is the chain's
    auto wait_for = [&] { return ready = wait2(cnt(P_ROW, I), cnt(K + 1 == C ? P_LAST : P_ROW, C), int(K + 1)); };
    if (K < J) {
        if (wait_for() < K + 1) return;
        fetch();
    }
    while (K < J) {
        to_lds_scaled(xs, xr, dr);
        to_lds(ys, yr);
        __syncthreads();
        ++K;
        const bool next = K < J && K < ready;   // known to be there: load it during the product
        if (next) fetch();
        TileAcc<R> acc;
        acc.product(xs, ys);
        acc.each_i([&](int, int, R v, int i) { c[i] -= v; });
        if (next || K >= J) {
            __syncthreads();
        } else {
            if (wait_for() < K + 1) return;
            fetch();
        }
    }
    TileAcc<R> acc;
    if (!near) {
        if (t == 0) {
            R* part = tile(tiles, I, I);
            acc.each_i([&](int row, int col, R, int i) { cst<true>(&part[col * T + row], c[i]); });
            publish(cnt(P_PART, I), 1);
        }
        acc.each_i([&](int row, int col, R, int i) { xs[col][row] = c[i]; });
        if (!wait1(cnt(P_DIAG, J), 1)) return;
        stage_linv(J);
        __syncthreads();
        acc.product_ylower(xs, ys);
        R* out = tile(tiles, I, J);
        acc.each_i([&](int row, int col, R v, int i) {
            c[i] = v * rdk[col];
            cst<true>(&out[col * T + row], c[i]);
        });
        publish(cnt(P_ROW, I), int(J + 1));
        acc.each_i([&](int row, int col, R, int i) { tt[row * T + col] = c[i]; });
        return;
    }
    // near(I): (I, I-2) as its owner and (I-1, I-2) as the chain got them
    R* t1 = tile(tiles_t, I - 1, J);
    if (!wait1(cnt(P_PART, I), 1)) return;
    stage<true>(xs, tile(tiles, I, I));
    if (I > 2) {
        if (!wait1(cnt(P_NEAR, I - 1), 1)) return;
        stage<true>(zs, t1);
    } else {
        stage<false>(zs, t1);
    }
    if (!wait1(cnt(P_DIAG, J), 1)) return;
    stage_linv(J);
    __syncthreads();
    TileAcc<R> acc1;
    acc.product_ylower(xs, ys);
    acc1.product_ylower(zs, ys);
    __syncthreads();
    R lv1[N];
    acc.each([&](int row, int col, R v) { xs[col][row] = v * rdk[col] * R(dk[col]); });
    acc1.each_i([&](int row, int col, R v, int i) {
        lv1[i] = v * rdk[col];
        ys[col][row] = lv1[i];
    });
    __syncthreads();
    acc.product(xs, ys);
    acc.each_i([&](int row, int col, R v, int i) { cst<true>(&tt[col * T + row], c[i] - v); });
    publish(cnt(P_NEAR, I), 1);
    // the chain has read (I-1, I-2) once it has published row I-1
    if (!wait1(cnt(P_LAST, I - 1), 1)) return;
    acc.each_i([&](int row, int col, R, int i) { t1[row * T + col] = lv1[i]; });
}

// ---- pipelined sweeps ---------------------------------------------------------
// One workgroup per tile row, taken in tile order (forward) or reverse tile
// order (backward) as the workgroups start (start_number).  A workgroup waits
// on earlier rows only, so the sweep makes progress.  A tile row's values are
// their own completion signal: before a sweep every slot holds SENT, a
// signalling-NaN bit pattern that no arithmetic produces; the producer writes
// the 64 values with system-scope stores (written through to memory) and a
// consumer polls them with system-scope loads until none is SENT.  There is
// no flag and no cache maintenance on the critical path.  Every lane polls
// its own value, one load at a time (several in flight, which sees a value
// sooner, made the sweeps slower: about 26 consumers poll each row, so the
// polls crowd the row's memory channel); polling slows down once a wait has
// lasted long, so the workgroups far ahead of the front load memory little.
// Each wait is bounded: past spin_limit polls the value reads as
// a quiet NaN and *err is raised, so every workgroup still finishes and the
// sweep drains.  Contributions of earlier rows are applied while the newest
// one is still pending, four rows at a time: each wavefront polls one of
// them, so a workgroup that is catching up pays one memory round trip per
// four rows rather than per row (one per row made the workgroups finish
// their older rows only just before the newest one arrived).  The newest
// off-diagonal tile and Linv stay in registers, so the critical path per row
// is one store-to-load hand-off and two 64x64 products.
constexpr unsigned long long SENT = 0x7FF4C0DE5E471E11ull;

__device__ __forceinline__ double poll_value(const double* p, long spin_limit, int* err) {
    const unsigned long long* q = reinterpret_cast<const unsigned long long*>(p);
    auto ld = [q] { return __hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM); };
    for (long n = 0;; ++n) {
        const unsigned long long a = ld();
        if (a != SENT) return __builtin_bit_cast(double, a);
        if (n >= spin_limit) {
            atomicOr(err, 1);
            return __builtin_nan("");
        }
        if (n >= 256) __builtin_amdgcn_s_sleep(4);   // far from the front: poll less often
    }
}

// vin[0..63] = the values of tile row J of v (wave 0 polls, a value per lane)
__device__ __forceinline__ void fetch_row(const double* v, long J, double* vin, long spin_limit, int* err) {
    if (threadIdx.x < T) vin[threadIdx.x] = poll_value(v + J * T + threadIdx.x, spin_limit, err);
    __syncthreads();
}

// Rows that the sweeps' older contributions need, polled side by side:
// wavefront c polls row J + dir * c (c < nc) into vch[c], so a chunk costs
// one memory round trip instead of one per row.
constexpr int NCH = 4;
__device__ __forceinline__ void fetch_rows(const double* v, long J, int dir, int nc, double (*vch)[T],
                                           long spin_limit, int* err) {
    const int c = threadIdx.x >> 6;
    if (c < nc) vch[c][threadIdx.x & 63] = poll_value(v + (J + dir * c) * T + (threadIdx.x & 63), spin_limit, err);
    __syncthreads();
}

__device__ __forceinline__ void put_value(double* p, double x) {
    __hip_atomic_store(p, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// y_I = Linv_I (r_I - sum_{J<I} L_IJ y_J).  r is read from xr, whose slot I
// is set to SENT for the backward sweep; y must hold SENT.
template <class R>
__global__ void __launch_bounds__(256) k_fwd_sweep(const R* __restrict__ tiles, const R* __restrict__ linv,
                                                   double* __restrict__ xr, double* y, long nt, int w,
                                                   int* started, bool by_count, long spin_limit, int* err) {
    __shared__ double vin[T];
    __shared__ double vch[NCH][T];
    __shared__ double part[4][T];
    const long I = start_number(started, by_count);
    const int tid = threadIdx.x, row = tid % T, q = tid / T, k0 = 16 * q;
    R lv[16], ln[16];
    const R* lvp = linv + I * (long)TT;
#pragma unroll
    for (int k = 0; k < 16; ++k) lv[k] = lvp[(k0 + k) * T + row];
    const long J0 = I - w > 0 ? I - w : 0;
    const bool has_prev = J0 <= I - 1;
    if (has_prev) {
        const R* lnp = tiles + (I * (w + 1) + (w - 1)) * (long)TT;   // tile (I, I-1)
#pragma unroll
        for (int k = 0; k < 16; ++k) ln[k] = lnp[(k0 + k) * T + row];
    }
    double acc = 0.0;
    if (q == 0) {
        acc = xr[I * T + row];
        xr[I * T + row] = __builtin_bit_cast(double, SENT);
    }
    // the older rows J < I - 1 in chunks of NCH, wavefront c polling row J + c
    for (long J = J0; J < I - 1; J += NCH) {
        const int nc = (I - 1 - J < NCH) ? int(I - 1 - J) : NCH;
        R lx[NCH][16];
#pragma unroll
        for (int c = 0; c < NCH; ++c)
            if (c < nc) {
                const R* l = tiles + (I * (w + 1) + (J + c - I + w)) * (long)TT;
#pragma unroll
                for (int k = 0; k < 16; ++k) lx[c][k] = l[(k0 + k) * T + row];
            }
        fetch_rows(y, J, 1, nc, vch, spin_limit, err);
#pragma unroll
        for (int c = 0; c < NCH; ++c)
            if (c < nc) {
#pragma unroll
                for (int k = 0; k < 16; ++k) acc -= double(lx[c][k]) * vch[c][k0 + k];
            }
        __syncthreads();
    }
    if (has_prev) {
        fetch_row(y, I - 1, vin, spin_limit, err);
#pragma unroll
        for (int k = 0; k < 16; ++k) acc -= double(ln[k]) * vin[k0 + k];
    }
    // every thread has read vin before it passes this barrier, so vin may be
    // overwritten after it
    part[q][row] = acc;
    __syncthreads();
    if (tid < T) vin[tid] = part[0][tid] + part[1][tid] + part[2][tid] + part[3][tid];
    __syncthreads();
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < 16; ++k) s += double(lv[k]) * vin[k0 + k];
    part[q][row] = s;
    __syncthreads();
    if (tid < T) put_value(&y[I * T + tid], part[0][tid] + part[1][tid] + part[2][tid] + part[3][tid]);
}

// x_I = Linv_I^T (y_I / D_I - sum_{J>I} L_JI^T x_J); workgroup g handles
// I = nt-1-g.  x must hold SENT.  The factor tiles are read from their
// transposed copies, so that consecutive lanes read consecutive entries.
template <class R>
__global__ void __launch_bounds__(256) k_bwd_sweep(const R* __restrict__ tiles_t, const R* __restrict__ linv,
                                                   const double* __restrict__ y, const double* __restrict__ piv,
                                                   double* x, long nt, int w, int* started, bool by_count,
                                                   long spin_limit, int* err) {
    __shared__ double vin[T];
    __shared__ double vch[NCH][T];
    __shared__ double part[4][T];
    const long I = nt - 1 - start_number(started, by_count);
    const int tid = threadIdx.x, col = tid % T, q = tid / T, k0 = 16 * q;
    R lv[16], ln[16];
    const R* lvp = linv + I * (long)TT;
#pragma unroll
    for (int k = 0; k < 16; ++k) lv[k] = lvp[col * T + k0 + k];   // Linv[k][col]
    const long J1 = (I + w < nt - 1) ? I + w : nt - 1;
    const bool has_next = I + 1 <= J1;
    if (has_next) {
        const R* lnp = tiles_t + ((I + 1) * (w + 1) + (w - 1)) * (long)TT;   // tile (I+1, I), transposed
#pragma unroll
        for (int k = 0; k < 16; ++k) ln[k] = lnp[(k0 + k) * T + col];
    }
    double acc = (q == 0) ? y[I * T + col] / piv[I * T + col] : 0.0;
    // the later rows J > I + 1 in chunks of NCH, wavefront c polling row J - c
    for (long J = J1; J > I + 1; J -= NCH) {
        const int nc = (J - (I + 1) < NCH) ? int(J - (I + 1)) : NCH;
        R lx[NCH][16];
#pragma unroll
        for (int c = 0; c < NCH; ++c)
            if (c < nc) {
                const R* l = tiles_t + ((J - c) * (w + 1) + (I - (J - c) + w)) * (long)TT;
#pragma unroll
                for (int k = 0; k < 16; ++k) lx[c][k] = l[(k0 + k) * T + col];
            }
        fetch_rows(x, J, -1, nc, vch, spin_limit, err);
#pragma unroll
        for (int c = 0; c < NCH; ++c)
            if (c < nc) {
#pragma unroll
                for (int k = 0; k < 16; ++k) acc -= double(lx[c][k]) * vch[c][k0 + k];
            }
        __syncthreads();
    }
    if (has_next) {
        fetch_row(x, I + 1, vin, spin_limit, err);
#pragma unroll
        for (int k = 0; k < 16; ++k) acc -= double(ln[k]) * vin[k0 + k];
    }
    part[q][col] = acc;
    __syncthreads();
    if (tid < T) vin[tid] = part[0][tid] + part[1][tid] + part[2][tid] + part[3][tid];
    __syncthreads();
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < 16; ++k) s += double(lv[k]) * vin[k0 + k];
    part[q][col] = s;
    __syncthreads();
    if (tid < T) put_value(&x[I * T + tid], part[0][tid] + part[1][tid] + part[2][tid] + part[3][tid]);
}

// ---- sweeps with a precomputed chain matrix ----------------------------------
// In the sweeps above the last step of a tile row waits for its predecessor
// and then applies two dependent 64x64 products (L_{I,I-1} y_{I-1}, then Linv_I).
// After each factorization k_sweep_chain forms per tile row
//   M_I = Linv_I L_{I,I-1}            (column-major, for the forward sweep)
//   G_I = L_{I+1,I} Linv_I            (row-major, for the backward sweep)
// so that y_I = U_I - M_I y_{I-1}, U_I = Linv_I (b_I - sum_{J <= I-2} L_IJ y_J),
// and x_I = U'_I - G_I^T x_{I+1}, U'_I = Linv_I^T (y_I / D_I - sum_{J >= I+2} L_JI^T x_J).
// U_I needs the rows up to I-2 only, which arrive one chain step before
// y_{I-1}; once y_{I-1} lands the row takes one 64x64 product and one
// reduction.  Each workgroup still reads only its own tile row (the older
// contributions' bandwidth per workgroup is that of the sweeps above).

// tile (I, J) of the factor, I > J, read as doubles; zero outside the band
template <class R> struct TileRd {
    const R* p;
    __device__ double operator()(int r, int c) const { return p ? double(p[c * T + r]) : 0.0; }
};
template <class R> __device__ inline TileRd<R> factor_tile(const R* tiles, long I, long J, long nt, int w) {
    if (J < 0 || I >= nt || I - J > w || I - J < 1) return TileRd<R>{nullptr};
    return TileRd<R>{tiles + tile_index(I, J, w) * TT};
}
template <class R> __device__ inline TileRd<R> linv_tile(const R* linv, long I, long nt) {
    return TileRd<R>{(I >= 0 && I < nt) ? linv + I * TT : nullptr};
}

// acc[j] += sum_k A(r, k) B(k, c0 + j), j < 16 (B's reads are uniform over a wavefront)
template <class FA, class FB> __device__ inline void mm64(const FA& A, const FB& B, int r, int c0, double* acc) {
    for (int k = 0; k < T; ++k) {
        const double a = A(r, k);
#pragma unroll
        for (int j = 0; j < 16; ++j) acc[j] += a * B(k, c0 + j);
    }
}

// M_I and G_I for every tile row: one workgroup per row, thread (r, c0)
// forming entries (r, c0..c0+15) of each product.
template <class R>
__global__ void __launch_bounds__(256) k_sweep_chain(const R* __restrict__ tiles, const R* __restrict__ linv,
                                                     R* __restrict__ mch, R* __restrict__ gch, long nt, int w) {
    const long I = blockIdx.x;
    const int r = threadIdx.x % T, c0 = 16 * (threadIdx.x / T);
    double acc[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) acc[j] = 0.0;
    mm64(linv_tile(linv, I, nt), factor_tile(tiles, I, I - 1, nt, w), r, c0, acc);
#pragma unroll
    for (int j = 0; j < 16; ++j) mch[I * TT + (c0 + j) * T + r] = R(acc[j]);
#pragma unroll
    for (int j = 0; j < 16; ++j) acc[j] = 0.0;
    mm64(factor_tile(tiles, I + 1, I, nt, w), linv_tile(linv, I, nt), r, c0, acc);
#pragma unroll
    for (int j = 0; j < 16; ++j) gch[I * TT + r * T + c0 + j] = R(acc[j]);
}

// y_I = U_I - M_I y_{I-1}.  r is read from xr, whose slot I is set to SENT for
// the backward sweep; y must hold SENT.
template <class R>
__global__ void __launch_bounds__(256) k_fwd_sweep_m(const R* __restrict__ tiles, const R* __restrict__ linv,
                                                     const R* __restrict__ mch, double* __restrict__ xr, double* y,
                                                     long nt, int w, int* started, bool by_count, long spin_limit, int* err) {
    __shared__ double vin[T];
    __shared__ double vch[NCH][T];
    __shared__ double part[4][T];
    const long I = start_number(started, by_count);
    const int tid = threadIdx.x, row = tid % T, q = tid / T, k0 = 16 * q;
    R lv[16], lm[16];
    const R* lvp = linv + I * (long)TT;
#pragma unroll
    for (int k = 0; k < 16; ++k) lv[k] = lvp[(k0 + k) * T + row];
    const bool has_prev = I >= 1;
    if (has_prev) {
        const R* lmp = mch + I * (long)TT;
#pragma unroll
        for (int k = 0; k < 16; ++k) lm[k] = lmp[(k0 + k) * T + row];
    }
    double acc = 0.0;
    if (q == 0) {
        acc = xr[I * T + row];
        xr[I * T + row] = __builtin_bit_cast(double, SENT);
    }
    // the older rows J <= I - 2 in chunks of NCH, wavefront c polling row J + c
    const long J0 = I - w > 0 ? I - w : 0;
    for (long J = J0; J < I - 1; J += NCH) {
        const int nc = (I - 1 - J < NCH) ? int(I - 1 - J) : NCH;
        R lx[NCH][16];
#pragma unroll
        for (int c = 0; c < NCH; ++c)
            if (c < nc) {
                const R* l = tiles + (I * (w + 1) + (J + c - I + w)) * (long)TT;
#pragma unroll
                for (int k = 0; k < 16; ++k) lx[c][k] = l[(k0 + k) * T + row];
            }
        fetch_rows(y, J, 1, nc, vch, spin_limit, err);
#pragma unroll
        for (int c = 0; c < NCH; ++c)
            if (c < nc) {
#pragma unroll
                for (int k = 0; k < 16; ++k) acc -= double(lx[c][k]) * vch[c][k0 + k];
            }
        __syncthreads();
    }
    // U_I = Linv_I S_I, formed before y_{I-1} is needed
    part[q][row] = acc;
    __syncthreads();
    if (tid < T) vin[tid] = part[0][tid] + part[1][tid] + part[2][tid] + part[3][tid];
    __syncthreads();
    double u = 0.0;
#pragma unroll
    for (int k = 0; k < 16; ++k) u += double(lv[k]) * vin[k0 + k];
    __syncthreads();
    part[q][row] = u;
    __syncthreads();
    double yi = (q == 0) ? part[0][row] + part[1][row] + part[2][row] + part[3][row] : 0.0;
    if (has_prev) {
        fetch_row(y, I - 1, vin, spin_limit, err);
        double m = 0.0;
#pragma unroll
        for (int k = 0; k < 16; ++k) m += double(lm[k]) * vin[k0 + k];
        part[q][row] = m;
        __syncthreads();
        if (q == 0) yi -= part[0][row] + part[1][row] + part[2][row] + part[3][row];
    }
    if (q == 0) put_value(&y[I * T + row], yi);
}

// x_I = U'_I - G_I^T x_{I+1}; workgroup g handles I = nt-1-g.  x must hold SENT.
template <class R>
__global__ void __launch_bounds__(256) k_bwd_sweep_m(const R* __restrict__ tiles_t, const R* __restrict__ linv,
                                                     const R* __restrict__ gch, const double* __restrict__ y,
                                                     const double* __restrict__ piv, double* x, long nt, int w,
                                                     int* started, bool by_count, long spin_limit, int* err) {
    __shared__ double vin[T];
    __shared__ double vch[NCH][T];
    __shared__ double part[4][T];
    const long I = nt - 1 - start_number(started, by_count);
    const int tid = threadIdx.x, col = tid % T, q = tid / T, k0 = 16 * q;
    R lv[16], lm[16];
    const R* lvp = linv + I * (long)TT;
#pragma unroll
    for (int k = 0; k < 16; ++k) lv[k] = lvp[col * T + k0 + k];   // Linv[k][col]
    const bool has_next = I + 1 < nt;
    if (has_next) {
        const R* lgp = gch + I * (long)TT;
#pragma unroll
        for (int k = 0; k < 16; ++k) lm[k] = lgp[(k0 + k) * T + col];   // G_I[k][col]
    }
    double acc = (q == 0) ? y[I * T + col] / piv[I * T + col] : 0.0;
    // the later rows J >= I + 2 in chunks of NCH, wavefront c polling row J - c
    const long J1 = (I + w < nt - 1) ? I + w : nt - 1;
    for (long J = J1; J > I + 1; J -= NCH) {
        const int nc = (J - (I + 1) < NCH) ? int(J - (I + 1)) : NCH;
        R lx[NCH][16];
#pragma unroll
        for (int c = 0; c < NCH; ++c)
            if (c < nc) {
                const R* l = tiles_t + ((J - c) * (w + 1) + (I - (J - c) + w)) * (long)TT;
#pragma unroll
                for (int k = 0; k < 16; ++k) lx[c][k] = l[(k0 + k) * T + col];
            }
        fetch_rows(x, J, -1, nc, vch, spin_limit, err);
#pragma unroll
        for (int c = 0; c < NCH; ++c)
            if (c < nc) {
#pragma unroll
                for (int k = 0; k < 16; ++k) acc -= double(lx[c][k]) * vch[c][k0 + k];
            }
        __syncthreads();
    }
    part[q][col] = acc;
    __syncthreads();
    if (tid < T) vin[tid] = part[0][tid] + part[1][tid] + part[2][tid] + part[3][tid];
    __syncthreads();
    double u = 0.0;
#pragma unroll
    for (int k = 0; k < 16; ++k) u += double(lv[k]) * vin[k0 + k];
    __syncthreads();
    part[q][col] = u;
    __syncthreads();
    double xi = (q == 0) ? part[0][col] + part[1][col] + part[2][col] + part[3][col] : 0.0;
    if (has_next) {
        fetch_row(x, I + 1, vin, spin_limit, err);
        double m = 0.0;
#pragma unroll
        for (int k = 0; k < 16; ++k) m += double(lm[k]) * vin[k0 + k];
        part[q][col] = m;
        __syncthreads();
        if (q == 0) xi -= part[0][col] + part[1][col] + part[2][col] + part[3][col];
    }
    if (q == 0) put_value(&x[I * T + col], xi);
}

// ---- block sweeps --------------------------------------------------------------
// Above, every tile row waits for the one before: about 1 us a row of store,
// poll and products, however fast the tiles stream.  The look-ahead schedules
// take SB tile rows at a time.  With Linv_B the inverse of a block's SB x SB
// tiles of L, formed after each factorization,
//   y_B = Linv_B S_B - M_B y_{B-1},  S_B = b_B - sum over the rows before block B-1,
//   M_B = Linv_B L_{B,B-1},
// so a block waits once for its predecessor, and everything else of it is
// formed meanwhile.  The backward sweep is the same on L^T: x_B = Linv_B^T S'_B -
// G_B x_{B+1}, G_B = Linv_B^T L_{B+1,B}^T, S'_B = y_B / D_B - sum over the rows past
// block B+1.
// The products of a block are spread over many workgroups, which load their
// tiles into registers before they wait: a sweep has few rows in progress
// at once, and one workgroup per row could not stream a row's tiles in the
// time the front takes to pass it.  A block has 4 (gh + 1) workgroups of 512
// threads: for each row gh helpers, each with up to HT tiles of the older
// rows, which leave partial sums, and one that finishes the row.
// 256 x 256 panel (6168 rows, 25 tiles below the diagonal): 2.46 / 2.44 ms
// forward / backward (2.2 TB/s of 5.3 GB) and 2.7 ms to form the matrices per
// factorization; one row at a time took 6.2 / 6.5 ms, and systems that
// decoupled each row from the one or two before 5.1 / 5.2 ms with 11 ms of
// forming.  A band of a single block has nothing to overlap and takes the
// chain matrices (BandLDLT::blocked).
constexpr int SB = 4;      // tile rows per block
constexpr int HT = 8;      // tiles per helper; a wavefront polls one of their rows
constexpr int SWT = 512;
constexpr int LB = SB * (SB - 1) / 2;   // off-diagonal tiles of Linv_B
__device__ __forceinline__ long lb_index(long b, int i, int k) { return (b * LB + i * (i - 1) / 2 + k) * TT; }   // i > k

// Linv_B below its diagonal tiles, column by column: workgroup (b, j) forms
// Linv_ij = -Linv_i sum_{k=j}^{i-1} L_ik Linv_kj for i = j+1 .. (FP64 products)
template <class R>
__global__ void __launch_bounds__(NTH) k_block_inverse(const R* __restrict__ tiles, const R* __restrict__ linv,
                                                       R* __restrict__ lb, long nt, int w) {
    __shared__ double xs[T][T], ys[T][T];
    __shared__ double vs[SB - 2][T][T];   // Linv_kj, k > j, row-major
    const long b = blockIdx.x / (SB - 1);
    const int j = int(blockIdx.x % (SB - 1)), nr = int(min(long(SB), nt - SB * b));
    for (int i = j + 1; i < nr; ++i) {
        const long I = SB * b + i;
        double sum[TileAcc<double>::N] = {};
        TileAcc<double> acc;
        for (int k = j; k < i; ++k) {
            if (i - k > w) continue;
            stage<false>(xs, tiles + tile_index(I, SB * b + k, w) * TT);
            if (k == j) stage_t(ys, linv + (SB * b + j) * (long)TT);
            __syncthreads();
            acc.product(xs, k == j ? ys : vs[k - j - 1]);
            acc.each_i([&](int, int, double v, int e) { sum[e] += v; });
            __syncthreads();
        }
        stage<false>(xs, linv + I * (long)TT);
        acc.each_i([&](int row, int col, double, int e) { ys[row][col] = sum[e]; });
        __syncthreads();
        acc.product(xs, ys);
        R* out = lb + lb_index(b, i, j);
        acc.each([&](int row, int col, double v) {
            out[col * T + row] = R(-v);
            if (i - j - 1 < SB - 2) vs[i - j - 1][row][col] = -v;
        });
        __syncthreads();
    }
}

// Whether M_B (dir 1) or G_B (dir -1) has a tile in column j of its block: the
// row or column of the band nearest to it reaches it.
__device__ __forceinline__ bool has_link(bool fwd, long b, int j, long nt, int w) {
    return fwd ? b >= 1 && SB - j <= w : SB * (b + 1) + j < nt && j < w;
}

// Tile (i, j) of M_B (the first half of the grid) or of G_B (the second),
// column-major, at [SB b + i][j]
template <class R>
__global__ void __launch_bounds__(NTH) k_block_link(const R* __restrict__ tiles, const R* __restrict__ tiles_t,
                                                    const R* __restrict__ linv, const R* __restrict__ lb,
                                                    R* __restrict__ mch, R* __restrict__ gch, long nt, int w) {
    __shared__ double xs[T][T], ys[T][T];
    const bool fwd = blockIdx.x < nt * SB;
    const long q = fwd ? blockIdx.x : blockIdx.x - nt * SB, I = q / SB, b = I / SB;
    const int i = int(I % SB), j = int(q % SB);
    if (!has_link(fwd, b, j, nt, w)) return;
    double sum[TileAcc<double>::N] = {};
    TileAcc<double> acc;
    for (int k = fwd ? 0 : i; k <= (fwd ? i : SB - 1); ++k) {
        const long K = SB * b + k;
        if ((fwd ? SB + k - j : SB + j - k) > w) continue;
        if (fwd) {
            stage<false>(xs, k == i ? linv + I * (long)TT : lb + lb_index(b, i, k));
            stage<false>(ys, tiles_t + tile_index(K, SB * (b - 1) + j, w) * TT);
        } else {
            stage_t(xs, k == i ? linv + I * (long)TT : lb + lb_index(b, k, i));
            stage<false>(ys, tiles + tile_index(SB * (b + 1) + j, K, w) * TT);
        }
        __syncthreads();
        acc.product(xs, ys);
        acc.each_i([&](int, int, double v, int e) { sum[e] += v; });
        __syncthreads();
    }
    R* out = (fwd ? mch : gch) + q * (long)TT;
    acc.each_i([&](int row, int col, double, int e) { out[col * T + row] = R(sum[e]); });
}

inline int helpers_per_row(int w) { return std::max(0, (w - SB + HT - 1) / HT); }

// One sweep: v = the solution, every slot SENT before; part [nt][gh][T], SENT.
// FWD: v = y from rhs = b.  Otherwise v = x from rhs = y and the pivots, with
// the transposed tiles.  Workgroups in the order of the blocks, a block's
// helpers (oldest rows first) before its finishing workgroups, so that each
// waits on ones that started before it only.
template <class R, bool FWD>
__global__ void __launch_bounds__(SWT) k_sweep_block(const R* __restrict__ tl, const R* __restrict__ linv,
                                                     const R* __restrict__ lb, const R* __restrict__ link,
                                                     const double* __restrict__ rhs, const double* __restrict__ piv,
                                                     double* v, double* part, long nt, int w, int gh, int* started,
                                                     long spin_limit, int* err) {
    __shared__ double vch[HT][T];
    __shared__ double red[SWT / T][T];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, k0 = 8 * wv;
    const long nb = (nt + SB - 1) / SB, per = SB * (gh + 1), number = start_by_count(started);
    const long b = FWD ? number / per : nb - 1 - number / per;
    const int r = int(number % per), i = r % SB;
    const long I = SB * b + i;
    if (I >= nt) return;
    // older rows of row I by groups of HT, group 0 the newest: first and last
    // row (towards older rows) of group g, none left when the count is <= 0
    const int dir = FWD ? -1 : 1;
    auto group = [&](long row, int g, long& first) {
        first = FWD ? SB * (b - 1) - 1 - HT * g : SB * (b + 2) + HT * g;
        const long last = FWD ? max(0L, row - w) : min(nt - 1, row + w);
        return int(min(long(HT), FWD ? first - last + 1 : last - first + 1));
    };
    auto finish = [&](double acc, double* out) {
        red[wv][lane] = acc;
        __syncthreads();
        if (wv == 0) {
            double s = red[0][lane];
#pragma unroll
            for (int q = 1; q < SWT / T; ++q) s += red[q][lane];
            put_value(out, s);
        }
    };
    if (r < SB * gh) {
        const int g = gh - 1 - r / SB;
        long first;
        const int n = group(I, g, first);
        if (n <= 0) return;
        R lx[HT][8];
#pragma unroll
        for (int c = 0; c < HT; ++c)
            if (c < n) {
                const long J = first + dir * c;
                const R* l = tl + (FWD ? tile_index(I, J, w) : tile_index(J, I, w)) * TT;
#pragma unroll
                for (int k = 0; k < 8; ++k) lx[c][k] = l[(k0 + k) * T + lane];
            }
        if (wv < n) vch[wv][lane] = poll_value(v + (first + dir * wv) * T + lane, spin_limit, err);
        __syncthreads();
        double acc = 0.0;
#pragma unroll
        for (int c = 0; c < HT; ++c)
            if (c < n) {
#pragma unroll
                for (int k = 0; k < 8; ++k) acc -= double(lx[c][k]) * vch[c][k0 + k];
            }
        finish(acc, &part[(I * gh + g) * T + lane]);
        return;
    }
    const int nr = int(min(long(SB), nt - SB * b));
    R li[SB][8], lm[SB][8];
    bool linked[SB];
#pragma unroll
    for (int k = 0; k < SB; ++k) {
        linked[k] = has_link(FWD, b, k, nt, w);
        if (linked[k]) {
            const R* l = link + (I * SB + k) * (long)TT;
#pragma unroll
            for (int e = 0; e < 8; ++e) lm[k][e] = l[(k0 + e) * T + lane];
        }
        if (FWD ? k <= i : k >= i && k < nr) {
            const R* l = k == i ? linv + I * (long)TT : lb + (FWD ? lb_index(b, i, k) : lb_index(b, k, i));
#pragma unroll
            for (int e = 0; e < 8; ++e) li[k][e] = FWD ? l[(k0 + e) * T + lane] : l[lane * T + k0 + e];
        }
    }
    // S of the block's rows that row I needs, a wavefront each
    if (wv < SB && (FWD ? wv <= i : wv >= i && wv < nr)) {
        const long K = SB * b + wv, e = K * T + lane;
        double s = FWD ? rhs[e] : rhs[e] / piv[e];
        for (int g = gh - 1; g >= 0; --g) {
            long first;
            if (group(K, g, first) > 0) s += poll_value(&part[(K * gh + g) * T + lane], spin_limit, err);
        }
        vch[wv][lane] = s;
    }
    __syncthreads();
    double acc = 0.0;
#pragma unroll
    for (int k = 0; k < SB; ++k)
        if (FWD ? k <= i : k >= i && k < nr) {
#pragma unroll
            for (int e = 0; e < 8; ++e) acc += double(li[k][e]) * vch[k][k0 + e];
        }
    if (wv >= SB) {   // the neighbouring block's rows
        const int k = wv - SB;
        if (has_link(FWD, b, k, nt, w))
            vch[wv][lane] = poll_value(v + ((FWD ? SB * (b - 1) : SB * (b + 1)) + k) * T + lane, spin_limit, err);
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < SB; ++k)
        if (linked[k]) {
#pragma unroll
            for (int e = 0; e < 8; ++e) acc -= double(lm[k][e]) * vch[SB + k][k0 + e];
        }
    finish(acc, &v[I * T + lane]);
}

// dst = rhs padded with zeros to ntot; y, x and the partial sums SENT
__global__ void k_sweep_block_prep(double* __restrict__ dst, const double* __restrict__ src, double* __restrict__ y,
                                   double* __restrict__ x, double* __restrict__ part, long n, long ntot, long npart) {
    const double sent = __builtin_bit_cast(double, SENT);
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < max(ntot, npart); i += (long)gridDim.x * blockDim.x) {
        if (i < ntot) {
            dst[i] = i < n ? src[i] : 0.0;
            y[i] = sent;
            x[i] = sent;
        }
        if (i < npart) part[i] = sent;
    }
}

// dst = rhs padded with zeros to ntot; y = SENT
__global__ void k_sweep_prep(double* __restrict__ dst, const double* __restrict__ src, double* __restrict__ y,
                             long n, long ntot) {
    long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i < ntot) {
        dst[i] = i < n ? src[i] : 0.0;
        y[i] = __builtin_bit_cast(double, SENT);
    }
}

// ---- batches of models ---------------------------------------------------------
// Identity rows for the equations no DOF slot maps to (the tail of each
// model's last tile).
// Fills by kernel rather than hipMemsetAsync, so that a captured HIP graph of a
// batch round holds no memset node.
__global__ void k_fill_f64(double* __restrict__ y, long n) {
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) y[i] = 0.0;
}
__global__ void k_fill_i32(int* __restrict__ y, long n) {
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) y[i] = 0;
}

__global__ void k_band_gap_pad(double* __restrict__ tiles, const int32_t* __restrict__ gaps, long ngap, int w) {
    long k = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (k >= ngap) return;
    const long i = gaps[k], I = i / T;
    tiles[tile_index(I, I, w) * TT + (i % T) * T + (i % T)] = 1.0;
}

// One workgroup factors one model, column by column, with the tile arithmetic
// of the single-model schedules (so the same factor): D_K, then P_{I,K} for
// the m tiles below it, then U_{I,J,K}.  Linv_K stays in LDS for the panels.
// While m <= 2 the panels also stay in LDS (P_{K+1,K} in ys, P_{K+2,K} in lk
// once Linv_K is no longer needed), the updates take their operands from
// there, and U_{K+1,K+1,K} is applied last and left in xs, where D_{K+1}
// starts.  Wider columns take the operands of the updates from memory.  The
// barrier after each task orders its LDS and memory writes before the next
// task reads them.
//
// A model with two tiles below the diagonal may instead be factored by a pair
// of workgroups (role ROLE_MAIN and ROLE_HELPER).  The main workgroup keeps the
// critical chain D_K -> P_{K+1,K} -> U_{K+1,K+1,K} -> D_{K+1}; the helper
// computes P_{K+2,K}, U_{K+2,K+1,K} and U_{K+2,K+2,K} meanwhile.  They hand
// over through memory with system-scope stores and loads and four progress
// counters per model (the main's D_K and P_{K+1,K}, the helper's two
// updates), each raised after the writer's stores have completed.  The main
// reads A_{K+1,K} after the helper's U_{K+1,K,K-1} and A_{K+1,K+1} after its
// U_{K+1,K+1,K-1}; the helper reads Linv_K, D_K and P_{K+1,K} after the main
// has published them.  Every task keeps its arithmetic, so the factor is the
// one a single workgroup computes.  The pairs come first in the grid, so both
// workgroups of a pair are resident together; every wait is bounded and ends
// early once any wait has failed (error bit 1).
constexpr int ROLE_SINGLE = 0, ROLE_MAIN = 1, ROLE_HELPER = 2;
enum { C_DIAG = 0, C_P1 = 1, C_U21 = 2, C_U22 = 3 };

// thread 0 waits until *c >= target (or an error is raised anywhere)
__device__ inline bool wait_count(const int* c, int target, long spin_limit, int* err, int* ok_s) {
    if (threadIdx.x == 0) *ok_s = poll_count(c, target, spin_limit, err) >= target;
    __syncthreads();
    return *ok_s != 0;
}

__global__ void __launch_bounds__(NTH) k_band_factor_models(double* __restrict__ tiles, double* __restrict__ linv,
                                                            double* __restrict__ piv, int w,
                                                            const BandSeg* __restrict__ segs,
                                                            const int* __restrict__ order,
                                                            const int* __restrict__ role, int* prog,
                                                            long spin_limit, int* err) {
    __shared__ double xs[T][T];
    __shared__ double ys[TT];
    __shared__ double lk[T][T];   // Linv_K as the panels' second operand (lk[k][row] = Linv(row, k))
    __shared__ double dd[T];
    __shared__ DiagScratch<double> sm;
    __shared__ int ok_s;
    const int mdl = order[blockIdx.x], rl = role[blockIdx.x];
    const BandSeg g = segs[mdl];
    int* pc = prog + long(mdl) * 4 * FLAG_STRIDE;   // the model's progress counters
    double(*yt)[T] = reinterpret_cast<double(*)[T]>(ys);
    const long Kend = g.t0 + g.nt;
    bool staged = false;   // xs already holds A_KK
    // xs = src * D_K by column (the scaled operand of the updates)
    auto scale_into_xs = [&](const double (*src)[T], const double* dk) {
        for (int idx = threadIdx.x; idx < TT; idx += NTH) xs[idx / T][idx % T] = src[idx / T][idx % T] * dk[idx / T];
    };
    if (rl == ROLE_HELPER) {
        // P_{K+2,K}, U_{K+2,K+1,K}, U_{K+2,K+2,K} for the columns with two tiles below
        for (long K = g.t0; K + 2 < Kend; ++K) {
            const int rel = int(K - g.t0);
            if (!wait_count(pc + C_DIAG * FLAG_STRIDE, rel + 1, spin_limit, err, &ok_s)) return;
            stage<true>(lk, linv + K * (long)TT);
            if (threadIdx.x < T) dd[threadIdx.x] = cld<true>(&piv[K * T + threadIdx.x]);
            double* p2 = tiles + tile_index(K + 2, K, w) * TT;
            stage<false>(xs, p2);
            __syncthreads();
            TileAcc<double> acc;
            acc.product_ylower(xs, lk);
            acc.each([&](int row, int col, double v) {
                const double p = v * (1.0 / dd[col]);
                p2[col * T + row] = p;
                yt[col][row] = p;
            });
            __syncthreads();
            if (!wait_count(pc + C_P1 * FLAG_STRIDE, rel + 1, spin_limit, err, &ok_s)) return;
            stage<true>(lk, tiles + tile_index(K + 1, K, w) * TT);   // P_{K+1,K}
            scale_into_xs(yt, dd);
            __syncthreads();
            acc.product(xs, lk);
            double* o21 = tiles + tile_index(K + 2, K + 1, w) * TT;
            acc.each([&](int row, int col, double v) { cst<true>(&o21[col * T + row], o21[col * T + row] - v); });
            publish(pc + C_U21 * FLAG_STRIDE, rel + 1);
            acc.product(xs, yt);
            double* o22 = tiles + tile_index(K + 2, K + 2, w) * TT;
            acc.each([&](int row, int col, double v) { cst<true>(&o22[col * T + row], o22[col * T + row] - v); });
            publish(pc + C_U22 * FLAG_STRIDE, rel + 1);
        }
        return;
    }
    for (long K = g.t0; K < Kend; ++K) {
        const long m = (Kend - 1 - K < g.w) ? Kend - 1 - K : g.w;
        const bool in_lds = m <= 2;
        // A workgroup that factors its model alone stages A_{K+1,K} after the
        // diagonal task; the previous column has written it, so it is loaded
        // into registers (in the staging layout) once the pivot steps are
        // done, and its latency overlaps the rest of the diagonal task.
        const bool pre = rl != ROLE_MAIN && in_lds && m >= 1;
        double pa[TT / NTH];
        if (!staged) {
            stage<false>(xs, tiles + tile_index(K, K, w) * TT);
            __syncthreads();
        }
        staged = false;
        diag_task(xs, ys, dd, sm, linv + K * (long)TT, piv, K, &lk[0][0], [&](int k, int) {
            if (pre && k == 4) {
                const double* t1 = tiles + tile_index(K + 1, K, w) * TT;
#pragma unroll
                for (int i = 0; i < TT / NTH; ++i) pa[i] = t1[threadIdx.x + NTH * i];
            }
        });
        __syncthreads();
        const double* dk = piv + K * T;
        if (rl == ROLE_MAIN) {
            const int rel = int(K - g.t0);
            if (m == 2) {
                // Linv_K and D_K for the helper, stored again through to memory
                for (int idx = threadIdx.x; idx < TT; idx += NTH)
                    cst<true>(&linv[K * (long)TT + idx], lk[idx / T][idx % T]);
                if (threadIdx.x < T) cst<true>(&piv[K * T + threadIdx.x], piv[K * T + threadIdx.x]);
                publish(pc + C_DIAG * FLAG_STRIDE, rel + 1);
            }
            if (m >= 1) {
                // P_{K+1,K}, after the helper's U_{K+1,K,K-1}
                if (K > g.t0 && !wait_count(pc + C_U21 * FLAG_STRIDE, rel, spin_limit, err, &ok_s)) return;
                double* p1 = tiles + tile_index(K + 1, K, w) * TT;
                stage<true>(xs, p1);
                __syncthreads();
                TileAcc<double> acc;
                acc.product_ylower(xs, lk);
                acc.each([&](int row, int col, double v) {
                    const double p = v * (1.0 / dk[col]);
                    cst<true>(&p1[col * T + row], p);
                    yt[col][row] = p;
                });
                if (m == 2) publish(pc + C_P1 * FLAG_STRIDE, rel + 1);
                else __syncthreads();
                // U_{K+1,K+1,K}, after the helper's U_{K+1,K+1,K-1}; left in xs for D_{K+1}
                if (K > g.t0 && !wait_count(pc + C_U22 * FLAG_STRIDE, rel, spin_limit, err, &ok_s)) return;
                scale_into_xs(yt, dk);
                __syncthreads();
                // symmetric, and the diagonal task reads only the lower part
                LowerAcc u;
                u.product(xs, yt);
                __syncthreads();
                const double* a11 = tiles + tile_index(K + 1, K + 1, w) * TT;
                u.each_i([&](int row, int col, double v, int) { xs[col][row] = cld<true>(&a11[col * T + row]) - v; });
                __syncthreads();
                staged = true;
            }
            continue;
        }
        for (long r = 1; r <= m; ++r) {
            // P_{K+r,K} as panel_task computes it, with Linv_K from LDS
            double* tile = tiles + tile_index(K + r, K, w) * TT;
            if (pre && r == 1) {
#pragma unroll
                for (int i = 0; i < TT / NTH; ++i) {
                    const int idx = threadIdx.x + NTH * i;
                    xs[idx / T][idx % T] = pa[i];
                }
            } else {
                stage<false>(xs, tile);
            }
            __syncthreads();
            TileAcc<double> acc;
            acc.product_ylower(xs, lk);
            if (in_lds) {
                __syncthreads();   // lk is free after the last panel's product
                double(*dst)[T] = (r == 1) ? yt : lk;
                acc.each([&](int row, int col, double v) {
                    const double p = v * (1.0 / dk[col]);
                    tile[col * T + row] = p;
                    dst[col][row] = p;
                });
            } else {
                acc.each([&](int row, int col, double v) { tile[col * T + row] = v * (1.0 / dk[col]); });
            }
            __syncthreads();
        }
        if (in_lds) {
            if (m == 2) {
                // U_{K+2,K+1,K} and U_{K+2,K+2,K}: (P_{K+2} D_K) P_{K+1}^T and (P_{K+2} D_K) P_{K+2}^T
                scale_into_xs(lk, dk);
                __syncthreads();
                TileAcc<double> acc;
                acc.product(xs, yt);
                double* o21 = tiles + tile_index(K + 2, K + 1, w) * TT;
                acc.each([&](int row, int col, double v) { o21[col * T + row] -= v; });
                acc.product(xs, lk);
                double* o22 = tiles + tile_index(K + 2, K + 2, w) * TT;
                acc.each([&](int row, int col, double v) { o22[col * T + row] -= v; });
                __syncthreads();
            }
            if (m >= 1) {
                // U_{K+1,K+1,K}, left in xs for D_{K+1}: symmetric, and the
                // diagonal task reads only the lower part
                scale_into_xs(yt, dk);
                __syncthreads();
                LowerAcc u;
                u.product(xs, yt);
                __syncthreads();
                const double* a11 = tiles + tile_index(K + 1, K + 1, w) * TT;
                u.each_i([&](int row, int col, double v, int) { xs[col][row] = a11[col * T + row] - v; });
                __syncthreads();
                staged = true;
            }
        } else {
            for (long r = 1; r <= m; ++r)
                for (long c = 1; c <= r; ++c) {
                    update_task<false, double>(tiles + tile_index(K + r, K + c, w) * TT,
                                               tiles + tile_index(K + r, K, w) * TT,
                                               tiles + tile_index(K + c, K, w) * TT, piv + K * T, xs, yt);
                    __syncthreads();
                }
        }
    }
}

// One 256-thread workgroup solves one model: the forward sweep into y, then
// the backward sweep into out, tile row by tile row.  Thread (row, q) keeps the
// partial sum over columns 16q..16q+15 and the partial sums are combined in
// the order of k_fwd_sweep / k_bwd_sweep, so a model's solution is the one
// those kernels give.  The last RING rows of the solution stay in LDS, where
// every thread reads the values it needs; the first RW off-diagonal tiles of
// a row and its Linv are loaded into registers when the row starts.  A row
// then costs three barriers.
__global__ void __launch_bounds__(256) k_band_solve_models(const double* __restrict__ tiles,
                                                           const double* __restrict__ linv,
                                                           const double* __restrict__ piv, int w,
                                                           const BandSeg* __restrict__ segs,
                                                           const int* __restrict__ order,
                                                           const double* __restrict__ rhs, double* y, double* out) {
    constexpr int RING = 8, RW = 2;
    __shared__ double vin[T];
    __shared__ double part[4][T];
    __shared__ double ring[RING][T];
    const BandSeg g = segs[order[blockIdx.x]];
    const int tid = threadIdx.x, row = tid % T, q = tid / T, k0 = 16 * q;
    const long Iend = g.t0 + g.nt, e0 = g.t0 * T;
    // acc -= sum_k a[k] * (row J of the solution)[k0 + k], from the ring when
    // row J is one of the last RING rows
    auto sub_row = [&](double& acc, const double* a, const double* v, long I, long J) {
        if (I - J < RING && J - I < RING) {
            const double* rj = &ring[J % RING][k0];
#pragma unroll
            for (int k = 0; k < 16; ++k) acc -= a[k] * rj[k];
        } else {
            const double* vj = v + J * T + k0;
#pragma unroll
            for (int k = 0; k < 16; ++k) acc -= a[k] * vj[k];
        }
    };
    // acc -> combined over q -> Linv-product (lv) -> combined; thread tid < T
    // returns entry tid of the row's result
    auto finish_row = [&](double acc, const double* lv) {
        part[q][row] = acc;
        __syncthreads();
        if (tid < T) vin[tid] = part[0][tid] + part[1][tid] + part[2][tid] + part[3][tid];
        __syncthreads();
        double t = 0.0;
#pragma unroll
        for (int k = 0; k < 16; ++k) t += lv[k] * vin[k0 + k];
        part[q][row] = t;
        __syncthreads();
        double s = 0.0;
        if (tid < T) s = part[0][tid] + part[1][tid] + part[2][tid] + part[3][tid];
        return s;
    };
    // The entries of a model's band more than bw below the diagonal are zero
    // in A and in L, and Linv is lower triangular: a thread whose 16 entries
    // of a tile are all such zeros takes zeros instead of reading them (the
    // products are the same up to the sign of zero).
    // a[k] = tile entry (r0, c0 + k) of a tile d tiles below the diagonal
    auto load16 = [&](double* a, const double* l, long d, int r0, int c0, int stride_r, int stride_c) {
        if (64 * d + r0 - (c0 + 15) > g.bw) {
#pragma unroll
            for (int k = 0; k < 16; ++k) a[k] = 0.0;
        } else {
#pragma unroll
            for (int k = 0; k < 16; ++k) a[k] = l[(c0 + k) * stride_c + r0 * stride_r];
        }
    };
    double lt[RW][16], lv[16];
    for (long I = g.t0; I < Iend; ++I) {
        const long J0 = (I - g.w > g.t0) ? I - g.w : g.t0;
        const int nJ = int(I - J0);
#pragma unroll
        for (int j = 0; j < RW; ++j)
            if (j < nJ) load16(lt[j], tiles + tile_index(I, J0 + j, w) * TT, I - J0 - j, row, k0, 1, T);
        if (k0 > row) {
#pragma unroll
            for (int k = 0; k < 16; ++k) lv[k] = 0.0;
        } else {
#pragma unroll
            for (int k = 0; k < 16; ++k) lv[k] = linv[I * (long)TT + (k0 + k) * T + row];
        }
        double acc = 0.0;
        if (q == 0) {
            const long e = I * T + row;
            acc = (e - e0 < g.neq) ? rhs[e] : 0.0;
        }
#pragma unroll
        for (int j = 0; j < RW; ++j)
            if (j < nJ) sub_row(acc, lt[j], y, I, J0 + j);
        for (long J = J0 + RW; J < I; ++J) {
            double a[16];
            load16(a, tiles + tile_index(I, J, w) * TT, I - J, row, k0, 1, T);
            sub_row(acc, a, y, I, J);
        }
        const double s = finish_row(acc, lv);
        if (tid < T) {
            y[I * T + tid] = s;
            ring[I % RING][tid] = s;
        }
        __syncthreads();
    }
    for (long I = Iend - 1; I >= g.t0; --I) {
        const int col = row;
        const long J1 = (I + g.w < Iend - 1) ? I + g.w : Iend - 1;
        const int nJ = int(J1 - I);
        // tile (J, I) read by columns: entry (k0 + k, col), 64 d + k0 + k - col
        // below the diagonal
#pragma unroll
        for (int j = 0; j < RW; ++j)
            if (j < nJ) {
                const double* l = tiles + tile_index(J1 - j, I, w) * TT;
                const long d = J1 - j - I;
                if (64 * d + k0 - col > g.bw) {
#pragma unroll
                    for (int k = 0; k < 16; ++k) lt[j][k] = 0.0;
                } else {
#pragma unroll
                    for (int k = 0; k < 16; ++k) lt[j][k] = l[col * T + k0 + k];
                }
            }
        if (k0 + 15 < col) {
#pragma unroll
            for (int k = 0; k < 16; ++k) lv[k] = 0.0;
        } else {
#pragma unroll
            for (int k = 0; k < 16; ++k) lv[k] = linv[I * (long)TT + col * T + k0 + k];
        }
        double acc = (q == 0) ? y[I * T + col] / piv[I * T + col] : 0.0;
#pragma unroll
        for (int j = 0; j < RW; ++j)
            if (j < nJ) sub_row(acc, lt[j], out, I, J1 - j);
        for (long J = J1 - RW; J > I; --J) {
            const double* l = tiles + tile_index(J, I, w) * TT;
            double a[16];
            if (64 * (J - I) + k0 - col > g.bw) {
#pragma unroll
                for (int k = 0; k < 16; ++k) a[k] = 0.0;
            } else {
#pragma unroll
                for (int k = 0; k < 16; ++k) a[k] = l[col * T + k0 + k];
            }
            sub_row(acc, a, out, I, J);
        }
        const double s = finish_row(acc, lv);
        if (tid < T) {
            out[I * T + tid] = s;
            ring[I % RING][tid] = s;
        }
        __syncthreads();
    }
}

}  // namespace

void KernelClock::begin(int f, hipStream_t s, long n) {
    if (used + 2 > ev.size()) {
        size_t old = ev.size();
        ev.resize(old + 4096);
        for (size_t i = old; i < ev.size(); ++i) CB_CHECK(hipEventCreate(&ev[i]));
    }
    fam.push_back(f);
    count.push_back(n);
    CB_CHECK(hipEventRecord(ev[used++], s));
}

void KernelClock::end(hipStream_t s) { CB_CHECK(hipEventRecord(ev[used++], s)); }

void KernelClock::collect() {
    for (size_t i = 0; i < fam.size(); ++i) {
        float t = 0;
        CB_CHECK(hipEventElapsedTime(&t, ev[2 * i], ev[2 * i + 1]));
        ms_timed[fam[i]] += t;
        n_timed[fam[i]] += count[i];
    }
    for (int f = 0; f < KT_N; ++f)
        ms[f] = n_timed[f] > 0 ? ms_timed[f] * double(launches[f]) / double(n_timed[f]) : 0.0;
    fam.clear();
    count.clear();
    used = 0;
}

void KernelClock::release() {
    for (hipEvent_t e : ev) (void)hipEventDestroy(e);
    ev.clear();
    fam.clear();
    count.clear();
    used = 0;
}

template <class R>
void BandLDLT<R>::setup(long n_, long bandwidth, hipStream_t s_) {
    release();
    n = n_;
    s = s_;
    nt = (n + T - 1) / T;
    w = int((std::max(bandwidth, 1L) + T - 1) / T);
    if (w > nt - 1) w = int(std::max(nt - 1, 0L));
    tiles = dalloc<R>(size_t(nt) * size_t(w + 1) * TT);
    tiles_t = dalloc<R>(size_t(nt) * size_t(w + 1) * TT);
    linv = dalloc<R>(size_t(nt) * TT);
    piv = dalloc<double>(size_t(nt) * T);
    xw = dalloc<double>(size_t(nt) * T);
    yw = dalloc<double>(size_t(nt) * T);
    flag = dalloc<int>(size_t(PSTRIDE + 2 * start_counters(nt)));
    prog = dalloc<int>(size_t(P_N * nt * PSTRIDE + start_counters(factor_workgroups(nt, w))));
    CB_CHECK(hipMemsetAsync(flag, 0, sizeof(int) * size_t(PSTRIDE + 2 * start_counters(nt)), s));
    piv_host.resize(size_t(n));
    CB_CHECK(hipStreamSynchronize(s));
}

template <class R>
void BandLDLT<R>::release() {
    void* ps[] = {tiles, tiles_t, linv, lb, mch, gch, cmat, gmat, piv, xw, yw, bw, part, flag, prog};
    for (void* p : ps)
        if (p) (void)hipFree(p);
    tiles = nullptr; tiles_t = nullptr; linv = nullptr; piv = nullptr; xw = nullptr; yw = nullptr; flag = nullptr;
    cmat = nullptr; gmat = nullptr;
    lb = nullptr; mch = nullptr; gch = nullptr; bw = nullptr; part = nullptr;
    prog = nullptr;
    factored = false;
    clock.release();
}

template <class R>
int BandLDLT<R>::factor(const Dev& d) {
    factored = false;
    // the fused schedule takes the matrix from tiles_t
    R* band = split ? tiles : tiles_t;
    CB_CHECK(hipMemsetAsync(band, 0, sizeof(R) * size_t(nt) * (w + 1) * TT, s));
    CB_CHECK(hipMemsetAsync(flag, 0, sizeof(int) * size_t(PSTRIDE + 2 * start_counters(nt)), s));
    if (src32)
        hipLaunchKernelGGL((k_band_from_bsr<R, float>), dim3(int((d.nslot + 255) / 256)), dim3(256), 0, s, band,
                           d.K32, d.rowptr, d.colidx, d.eq_of_slot, d.nj, d.bs, w, flag);
    else
        hipLaunchKernelGGL((k_band_from_bsr<R>), dim3(int((d.nslot + 255) / 256)), dim3(256), 0, s, band,
                           d.K, d.rowptr, d.colidx, d.eq_of_slot, d.nj, d.bs, w, flag);
    if (nt * T > n)
        hipLaunchKernelGGL((k_band_pad<R>), dim3(1), dim3(T), 0, s, band, n, nt, w);
    CB_CHECK(hipGetLastError());
    if (!split) {
        const long grid = factor_workgroups(nt, w);
        CB_CHECK(hipMemsetAsync(prog, 0, sizeof(int) * size_t(P_N * nt * PSTRIDE + start_counters(grid)), s));
        const bool tk_column = clock.on(KT_COLUMN);
        if (tk_column) {
            clock.launches[KT_COLUMN] += nt;
            clock.begin(KT_COLUMN, s, nt);
        }
        hipLaunchKernelGGL((k_band_factor<R>), dim3(unsigned(grid)), dim3(NTH), 0, s, tiles,
                           tiles_t, linv, piv, w, nt, prog, prog + P_N * nt * PSTRIDE, by_count(grid), spin_limit, flag);
        if (tk_column) clock.end(s);
    } else {
        for (long Kt = 0; Kt < nt; ++Kt) {
            const bool tk_diag = clock.take(KT_DIAG);
            if (tk_diag) clock.begin(KT_DIAG, s);
            hipLaunchKernelGGL((k_tile_diag<R>), dim3(1), dim3(NTH), 0, s, tiles, linv, piv, Kt, w);
            if (tk_diag) clock.end(s);
            const long m = std::min<long>(w, nt - 1 - Kt);
            if (m > 0) {
                const bool tk_panel = clock.take(KT_PANEL);
                if (tk_panel) clock.begin(KT_PANEL, s);
                hipLaunchKernelGGL((k_tile_panel<R>), dim3(int(m)), dim3(NTH), 0, s, tiles, tiles_t, linv, piv, Kt,
                                   w);
                if (tk_panel) clock.end(s);
                const bool tk_update = clock.take(KT_UPDATE);
                if (tk_update) clock.begin(KT_UPDATE, s);
                hipLaunchKernelGGL((k_tile_update<R>), dim3(int(m * (m + 1) / 2)), dim3(NTH), 0, s, tiles, piv,
                                   Kt, w);
                if (tk_update) clock.end(s);
            }
        }
    }
    CB_CHECK(hipGetLastError());
    // each by itself: one that fails leaves the others for the next factorization
    auto need = [](auto*& p, long count) {
        if (!p) p = dalloc<std::remove_reference_t<decltype(*p)>>(size_t(count));
    };
    if (chained && !blocked()) {
        need(cmat, nt * TT);
        need(gmat, nt * TT);
        const bool tk_prep = clock.take(KT_PREP);
        if (tk_prep) clock.begin(KT_PREP, s);
        hipLaunchKernelGGL((k_sweep_chain<R>), dim3(int(nt)), dim3(256), 0, s, tiles, linv, cmat, gmat, nt, w);
        if (tk_prep) clock.end(s);
        CB_CHECK(hipGetLastError());
    }
    if (blocked()) {
        const bool tk_prep = clock.take(KT_PREP);
        if (tk_prep) clock.begin(KT_PREP, s);
        const long nb = (nt + SB - 1) / SB;
        need(lb, nb * LB * TT);
        need(mch, nt * SB * TT);
        need(gch, nt * SB * TT);
        need(bw, nt * T);
        need(part, 2 * nt * helpers_per_row(w) * T);
        hipLaunchKernelGGL((k_block_inverse<R>), dim3(unsigned(nb * (SB - 1))), dim3(NTH), 0, s, tiles, linv, lb, nt,
                           w);
        hipLaunchKernelGGL((k_block_link<R>), dim3(unsigned(2 * nt * SB)), dim3(NTH), 0, s, tiles, tiles_t, linv, lb,
                           mch, gch, nt, w);
        if (tk_prep) clock.end(s);
        CB_CHECK(hipGetLastError());
    }
    int bad = 0;
    CB_CHECK(hipMemcpyAsync(&bad, flag, sizeof(int), hipMemcpyDeviceToHost, s));
    CB_CHECK(hipMemcpyAsync(piv_host.data(), piv, sizeof(double) * size_t(n), hipMemcpyDeviceToHost, s));
    CB_CHECK(hipStreamSynchronize(s));
    clock.collect();
    if (bad & 1) throw DeviceError("band factorization: a wait exceeded its bound");
    if (bad & 2) return 2;
    factored = true;
    for (long i = 0; i < n; ++i)
        if (piv_host[i] == 0.0 || !std::isfinite(piv_host[i])) return 1;
    return 0;
}

template <class R>
void BandLDLT<R>::solve(const double* rhs, double* out) {
    if (!factored) throw DeviceError("band solve: there is no factorization to solve with");
    CB_CHECK(hipMemsetAsync(flag, 0, sizeof(int) * size_t(PSTRIDE + 2 * start_counters(nt)), s));
    const long ntot = nt * T;
    const int gh = helpers_per_row(w);
    const long npart = nt * gh * T;
    const unsigned grid = unsigned((nt + SB - 1) / SB * SB * (gh + 1));
    if (blocked())
        hipLaunchKernelGGL(k_sweep_block_prep, dim3(int(std::min(2048L, (std::max(ntot, 2 * npart) + 255) / 256))),
                           dim3(256), 0, s, bw, rhs, yw, xw, part, n, ntot, 2 * npart);
    else
        hipLaunchKernelGGL(k_sweep_prep, dim3(int((ntot + 255) / 256)), dim3(256), 0, s, xw, rhs, yw, n, ntot);
    const bool tk_fwd = clock.take(KT_FWD);
    if (tk_fwd) clock.begin(KT_FWD, s);
    if (blocked())
        hipLaunchKernelGGL((k_sweep_block<R, true>), dim3(grid), dim3(SWT), 0, s, tiles, linv, lb, mch, bw, piv, yw,
                           part, nt, w, gh, flag + PSTRIDE, spin_limit, flag);
    else if (chained)
        hipLaunchKernelGGL((k_fwd_sweep_m<R>), dim3(int(nt)), dim3(256), 0, s, tiles, linv, cmat, xw, yw, nt, w,
                           flag + PSTRIDE, by_count(nt), spin_limit, flag);
    else
        hipLaunchKernelGGL((k_fwd_sweep<R>), dim3(int(nt)), dim3(256), 0, s, tiles, linv, xw, yw, nt, w,
                           flag + PSTRIDE, by_count(nt), spin_limit, flag);
    if (tk_fwd) clock.end(s);
    const bool tk_bwd = clock.take(KT_BWD);
    if (tk_bwd) clock.begin(KT_BWD, s);
    if (blocked())
        hipLaunchKernelGGL((k_sweep_block<R, false>), dim3(grid), dim3(SWT), 0, s, tiles_t, linv, lb, gch, yw, piv, xw,
                           part + npart, nt, w, gh, flag + PSTRIDE + start_counters(nt), spin_limit, flag);
    else if (chained)
        hipLaunchKernelGGL((k_bwd_sweep_m<R>), dim3(int(nt)), dim3(256), 0, s, tiles_t, linv, gmat, yw, piv, xw, nt, w,
                           flag + PSTRIDE + start_counters(nt), by_count(nt), spin_limit, flag);
    else
        hipLaunchKernelGGL((k_bwd_sweep<R>), dim3(int(nt)), dim3(256), 0, s, tiles_t, linv, yw, piv, xw, nt, w,
                           flag + PSTRIDE + start_counters(nt), by_count(nt), spin_limit, flag);
    if (tk_bwd) clock.end(s);
    CB_CHECK(hipGetLastError());
    CB_CHECK(hipMemcpyAsync(out, xw, sizeof(double) * size_t(n), hipMemcpyDeviceToDevice, s));
    int bad = 0;
    CB_CHECK(hipMemcpyAsync(&bad, flag, sizeof(int), hipMemcpyDeviceToHost, s));
    CB_CHECK(hipStreamSynchronize(s));
    clock.collect();
    if (bad & 1) throw DeviceError("band solve: a tile-row wait exceeded its bound");
}

template struct BandLDLT<double>;
template struct BandLDLT<float>;

void BandBatch::setup(const std::vector<BandSeg>& sg, long n_total, int w_band, const std::vector<int32_t>& gap_eqs,
                      hipStream_t s_) {
    release();
    s = s_;
    n = n_total;
    if (n % T) throw DeviceError("band batch: the equations of a batch fill whole tiles");
    nt = n / T;
    w = w_band;
    segs_host = sg;
    nseg = int(sg.size());
    for (const BandSeg& g : sg)
        if (g.t0 < 0 || g.t0 + g.nt > nt || g.w > w || g.w < 0 || g.neq > g.nt * T)
            throw DeviceError("band batch: a model's tile range does not fit the band");
    // models in decreasing order of their tile work, so the longest
    // factorizations start first; the models with two tiles below the
    // diagonal (as many as fit with their helpers into the first workgroups
    // the GPU holds at once) get a helper workgroup and come first, in pairs
    std::vector<int> mo(sg.size());
    for (size_t i = 0; i < mo.size(); ++i) mo[i] = int(i);
    auto work = [&](int i) { return double(sg[i].nt) * double((sg[i].w + 1) * (sg[i].w + 2) / 2); };
    std::stable_sort(mo.begin(), mo.end(), [&](int a, int b) { return work(a) > work(b); });
    work_order = mo;
    // the factor kernel's LDS allows one workgroup per CU: the pairs stay
    // within the first CUs - 32 workgroups of the grid
    int dev = 0, ncu = 0;
    CB_CHECK(hipGetDevice(&dev));
    CB_CHECK(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
    int eligible = 0;
    for (const BandSeg& g : sg) eligible += (g.w == 2 && g.nt >= 3);
    max_pairs = std::max(0, std::min({96, (ncu - 32) / 2, eligible}));
    tiles = dalloc<double>(size_t(nt) * size_t(w + 1) * TT);
    linv = dalloc<double>(size_t(nt) * TT);
    piv = dalloc<double>(size_t(nt) * T);
    yw = dalloc<double>(size_t(nt) * T);
    flag = dalloc<int>(1);
    CB_CHECK(hipHostMalloc(&flag_host, sizeof(int), hipHostMallocDefault));
    *flag_host = 0;
    segs = dalloc<BandSeg>(sg.size());
    order = dalloc<int>(sg.size() + size_t(max_pairs));
    role = dalloc<int>(sg.size() + size_t(max_pairs));
    sorder = dalloc<int>(mo.size());
    prog = dalloc<int>(sg.size() * 4 * FLAG_STRIDE);
    ngap = long(gap_eqs.size());
    gaps = dalloc<int32_t>(size_t(ngap));
    h2d(segs, sg.data(), sg.size(), s);
    set_pairs(max_pairs);
    h2d(sorder, mo.data(), mo.size(), s);
    h2d(gaps, gap_eqs.data(), gap_eqs.size(), s);
    CB_CHECK(hipMemsetAsync(piv, 0, sizeof(double) * size_t(nt) * T, s));
    for (hipEvent_t& e : ev) CB_CHECK(hipEventCreate(&e));
    CB_CHECK(hipStreamSynchronize(s));
}

void BandBatch::release() {
    for (hipEvent_t& e : ev)
        if (e) {
            (void)hipEventDestroy(e);
            e = nullptr;
        }
    void* ps[] = {tiles, linv, piv, yw, flag, segs, order, role, sorder, prog, gaps};
    for (void* p : ps)
        if (p) (void)hipFree(p);
    if (flag_host) (void)hipHostFree(flag_host);
    tiles = linv = piv = yw = nullptr;
    flag = nullptr;
    flag_host = nullptr;
    segs = nullptr;
    order = nullptr;
    role = nullptr;
    sorder = nullptr;
    prog = nullptr;
    gaps = nullptr;
}

void BandBatch::zero() {
    const long nv = nt * long(w + 1) * TT;
    hipLaunchKernelGGL(k_fill_f64, dim3(int(std::min<long>(8192, (nv + 255) / 256))), dim3(256), 0, s, tiles, nv);
    hipLaunchKernelGGL(k_fill_i32, dim3(1), dim3(64), 0, s, flag, 1L);
    CB_CHECK(hipGetLastError());
}

void BandBatch::factor(const Dev& d) {
    if (!nseg) return;
    zero();
    hipLaunchKernelGGL((k_band_from_bsr<double>), dim3(int((d.nslot + 255) / 256)), dim3(256), 0, s, tiles, d.K,
                       d.rowptr, d.colidx, d.eq_of_slot, d.nj, d.bs, w, flag);
    factor_filled();
}

void BandBatch::factor_filled(bool fetch_flag) {
    if (!nseg) return;
    if (ngap)
        hipLaunchKernelGGL(k_band_gap_pad, dim3(int((ngap + 255) / 256)), dim3(256), 0, s, tiles, gaps, ngap, w);
    const long np = long(nseg) * 4 * FLAG_STRIDE;
    hipLaunchKernelGGL(k_fill_i32, dim3(int(std::min<long>(1024, (np + 255) / 256))), dim3(256), 0, s, prog, np);
    const long spin_limit = 1L << 22;
    if (timing) CB_CHECK(hipEventRecord(ev[0], s));
    hipLaunchKernelGGL(k_band_factor_models, dim3(nwg), dim3(NTH), 0, s, tiles, linv, piv, w, segs, order, role, prog,
                       spin_limit, flag);
    if (timing) CB_CHECK(hipEventRecord(ev[1], s));
    CB_CHECK(hipGetLastError());
    if (fetch_flag) this->fetch_flag();
}

void BandBatch::fetch_flag() {
    CB_CHECK(hipMemcpyAsync(flag_host, flag, sizeof(int), hipMemcpyDeviceToHost, s));
}

void BandBatch::set_pairs(int np) {
    np = std::max(0, std::min(np, max_pairs));
    std::vector<int> ord, rol;
    std::vector<char> paired(segs_host.size(), 0);
    npair = 0;
    for (int i : work_order)
        if (segs_host[size_t(i)].w == 2 && segs_host[size_t(i)].nt >= 3 && npair < np) {
            ord.push_back(i);
            rol.push_back(ROLE_MAIN);
            ord.push_back(i);
            rol.push_back(ROLE_HELPER);
            paired[size_t(i)] = 1;
            ++npair;
        }
    for (int i : work_order)
        if (!paired[size_t(i)]) {
            ord.push_back(i);
            rol.push_back(ROLE_SINGLE);
        }
    nwg = int(ord.size());
    h2d(order, ord.data(), ord.size(), s);
    h2d(role, rol.data(), rol.size(), s);
    CB_CHECK(hipStreamSynchronize(s));
}

std::vector<std::pair<int, double>> BandBatch::tune_pairs(const std::vector<int>& cand) {
    std::vector<std::pair<int, double>> out;
    if (!nseg || cand.empty()) return out;
    const size_t nbytes = sizeof(double) * size_t(nt) * size_t(w + 1) * TT;
    double* save = dalloc<double>(nbytes / sizeof(double));
    CB_CHECK(hipMemcpyAsync(save, tiles, nbytes, hipMemcpyDeviceToDevice, s));
    hipEvent_t e0 = nullptr, e1 = nullptr;
    CB_CHECK(hipEventCreate(&e0));
    CB_CHECK(hipEventCreate(&e1));
    const bool keep_timing = timing;
    timing = false;
    int best = max_pairs;
    double best_ms = 1e300;
    for (int c : cand) {
        double ms = 1e300;
        bool bad = false;
        for (int rep = 0; rep < 2 && !bad; ++rep) {
            CB_CHECK(hipMemcpyAsync(tiles, save, nbytes, hipMemcpyDeviceToDevice, s));
            CB_CHECK(hipMemsetAsync(flag, 0, sizeof(int), s));
            set_pairs(c);
            CB_CHECK(hipEventRecord(e0, s));
            factor_filled(true);
            CB_CHECK(hipEventRecord(e1, s));
            CB_CHECK(hipStreamSynchronize(s));
            float t = 0;
            CB_CHECK(hipEventElapsedTime(&t, e0, e1));
            if (*flag_host & 1) bad = true;
            ms = std::min(ms, double(t));
        }
        out.emplace_back(npair, bad ? -1.0 : ms);
        if (!bad && ms < best_ms) {
            best_ms = ms;
            best = npair;
        }
    }
    timing = keep_timing;
    CB_CHECK(hipMemcpyAsync(tiles, save, nbytes, hipMemcpyDeviceToDevice, s));
    CB_CHECK(hipMemsetAsync(flag, 0, sizeof(int), s));
    CB_CHECK(hipStreamSynchronize(s));
    (void)hipFree(save);
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    set_pairs(best);
    return out;
}

void BandBatch::solve(const double* rhs, double* out) {
    if (!nseg) return;
    if (timing) CB_CHECK(hipEventRecord(ev[2], s));
    hipLaunchKernelGGL(k_band_solve_models, dim3(nseg), dim3(256), 0, s, tiles, linv, piv, w, segs, sorder, rhs, yw,
                       out);
    if (timing) CB_CHECK(hipEventRecord(ev[3], s));
    CB_CHECK(hipGetLastError());
}

}  // namespace cb
