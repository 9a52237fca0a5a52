// MFMA tile engine shared by the K contraction and the metric solve.
//
// One workgroup (256 threads = 4 wavefronts as 2 x 2) computes a BM x BN
// tile of C = sum_k A[m, k] B[k, n] over nk K-steps of BK = 16.  Operands are
// staged through double-buffered LDS (A as As[k][m], B as Bs[k][n]) with the
// K-step after the next held in registers while the current step's MFMAs
// run, so there is one barrier per K-step.  Loaders decide where a tile comes
// from (packed triangle, row-major matrix, transformed block ...) and convert
// to the engine's element type T on the way into LDS:
//
//   struct Loader {
//     using reg_t = ...;                      // register type (the source type)
//     static constexpr int N;                 // elements per thread per K-step
//     void load(int kt, reg_t (&r)[N]);       // global -> registers
//     static constexpr int SWZ;               // swizzle of its LDS rows
//     void store(const reg_t (&r)[N], T *lds, int pitch);   // convert -> LDS
//   };
//
// Prefetched values stay in the source type until the store, so converting
// them never makes the current K-step's MFMAs wait on the prefetch.
//
// T = double: v_mfma_f64_16x16x4_f64; T = float: v_mfma_f32_16x16x4_f32.
// Lane layouts measured on gfx950 with one-hot probes: A lane = m + 16 k,
// B lane = n + 16 k for both; the result element v of lane l is row
// l/16 + 4 v (f64) or 4 (l/16) + v (f32), column l % 16.
#pragma once
#include "mdf_common.h"

typedef float float4_t __attribute__((ext_vector_type(4)));

// LDS (address space 3) pointers: operand reads through them compile to
// ds_read; through a generic pointer they become flat loads that wait on the
// in-flight global prefetch (s_waitcnt vmcnt(0)) and break the pipeline.
#define MDF_LDS __attribute__((address_space(3)))

namespace mdf {

constexpr int G_THREADS = 256;
constexpr int G_BK = 16;

template <typename T>
struct Mfma;

template <>
struct Mfma<double> {
    using acc_t = double4_t;
    __device__ __forceinline__ static acc_t mma(double a, double b, acc_t c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    __device__ __forceinline__ static int row(int lane, int v) { return (lane >> 4) + 4 * v; }
};

template <>
struct Mfma<float> {
    using acc_t = float4_t;
    __device__ __forceinline__ static acc_t mma(float a, float b, acc_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    __device__ __forceinline__ static int row(int lane, int v) { return 4 * (lane >> 4) + v; }
};

__device__ __forceinline__ double4_t mfma16(double a, double b, double4_t c) { return Mfma<double>::mma(a, b, c); }

// Row k of an operand's LDS tile may hold its elements permuted, element m at
// m ^ swizzle<SWZ>(k), so that the stores of a loader whose lanes run along k
// spread over the banks (the pitch, 32 banks modulo 64, keeps the reads free
// of conflicts either way).  SWZ, the loader's: 0 none; 1 lanes of 16 single
// k by 4 rows; 2 of 8 k pairs (16 bytes of double) by 8 rows; 3 of 4 k
// quadruples (16 bytes of float) by 16 rows.
template <int SWZ>
__device__ __forceinline__ constexpr int swizzle(int k) {
    return SWZ == 1 ? ((k >> 1) & 3) << 2 : SWZ == 2 ? ((k >> 1) & 3) << 3 : SWZ == 3 ? ((k >> 2) & 3) << 4 : 0;
}

// A workgroup of WGM x WGN wavefronts (64 WGM WGN threads) computes a
// BM x BN tile; wavefront w owns sub-tile (w % WGM, w / WGM).
template <int BM, int BN, int WGM = 2, int WGN = 2>
struct TileShape {
    static constexpr int THREADS = 64 * WGM * WGN;
    static constexpr int WM = BM / WGM, WN = BN / WGN;   // per-wave tile
    static constexpr int MI = WM / 16, NI = WN / 16;     // MFMA tiles per wave
    static_assert(MI * 16 == WM && NI * 16 == WN, "wave tile must be a multiple of 16");
    static constexpr int PA = BM + 16, PB = BN + 16;     // LDS pitches (elements)
    static constexpr int LDS_ELEMS = 2 * G_BK * (PA + PB);
    static constexpr int LDS_DOUBLES = LDS_ELEMS;
};

// Accumulator tile of one wavefront.
template <int MI, int NI, typename T = double>
struct Acc {
    typename Mfma<T>::acc_t v[MI][NI];
    __device__ __forceinline__ void zero() {
#pragma unroll
        for (int a = 0; a < MI; a++)
#pragma unroll
            for (int b = 0; b < NI; b++) v[a][b] = typename Mfma<T>::acc_t{0, 0, 0, 0};
    }
};

// Runs the K loop.  `lds` must hold TileShape<BM,BN,WGM,WGN>::LDS_ELEMS
// elements of T.
template <int BM, int BN, class LA, class LB, typename T = double, int WGM = 2, int WGN = 2>
__device__ __forceinline__ void gemm_mainloop(LA &la, LB &lb, int nk, T *lds,
                                     Acc<TileShape<BM, BN, WGM, WGN>::MI, TileShape<BM, BN, WGM, WGN>::NI, T> &acc) {
    using S = TileShape<BM, BN, WGM, WGN>;
    constexpr int SA = G_BK * S::PA, SB = G_BK * S::PB;
    static_assert(LA::SWZ < 2 || (S::MI & (S::MI - 1)) == 0, "a swizzled operand has 2^n blocks a wavefront");
    static_assert(LB::SWZ < 2 || (S::NI & (S::NI - 1)) == 0, "a swizzled operand has 2^n blocks a wavefront");
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wm = wave % WGM, wn = wave / WGM;
    T *const Bbase = lds + 2 * SA;
    const MDF_LDS T *const Ar = (const MDF_LDS T *)lds, *const Br = (const MDF_LDS T *)Bbase;
    const int q4 = lane >> 4;
    const int la15 = (lane & 15) ^ swizzle<LA::SWZ>(q4), lb15 = (lane & 15) ^ swizzle<LB::SWZ>(q4);
    typename LA::reg_t ra[LA::N];
    typename LB::reg_t rb[LB::N];
    if (nk <= 0) return;
    T a[2][S::MI], b[2][S::NI];
    auto read = [&](int buf, int kq, int s) {
        // the swizzle of k = 4 kq + q4 is that of q4 (lane bits) and of 4 kq
        // (a constant here: lane bits below 16, MFMA blocks above)
        const int kk = kq * 4 + q4, xa = swizzle<LA::SWZ>(kq * 4), xb = swizzle<LB::SWZ>(kq * 4);
        const int ba = xa >> 4, bb = xb >> 4;
        const MDF_LDS T *A = Ar + buf * SA + kk * S::PA + (wm ^ (ba / S::MI)) * S::WM + (la15 ^ (xa & 15));
        const MDF_LDS T *B = Br + buf * SB + kk * S::PB + (wn ^ (bb / S::NI)) * S::WN + (lb15 ^ (xb & 15));
#pragma unroll
        for (int mi = 0; mi < S::MI; mi++) a[s][mi] = A[(ba ? mi ^ (ba % S::MI) : mi) * 16];
#pragma unroll
        for (int ni = 0; ni < S::NI; ni++) b[s][ni] = B[(bb ? ni ^ (bb % S::NI) : ni) * 16];
    };
    la.load(0, ra);
    lb.load(0, rb);
    la.store(ra, lds, S::PA);
    lb.store(rb, Bbase, S::PB);
    if (nk > 1) {
        la.load(1, ra);
        lb.load(1, rb);
    }
    __syncthreads();
    read(0, 0, 0);
    for (int kt = 0; kt < nk; kt++) {
        const int cur = kt & 1;
        const bool more = kt + 1 < nk;
#pragma unroll
        for (int kq = 0; kq < G_BK / 4; kq++) {
            // the operands of the next MFMA group are read before this
            // group's MFMAs issue, so they arrive under them; the step's
            // barrier stands before its last group, whose operands are in
            // registers: the next step's first reads run under that group
            if (kq < G_BK / 4 - 1) {
                read(cur, kq + 1, (kq + 1) & 1);
            } else if (more) {
                __syncthreads();
                read(cur ^ 1, 0, (kq + 1) & 1);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int mi = 0; mi < S::MI; mi++)
#pragma unroll
                for (int ni = 0; ni < S::NI; ni++)
                    acc.v[mi][ni] = Mfma<T>::mma(a[kq & 1][mi], b[kq & 1][ni], acc.v[mi][ni]);
            __builtin_amdgcn_sched_barrier(0);
            // halfway through a step's MFMAs the next step's tile goes into
            // the other buffer (read by no wave since the last barrier) and
            // the loads of the step after it start: they have a whole step,
            // from here to the next one's middle, to arrive
            if (kq == G_BK / 8 - 1 && more) {
                la.store(ra, lds + (cur ^ 1) * SA, S::PA);
                lb.store(rb, Bbase + (cur ^ 1) * SB, S::PB);
                if (kt + 2 < nk) {
                    la.load(kt + 2, ra);
                    lb.load(kt + 2, rb);
                }
            }
        }
    }
    __syncthreads();        // the LDS may be reused by the caller
}

// Visits every accumulator element with its tile-local (row, col); the
// element-to-row layout is that of the MFMA type LT (an FP64 shadow of an
// FP32 accumulator keeps the FP32 layout).
template <int BM, int BN, typename LT, class AccT, class F, int WGM = 2, int WGN = 2>
__device__ __forceinline__ void gemm_epilogue_layout(const AccT &acc, F &&f) {
    using S = TileShape<BM, BN, WGM, WGN>;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wm = wave % WGM, wn = wave / WGM;
#pragma unroll
    for (int mi = 0; mi < S::MI; mi++)
#pragma unroll
        for (int ni = 0; ni < S::NI; ni++) {
            const int c = wn * S::WN + ni * 16 + (lane & 15);
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int r = wm * S::WM + mi * 16 + Mfma<LT>::row(lane, v);
                f(r, c, acc.v[mi][ni][v]);
            }
        }
}

template <int BM, int BN, typename T = double, class F>
__device__ __forceinline__ void gemm_epilogue(const Acc<TileShape<BM, BN>::MI, TileShape<BM, BN>::NI, T> &acc, F &&f) {
    gemm_epilogue_layout<BM, BN, T>(acc, f);
}

// ---------------------------------------------------------------- loaders
// Two or four neighbouring elements loaded at once, at the alignment of one.
template <typename S, int N>
struct alignas(sizeof(S)) Piece {
    S v[N];
};

// Row-major matrix M[row][k] (k contiguous, element type Src) as the A or B
// operand: tile rows r0 .. r0+R-1, K-step kt covers k = kt*BK .. +BK-1, out of
// range k read 0.  Eight lanes take the 16 k of one row in pairs, so a load
// instruction reads whole 128-byte rows (a thread per 8 k of a row touched
// every line four times: 3.2 times the cache accesses in K's step 2).
// Rows past the last repeat it (their results are not used).
template <int R, typename T = double, typename Src = double, int THREADS = G_THREADS>
struct RowsLoader {
    using reg_t = Src;
    static constexpr int N = R * G_BK / THREADS, Q = N / 2;
    static constexpr int RPP = THREADS / 8;              // rows per piece
    static constexpr int SWZ = 2;
    static_assert(Q >= 1 && Q * RPP == R, "RowsLoader shape");
    const Src *p[Q];          // this thread's rows, at k0
    int nk;                   // k in range from there
    __device__ __forceinline__ RowsLoader(const Src *base, long ld, int r0, int nrows, int k0, int kmax) {
#pragma unroll
        for (int q = 0; q < Q; q++)
            p[q] = base + (long)min(r0 + (int)(threadIdx.x >> 3) + q * RPP, nrows - 1) * ld + k0;
        nk = kmax - k0;
    }
    __device__ __forceinline__ void load(int kt, Src (&r)[N]) const {
        const int k = kt * G_BK + 2 * (int)(threadIdx.x & 7);
        if ((kt + 1) * G_BK <= nk) {
#pragma unroll
            for (int q = 0; q < Q; q++) {
                const Piece<Src, 2> x = *(const Piece<Src, 2> *)(p[q] + k);
                r[2 * q] = x.v[0];
                r[2 * q + 1] = x.v[1];
            }
            return;
        }
#pragma unroll
        for (int q = 0; q < Q; q++)
#pragma unroll
            for (int v = 0; v < 2; v++) {
                const Src x = p[q][min(k + v, nk - 1)];
                r[2 * q + v] = k + v < nk ? x : (Src)0;
            }
    }
    __device__ __forceinline__ void store(const Src (&r)[N], T *lds, int pitch) const {
        const int k = 2 * (threadIdx.x & 7);
        T *d = lds + k * pitch + ((int)(threadIdx.x >> 3) ^ swizzle<SWZ>(k));
#pragma unroll
        for (int q = 0; q < Q; q++) {
            d[q * RPP] = (T)r[2 * q];
            d[q * RPP + pitch] = (T)r[2 * q + 1];
        }
    }
};

// Row-major matrix M[k][col] (col contiguous) as the B operand: tile columns
// c0 .. c0+C-1.  The lanes of a k row take column pairs at a stride of the
// whole row of lanes, so loads and LDS stores run along rows.  Columns past
// the last repeat one in range (their results are not used).
template <int C, typename T = double, typename Src = double, int THREADS = G_THREADS>
struct ColsLoader {
    using reg_t = Src;
    static constexpr int N = C * G_BK / THREADS, Q = N / 2;
    static constexpr int TPR = THREADS / G_BK;           // threads per k row
    static constexpr int SWZ = 0;
    static_assert(Q >= 1 && Q * 2 * TPR == C, "ColsLoader shape");
    const Src *base;          // row k0
    long ld;
    int c, ncols, nk;
    __device__ __forceinline__ ColsLoader(const Src *b, long ld_, int c0, int ncols_, int k0, int kmax)
        : base(b + (long)k0 * ld_), ld(ld_), c(c0 + 2 * (int)(threadIdx.x % TPR)), ncols(ncols_), nk(kmax - k0) {}
    __device__ __forceinline__ void load(int kt, Src (&r)[N]) const {
        const int k = kt * G_BK + (int)(threadIdx.x / TPR);
        const int cl = c - 2 * (int)(threadIdx.x % TPR);          // the tile's first column
        if ((kt + 1) * G_BK <= nk && cl + C <= ncols) {
            const Src *src = base + (long)k * ld + c;
#pragma unroll
            for (int q = 0; q < Q; q++) {
                const Piece<Src, 2> x = *(const Piece<Src, 2> *)(src + q * 2 * TPR);
                r[2 * q] = x.v[0];
                r[2 * q + 1] = x.v[1];
            }
            return;
        }
        const Src *src = base + (long)min(k, nk - 1) * ld;
#pragma unroll
        for (int e = 0; e < N; e++) {
            const Src x = src[min(c + (e >> 1) * 2 * TPR + (e & 1), ncols - 1)];
            r[e] = k < nk ? x : (Src)0;
        }
    }
    __device__ __forceinline__ void store(const Src (&r)[N], T *lds, int pitch) const {
        struct alignas(2 * sizeof(T)) Pair { T x, y; };
        T *d = lds + (threadIdx.x / TPR) * pitch + 2 * (threadIdx.x % TPR);
#pragma unroll
        for (int q = 0; q < Q; q++) *(Pair *)(d + q * 2 * TPR) = Pair{(T)r[2 * q], (T)r[2 * q + 1]};
    }
};

}  // namespace mdf
