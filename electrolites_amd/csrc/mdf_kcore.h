// Tile bodies of the exchange (K) contraction, shared by the single-item
// launches (mdf_k.hip) and the grouped persistent launch (mdf_grouped.hip),
// so an item gives bit-identical results alone and in a batch.
//
//     R[L, i, k] = sum_j A_L[i, j] F[j, k]                 (step 1)
//     K[i, j]   += sum_{L,k} R_l[L, i, k] R_r[L, j, k]     (step 2)
#pragma once
#include <cstdlib>
#include <type_traits>

#include "mdf_common.h"
#include "mdf_gemm.h"
#include "mdf_b3.h"
#include "mdf_tiles.h"

namespace mdf {
namespace kcore {

__device__ __forceinline__ long tri(long i) { return i * (i + 1) / 2; }

// ---------------------------------------------------------------- step 1
// A operand of step 1: rows i0..i0+127 of the unpacked A_L, K-step kt covers
// j = 16 kt .. 16 kt + 15.  TRI: the lower triangle of A_L with its
// diagonal halved (A_L = T + T^T), zero above the diagonal.
template <bool MAPPED, typename T = double, typename Src = double, int THREADS = G_THREADS, bool TRI = false>
struct PackedALoader {
    using reg_t = Src;                                   // the cderi storage type
    static constexpr int N = 128 * G_BK / THREADS;       // 8 (256 threads) or 4 (512)
    static constexpr int SWZ = 0;
    static constexpr int TPJ = THREADS / G_BK;           // threads per j row (upper)
    static constexpr int TPR = G_BK / N;                 // threads per i row (lower)
    const Src *row;      // cderi row L
    const int *pmap;     // MAPPED: pair index of (i, j), -1 if not stored
    int nao, i0;
    int upper;           // layout used by the last load()
    // MAPPED: the pair indices of the next K-step, loaded one call ahead so
    // the value gathers do not wait on the map (calls come with kt = 0, 1, ...)
    int pm[N];
    __device__ __forceinline__ void map_step(int kt, int (&p)[N]) const {
        const int t = threadIdx.x, i = i0 + t / TPR, jb = kt * G_BK + (t % TPR) * N;
        if ((nao & 3) == 0 && i < nao && jb + N <= nao) {
            // a thread's N map entries as 16-byte loads (N is 4 or 8, jb a
            // multiple of 4, so the row start i nao + jb is one too)
            const int4 *src = reinterpret_cast<const int4 *>(pmap + (long)i * nao + jb);
#pragma unroll
            for (int q = 0; q < N / 4; q++) {
                const int4 m = src[q];
                p[4 * q] = m.x;
                p[4 * q + 1] = m.y;
                p[4 * q + 2] = m.z;
                p[4 * q + 3] = m.w;
            }
            if (TRI) {
#pragma unroll
                for (int v = 0; v < N; v++)
                    if (jb + v > i) p[v] = -1;
            }
            return;
        }
#pragma unroll
        for (int v = 0; v < N; v++)
            p[v] = (i < nao && jb + v < nao && (!TRI || jb + v <= i)) ? pmap[(long)i * nao + jb + v] : -1;
    }
    __device__ __forceinline__ void load(int kt, Src (&r)[N]) {
        const int t = threadIdx.x, j0 = kt * G_BK;
        if (MAPPED) {
            // lanes run along j of one row i in every K-step (the transposed
            // layout above the diagonal measured no faster here)
            upper = 0;
            if (kt == 0) map_step(0, pm);
#pragma unroll
            for (int v = 0; v < N; v++) r[v] = pm[v] >= 0 ? row[pm[v]] : (Src)0;
            if (TRI) {
                const int i = i0 + t / TPR, jb = j0 + (t % TPR) * N;
#pragma unroll
                for (int v = 0; v < N; v++)
                    if (jb + v == i) r[v] *= (Src)0.5;
            }
            map_step(kt + 1, pm);
            return;
        }
        if (TRI && j0 >= i0 + 127) {
            // above the diagonal: zero (the K-loop of a TRI tile stops at
            // the diagonal block, so this is only a guard)
            upper = 0;
#pragma unroll
            for (int v = 0; v < N; v++) r[v] = (Src)0;
            return;
        }
        if (!MAPPED && j0 >= i0 + 127) {
            // every j > every i: (i, j) at tri(j) + i, contiguous in i
            upper = 1;
            const int j = j0 + t / TPJ, ib = i0 + (t % TPJ) * N;
            const Src *src = row + tri(j) + ib;
#pragma unroll
            for (int v = 0; v < N; v++) r[v] = (j < nao && ib + v < nao) ? src[v] : (Src)0;
            return;
        }
        upper = 0;
        const int i = i0 + t / TPR, jb = j0 + (t % TPR) * N;
        if (!MAPPED && i0 >= j0 + G_BK - 1) {
            // every i >= every j: contiguous in j
            const Src *src = row + tri(i) + jb;
#pragma unroll
            for (int v = 0; v < N; v++) r[v] = (i < nao) ? src[v] : (Src)0;
            return;
        }
#pragma unroll
        for (int v = 0; v < N; v++) {
            const int j = jb + v;
            Src x = 0;
            if (i < nao && j < nao) {
                if (MAPPED) {
                    const int p = pmap[(long)i * nao + j];
                    x = p >= 0 ? row[p] : 0.;
                } else if (TRI) {
                    x = i > j ? row[tri(i) + j] : i == j ? (Src)0.5 * row[tri(i) + i] : (Src)0;
                } else {
                    x = row[i >= j ? tri(i) + j : tri(j) + i];
                }
            }
            r[v] = x;
        }
    }
    __device__ __forceinline__ void store(const Src (&r)[N], T *lds, int pitch) const {
        const int t = threadIdx.x;
        if (upper) {
            const int jj = t / TPJ, ib = (t % TPJ) * N;
#pragma unroll
            for (int v = 0; v < N; v++) lds[jj * pitch + ib + v] = (T)r[v];
        } else {
            const int ii = t / TPR, jb = (t % TPR) * N;
#pragma unroll
            for (int v = 0; v < N; v++) lds[(jb + v) * pitch + ii] = (T)r[v];
        }
    }
};

// Step-1 tile widths: 64, 128 and 160 columns on 2 x 2 wavefronts, 256 and
// 320 on 2 x 4 (a workgroup of 512 threads then covers up to 320 occupied
// columns, so each cderi tile is read once per 320 columns instead of once
// per 128 or 160).
template <int BN>
struct Step1Shape {
    static constexpr int WGN = BN >= 192 ? 4 : 2;
    static constexpr int THREADS = 128 * WGN;
    using S = TileShape<128, BN, 2, WGN>;
};

// One 128 x BN tile of step 1 for aux row `row` (the cderi row L): rows
// i0.., columns (occupied index) k0.. of R_L.
// TRI: A_L replaced by its lower triangle with the diagonal halved, and the
// K loop stops after the tile's diagonal block (about half the work; for a
// symmetric bilinear form F^T A_L F = G + G^T with G = F^T (TRI product)).
template <int BN, bool MAPPED, typename T, typename Src = double, bool TRI = false>
__device__ __forceinline__ void step1_tile(const Src *__restrict__ row, const int *__restrict__ pmap, int nao,
                                  const double *__restrict__ F, long ldf, int nocc, T *__restrict__ Rl, long ldr,
                                  int i0, int k0, T *lds) {
    using C = Step1Shape<BN>;
    using S = typename C::S;
    PackedALoader<MAPPED, T, Src, C::THREADS, TRI> la{row, pmap, nao, i0, 0};
    ColsLoader<BN, T, double, C::THREADS> lb{F, ldf, k0, nocc, 0, nao};
    Acc<S::MI, S::NI, T> acc;
    acc.zero();
    const int jend = TRI ? min(nao, i0 + 128) : nao;
    gemm_mainloop<128, BN, decltype(la), decltype(lb), T, 2, C::WGN>(la, lb, (jend + G_BK - 1) / G_BK, lds, acc);
    auto emit = [&](int r, int c, T v) {
        const int i = i0 + r, k = k0 + c;
        if (i < nao && k < nocc) Rl[(long)i * ldr + k] = v;
    };
    gemm_epilogue_layout<128, BN, T, decltype(acc), decltype(emit) &, 2, C::WGN>(acc, emit);
}

// The step-1 tile of one group of pair tiles: its 16 AO rows of the nl (1..8)
// aux rows at c, occupied columns k0..k0+BN-1, into the R blocks of those aux
// rows.  `fp` is the packed factor (tiles::pack_factor_range, row stride ldp).
template <int BN, typename T, typename Src, bool HALVES>
__device__ __forceinline__ void step1_pairs_tile(const Src *__restrict__ c, long ld, int nl, const tiles::View &tv, int g,
                                        const T *__restrict__ fp, unsigned ldp, int nocc, T *__restrict__ R, long ldr,
                                        long strideL, int k0, T *lds) {
    using C = Step1Shape<BN>;
    using S = typename C::S;
    tiles::ALoader<T, Src, C::THREADS, HALVES> la;
    tiles::BLoader<BN, T, C::THREADS> lb;
    la.init(c, ld, nl, tv.map + (long)g * tv.ccap * tiles::RB);
    lb.init(fp, ldp, k0, tv.cols + (long)g * tv.ccap);
    Acc<S::MI, S::NI, T> acc;
    acc.zero();
    gemm_mainloop<128, BN, decltype(la), decltype(lb), T, 2, C::WGN>(la, lb, tv.nstep[g], lds, acc);
    // a wavefront's 16-row MFMA blocks are whole aux rows
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int l0 = (wave % 2) * S::MI, c0 = k0 + (wave / 2) * S::WN + (lane & 15);
#pragma unroll
    for (int v = 0; v < 4; v++) {
        const int i = tv.rows[g * tiles::RB + Mfma<T>::row(lane, v)];
        if (i < 0) continue;
        T *Ri = R + (long)i * ldr + c0;
#pragma unroll
        for (int mi = 0; mi < S::MI; mi++)
            if (l0 + mi < nl) {
                T *Rl = Ri + (l0 + mi) * strideL;
#pragma unroll
                for (int ni = 0; ni < S::NI; ni++)
                    if (c0 + ni * 16 < nocc) Rl[ni * 16] = acc.v[mi][ni][v];
            }
    }
}

// ---------------------------------------------------------------- step 2
// The transformed blocks: the occupied columns of 8 aux rows side by side,
// R[L / 8][i][(L % 8) nocc + k], row stride ldr = 8 nocc (of a pass of fewer
// rows, one block as wide as those).  Step 2's reduction
// runs over a block's 8 nocc columns in K-steps of 16 (one aux row at a time
// it computed nocc rounded up to 16: 96 columns for 81, 64 for 50).
constexpr int RL = tiles::NL;

// Columns a factor may have in one contraction: TransformedLoader's and the
// packed factor's 32-bit offsets reach that far (at least 92,000 columns
// at the functions that int32 pair addresses hold).
inline long max_cols(int nao) {
    const long packed = (1L << 32) / (nao + 1L) - 320;
    return packed < 1 ? 1 : packed < 1L << 22 ? packed : 1L << 22;
}

// Aux rows a block holds in passes of nL rows, and its row stride (whole 16-byte
// pieces of float).
__host__ __device__ __forceinline__ int block_of(long nL) { return nL < RL ? (int)nL : RL; }
__host__ __device__ __forceinline__ long block_ld(int rl, int nocc) { return ((long)rl * nocc + 3) / 4 * 4; }

// FP32 step 2 adds its MFMA accumulators into an FP64 shadow every S2_FLUSH
// K-steps of one aux row's columns rounded up to 16 (at nocc = 81, 32 steps of
// 13.5 products on average), so the rounding error of the long (L, k) reduction
// grows with the flush length, not with naux * nocc.
constexpr int S2_FLUSH = 32;

// A pass of nL aux rows in blocks of rl (block_of the plan's passes, in the
// last, shorter one too): columns of a block's row that hold values, fewer in
// the last block; and the K-steps, of 16 products each here, between two
// flushes.
struct RShape {
    int ldr, cols, kchunks, nfull, lastcols, flush;
    __host__ __device__ __forceinline__ RShape(long nL, int nocc, int rl)
        : ldr((int)block_ld(rl, nocc)), cols(rl * nocc), kchunks((cols + G_BK - 1) / G_BK), nfull((int)(nL / rl)),
          lastcols((int)(nL % rl) * nocc) {
        const long f = (long)S2_FLUSH * nocc / ((nocc + G_BK - 1L) / G_BK * G_BK);
        flush = f > 1 ? (int)f : 1;
    }
    __host__ __device__ __forceinline__ long steps() const {
        return (long)nfull * kchunks + (lastcols + G_BK - 1) / G_BK;
    }
};

// Rows r0..r0+ROWS-1 of the blocks; K-step kt of this split is (block, kc) =
// divmod(s0 + kt, kchunks), columns kc*16 .. kc*16 + 15.  The lanes of a row
// take its 16-byte pieces, as in RowsLoader.
template <typename T, int ROWS>
struct TransformedLoader {
    using reg_t = T;
    static constexpr int N = ROWS * G_BK / G_THREADS;
    static constexpr int EPV = 16 / (int)sizeof(T);      // elements per 16-byte piece
    static constexpr int Q = N / EPV, LPR = G_BK / EPV, RPP = G_THREADS / LPR;
    static constexpr int SWZ = sizeof(T) == 8 ? 2 : 3;
    static_assert(Q >= 1 && Q * RPP == ROWS, "TransformedLoader shape");
    const T *R;          // row r0 of block 0
    long strideB;
    RShape y;
    // this thread's rows, from row r0: 32 bits hold the 127 rows of a tile up
    // to max_cols columns, where a row's place in the whole block outgrows
    // them from nao nocc = 2^29
    unsigned off[Q];
    int last;            // its column in a row's last, ragged chunk
    long b;              // block and
    int kc;              // chunk of the next load()
    int left;            // columns in range of the loaded chunk
    __device__ __forceinline__ TransformedLoader(const T *R_, long strideB_, const RShape &y_, int r0, int nao, long b_,
                                                 int kc_)
        : R(R_ + (long)r0 * y_.ldr), strideB(strideB_), y(y_), b(b_), kc(kc_) {
        const int c = (int)(threadIdx.x % LPR) * EPV;
#pragma unroll
        for (int q = 0; q < Q; q++)
            off[q] = (unsigned)min((int)(threadIdx.x / LPR) + q * RPP, nao - 1 - r0) * (unsigned)y.ldr + c;
        last = min((y.kchunks - 1) * G_BK + c, y.ldr - EPV) - c;
    }
    __device__ __forceinline__ void load(int, T (&r)[N]) {
        // called for kt = 0, 1, 2, ... in order: advance (b, kc) in place
        const T *src = R + b * strideB + ((kc + 1) * G_BK > y.ldr ? last : kc * G_BK);
#pragma unroll
        for (int q = 0; q < Q; q++) {
            const Piece<T, EPV> x = *(const Piece<T, EPV> *)(src + off[q]);
#pragma unroll
            for (int e = 0; e < EPV; e++) r[q * EPV + e] = x.v[e];
        }
        left = (b < y.nfull ? y.cols : y.lastcols) - kc * G_BK;
        if (++kc == y.kchunks) {
            kc = 0;
            ++b;
        }
    }
    __device__ __forceinline__ void store(T (&r)[N], T *lds, int pitch) const {
        const int k = (int)(threadIdx.x % LPR) * EPV;
        if (left < G_BK) {
            // columns past the last hold nothing: zero, whatever is there
#pragma unroll
            for (int e = 0; e < N; e++)
                if (k + e % EPV >= left) r[e] = (T)0;
        }
        T *d = lds + k * pitch + ((int)(threadIdx.x / LPR) ^ swizzle<SWZ>(k));
#pragma unroll
        for (int e = 0; e < N; e++) d[(e % EPV) * pitch + e / EPV * RPP] = r[e];
    }
};

constexpr double S2_64_COST = 1.25;
constexpr int S2_B = 128;              // split-BF16 step-2 tile; FP64/FP32: KPlan::s2 (64 or 128)

// One B x B output tile (i0, j0) of step 2 over the K-steps [s0, s1) of the
// (block, chunk) reduction; writes (beta = 0) or adds (beta = 1) into o.
template <int B, typename T>
__device__ __forceinline__ void step2_tile(const T *__restrict__ Rl, const T *__restrict__ Rr, int nao, const RShape &y,
                                  int i0, int j0, long s0, long s1, double *__restrict__ o, int beta, T *lds) {
    using S = TileShape<B, B>;
    const long b0 = s0 / y.kchunks, strideB = (long)nao * y.ldr;
    const int kc0 = (int)(s0 - b0 * y.kchunks);
    TransformedLoader<T, B> la{Rl, strideB, y, i0, nao, b0, kc0};
    TransformedLoader<T, B> lb{Rr, strideB, y, j0, nao, b0, kc0};
    Acc<S::MI, S::NI, T> acc;
    auto emit = [&](int r, int c, double v) {
        const int i = i0 + r, j = j0 + c;
        if (i < nao && j < nao) {
            double *dst = o + (long)i * nao + j;
            *dst = beta ? *dst + v : v;
        }
    };
    if constexpr (sizeof(T) == 8) {
        acc.zero();
        gemm_mainloop<B, B>(la, lb, (int)(s1 - s0), lds, acc);
        gemm_epilogue<B, B, T>(acc, emit);
    } else {
        Acc<S::MI, S::NI, double> sum;
        sum.zero();
        for (long s = s0; s < s1; s += y.flush) {
            acc.zero();
            // the loaders advance in place, so consecutive calls continue the
            // reduction where the previous one stopped
            gemm_mainloop<B, B>(la, lb, (int)min((long)y.flush, s1 - s), lds, acc);
#pragma unroll
            for (int a = 0; a < S::MI; a++)
#pragma unroll
                for (int b = 0; b < S::NI; b++)
#pragma unroll
                    for (int v = 0; v < 4; v++) sum.v[a][b][v] += (double)acc.v[a][b][v];
        }
        gemm_epilogue_layout<B, B, T>(sum, emit);
    }
}

// Lower-triangle tile index x -> (ti >= tj), row-major.
__device__ __forceinline__ void tri_tile(int x, int &ti, int &tj) {
    ti = (int)((sqrt(8.0 * x + 1.0) - 1.0) * 0.5);
    while (ti * (ti + 1) / 2 > x) ti--;
    while ((ti + 1) * (ti + 2) / 2 <= x) ti++;
    tj = x - ti * (ti + 1) / 2;
}

// vk[i, j] (+)= sum_s part[s, I, J] for the flat range [e0, e1); sym, the
// step-2 tile width or 0, reads the lower-tile copy for upper-tile entries.
__device__ __forceinline__ void finalize_range(const double *__restrict__ part, int ksplit, long part_stride, int nao,
                                      int sym, double *__restrict__ vk, long ldvk, int accumulate, long e0, long e1) {
    for (long t = e0 + threadIdx.x; t < e1; t += 256) {
        const int i = (int)(t / nao), j = (int)(t % nao);
        int I = i, J = j;
        if (sym && (i / sym) < (j / sym)) { I = j; J = i; }
        const double *src = part + (long)I * nao + J;
        double s = 0.;
        for (int k = 0; k < ksplit; k += 8) {        // ksplit is a multiple of 8
            double x[8];
#pragma unroll
            for (int v = 0; v < 8; v++) x[v] = src[(k + v) * part_stride];
#pragma unroll
            for (int v = 0; v < 8; v++) s += x[v];
        }
        double *dst = vk + (long)i * ldvk + j;
        *dst = accumulate ? *dst + s : s;
    }
}

// step-1 tile width: each k-tile re-reads the cderi tile (worth about 64
// columns of MFMA work), so minimise nkt * (64 + BN) over the widths; ties
// go to the wider tile
inline int pick_bn(int nocc) {
    const int cand[8] = {32, 64, 96, 128, 160, 192, 256, 320};
    // MDF_K_STEP1_BN forces one of the widths (for tuning runs)
    if (const char *e = getenv("MDF_K_STEP1_BN")) {
        const int v = atoi(e);
        for (int b : cand)
            if (b == v) return b;
    }
    int best = 64;
    long best_cost = 1L << 40;
    for (int b : cand) {
        const long cost = (long)((nocc + b - 1) / b) * (64 + b);
        if (cost <= best_cost) { best_cost = cost; best = b; }
    }
    return best;
}

// f(integral constant of the step-1 tile width)
template <class F>
void with_bn(int bn, F &&f) {
    switch (bn) {
    case 320: f(std::integral_constant<int, 320>{}); break;
    case 256: f(std::integral_constant<int, 256>{}); break;
    case 192: f(std::integral_constant<int, 192>{}); break;
    case 160: f(std::integral_constant<int, 160>{}); break;
    case 128: f(std::integral_constant<int, 128>{}); break;
    case 96: f(std::integral_constant<int, 96>{}); break;
    case 64: f(std::integral_constant<int, 64>{}); break;
    default: f(std::integral_constant<int, 32>{}); break;
    }
}

struct KPlan {
    int ntile, ntiles_grid, ksplit, bn;
    int s2;             // step-2 tile width
    long nL;            // aux rows per pass
    size_t r_words;     // one R buffer
    size_t part_words;
};

inline int cu_count() {
    static int cached[64] = {0};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    if (!cached[dev]) {
        int cu = 0;
        if (hipDeviceGetAttribute(&cu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cu <= 0)
            cu = 256;
        cached[dev] = cu;
    }
    return cached[dev];
}

// Split of the (L, k) reduction of nsteps K-steps: a multiple of the XCD
// count, so that each XCD takes whole splits (step2_coords) and the output
// tiles running on one XCD at a time read the same R panels through its L2.
// Of the splits of at least 8 K-steps, the one of least estimated time: the
// rounds of resident workgroups (slots per XCD) each over its K-steps and
// about 6 more to start and end, plus the partials written and read again
// (nao^2 words each, 1.5e-6 K-steps a word; 3e-6 of split BF16's, which take
// half the time).  Against the best of 8, 16, 24, 32, 48, 64, 96, 128, 192 and
// 256 splits, whole K at 48 to 768 functions: FP64 within 9 % (nao 192: 189 us
// for 173; 768: 13.94 ms for 13.96), two factors within 4 % of the chosen
// width's best, FP32 within 18 % (192: 143 us for 123; from 288 on 5 %), split
// BF16 within 7 % (from 192 on 5 %); a fixed 32 loses up to 36 % (48 functions)
// and 21 % (768).
inline int pick_ksplit(int ntiles_grid, long nsteps, int nao, int slots, double word) {
    int best = N_XCD;
    double best_t = 1e300;
    for (int ks = N_XCD; ks <= 256 && (ks == N_XCD || nsteps >= 8L * ks); ks += N_XCD) {
        const long rounds = ((long)ntiles_grid * ks / N_XCD + slots - 1) / slots;
        const double t = rounds * ((double)nsteps / ks + 6.) + word * ks * nao * nao;
        if (t < best_t) { best_t = t; best = ks; }
    }
    return best;
}

// (output tile, split) of workgroup w of a 1-D step-2 grid of ntiles_grid *
// ksplit workgroups (ksplit a multiple of N_XCD).  Workgroups reach the XCDs
// round-robin (w % N_XCD); XCD x takes splits x, x + N_XCD, ..., every
// output tile of one split before the next, so the tiles resident on an XCD
// together mostly share one split's K range: each R panel of that range is
// fetched into the XCD's L2 once and read there by every tile of its row
// and column.
__device__ __forceinline__ void step2_coords(long w, int ntiles_grid, int &tile, int &split) {
    const int xcd = (int)(w % N_XCD);
    const long l = w / N_XCD;
    split = xcd + N_XCD * (int)(l / ntiles_grid);
    tile = (int)(l % ntiles_grid);
}

// Aux rows per pass: the transformed blocks of one pass (R_l and R_r) stay
// within K_BLOCK_BYTES.  A function of the item's shape only, so the single
// entry and the grouped launch cut an item into the same passes.
// The environment variable MDF_K_BLOCK_BYTES overrides the bound (read on
// every plan, so tests can force several passes on small items).
constexpr size_t K_BLOCK_BYTES = 8ull << 30;

inline size_t k_block_bytes() {
    const char *e = getenv("MDF_K_BLOCK_BYTES");
    if (e && *e) {
        const long long v = atoll(e);
        if (v > 0) return (size_t)v;
    }
    return K_BLOCK_BYTES;
}

// The most of naux aux rows whose transformed blocks take no more than cap rows'
// space: all of them, whole blocks, or one block of fewer rows (at least one).
// Split BF16's rows stand alone (b3): no space goes to a last block's missing ones.
inline long rows_within(long naux, long cap, bool b3) {
    const long all = b3 || naux < RL ? naux : (naux + RL - 1) / RL * RL;
    const long r = cap >= all ? naux : cap >= RL ? cap / RL * RL : cap;
    return r < 1 ? 1 : r;
}

inline long block_rows(long naux, int nao, int nocc, bool two, bool b3, size_t elem) {
    const size_t per_row = (size_t)nao * nocc * elem * (two ? 2 : 1);
    return rows_within(naux, per_row ? (long)(k_block_bytes() / per_row) : naux + RL, b3);
}

// Words of one factor's transformed blocks of a pass of nL aux rows.
inline size_t r_words(long nL, int nao, int nocc) {
    const int rl = block_of(nL);
    return (size_t)((nL + rl - 1) / rl) * nao * block_ld(rl, nocc);
}

// b3: the split-BF16 kernels' plan (128-wide step-2 tiles).
inline KPlan plan_k(long naux, int nao, int nocc, bool two, long max_rows, bool b3) {
    KPlan p;
    p.nL = max_rows < naux ? max_rows : naux;
    if (p.nL < 1) p.nL = 1;
    auto tiles = [&](int b) {
        const int n = (nao + b - 1) / b;
        return two ? n * n : n * (n + 1) / 2;
    };
    // 64-wide tiles cover a small result with less padding, at S2_64_COST
    // times the time of a 128-wide tile's product per element: a whole FP64 K,
    // one factor, 64 against 128 wide, each at its best split, at nao 72 29/37
    // us, 96 42/47, 144 78/92, 192 173/206, 288 522/637, 384 1304/1319, 489
    // 3293/3213, 576 5120/5330, 768 14972/13935; the rule takes 128 at 144,
    // 249, 384, 489 and 768
    p.s2 = !b3 && S2_64_COST * tiles(64) * 64 * 64 < (double)tiles(128) * 128 * 128 ? 64 : 128;
    p.ntile = (nao + p.s2 - 1) / p.s2;
    p.ntiles_grid = tiles(p.s2);
    const long nsteps = b3 ? p.nL * ((nocc + 31) / 32) : RShape(p.nL, nocc, block_of(p.nL)).steps();
    p.ksplit = pick_ksplit(p.ntiles_grid, nsteps, nao, (p.s2 == 64 ? 4 : 2) * cu_count() / N_XCD,
                           b3 ? 3e-6 : 1.5e-6);
    p.bn = pick_bn(nocc);
    p.r_words = r_words(p.nL, nao, nocc);
    p.part_words = (size_t)p.ksplit * nao * nao;
    return p;
}

// Packed factor of the pair-tile step 1: nao + 1 rows of whole tile widths.
inline unsigned pack_ld(const KPlan &p, int nocc) { return (unsigned)((nocc + p.bn - 1) / p.bn * p.bn); }
inline size_t pack_words(const KPlan &p, int nao, int nocc) { return (size_t)(nao + 1) * pack_ld(p, nocc); }

// ------------------------------------------------- split-BF16 (prec 2)
// The same two steps on the three-term split-BF16 engine (mdf_b3.h).  The
// factors are pre-split into transposed planes FT[k][j] (j zero-padded to
// ldft = a multiple of 32 >= nao); R is stored split, as two planes of
// [L][i][k] bfloat16 with k zero-padded to ldr = a multiple of 32 >= nocc,
// so step 2 copies it into LDS without conversion.  Both are stored in
// chunks of 32 along their contiguous index (FT: (j / 32, k, j % 32); R:
// r_index), so each K-step reads its tile of a plane as one contiguous run.
namespace kb3 {

using b3::u16;
constexpr int BM = 128;               // step-1 rows per tile (step 2: S2_B x S2_B)
// step 2 adds its FP32 accumulators into the FP64 partial in global memory
// every S2_FLUSH K-steps (S2_FLUSH * 32 reduction terms)
constexpr int S2_FLUSH = 64;

__host__ __device__ inline long pad32(long n) { return (n + 31) / 32 * 32; }

// Element (i, k) of one aux row's split R plane (nao rows, ldr = pad32(nocc)
// columns): stored as ldr / 32 chunks of 32 columns, each chunk nao rows of
// 32 contiguous values, so the 128 rows x 32 columns a step-2 K-step reads
// are one contiguous 8 KB run per plane (row-major rows would give 128 runs
// of 64 bytes, half a cache line each).  The plane's size is nao * ldr, as
// row-major.
__host__ __device__ inline long r_index(int nao, int i, int k) {
    return ((long)(k >> 5) * nao + i) * 32 + (k & 31);
}

// A operand: rows i0..i0+127 of the unpacked A_L; K-step kt covers
// j = 32 kt .. 32 kt + 31.  THREADS threads, N = 4096 / THREADS values each.
template <bool MAPPED, int THREADS, typename Src = double>
struct PackedA32 {
    using reg_t = Src;
    static constexpr int N = 128 * b3::BK / THREADS;
    static constexpr int TPR = b3::BK / N;           // threads per row (lower layout)
    const Src *row;
    const int *pmap;
    int nao, i0;
    int upper;
    int pm[N];           // MAPPED: the next K-step's pair indices (one call ahead)
    int pm_upper;        // and their layout
    // Above the diagonal (every j > every i) the transposed layout of the
    // packed loader: thread t takes i = i0 + t % 128 and j = j0 + N (t / 128)
    // + v, so a load instruction reads consecutive i of the map row j and of
    // the stored pairs (j, i).
    __device__ __forceinline__ void map_step(int kt, int (&p)[N], int &up) const {
        const int t = threadIdx.x, j0 = kt * b3::BK;
        up = j0 >= i0 + 127;
        if (up) {
            const int i = i0 + (t & 127), jb = j0 + (t >> 7) * N;
#pragma unroll
            for (int v = 0; v < N; v++) p[v] = (i < nao && jb + v < nao) ? pmap[(long)(jb + v) * nao + i] : -1;
        } else {
            const int i = i0 + t / TPR, jb = j0 + (t % TPR) * N;
            if ((nao & 3) == 0 && i < nao && jb + N <= nao) {
                // N (a multiple of 4) map entries as 16-byte loads
                const int4 *src = reinterpret_cast<const int4 *>(pmap + (long)i * nao + jb);
#pragma unroll
                for (int q = 0; q < N / 4; q++) {
                    const int4 m = src[q];
                    p[4 * q] = m.x;
                    p[4 * q + 1] = m.y;
                    p[4 * q + 2] = m.z;
                    p[4 * q + 3] = m.w;
                }
                return;
            }
#pragma unroll
            for (int v = 0; v < N; v++) p[v] = (i < nao && jb + v < nao) ? pmap[(long)i * nao + jb + v] : -1;
        }
    }
    __device__ __forceinline__ void load(int kt, Src (&r)[N]) {
        const int t = threadIdx.x, j0 = kt * b3::BK;
        if (MAPPED) {
            if (kt == 0) map_step(0, pm, pm_upper);
            upper = pm_upper;
#pragma unroll
            for (int v = 0; v < N; v++) r[v] = pm[v] >= 0 ? row[pm[v]] : (Src)0;
            map_step(kt + 1, pm, pm_upper);
            return;
        }
        if (!MAPPED && j0 >= i0 + 127) {
            // every j > every i: (i, j) at tri(j) + i, contiguous in i.  Thread
            // t takes row i = i0 + t % 128 and j = j0 + N (t / 128) + v: each
            // load instruction reads 64 consecutive i of one j (coalesced), and
            // the row lands in LDS as N contiguous k (16-byte stores).
            upper = 1;
            const int i = i0 + (t & 127), jb = j0 + (t >> 7) * N;
#pragma unroll
            for (int v = 0; v < N; v++) r[v] = (i < nao && jb + v < nao) ? row[tri(jb + v) + i] : (Src)0;
            return;
        }
        upper = 0;
        const int i = i0 + t / TPR, jb = j0 + (t % TPR) * N;
        if (!MAPPED && i0 >= j0 + b3::BK - 1) {
            // every i >= every j: contiguous in j
            const Src *src = row + tri(i) + jb;
#pragma unroll
            for (int v = 0; v < N; v++) r[v] = (i < nao) ? src[v] : (Src)0;
            return;
        }
#pragma unroll
        for (int v = 0; v < N; v++) {
            const int j = jb + v;
            Src x = 0;
            if (i < nao && j < nao) {
                if (MAPPED) {
                    const int p = pmap[(long)i * nao + j];
                    x = p >= 0 ? row[p] : 0.;
                } else {
                    x = row[i >= j ? tri(i) + j : tri(j) + i];
                }
            }
            r[v] = x;
        }
    }
    __device__ __forceinline__ void store(const Src (&r)[N], u16 *hi, u16 *lo) const {
        const int t = threadIdx.x;
        if (upper)
            b3::put<N>(r, hi, lo, t & 127, (t >> 7) * N);
        else
            b3::put<N>(r, hi, lo, t / TPR, (t % TPR) * N);
    }
};

// B operand of step 1: rows k0..k0+BN-1 of the split FT planes.
template <int BN, int THREADS>
struct FTLoader {
    using P = b3::PlaneRowsN<BN, THREADS>;
    using reg_t = uint4;
    static constexpr int N = P::N;
    const u16 *hi, *lo;
    long ld;
    int k0, nocc;
    // the planes are chunk-major (split_ft_range): K-step kt is chunk kt,
    // nocc rows of 32 values
    __device__ __forceinline__ void load(int kt, uint4 (&r)[N]) const {
        P::fetch(hi, lo, b3::BK, (long)kt * b3::BK * nocc, k0, nocc, r);
    }
    __device__ __forceinline__ void store(const uint4 (&r)[N], u16 *h, u16 *l) const { P::put(r, h, l); }
};

// Step-1 tile widths: 128 columns on 2 x 2 wavefronts, 192, 256 or 320 on
// 2 x 4 (one workgroup then covers up to 320 occupied columns, so each cderi tile
// is read once per factor instead of once per 128 columns).
template <int BN>
struct Step1Cfg {
    static constexpr int WGN = BN == 128 ? 2 : 4;
    static constexpr int THREADS = 128 * WGN;
    using S = b3::Shape<BM, BN, 2, WGN>;
};

inline int pick_bn(long ldr) {
    int best = 128;
    long pad = -1;
    for (int bn : {128, 192, 256, 320}) {
        const long p = (ldr + bn - 1) / bn * bn - ldr;
        if (pad < 0 || p < pad || (p == pad && bn > best)) {
            best = bn;
            pad = p;
        }
    }
    return best;
}

// Writes one plane at a time: the split 128 x BN tile through LDS (freed by
// the mainloop's last barrier), then whole 16-byte runs of 8 columns at
// dst(row) + chunk-major offset of (AO row, column).
template <int BN, class AccT, class Row>
__device__ __forceinline__ void put_split_tile(const AccT &acc, u16 *Rhi, u16 *Rlo, int nao, long ldr, int k0, u16 *lds,
                                               Row &&row) {
    using C = Step1Cfg<BN>;
    constexpr int P = BN + 8;                  // row pitch (u16), 16-byte multiple
    constexpr int CH = BN / 8;                 // 16-byte runs per row
    static_assert(BM * P <= C::S::LDS_ELEMS, "one output plane must fit the tile's LDS");
    for (int plane = 0; plane < 2; plane++) {
        u16 *R = plane ? Rlo : Rhi;
        b3::epilogue<BM, BN, 2, C::WGN>(acc, [&](int r, int c, float v) {
            u16 h, l;
            b3::split(v, h, l);
            lds[r * P + c] = plane ? l : h;
        });
        __syncthreads();
        // ldr and k0 are multiples of 32: a run lies inside or outside ldr
        for (int u = threadIdx.x; u < BM * CH; u += C::THREADS) {
            const int r = u / CH, c = (u % CH) * 8, k = k0 + c;
            long off;
            const int i = row(r, off);
            if (i >= 0 && k < ldr)
                *reinterpret_cast<uint4 *>(R + off + r_index(nao, i, k)) = *reinterpret_cast<const uint4 *>(lds + r * P + c);
        }
        __syncthreads();
    }
}

// One 128 x BN tile of step 1 for the cderi row `row`: rows i0.., columns
// k0.. of the split R planes (row stride ldr; columns nocc..ldr-1 get zeros).
template <bool MAPPED, int BN, typename Src = double>
__device__ __forceinline__ void step1_tile(const Src *__restrict__ row, const int *__restrict__ pmap, int nao,
                                           const u16 *fthi, const u16 *ftlo, long ldft, int nocc, u16 *Rhi,
                                           u16 *Rlo, long ldr, int i0, int k0, u16 *lds) {
    using C = Step1Cfg<BN>;
    PackedA32<MAPPED, C::THREADS, Src> la{row, pmap, nao, i0, 0};
    FTLoader<BN, C::THREADS> lb{fthi, ftlo, ldft, k0, nocc};
    b3::Acc32<C::S::MI, C::S::NI> acc;
    acc.zero();
    b3::mainloop<BM, BN, 2, C::WGN>(la, lb, (nao + b3::BK - 1) / b3::BK, lds, acc);
    put_split_tile<BN>(acc, Rhi, Rlo, nao, ldr, k0, lds, [&](int r, long &off) {
        off = 0;
        return i0 + r < nao ? i0 + r : -1;
    });
}

// ---- step 1 on pair tiles (mdf_tiles.h): a K-step is 32 columns of the
// group, two steps of its map.
// A operand: a thread owns two neighbouring columns of one AO row and N of the
// 8 aux rows, so its LDS stores are whole 4-byte pairs and 16 lanes read 32
// consecutive columns.  As in tiles::ALoader every lane loads.
template <int THREADS, typename Src>
struct PairsA32 {
    using reg_t = Src;
    static constexpr int NLT = 2048 / THREADS;           // aux rows: 4 (512 threads) or 8 (256)
    static constexpr int N = 2 * NLT;
    const char *row[NLT];
    const int *map;
    int ii, jp, l0;
    int2 pm;                  // the next step's map entries, read one call ahead
    bool s0, s1;              // the loaded step's: stored
    __device__ __forceinline__ void init(const Src *c, long ld, int nl, const int *gmap) {
        const int t = threadIdx.x;
        jp = t & 15;
        ii = (t >> 4) & 15;
        l0 = (__builtin_amdgcn_readfirstlane(t >> 6) >> 2) * NLT;
#pragma unroll
        for (int v = 0; v < NLT; v++) row[v] = (const char *)(c + (long)min(l0 + v, nl - 1) * ld);
        map = gmap + (jp >> 3) * 256 + ii * 16 + (2 * jp & 15);
        pm = *(const int2 *)map;
    }
    __device__ __forceinline__ void load(int kt, Src (&r)[N]) {
        const unsigned o0 = (unsigned)max(pm.x, 0) * (unsigned)sizeof(Src);
        const unsigned o1 = (unsigned)max(pm.y, 0) * (unsigned)sizeof(Src);
#pragma unroll
        for (int v = 0; v < NLT; v++) {
            r[2 * v] = *(const Src *)(row[v] + o0);
            r[2 * v + 1] = *(const Src *)(row[v] + o1);
        }
        s0 = pm.x >= 0;
        s1 = pm.y >= 0;
        pm = *(const int2 *)(map + (kt + 1) * 512);
    }
    __device__ __forceinline__ void store(const Src (&r)[N], u16 *hi, u16 *lo) const {
#pragma unroll
        for (int v = 0; v < NLT; v++) {
            unsigned h, m;
            b3::split2(s0 ? (float)r[2 * v] : 0.f, s1 ? (float)r[2 * v + 1] : 0.f, h, m);
            const int at = ((l0 + v) * tiles::RB + ii) * b3::PK + 2 * jp;
            *(unsigned *)(hi + at) = h;
            *(unsigned *)(lo + at) = m;
        }
    }
};

// B operand: eight factor rows (columns of the group, uniform over a
// wavefront) at one occupied index per unit, each value hi << 16 | lo of the
// packed factor; the octet leaves as 16 bytes of each plane.
template <int BN, int THREADS>
struct PairsB32 {
    using reg_t = unsigned;
    static constexpr int UNITS = 4 * BN, Q = (UNITS + THREADS - 1) / THREADS;
    static constexpr int N = 8 * Q;
    static_assert(BN % 64 == 0, "a wavefront stays in one octet");
    const unsigned *base;     // packed factor at the tile's first column
    const int *cols;
    unsigned ldp;
    int oct[Q], n[Q];         // this thread's units (the last repeated past the end)
    __device__ __forceinline__ void init(const unsigned *fp, unsigned ldp_, int k0, const int *gcols) {
        base = fp + k0;
        cols = gcols;
        ldp = ldp_;
#pragma unroll
        for (int q = 0; q < Q; q++) {
            const int w = min(__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) + q * (THREADS / 64), UNITS / 64 - 1);
            oct[q] = w / (BN / 64);
            n[q] = w % (BN / 64) * 64 + (threadIdx.x & 63);
        }
    }
    __device__ __forceinline__ void load(int kt, unsigned (&r)[N]) const {
#pragma unroll
        for (int q = 0; q < Q; q++) {
            const int *c = cols + kt * b3::BK + oct[q] * 8;
#pragma unroll
            for (int e = 0; e < 8; e++) r[q * 8 + e] = (base + (unsigned long)((unsigned)c[e] * ldp))[n[q]];
        }
    }
    __device__ __forceinline__ void store(const unsigned (&r)[N], u16 *hi, u16 *lo) const {
#pragma unroll
        for (int q = 0; q < Q; q++) {
            uint4 h, m;
            unsigned *hs = (unsigned *)&h, *ms = (unsigned *)&m;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                hs[e] = __builtin_amdgcn_perm(r[q * 8 + 2 * e + 1], r[q * 8 + 2 * e], 0x07060302);
                ms[e] = __builtin_amdgcn_perm(r[q * 8 + 2 * e + 1], r[q * 8 + 2 * e], 0x05040100);
            }
            *(uint4 *)(hi + n[q] * b3::PK + oct[q] * 8) = h;
            *(uint4 *)(lo + n[q] * b3::PK + oct[q] * 8) = m;
        }
    }
};

// The step-1 tile of one group of pair tiles, as kcore::step1_pairs_tile;
// strideL between the planes of aux rows.
template <int BN, typename Src>
__device__ __forceinline__ void step1_pairs_tile(const Src *__restrict__ c, long ld, int nl, const tiles::View &tv, int g,
                                                 const unsigned *__restrict__ fp, unsigned ldp, u16 *Rhi, u16 *Rlo,
                                                 long ldr, long strideL, int k0, u16 *lds) {
    using C = Step1Cfg<BN>;
    PairsA32<C::THREADS, Src> la;
    PairsB32<BN, C::THREADS> lb;
    la.init(c, ld, nl, tv.map + (long)g * tv.ccap * tiles::RB);
    lb.init(fp, ldp, k0, tv.cols + (long)g * tv.ccap);
    b3::Acc32<C::S::MI, C::S::NI> acc;
    acc.zero();
    b3::mainloop<BM, BN, 2, C::WGN>(la, lb, (tv.nstep[g] + 1) / 2, lds, acc);
    const int *rows = tv.rows + g * tiles::RB;
    put_split_tile<BN>(acc, Rhi, Rlo, tv.nao, ldr, k0, lds, [&](int r, long &off) {
        const int l = r / tiles::RB;
        off = l * strideL;
        return l < nl ? rows[r % tiles::RB] : -1;
    });
}

// Fp[j][k] = F[j][k] split, hi << 16 | lo; zero for k in nocc..ldp-1 and in
// row nao.
__device__ __forceinline__ void pack_split_range(const double *__restrict__ F, long ldf, int nao, int nocc, unsigned *fp,
                                                 long ldp, long e0, long e1) {
    for (long e = e0 + threadIdx.x; e < e1; e += blockDim.x) {
        const int j = (int)(e / ldp), k = (int)(e - (long)j * ldp);
        u16 h, l;
        b3::split(j < nao && k < nocc ? (float)F[(long)j * ldf + k] : 0.f, h, l);
        fp[e] = (unsigned)h << 16 | l;
    }
}

// Rows r0..r0+127 of the R planes; K-step kt of this split is
// (L, kc) = divmod(s0 + kt, ldr / 32), advanced in place by load().  A
// K-step's 128 rows x 32 k of one plane are 8 KB in one piece (r_index).
struct RLoader {
    using reg_t = uint4;
    static constexpr int N = b3::PlaneRows128::N;
    const u16 *hi, *lo;
    long strideL, ldr;
    int r0, nao, kchunks;
    long L;
    int kc;
    __device__ __forceinline__ void load(int, uint4 (&r)[N]) {
        const int t = threadIdx.x, row = r0 + (t >> 1);
        const bool ok = row < nao;
        const long off = L * strideL + r_index(nao, row, kc * b3::BK) + (t & 1) * 16;
        b3::PlaneRows128::fetch(ok ? hi + off : hi, ok ? lo + off : lo, ok, r);
        if (++kc == kchunks) {
            kc = 0;
            ++L;
        }
    }
    __device__ __forceinline__ void store(const uint4 (&r)[N], u16 *h, u16 *l) const {
        b3::PlaneRows128::put(r, h, l);
    }
};

// One 128 x 128 output tile (i0, j0) of step 2 over the K-steps [s0, s1);
// writes (beta = 0) or adds (beta = 1) into the FP64 partial o.
__device__ __forceinline__ void step2_tile(const u16 *lhi, const u16 *llo, const u16 *rhi, const u16 *rlo, int nao,
                                           long ldr, long strideL, int i0, int j0, long s0, long s1,
                                           double *__restrict__ o, int beta, u16 *lds) {
    const int kchunks = (int)(ldr / b3::BK);
    const long Ls = s0 / kchunks;
    const int kcs = (int)(s0 - Ls * kchunks);
    RLoader la{lhi, llo, strideL, ldr, i0, nao, kchunks, Ls, kcs};
    RLoader lb{rhi, rlo, strideL, ldr, j0, nao, kchunks, Ls, kcs};
    b3::Acc32<b3::Shape<S2_B, S2_B>::MI, b3::Shape<S2_B, S2_B>::NI> acc;
    bool first = true;
    long s = s0;
    do {
        const int n = (int)min((long)S2_FLUSH, s1 - s);
        acc.zero();
        b3::mainloop<S2_B, S2_B, 2, 2>(la, lb, n, lds, acc);
        const bool add = beta || !first;
        b3::epilogue<S2_B, S2_B, 2, 2>(acc, [&](int r, int c, float v) {
            const int i = i0 + r, j = j0 + c;
            if (i < nao && j < nao) {
                double *dst = o + (long)i * nao + j;
                *dst = add ? *dst + (double)v : (double)v;
            }
        });
        first = false;
        s += n;
    } while (s < s1);
}

// FT[k][j] = F[j][k] split into two planes, j zero-padded to ldft, stored
// chunk-major: (j / 32, k, j % 32).
__device__ __forceinline__ void split_ft_range(const double *__restrict__ F, long ldf, int nao, int nocc, u16 *hi,
                                               u16 *lo, long ldft, long e0, long e1) {
    // e runs over the planes in storage order: chunks of 32 j, each nocc
    // rows k of 32 contiguous j (a step-1 K-step then reads BN rows x 32 j
    // of a plane as one contiguous run)
    for (long e = e0 + threadIdx.x; e < e1; e += blockDim.x) {
        const long chunk = e / ((long)nocc * 32), rem = e % ((long)nocc * 32);
        const int k = (int)(rem / 32), j = (int)(chunk * 32 + rem % 32);
        const double x = j < nao ? F[(long)j * ldf + k] : 0.;
        u16 h, l;
        b3::split((float)x, h, l);
        hi[e] = h;
        lo[e] = l;
    }
}

// Workspace layout of one item (bytes from its base): step-2 partials, then
// per factor side the FT planes and the R planes.
struct Layout {
    long ldr, ldft, ldp;
    size_t ft_elems, r_elems;        // per plane
    size_t ft_bytes, part_bytes, side_bytes, total;
};

// pairs: the packed factor of the pair tiles (rows of ldp) in the place of
// the FT planes
inline Layout layout(int nao, int nocc, long nL, int ksplit, bool two, bool pairs) {
    Layout y;
    y.ldr = pad32(nocc);
    y.ldft = pad32(nao);
    y.ft_elems = (size_t)nocc * y.ldft;
    y.r_elems = (size_t)nL * nao * y.ldr;
    const int bn = pick_bn(y.ldr);
    y.ldp = (y.ldr + bn - 1) / bn * bn;
    y.ft_bytes = align_up(pairs ? (size_t)(nao + 1) * y.ldp * sizeof(unsigned) : 2 * y.ft_elems * sizeof(u16), 256);
    y.part_bytes = align_up((size_t)ksplit * nao * nao * sizeof(double), 256);
    y.side_bytes = y.ft_bytes + align_up(2 * y.r_elems * sizeof(u16), 256);
    y.total = y.part_bytes + (two ? 2 : 1) * y.side_bytes;
    return y;
}

// pointers of one side (0 left, 1 right) inside an item's workspace
struct Side {
    u16 *fthi, *ftlo, *rhi, *rlo;    // fthi: the packed factor with pair tiles
};
inline Side side_ptrs(char *base, const Layout &y, int side) {
    char *b = base + y.part_bytes + side * y.side_bytes;
    Side s;
    s.fthi = (u16 *)b;
    s.ftlo = s.fthi + y.ft_elems;
    s.rhi = (u16 *)(b + y.ft_bytes);
    s.rlo = s.rhi + y.r_elems;
    return s;
}

}  // namespace kb3

}  // namespace kcore
}  // namespace mdf
