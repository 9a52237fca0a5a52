// Pair tiles: the stored pairs of a screened cderi as blocks of 16 AO rows,
// each with the list of the columns any of its rows is paired with.
//
// K's step 1, R[L, i, k] = sum_j A_L[i, j] F[j, k], multiplies a symmetric A_L
// that is mostly zero: 32 % of its entries are stored for 64 waters, 47 % for
// 32.  In AO order every 128 x 16 block of it holds a stored pair, so nothing
// can be skipped.  What is sparse is the rows by kind: tight functions pair
// only with near ones, diffuse ones with all.  Grouping rows whose partners
// agree (greedily: the next row of a group is the one that adds the fewest
// columns) and compacting each group's columns leaves 44 % of nao^2 at 64
// waters, 60 % at 32, 87 % at 8 (16-row groups; 32-row ones 50, 67, 92 %, 64-
// row ones 58, 75, 97 %).  A workgroup takes 16 rows x 8 aux rows as its 128
// tile rows: the map entry and the factor rows of a K-step serve 8 aux rows.
//
// One device buffer holds a molecule's tiles (built from its pair map on the
// device, no transfer to the host):
//   rows[G][16]       AO index of each row, -1 past the last
//   nstep[G]          K-steps of 16 columns
//   cols[G][C]        AO index of each column, ascending; nao past the last
//   map[G][C/16][256] column of the cderi of (row, col), -1 where not stored;
//                     entry 16 ii + jj of a step
// with G = ceil(nao / 16) groups and C = nao rounded up to 32, plus 32 (a
// loader reads one step ahead).
#pragma once
#include "mdf_common.h"
#include "mdf_gemm.h"

namespace mdf {
namespace tiles {

constexpr int RB = 16;      // rows of a group
constexpr int NL = 8;       // aux rows of a workgroup
constexpr int MAX_NAO = 32768;
//: a `lower` map entry carries the factor 1/2 (pairs inside one group)
constexpr int HALF = 1 << 30;
constexpr int INDEX = HALF - 1;

struct View {
    int nao, ngroup, ccap;
    const int *rows, *nstep, *cols, *map;
};

__host__ __device__ inline int groups(int nao) { return (nao + RB - 1) / RB; }
__host__ __device__ inline int col_cap(int nao) { return (nao + 31) / 32 * 32 + 32; }

// Offsets (ints) of the parts of the buffer; `scratch` holds the build's group
// of each AO and bit rows.
struct Offsets {
    long rows, nstep, cols, map, scratch, total;
};
__host__ __device__ inline Offsets offsets(int nao) {
    const long g = groups(nao), c = col_cap(nao), w = (nao + 63) / 64;
    Offsets o;
    o.rows = 0;
    o.nstep = o.rows + g * RB;
    o.cols = (o.nstep + g + 63) / 64 * 64;
    o.map = (o.cols + g * c + 63) / 64 * 64;
    o.scratch = o.map + g * c * RB;
    o.total = o.scratch + nao + 2 + 2 * w * nao;
    return o;
}
__host__ __device__ inline View view(const void *buf, int nao) {
    const Offsets o = offsets(nao);
    const int *b = (const int *)buf;
    return View{nao, groups(nao), col_cap(nao), b + o.rows, b + o.nstep, b + o.cols, b + o.map};
}

// A operand: K-step kt of the group covers 16 of its columns; tile row
// 16 l + ii is AO row ii of aux row l.  A thread owns one (ii, jj) of the
// step, one map entry, and N of the 8 aux rows: its N loads share the index
// and one branch.  16 lanes run along jj, contiguous in the cderi where the
// columns are consecutive and below the row.
template <typename T, typename Src, int THREADS, bool HALVES>
struct ALoader {
    using reg_t = Src;
    static constexpr int N = RB * NL * G_BK / THREADS;      // 8 (256 threads) or 4 (512)
    static constexpr int SWZ = 1;
    const char *row[N];       // this thread's aux rows
    const int *map;           // the group's map, at this thread's entry
    int e, l0;                // entry 16 ii + jj, first aux row
    int pm;                   // the next step's map entry, read one call ahead
    bool stored, half;        // the loaded step's entry
    __device__ __forceinline__ void init(const Src *c, long ld, int nl, const int *gmap) {
        e = threadIdx.x & 255;
        l0 = (__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) >> 2) * N;   // uniform: the rows stay in SGPRs
#pragma unroll
        for (int v = 0; v < N; v++) row[v] = (const char *)(c + (long)min(l0 + v, nl - 1) * ld);
        map = gmap + e;
        pm = map[0];
    }
    // Every lane loads (one not stored the row's first value, then zeroed): a
    // branch around the loads would make each later wait drain them all.
    __device__ __forceinline__ void load(int kt, Src (&r)[N]) {
        const int p = pm;
        const unsigned off = (unsigned)(p >= 0 ? (HALVES ? p & INDEX : p) : 0) * (unsigned)sizeof(Src);
#pragma unroll
        for (int v = 0; v < N; v++) r[v] = *(const Src *)(row[v] + off);
        stored = p >= 0;
        if (HALVES) half = p & HALF;
        pm = map[(kt + 1) * 256];
    }
    __device__ __forceinline__ void store(const Src (&r)[N], T *lds, int pitch) const {
        T *d = lds + (e & 15) * pitch + ((e >> 4) ^ swizzle<SWZ>(e & 15)) + l0 * RB;
        const Src f = HALVES && half ? (Src)0.5 : (Src)1;
#pragma unroll
        for (int v = 0; v < N; v++) d[v * RB] = stored ? (T)(HALVES ? f * r[v] : r[v]) : (T)0;
    }
};

// B operand: the factor rows of the group's columns, from the packed factor
// (rows of ldp = whole tile widths, row nao zero).  Pieces of two values at
// a stride of a whole row of threads: loads and LDS stores run along rows.
template <int BN, typename T, int THREADS>
struct BLoader {
    using reg_t = T;
    static constexpr int N = BN * G_BK / THREADS;
    static constexpr int SWZ = 0;
    static constexpr int TPR = THREADS / G_BK;          // threads per k row
    static constexpr int Q = N / 2;
    static_assert(Q * 2 == N && Q * 2 * TPR == BN, "BLoader shape");
    struct alignas(2 * sizeof(T)) Pair { T x, y; };
    const T *base;            // packed factor at this thread's first column
    const int *cols;          // the group's columns, at this thread's k row
    unsigned ldp;
    int j;                    // the next step's column, read one call ahead
    __device__ __forceinline__ void init(const T *fp, unsigned ldp_, int k0, const int *gcols) {
        base = fp + k0 + 2 * (threadIdx.x % TPR);
        cols = gcols + threadIdx.x / TPR;
        ldp = ldp_;
        j = cols[0];
    }
    __device__ __forceinline__ void load(int kt, T (&r)[N]) {
        const T *src = base + (unsigned long)((unsigned)j * ldp);
        j = cols[(kt + 1) * G_BK];
#pragma unroll
        for (int q = 0; q < Q; q++) {
            const Pair p = *(const Pair *)(src + q * 2 * TPR);
            r[2 * q] = p.x;
            r[2 * q + 1] = p.y;
        }
    }
    __device__ __forceinline__ void store(const T (&r)[N], T *lds, int pitch) const {
        T *d = lds + (threadIdx.x / TPR) * pitch + 2 * (threadIdx.x % TPR);
#pragma unroll
        for (int q = 0; q < Q; q++) *(Pair *)(d + q * 2 * TPR) = Pair{r[2 * q], r[2 * q + 1]};
    }
};

// Fp[j][k] = F[j][k] in T, zero for k in nocc..ldp-1 and in row nao.
template <typename T>
__device__ __forceinline__ void pack_factor_range(const double *__restrict__ F, long ldf, int nao, int nocc,
                                                  T *__restrict__ fp, long ldp, long e0, long e1) {
    for (long e = e0 + threadIdx.x; e < e1; e += blockDim.x) {
        const int j = (int)(e / ldp), k = (int)(e - (long)j * ldp);
        fp[e] = j < nao && k < nocc ? (T)F[(long)j * ldf + k] : (T)0;
    }
}

}  // namespace tiles
}  // namespace mdf
