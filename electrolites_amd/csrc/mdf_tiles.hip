// Building the pair tiles of a molecule from its pair map (mdf_tiles.h).
#include "mdf_tiles.h"

#include "../../include/mi355df.h"

using namespace mdf;
using namespace mdf::tiles;

namespace {

typedef unsigned long long u64;

// bits[w][i], bit b: (i, 64 w + b) is stored; a wavefront per word.
__global__ __launch_bounds__(256) void tiles_bits_kernel(const int *__restrict__ pmap, int nao, u64 *bits) {
    const int i = blockIdx.x, lane = threadIdx.x & 63;
    for (int w = threadIdx.x >> 6; w * 64 < nao; w += 4) {
        const int j = w * 64 + lane;
        const u64 b = __ballot(j < nao && pmap[(long)i * nao + j] >= 0);
        if (lane == 0) bits[(long)w * nao + i] = b;
    }
}

constexpr int MAX_WORDS = MAX_NAO / 64;

// The least key of a wavefront, in lane 63.
template <int CTRL>
__device__ __forceinline__ u64 dpp_min(u64 k) {
    const int lo = __builtin_amdgcn_update_dpp((int)k, (int)k, CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp((int)(k >> 32), (int)(k >> 32), CTRL, 0xf, 0xf, false);
    const u64 o = (u64)(unsigned)hi << 32 | (unsigned)lo;
    return o < k ? o : k;
}
__device__ __forceinline__ u64 wave_min63(u64 k) {
    k = dpp_min<0x111>(k);      // row_shr 1, 2, 4, 8, then the rows' last lanes
    k = dpp_min<0x112>(k);
    k = dpp_min<0x114>(k);
    k = dpp_min<0x118>(k);
    k = dpp_min<0x142>(k);      // row_bcast 15, 31
    return dpp_min<0x143>(k);
}

// The row order, by one workgroup: a group starts with the unplaced row of
// fewest partners and takes, until it holds 16, the row that adds the fewest
// columns to the group's (ties: the most columns in common, then the lowest
// index), and with it the AOs that follow it and add none (the rest of its
// shell).  About one step per shell, each four barriers and two reads of the
// bit rows long, once per molecule.  A thread keeps its rows' counts in
// registers.
template <int GT, int ROWS>
__global__ __launch_bounds__(GT) void tiles_order_kernel(const u64 *__restrict__ bits, int nao, int nwords, int *rows,
                                                         int nrows) {
    __shared__ u64 U[MAX_WORDS], dval[MAX_WORDS], red[GT / 64];
    __shared__ int dw[MAX_WORDS];
    __shared__ int nd, none[RB];
    const int t = threadIdx.x;
    int deg[ROWS], cnt[ROWS];                  // partners (-1: placed or past the last), those in the group
#pragma unroll
    for (int r = 0; r < ROWS; r++) {
        const int i = t + r * GT;
        deg[r] = i < nao ? 0 : -1;
        cnt[r] = 0;
        if (i < nao)
            for (int w = 0; w < nwords; w++) deg[r] += __popcll(bits[(long)w * nao + i]);
    }
    for (int n = 0; n < nao;) {
        if (n % RB == 0) {
            for (int w = t; w < nwords; w += GT) U[w] = 0;
#pragma unroll
            for (int r = 0; r < ROWS; r++) cnt[r] = 0;
        }
        u64 key = ~0ull;
#pragma unroll
        for (int r = 0; r < ROWS; r++) {
            const u64 k = (u64)(deg[r] - cnt[r]) << 40 | (u64)(MAX_NAO - cnt[r]) << 20 | (u64)(t + r * GT);
            key = deg[r] >= 0 && k < key ? k : key;
        }
        key = wave_min63(key);
        if ((t & 63) == 63) red[t >> 6] = key;
        if (t == 0) nd = 0;
        if (t < RB) none[t] = 0;
        __syncthreads();
        key = red[0];
#pragma unroll
        for (int q = 1; q < GT / 64; q++) key = red[q] < key ? red[q] : key;
        const int best = (int)(key & ((1 << 20) - 1));
        for (int w = t; w < nwords; w += GT) {
            const u64 b = bits[(long)w * nao + best], d = b & ~U[w];
            if (d) {
                U[w] |= b;
                const int q = atomicAdd(&nd, 1);
                dw[q] = w;
                dval[q] = d;
            }
        }
        __syncthreads();
        const int m = nd;
        // four words at a time, every load of them in flight together
        for (int q0 = 0; q0 < m; q0 += 4) {
            u64 v[4][ROWS];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const u64 *b = bits + (long)dw[min(q0 + q, m - 1)] * nao;
#pragma unroll
                for (int r = 0; r < ROWS; r++) v[q][r] = b[min(t + r * GT, nao - 1)];
            }
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const u64 d = q0 + q < m ? dval[q0 + q] : 0;
#pragma unroll
                for (int r = 0; r < ROWS; r++) cnt[r] += __popcll(v[q][r] & d);
            }
        }
#pragma unroll
        for (int r = 0; r < ROWS; r++) {
            const int a = t + r * GT - best;     // AOs after the placed one
            if (a >= 0 && a < RB && deg[r] >= 0 && deg[r] == cnt[r]) none[a] = 1;
        }
        __syncthreads();
        const int left = RB - n % RB;            // room in the group
        int take = 1;
        while (take < left && none[take]) take++;
#pragma unroll
        for (int r = 0; r < ROWS; r++) {
            const int a = t + r * GT - best;
            if (a >= 0 && a < take) deg[r] = -1;
        }
        if (t < take) rows[n + t] = best + t;
        n += take;
        __syncthreads();
    }
    for (int n = nao + t; n < nrows; n += GT) rows[n] = -1;
}

// grp[i]: the group of AO i.
__global__ __launch_bounds__(256) void tiles_groups_kernel(const int *__restrict__ rows, int nrows, int *grp) {
    const int n = blockIdx.x * 256 + threadIdx.x;
    if (n < nrows && rows[n] >= 0) grp[rows[n]] = n / RB;
}

// One workgroup per group: its columns (of its own and later groups with
// LOWER), their count in steps and the map.
template <bool LOWER>
__global__ __launch_bounds__(256) void tiles_map_kernel(const int *__restrict__ pmap, int nao,
                                                        const int *__restrict__ grp, const int *__restrict__ rows,
                                                        int *nstep, int *cols, int *map, int ccap) {
    __shared__ int row[RB];
    __shared__ int wsum[4];
    const int g = blockIdx.x, t = threadIdx.x, lane = t & 63, wave = t >> 6;
    if (t < RB) row[t] = rows[g * RB + t];
    cols += (long)g * ccap;
    map += (long)g * ccap * RB;
    __syncthreads();
    int n = 0;                                 // columns so far
    for (int j0 = 0; j0 < nao; j0 += 256) {
        const int j = j0 + t;
        bool in = false;
        if (j < nao && (!LOWER || grp[j] >= g))
            for (int r = 0; r < RB; r++) in = in || (row[r] >= 0 && pmap[(long)row[r] * nao + j] >= 0);
        const u64 b = __ballot(in);
        if (lane == 0) wsum[wave] = __popcll(b);
        __syncthreads();
        int at = n + __popcll(b & ((1ull << lane) - 1));
        for (int q = 0; q < wave; q++) at += wsum[q];
        if (in) cols[at] = j;
        n += wsum[0] + wsum[1] + wsum[2] + wsum[3];
        __syncthreads();
    }
    for (int c = n + t; c < ccap; c += 256) cols[c] = nao;
    if (t == 0) nstep[g] = (n + G_BK - 1) / G_BK;
    __syncthreads();
    const int i = row[t >> 4];
    for (int s = 0; s * 16 < ccap; s++) {
        const int j = cols[s * 16 + (t & 15)];
        int p = i >= 0 && j < nao ? pmap[(long)i * nao + j] : -1;
        if (LOWER && p >= 0 && grp[j] == g) p |= HALF;
        map[s * 256 + t] = p;
    }
}

}  // namespace

extern "C" size_t mdf_pair_tiles_bytes(int nao) {
    return nao > 0 && nao <= MAX_NAO ? (size_t)offsets(nao).total * sizeof(int) : 0;
}

extern "C" int mdf_build_pair_tiles(const int *pair_map, int nao, int lower, const void *order_of, void *tiles,
                                    size_t tiles_bytes, void *stream) {
    MDF_CHECK_ARG(nao > 0 && nao <= MAX_NAO, "mdf_build_pair_tiles: nao %d not in 1..%d", nao, MAX_NAO);
    MDF_CHECK_ARG(pair_map && tiles && tiles_bytes >= mdf_pair_tiles_bytes(nao),
                  "mdf_build_pair_tiles: null pointer or %zu bytes < %zu", tiles_bytes, mdf_pair_tiles_bytes(nao));
    hipStream_t st = as_stream(stream);
    const Offsets o = offsets(nao);
    int *b = (int *)tiles;
    const int nw = (nao + 63) / 64, ng = groups(nao), nrows = ng * RB;
    int *rows = b + o.rows, *grp = b + o.scratch;
    u64 *bits = (u64 *)(b + (o.scratch + nao + 1) / 2 * 2);
    const unsigned gr = (unsigned)cdiv(nrows, 256);
    if (order_of) {
        MDF_HIP(hipMemcpyAsync(rows, (const int *)order_of + o.rows, nrows * sizeof(int), hipMemcpyDeviceToDevice, st));
    } else {
        hipLaunchKernelGGL(tiles_bits_kernel, dim3((unsigned)nao), dim3(256), 0, st, pair_map, nao, bits);
        MDF_LAUNCHED("tiles_bits_kernel");
        if (nao <= 512)
            hipLaunchKernelGGL((tiles_order_kernel<256, 2>), dim3(1), dim3(256), 0, st, bits, nao, nw, rows, nrows);
        else if (nao <= 2048)
            hipLaunchKernelGGL((tiles_order_kernel<512, 4>), dim3(1), dim3(512), 0, st, bits, nao, nw, rows, nrows);
        else if (nao <= 8192)
            hipLaunchKernelGGL((tiles_order_kernel<1024, 8>), dim3(1), dim3(1024), 0, st, bits, nao, nw, rows, nrows);
        else
            hipLaunchKernelGGL((tiles_order_kernel<1024, MAX_NAO / 1024>), dim3(1), dim3(1024), 0, st, bits, nao, nw, rows, nrows);
        MDF_LAUNCHED("tiles_order_kernel");
    }
    hipLaunchKernelGGL(tiles_groups_kernel, dim3(gr), dim3(256), 0, st, rows, nrows, grp);
    MDF_LAUNCHED("tiles_groups_kernel");
    if (lower)
        hipLaunchKernelGGL(tiles_map_kernel<true>, dim3((unsigned)ng), dim3(256), 0, st, pair_map, nao, grp, rows,
                           b + o.nstep, b + o.cols, b + o.map, col_cap(nao));
    else
        hipLaunchKernelGGL(tiles_map_kernel<false>, dim3((unsigned)ng), dim3(256), 0, st, pair_map, nao, grp, rows,
                           b + o.nstep, b + o.cols, b + o.map, col_cap(nao));
    MDF_LAUNCHED("tiles_map_kernel");
    return MDF_OK;
}
