// Exchange (K) contraction over the packed cderi on FP64 MFMA.
//
// Restates electrolites/fastdf.py:974-1005 (unpack + step 1 + step 2) and
// :330-335 (_syrk):
//     R[L, i, k] = sum_j A_L[i, j] F[j, k]                 (step 1)
//     K[i, j]   += sum_{L,k} R_l[L, i, k] R_r[L, j, k]     (step 2)
// where A_L is row L of the cderi unpacked to a symmetric nao x nao matrix.
// The reference materialises A_L with GPU4PySCF's fill_symmetric before the
// GEMM; here the unpack is fused into the step-1 A-operand load: each 128x16
// A tile is read straight from the packed triangle (row-contiguous below the
// diagonal, column-contiguous above it, so both halves load coalesced).
//
// Mode 0 (one factor, fr == NULL): step 2 is a symmetric rank-k update and
// only lower-triangle 128x128 output tiles are computed.  Mode 1: general
// GEMM.  Step 2 splits the (L, k) reduction across workgroups (ksplit); the
// per-split partials are summed in a fixed order by k_finalize, so results do
// not depend on scheduling.
//
// Precision: prec = 0 runs both steps on FP64 MFMA; prec = 1 converts the
// packed cderi and the factors to FP32 on the way into LDS, runs both steps
// on FP32 MFMA with FP32 accumulation and stores R in FP32 (the mixed-
// precision SCF cycles); the cross-split sum and the output stay FP64.
#include <algorithm>

#include "mdf_common.h"
#include "mdf_gemm.h"
#include "mdf_kcore.h"
#include "../../include/mi355df.h"

using namespace mdf;
using namespace mdf::kcore;

namespace {

// 1-D grid of round_xcd(nkt * nit * nL) workgroups in XCD order; tile
// (k-tile fastest, then i-tile, then aux row) so the k-tiles of one A tile
// share an L2.
template <int BN, bool MAPPED, typename T, typename Src, bool TRI = false>
__global__ __launch_bounds__(Step1Shape<BN>::THREADS) void k_step1(
    const Src *__restrict__ cderi, long ld, const int *__restrict__ pmap, int nao,
    const double *__restrict__ F, long ldf, int nocc, T *__restrict__ R, long ldr,
    long strideL, long strideB, int nkt, int nit, long ntiles) {
    __shared__ T lds[Step1Shape<BN>::S::LDS_ELEMS];
    const long x = xcd_tile(blockIdx.x, gridDim.x);
    if (x >= ntiles) return;
    const int kt = (int)(x % nkt), it = (int)((x / nkt) % nit);
    const long L = x / ((long)nkt * nit);
    step1_tile<BN, MAPPED, T, Src, TRI>(cderi + L * ld, pmap, nao, F, ldf, nocc,
                                        R + L / RL * strideB + L % RL * strideL, ldr, it * 128, kt * BN, lds);
}

// The pair-tile step 1: 1-D grid of round_xcd(nkt * ngroup * blocks of 8 aux
// rows) workgroups in XCD order, k-tile fastest, then group (the longest, the
// last placed, first), then aux rows: the groups of one aux block read the
// same cderi rows.
template <int BN, typename T, typename Src, bool HALVES>
__global__ __launch_bounds__(Step1Shape<BN>::THREADS, 2) void k_step1_pairs(
    const Src *__restrict__ cderi, long ld, int nL, tiles::View tv, const T *__restrict__ fp, unsigned ldp, int nocc,
    T *__restrict__ R, long ldr, long strideL, long strideB, int nkt, long ntiles) {
    __shared__ T lds[Step1Shape<BN>::S::LDS_ELEMS];
    const long x = xcd_tile(blockIdx.x, gridDim.x);
    if (x >= ntiles) return;
    const int kt = (int)(x % nkt);
    const long y = x / nkt;
    const int g = tv.ngroup - 1 - (int)(y % tv.ngroup);
    const long b = y / tv.ngroup, L = b * tiles::NL;
    step1_pairs_tile<BN, T, Src, HALVES>(cderi + L * ld, ld, (int)min((long)tiles::NL, nL - L), tv, g, fp, ldp, nocc,
                                         R + b * strideB, ldr, strideL, kt * BN, lds);
}

template <typename T>
__global__ __launch_bounds__(256) void k_pack_factor(const double *__restrict__ F, long ldf, int nao, int nocc,
                                                     T *__restrict__ fp, long ldp) {
    const long e0 = (long)blockIdx.x * 1024;
    tiles::pack_factor_range(F, ldf, nao, nocc, fp, ldp, e0, min(e0 + 1024, (long)(nao + 1) * ldp));
}

// 1-D grid of ntiles_grid * ksplit workgroups, (tile, split) by step2_coords.
template <int B, bool SYM, typename T>
__global__ __launch_bounds__(G_THREADS, B == 64 ? 4 : 2) void k_step2(
    const T *__restrict__ Rl, const T *__restrict__ Rr, int nao, RShape y, int ntile, int ntiles_grid, int ksplit,
    double *__restrict__ part, long part_stride, int beta) {
    __shared__ T lds[TileShape<B, B>::LDS_ELEMS];
    int tile, split, ti, tj;
    step2_coords(blockIdx.x, ntiles_grid, tile, split);
    if (SYM) {
        tri_tile(tile, ti, tj);
    } else {
        ti = tile / ntile;
        tj = tile % ntile;
    }
    const long nsteps = y.steps();
    const long s0 = nsteps * split / ksplit, s1 = nsteps * (split + 1) / ksplit;
    step2_tile<B, T>(Rl, Rr, nao, y, ti * B, tj * B, s0, s1, part + (long)split * part_stride, beta, lds);
}

__global__ __launch_bounds__(256) void k_finalize(
    const double *__restrict__ part, int ksplit, long part_stride, int nao, int sym,
    double *__restrict__ vk, long ldvk, int accumulate) {
    const long e0 = (long)blockIdx.x * 256;
    finalize_range(part, ksplit, part_stride, nao, sym, vk, ldvk, accumulate, e0,
                   min(e0 + 256, (long)nao * nao));
}

// ---- split-BF16 (prec 2)
__global__ __launch_bounds__(256) void k_split_ft(const double *__restrict__ F, long ldf, int nao, int nocc,
                                                  b3::u16 *hi, b3::u16 *lo, long ldft) {
    const long e0 = (long)blockIdx.x * 1024;
    kb3::split_ft_range(F, ldf, nao, nocc, hi, lo, ldft, e0, min(e0 + 1024, (long)nocc * ldft));
}

template <bool MAPPED, int BN, typename Src>
__global__ __launch_bounds__(kb3::Step1Cfg<BN>::THREADS) void k_step1_b3(
    const Src *__restrict__ cderi, long ld, const int *__restrict__ pmap, int nao, const b3::u16 *fthi,
    const b3::u16 *ftlo, long ldft, int nocc, b3::u16 *Rhi, b3::u16 *Rlo, long ldr, long strideL, int nkt,
    int nit, long ntiles) {
    __shared__ b3::u16 lds[kb3::Step1Cfg<BN>::S::LDS_ELEMS];
    const long x = xcd_tile(blockIdx.x, gridDim.x);
    if (x >= ntiles) return;
    const int kt = (int)(x % nkt), it = (int)((x / nkt) % nit);
    const long z = x / ((long)nkt * nit);
    kb3::step1_tile<MAPPED, BN, Src>(cderi + z * ld, pmap, nao, fthi, ftlo, ldft, nocc, Rhi + z * strideL,
                                Rlo + z * strideL, ldr, it * kb3::BM, kt * BN, lds);
}

// The pair-tile step 1, tiles ordered as k_step1_pairs.
template <int BN, typename Src>
__global__ __launch_bounds__(kb3::Step1Cfg<BN>::THREADS) void k_step1_pairs_b3(
    const Src *__restrict__ cderi, long ld, int nL, tiles::View tv, const unsigned *__restrict__ fp, unsigned ldp,
    b3::u16 *Rhi, b3::u16 *Rlo, long ldr, long strideL, int nkt, long ntiles) {
    __shared__ b3::u16 lds[kb3::Step1Cfg<BN>::S::LDS_ELEMS];
    const long x = xcd_tile(blockIdx.x, gridDim.x);
    if (x >= ntiles) return;
    const int kt = (int)(x % nkt);
    const long y = x / nkt;
    const int g = tv.ngroup - 1 - (int)(y % tv.ngroup);
    const long L = y / tv.ngroup * tiles::NL;
    kb3::step1_pairs_tile<BN, Src>(cderi + L * ld, ld, (int)min((long)tiles::NL, nL - L), tv, g, fp, ldp,
                                   Rhi + L * strideL, Rlo + L * strideL, ldr, strideL, kt * BN, lds);
}

__global__ __launch_bounds__(256) void k_pack_split(const double *__restrict__ F, long ldf, int nao, int nocc,
                                                    unsigned *fp, long ldp) {
    const long e0 = (long)blockIdx.x * 1024;
    kb3::pack_split_range(F, ldf, nao, nocc, fp, ldp, e0, min(e0 + 1024, (long)(nao + 1) * ldp));
}

template <int BN, typename Src>
void launch_step1_pairs_b3(int nL, hipStream_t st, const Src *blk, long ld, const tiles::View &tv, const kb3::Side &q,
                           const kb3::Layout &y, long strideL) {
    const int nkt = (int)(y.ldp / BN);
    const long ntiles = (long)nkt * tv.ngroup * cdiv(nL, tiles::NL);
    hipLaunchKernelGGL((k_step1_pairs_b3<BN, Src>), dim3((unsigned)round_xcd(ntiles)),
                       dim3(kb3::Step1Cfg<BN>::THREADS), 0, st, blk, ld, nL, tv, (const unsigned *)q.fthi,
                       (unsigned)y.ldp, q.rhi, q.rlo, y.ldr, strideL, nkt, ntiles);
}

template <int BN, typename Src>
void launch_step1_b3(int nL, hipStream_t st, const Src *blk, long ld, const int *pmap, int nao,
                     const b3::u16 *fthi, const b3::u16 *ftlo, long ldft, int nocc, b3::u16 *rhi, b3::u16 *rlo,
                     long ldr, long strideL) {
    const int nkt = (int)cdiv(ldr, (long)BN), nit = (int)cdiv(nao, kb3::BM);
    const long ntiles = (long)nkt * nit * nL;
    const dim3 g((unsigned)round_xcd(ntiles)), b(kb3::Step1Cfg<BN>::THREADS);
    if (pmap)
        hipLaunchKernelGGL((k_step1_b3<true, BN, Src>), g, b, 0, st, blk, ld, pmap, nao, fthi, ftlo, ldft, nocc, rhi,
                           rlo, ldr, strideL, nkt, nit, ntiles);
    else
        hipLaunchKernelGGL((k_step1_b3<false, BN, Src>), g, b, 0, st, blk, ld, pmap, nao, fthi, ftlo, ldft, nocc, rhi,
                           rlo, ldr, strideL, nkt, nit, ntiles);
}

template <bool SYM>
__global__ __launch_bounds__(G_THREADS, 2) void k_step2_b3(
    const b3::u16 *lhi, const b3::u16 *llo, const b3::u16 *rhi, const b3::u16 *rlo, int nao, long ldr,
    long strideL, int nL, int ntile, int ntiles_grid, int ksplit, double *__restrict__ part, long part_stride,
    int beta) {
    __shared__ b3::u16 lds[b3::Shape<S2_B, S2_B>::LDS_ELEMS];
    int tile, split, ti, tj;
    step2_coords(blockIdx.x, ntiles_grid, tile, split);
    if (SYM) {
        tri_tile(tile, ti, tj);
    } else {
        ti = tile / ntile;
        tj = tile % ntile;
    }
    const long nsteps = (long)nL * (ldr / b3::BK);
    const long s0 = nsteps * split / ksplit, s1 = nsteps * (split + 1) / ksplit;
    kb3::step2_tile(lhi, llo, rhi, rlo, nao, ldr, strideL, ti * S2_B, tj * S2_B, s0, s1,
                    part + (long)split * part_stride, beta, lds);
}

template <int BN, typename T, typename Src, bool TRI = false>
void launch_step1(int nL, hipStream_t st, const Src *blk, long ld, const int *pmap, int nao,
                  const double *f, long ldf, int nocc, T *r, long ldr, long strideL, long strideB) {
    const int nkt = (int)cdiv(nocc, BN), nit = (int)cdiv(nao, 128);
    const long ntiles = (long)nkt * nit * nL;
    const dim3 g((unsigned)round_xcd(ntiles)), b(Step1Shape<BN>::THREADS);
    if (pmap)
        hipLaunchKernelGGL((k_step1<BN, true, T, Src, TRI>), g, b, 0, st, blk, ld, pmap, nao, f, ldf,
                           nocc, r, ldr, strideL, strideB, nkt, nit, ntiles);
    else
        hipLaunchKernelGGL((k_step1<BN, false, T, Src, TRI>), g, b, 0, st, blk, ld, pmap, nao, f, ldf,
                           nocc, r, ldr, strideL, strideB, nkt, nit, ntiles);
}

template <typename T, typename Src, bool TRI = false>
int step1(const KPlan &p, int nL, hipStream_t st, const Src *blk, long ld, const int *pmap, int nao,
          const double *f, long ldf, int nocc, T *r, long ldr, long strideL, long strideB) {
    with_bn(p.bn, [&](auto w) {
        launch_step1<decltype(w)::value, T, Src, TRI>(nL, st, blk, ld, pmap, nao, f, ldf, nocc, r, ldr, strideL,
                                                      strideB);
    });
    MDF_LAUNCHED("k_step1");
    return MDF_OK;
}

template <int BN, typename T, typename Src, bool HALVES>
void launch_step1_pairs(int nL, hipStream_t st, const Src *blk, long ld, const tiles::View &tv, const T *fp,
                        unsigned ldp, int nocc, T *r, long ldr, long strideL, long strideB) {
    const int nkt = (int)cdiv(nocc, BN);
    const long ntiles = (long)nkt * tv.ngroup * cdiv(nL, tiles::NL);
    hipLaunchKernelGGL((k_step1_pairs<BN, T, Src, HALVES>), dim3((unsigned)round_xcd(ntiles)),
                       dim3(Step1Shape<BN>::THREADS), 0, st, blk, ld, nL, tv, fp, ldp, nocc, r, ldr, strideL, strideB,
                       nkt, ntiles);
}

template <typename T, typename Src, bool HALVES = false>
int step1_pairs(const KPlan &p, int nL, hipStream_t st, const Src *blk, long ld, const tiles::View &tv, const T *fp,
                int nocc, T *r, long ldr, long strideL, long strideB) {
    with_bn(p.bn, [&](auto w) {
        launch_step1_pairs<decltype(w)::value, T, Src, HALVES>(nL, st, blk, ld, tv, fp, pack_ld(p, nocc), nocc, r, ldr,
                                                               strideL, strideB);
    });
    MDF_LAUNCHED("k_step1_pairs");
    return MDF_OK;
}

template <typename T>
int pack_factor(const KPlan &p, hipStream_t st, const double *f, long ldf, int nao, int nocc, T *fp) {
    const long n = (long)pack_words(p, nao, nocc);
    hipLaunchKernelGGL(k_pack_factor<T>, dim3((unsigned)cdiv(n, 1024L)), dim3(256), 0, st, f, ldf, nao, nocc, fp,
                       (long)pack_ld(p, nocc));
    MDF_LAUNCHED("k_pack_factor");
    return MDF_OK;
}

template <int B, typename T>
void launch_step2(const KPlan &p, int nL, bool two, hipStream_t st, const T *rl, const T *rr, int nao, int nocc,
                  double *part, long part_stride, int beta) {
    const dim3 g2((unsigned)((long)p.ntiles_grid * p.ksplit));
    const RShape y(nL, nocc, block_of(p.nL));
    if (two)
        hipLaunchKernelGGL((k_step2<B, false, T>), g2, dim3(G_THREADS), 0, st, rl, rr, nao, y, p.ntile, p.ntiles_grid,
                           p.ksplit, part, part_stride, beta);
    else
        hipLaunchKernelGGL((k_step2<B, true, T>), g2, dim3(G_THREADS), 0, st, rl, rl, nao, y, p.ntile, p.ntiles_grid,
                           p.ksplit, part, part_stride, beta);
}

template <typename T>
int step2(const KPlan &p, int nL, bool two, hipStream_t st, const T *rl, const T *rr, int nao, int nocc, double *part,
          long part_stride, int beta) {
    if (p.s2 == 64)
        launch_step2<64, T>(p, nL, two, st, rl, rr, nao, nocc, part, part_stride, beta);
    else
        launch_step2<128, T>(p, nL, two, st, rl, rr, nao, nocc, part, part_stride, beta);
    MDF_LAUNCHED("k_step2");
    return MDF_OK;
}

// The block loop of mdf_get_k for element type T.  Step 1 runs on the pair
// tiles where the caller has them, else from the pair map or the packed
// triangle.
template <typename T, typename Src>
int run_k(const KPlan &p, const Src *cderi, long naux, long ld, const int *pair_map, const void *pair_tiles, int nao,
          const double *fl, const double *fr, int nocc, long ldf, double *vk, long ldvk, int accumulate,
          void *work, hipStream_t st) {
    const bool two = fr != nullptr;
    double *part = (double *)work;
    T *rl = (T *)(part + align_up(p.part_words, 64));
    T *rr = two ? rl + align_up(p.r_words, 64) : rl;
    T *fp[2];
    fp[0] = rr + align_up(p.r_words, 64);
    fp[1] = fp[0] + align_up(pack_words(p, nao, nocc), 64);
    if (pair_tiles)
        for (int side = 0; side < (two ? 2 : 1); side++)
            if (int rc = pack_factor<T>(p, st, side ? fr : fl, ldf, nao, nocc, fp[side])) return rc;
    const long ldr = block_ld(block_of(p.nL), nocc), strideB = (long)nao * ldr;
    const long part_stride = (long)nao * nao;
    for (long L0 = 0; L0 < naux; L0 += p.nL) {
        const int nL = (int)(naux - L0 < p.nL ? naux - L0 : p.nL);
        const Src *blk = cderi + L0 * ld;
        int rc;
        for (int side = 0; side < (two ? 2 : 1); side++) {
            T *r = side ? rr : rl;
            rc = pair_tiles ? step1_pairs<T, Src>(p, nL, st, blk, ld, tiles::view(pair_tiles, nao), fp[side], nocc, r,
                                                  ldr, nocc, strideB)
                            : step1<T, Src>(p, nL, st, blk, ld, pair_map, nao, side ? fr : fl, ldf, nocc, r, ldr,
                                            nocc, strideB);
            if (rc) return rc;
        }
        rc = step2<T>(p, nL, two, st, rl, rr, nao, nocc, part, part_stride, L0 > 0);
        if (rc) return rc;
    }
    long nt = (long)nao * nao;
    hipLaunchKernelGGL(k_finalize, dim3((unsigned)cdiv(nt, 256L)), dim3(256), 0, st,
                       part, p.ksplit, part_stride, nao, two ? 0 : p.s2, vk, ldvk, accumulate);
    MDF_LAUNCHED("k_finalize");
    return MDF_OK;
}

// The block loop of mdf_get_k on the split-BF16 engine.
template <typename Src>
int run_k_b3(const KPlan &p, const Src *cderi, long naux, long ld, const int *pair_map, const void *pair_tiles, int nao,
             const double *fl, const double *fr, int nocc, long ldf, double *vk, long ldvk, int accumulate,
             void *work, hipStream_t st) {
    const bool two = fr != nullptr;
    const kb3::Layout y = kb3::layout(nao, nocc, p.nL, p.ksplit, two, pair_tiles != nullptr);
    double *part = (double *)work;
    kb3::Side sd[2] = {kb3::side_ptrs((char *)work, y, 0), kb3::side_ptrs((char *)work, y, two ? 1 : 0)};
    const long strideL = (long)nao * y.ldr, part_stride = (long)nao * nao;
    const long nft = pair_tiles ? (long)(nao + 1) * y.ldp : (long)nocc * y.ldft;
    for (int side = 0; side < (two ? 2 : 1); side++) {
        if (pair_tiles)
            hipLaunchKernelGGL(k_pack_split, dim3((unsigned)cdiv(nft, 1024L)), dim3(256), 0, st, side ? fr : fl, ldf,
                               nao, nocc, (unsigned *)sd[side].fthi, y.ldp);
        else
            hipLaunchKernelGGL(k_split_ft, dim3((unsigned)cdiv(nft, 1024L)), dim3(256), 0, st, side ? fr : fl, ldf,
                               nao, nocc, sd[side].fthi, sd[side].ftlo, y.ldft);
        MDF_LAUNCHED("k_split_ft");
    }
    auto step1 = [&](auto width, int nL, const Src *blk, const kb3::Side &q) {
        constexpr int BN = decltype(width)::value;
        if (pair_tiles)
            launch_step1_pairs_b3<BN>(nL, st, blk, ld, tiles::view(pair_tiles, nao), q, y, strideL);
        else
            launch_step1_b3<BN>(nL, st, blk, ld, pair_map, nao, q.fthi, q.ftlo, y.ldft, nocc, q.rhi, q.rlo, y.ldr,
                                strideL);
    };
    for (long L0 = 0; L0 < naux; L0 += p.nL) {
        const int nL = (int)(naux - L0 < p.nL ? naux - L0 : p.nL);
        const Src *blk = cderi + L0 * ld;
        for (int side = 0; side < (two ? 2 : 1); side++) {
            switch (kb3::pick_bn(y.ldr)) {
            case 320: step1(std::integral_constant<int, 320>{}, nL, blk, sd[side]); break;
            case 256: step1(std::integral_constant<int, 256>{}, nL, blk, sd[side]); break;
            case 192: step1(std::integral_constant<int, 192>{}, nL, blk, sd[side]); break;
            default: step1(std::integral_constant<int, 128>{}, nL, blk, sd[side]); break;
            }
            MDF_LAUNCHED("k_step1_b3");
        }
        const dim3 g2((unsigned)((long)p.ntiles_grid * p.ksplit));
        const kb3::Side &a = sd[0], &b = sd[two ? 1 : 0];
        if (two)
            hipLaunchKernelGGL(k_step2_b3<false>, g2, dim3(G_THREADS), 0, st, a.rhi, a.rlo, b.rhi, b.rlo, nao, y.ldr,
                               strideL, nL, p.ntile, p.ntiles_grid, p.ksplit, part, part_stride, (int)(L0 > 0));
        else
            hipLaunchKernelGGL(k_step2_b3<true>, g2, dim3(G_THREADS), 0, st, a.rhi, a.rlo, b.rhi, b.rlo, nao, y.ldr,
                               strideL, nL, p.ntile, p.ntiles_grid, p.ksplit, part, part_stride, (int)(L0 > 0));
        MDF_LAUNCHED("k_step2_b3");
    }
    long nt = (long)nao * nao;
    hipLaunchKernelGGL(k_finalize, dim3((unsigned)cdiv(nt, 256L)), dim3(256), 0, st,
                       part, p.ksplit, part_stride, nao, two ? 0 : p.s2, vk, ldvk, accumulate);
    MDF_LAUNCHED("k_finalize");
    return MDF_OK;
}

}  // namespace

static size_t k_workspace(const KPlan &p, bool two, size_t elem, size_t pack) {
    return align_up(p.part_words, 64) * sizeof(double) +
           (two ? 2 : 1) * (align_up(p.r_words, 64) + align_up(pack, 64)) * elem;
}

// Aux rows per pass and workspace of one call for any precision.
static long k_rows_rule(long naux, int nao, int nocc, bool two, int prec) {
    if (prec == MDF_PREC_BF16X3) return block_rows(naux, nao, (int)kb3::pad32(nocc), two, true, 4);
    return block_rows(naux, nao, nocc, two, false, prec == MDF_PREC_FP32 ? sizeof(float) : sizeof(double));
}
static size_t k_bytes(long naux, int nao, int nocc, bool two, int prec, long rows, bool pairs) {
    KPlan p = plan_k(naux, nao, nocc, two, rows, prec == MDF_PREC_BF16X3);
    if (prec == MDF_PREC_BF16X3) return kb3::layout(nao, nocc, p.nL, p.ksplit, two, pairs).total;
    return k_workspace(p, two, prec == MDF_PREC_FP32 ? sizeof(float) : sizeof(double),
                       pairs ? pack_words(p, nao, nocc) : 0);
}

static size_t k_workspace_rule(long naux, int nao, int nocc, bool two, int prec, long max_block_rows, bool pairs) {
    long rows = k_rows_rule(naux, nao, nocc, two, prec);
    if (max_block_rows > 0) rows = std::min(rows, rows_within(naux, max_block_rows, prec == MDF_PREC_BF16X3));
    return k_bytes(naux, nao, nocc, two, prec, rows, pairs);
}

extern "C" size_t mdf_get_k_workspace(long naux, int nao, int nocc, int two_factors, int prec,
                                      long max_block_rows) {
    return k_workspace_rule(naux, nao, nocc, two_factors != 0, prec, max_block_rows, false);
}

extern "C" size_t mdf_get_k_tiles_workspace(long naux, int nao, int nocc, int two_factors, int prec,
                                            long max_block_rows) {
    return k_workspace_rule(naux, nao, nocc, two_factors != 0, prec, max_block_rows, true);
}

extern "C" int mdf_get_k(const void *cderi, int cderi_dtype, long naux, long npairs, long ld, const int *pair_map,
                         int nao, const double *fl, const double *fr, int nocc, long ldf, int prec,
                         double *vk, long ldvk, int accumulate, void *work, size_t work_bytes,
                         void *stream) {
    return mdf_get_k_tiles(cderi, cderi_dtype, naux, npairs, ld, pair_map, nullptr, nao, fl, fr, nocc, ldf, prec, vk,
                           ldvk, accumulate, work, work_bytes, stream);
}

extern "C" int mdf_get_k_tiles(const void *cderi, int cderi_dtype, long naux, long npairs, long ld,
                               const int *pair_map, const void *pair_tiles, int nao, const double *fl,
                               const double *fr, int nocc, long ldf, int prec, double *vk, long ldvk, int accumulate,
                               void *work, size_t work_bytes, void *stream) {
    MDF_CHECK_ARG(naux >= 0 && nao >= 0 && nocc >= 0, "mdf_get_k: bad sizes");
    MDF_CHECK_ARG(cderi && fl && vk, "mdf_get_k: null pointer");
    MDF_CHECK_ARG(ld >= npairs && ldf >= nocc && ldvk >= nao, "mdf_get_k: leading dimension too small");
    MDF_CHECK_ARG(prec == MDF_PREC_FP64 || prec == MDF_PREC_FP32 || prec == MDF_PREC_BF16X3,
                  "mdf_get_k: unknown precision %d", prec);
    MDF_CHECK_ARG(cderi_dtype == MDF_DTYPE_F64 || cderi_dtype == MDF_DTYPE_F32, "mdf_get_k: cderi dtype %d",
                  cderi_dtype);
    MDF_CHECK_ARG(pair_map || npairs == (long)nao * (nao + 1) / 2,
                  "mdf_get_k: without a pair map the cderi must hold the full packed triangle "
                  "(npairs=%ld, nao=%d)", npairs, nao);
    MDF_CHECK_ARG(!pair_tiles || (nao <= tiles::MAX_NAO && npairs < (1L << 29)),
                  "mdf_get_k: pair tiles hold up to %d functions and 2^29 pairs (nao=%d, npairs=%ld)", tiles::MAX_NAO,
                  nao, npairs);
    hipStream_t st = as_stream(stream);
    if (nao == 0) return MDF_OK;
    const bool two = fr != nullptr, pairs = pair_tiles != nullptr;
    if (nocc == 0 || naux == 0) {
        if (!accumulate)
            for (int i = 0; i < nao; i++) MDF_HIP(hipMemsetAsync(vk + (long)i * ldvk, 0, nao * sizeof(double), st));
        return MDF_OK;
    }
    const long most = max_cols(nao);
    if (nocc > most) {
        // the sum over the columns in parts
        for (long k0 = 0; k0 < nocc; k0 += most)
            if (int rc = mdf_get_k_tiles(cderi, cderi_dtype, naux, npairs, ld, pair_map, pair_tiles, nao, fl + k0,
                                         two ? fr + k0 : nullptr, (int)(nocc - k0 < most ? nocc - k0 : most), ldf, prec,
                                         vk, ldvk, accumulate || k0 > 0, work, work_bytes, stream))
                return rc;
        return MDF_OK;
    }
    MDF_CHECK_ARG(work != nullptr, "mdf_get_k: workspace is null");
    size_t need1 = k_bytes(naux, nao, nocc, two, prec, 1, pairs);
    if (work_bytes < need1) {
        set_error("mdf_get_k: workspace %zu bytes < %zu required", work_bytes, need1);
        return MDF_EWORKSPACE;
    }
    // passes of the shape rule's aux rows (the grouped launch cuts the same
    // way); shorter when the workspace is smaller
    long rows = k_rows_rule(naux, nao, nocc, two, prec);
    if (k_bytes(naux, nao, nocc, two, prec, rows, pairs) > work_bytes) {
        long lo = 1, hi = rows;          // largest rows that fit
        while (lo < hi) {
            const long mid = (lo + hi + 1) / 2;
            if (k_bytes(naux, nao, nocc, two, prec, mid, pairs) <= work_bytes) lo = mid; else hi = mid - 1;
        }
        rows = lo;
    }
    KPlan p = plan_k(naux, nao, nocc, two, rows, prec == MDF_PREC_BF16X3);
    if (cderi_dtype == MDF_DTYPE_F32) {
        const float *c = (const float *)cderi;
        if (prec == MDF_PREC_BF16X3)
            return run_k_b3(p, c, naux, ld, pair_map, pair_tiles, nao, fl, fr, nocc, ldf, vk, ldvk, accumulate, work,
                            st);
        if (prec == MDF_PREC_FP32)
            return run_k<float>(p, c, naux, ld, pair_map, pair_tiles, nao, fl, fr, nocc, ldf, vk, ldvk, accumulate,
                                 work, st);
        return run_k<double>(p, c, naux, ld, pair_map, pair_tiles, nao, fl, fr, nocc, ldf, vk, ldvk, accumulate,
                                 work, st);
    }
    const double *c = (const double *)cderi;
    if (prec == MDF_PREC_BF16X3)
        return run_k_b3(p, c, naux, ld, pair_map, pair_tiles, nao, fl, fr, nocc, ldf, vk, ldvk, accumulate, work,
                            st);
    if (prec == MDF_PREC_FP32)
        return run_k<float>(p, c, naux, ld, pair_map, pair_tiles, nao, fl, fr, nocc, ldf, vk, ldvk, accumulate,
                                 work, st);
    return run_k<double>(p, c, naux, ld, pair_map, pair_tiles, nao, fl, fr, nocc, ldf, vk, ldvk, accumulate,
                                 work, st);
}

// The first step of mdf_get_k alone, FP64: R[L] = A_L F for the nL aux rows
// of one block (A_L the unpacked symmetric row L), R[L * strideL + i * ldr +
// k] for i < nao, k < nocc.  The DF gradient's rhok = F_r^T A_L F_l takes its
// inner product from here.
namespace {
template <bool TRI>
int k_step1_entry(const char *name, const void *cderi, int cderi_dtype, long nL, long npairs, long ld,
                  const int *pair_map, int nao, const double *f, long ldf, int nocc, double *R, long ldr,
                  long strideL, void *stream) {
    MDF_CHECK_ARG(nL >= 0 && nao >= 0 && nocc >= 0 && nL < (1L << 31), "%s: bad sizes", name);
    MDF_CHECK_ARG(cderi && f && R, "%s: null pointer", name);
    MDF_CHECK_ARG(ld >= npairs && ldf >= nocc && ldr >= nocc && strideL >= (long)nao * ldr,
                  "%s: leading dimension too small", name);
    MDF_CHECK_ARG(cderi_dtype == MDF_DTYPE_F64 || cderi_dtype == MDF_DTYPE_F32, "%s: cderi dtype %d", name,
                  cderi_dtype);
    MDF_CHECK_ARG(pair_map || npairs == (long)nao * (nao + 1) / 2,
                  "%s: without a pair map the cderi must hold the full packed triangle "
                  "(npairs=%ld, nao=%d)", name, npairs, nao);
    if (nL == 0 || nao == 0 || nocc == 0) return MDF_OK;
    KPlan p{};
    p.bn = pick_bn(nocc);
    hipStream_t st = as_stream(stream);
    if (cderi_dtype == MDF_DTYPE_F32)
        return step1<double, float, TRI>(p, (int)nL, st, (const float *)cderi, ld, pair_map, nao, f, ldf, nocc, R,
                                         ldr, strideL, RL * strideL);
    return step1<double, double, TRI>(p, (int)nL, st, (const double *)cderi, ld, pair_map, nao, f, ldf, nocc, R,
                                         ldr, strideL, RL * strideL);
}
}  // namespace

extern "C" int mdf_k_step1_lower(const void *cderi, int cderi_dtype, long nL, long npairs, long ld,
                                 const int *pair_map, int nao, const double *f, long ldf, int nocc, double *R,
                                 long ldr, long strideL, void *stream) {
    return k_step1_entry<true>("mdf_k_step1_lower", cderi, cderi_dtype, nL, npairs, ld, pair_map, nao, f, ldf,
                               nocc, R, ldr, strideL, stream);
}

extern "C" int mdf_k_step1(const void *cderi, int cderi_dtype, long nL, long npairs, long ld, const int *pair_map,
                           int nao, const double *f, long ldf, int nocc, double *R, long ldr, long strideL,
                           void *stream) {
    return k_step1_entry<false>("mdf_k_step1", cderi, cderi_dtype, nL, npairs, ld, pair_map, nao, f, ldf, nocc, R,
                                ldr, strideL, stream);
}

extern "C" size_t mdf_k_step1_tiles_workspace(int nao, int nocc) {
    KPlan p{};
    p.bn = pick_bn(nocc);
    return pack_words(p, nao, nocc) * sizeof(double);
}

extern "C" int mdf_k_step1_tiles(const void *cderi, int cderi_dtype, long nL, long npairs, long ld,
                                 const void *pair_tiles, int lower, int nao, const double *f, long ldf, int nocc,
                                 double *R, long ldr, long strideL, void *work, size_t work_bytes, void *stream) {
    MDF_CHECK_ARG(nL >= 0 && nao >= 0 && nocc >= 0 && nL < (1L << 31), "mdf_k_step1_tiles: bad sizes");
    MDF_CHECK_ARG(cderi && pair_tiles && f && R, "mdf_k_step1_tiles: null pointer");
    MDF_CHECK_ARG(ld >= npairs && ldf >= nocc && ldr >= nocc && strideL >= (long)nao * ldr,
                  "mdf_k_step1_tiles: leading dimension too small");
    MDF_CHECK_ARG(cderi_dtype == MDF_DTYPE_F64 || cderi_dtype == MDF_DTYPE_F32, "mdf_k_step1_tiles: cderi dtype %d",
                  cderi_dtype);
    MDF_CHECK_ARG(nao <= tiles::MAX_NAO && npairs < (1L << 29),
                  "mdf_k_step1_tiles: pair tiles hold up to %d functions and 2^29 pairs", tiles::MAX_NAO);
    MDF_CHECK_ARG(nocc <= max_cols(nao), "mdf_k_step1_tiles: nocc %d > %ld", nocc, max_cols(nao));
    if (nL == 0 || nao == 0 || nocc == 0) return MDF_OK;
    const size_t need = mdf_k_step1_tiles_workspace(nao, nocc);
    if (!work || work_bytes < need) {
        set_error("mdf_k_step1_tiles: workspace %zu bytes < %zu required", work ? work_bytes : (size_t)0, need);
        return MDF_EWORKSPACE;
    }
    KPlan p{};
    p.bn = pick_bn(nocc);
    hipStream_t st = as_stream(stream);
    double *fp = (double *)work;
    if (int rc = pack_factor<double>(p, st, f, ldf, nao, nocc, fp)) return rc;
    const tiles::View tv = tiles::view(pair_tiles, nao);
    const long sB = RL * strideL;
    if (cderi_dtype == MDF_DTYPE_F32) {
        const float *c = (const float *)cderi;
        return lower ? step1_pairs<double, float, true>(p, (int)nL, st, c, ld, tv, fp, nocc, R, ldr, strideL, sB)
                     : step1_pairs<double, float, false>(p, (int)nL, st, c, ld, tv, fp, nocc, R, ldr, strideL, sB);
    }
    const double *c = (const double *)cderi;
    return lower ? step1_pairs<double, double, true>(p, (int)nL, st, c, ld, tv, fp, nocc, R, ldr, strideL, sB)
                 : step1_pairs<double, double, false>(p, (int)nL, st, c, ld, tv, fp, nocc, R, ldr, strideL, sB);
}
