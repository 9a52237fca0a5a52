// Shared declarations of the Rys integral kernels (hand-written entry points
// in mdf_int.hip, generated kernels in mdf_int_gen.hip).
#pragma once
#include "mdf_common.h"
#include "mdf_rys.h"

namespace mdf {

constexpr double TWO_PI_2P5 = 34.986836655249725;   // 2 pi^(5/2)
constexpr double TWO_PI = 6.283185307179586;        // 2 pi
constexpr double PI_1P5 = 5.568327996831708;        // pi^(3/2)
constexpr double PRIM_SCREEN = 1e-20;               // |c_a c_b exp(-ab/p R^2)| cutoff
constexpr int LMAX_AO = 2;
constexpr int LMAX_AUX = 4;

// Device view of one basis (all pointers are device memory).
struct BasisDev {
    const int *nprim, *poff, *aooff;
    const double *xyz, *exps, *coefs;
};

// Spreads the launches of one call, one small kernel per angular class and
// component, over the caller's stream and three of the library's own
// (default priority; a set for each of the streams that called last, so that
// callers on different streams do not wait for each other: two of 4 waters,
// a call each of int3c2e, 0.9 to 1.4 ms, 1.4 to 2.0 with one set for all and 1.5
// on the callers' streams alone; of 24 waters 8.8, 9.4 and 9.4), so one kernel's
// last workgroups run under the next ones: the own streams start after the
// caller's work queued so far and the caller's stream goes on after all of
// them (join, also in the destructor).  A capturing caller's launches stay on
// its stream.
class ForkJoin {
public:
    explicit ForkJoin(hipStream_t st);
    ~ForkJoin() { (void)join(); }
    ForkJoin(const ForkJoin &) = delete;
    ForkJoin &operator=(const ForkJoin &) = delete;
    hipStream_t next();
    int join();

private:
    static constexpr int SIDE = 3;
    hipStream_t st_, side_[SIDE];
    hipEvent_t ev_ = nullptr;
    int n_ = 0, rc_ = MDF_OK, at_ = 0;
    bool used_[SIDE] = {};
};

int launch_int3c(int la, int lb, int lc, const BasisDev &ao, const BasisDev &aux, const int *pairs, int np,
                 const int *kl, int nk, double *out, long ldo, long p0, const int *cmap, hipStream_t st);
int launch_int1e(int la, int lb, const BasisDev &ao, const int *pairs, int np, int natm, const double *charges,
                 const double *atom_xyz, double *S, double *T, double *V, int nao, hipStream_t st);
int launch_int2c(int la, int lc, const BasisDev &aux, const int *pl, int np, const int *ql, int nq,
                 double *out, long ldo, hipStream_t st);
int launch_int3c_ip(int la, int lb, int lc, const BasisDev &ao, const BasisDev &aux, const int *pairs, int np,
                    const int *kl, int nk, const double *W, long ldw, const int *cmap, const int *ao_atom,
                    const int *aux_atom, int natm, double *grad, double *grad_aux, ForkJoin &fj);
int launch_int2c_ip(int la, int lc, const BasisDev &aux, const int *pl, int np, const int *ql, int nq,
                    const double *Z, long ldz, const int *aux_atom, int natm, double *grad, ForkJoin &fj);

}  // namespace mdf
