// Node sums of an evaluation's pullback (pullback.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define RC_LIN_OUTS 6
#define RC_LIN_SRCS 6

// The contribution of one pair of channels to a term's sums over the nodes i < nn:
//   T1 += op(F_i) M_i,  M_i = w_i B op(A_i) + jk j_i D_i;   T2 += w_i op(F_i) op(A_i)
// (op: identity, or the conjugate transpose; F_i = F + i sF complex, A_i, D_i likewise at i sA)
struct RcPullEntry {
    const double *F, *A, *D;   // D null: no second summand
    long long sF, sA;
    double jk;
    int conj, pad;
};
// one pair of sums: entries first .. last - 1 on workgroups wg0 .. wg0 + nwg - 1, B their constant matrix
struct RcPullTerm {
    const double* B;
    double c;                  // weight of the term where terms are summed
    int first, last, wg0, nwg;
};
struct RcPullArgs {
    const RcPullEntry* e;        // device arrays
    const RcPullTerm* t;
    const double *wn, *jn;       // node weights w and j
    int nn, nterms, nwg, pad;
    double* partial;             // two Dp x Dp matrices per stream of nodes
};
// streams of nodes of one workgroup (each forms whole partial matrices)
__host__ __device__ inline int rc_pull_streams(int nb) { return nb == 1 ? 4 : nb == 2 ? 2 : 1; }

// out = sum over the sources of c sum_i weight_i op(X_i) (kind 0: w, 1: j, 2: the one matrix X)
struct RcLinSource {
    const double* X;
    long long s;
    double c;
    int kind, conj;
};
struct RcLinArgs {
    RcLinSource src[RC_LIN_OUTS][RC_LIN_SRCS];
    int nsrc[RC_LIN_OUTS];
    double* out[RC_LIN_OUTS];
    const double *wn, *jn;
    int nn, nouts;
};

hipError_t rc_launch_lin(int Dp, const RcLinArgs& a, hipStream_t stream);
// the partial sums, then XR = W + sum_t c_t T1_t, XQ = sum_t c_t T2_t
hipError_t rc_launch_pullback(int nb, const RcPullArgs& a, const double* W, double* XR, double* XQ, hipStream_t stream);
// the partial sums, then every term's T1 and T2 by itself: sums + 2 t Dp^2 complex, T2 behind T1
hipError_t rc_launch_pullback_terms(int nb, const RcPullArgs& a, double* sums, hipStream_t stream);
// out_a += g (T1 of terms 2 a and 2 a + 1) - g tr(T2 of term 2 a + 1) wrho_a, a < na (out, wrho at complex stride ts)
hipError_t rc_launch_action_pull(int Dp, int na, const double* sums, double g, const double* wrho, double* out,
                                 long long ts, hipStream_t stream);
