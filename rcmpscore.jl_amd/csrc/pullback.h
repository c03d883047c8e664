// Node sums of an evaluation's pullback (pullback.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define RC_PULL_ENTRIES 7
#define RC_PULL_TERMS 3
#define RC_LIN_OUTS 6
#define RC_LIN_SRCS 6

// The contribution of one pair of channels to a term's sums over the nodes i < nn:
//   T1 += op(F_i) M_i,  M_i = w_i R^+ op(A_i) + jk j_i D_i;   T2 += w_i op(F_i) op(A_i)
// (op: identity, or the conjugate transpose; F_i = F + i sF complex, A_i, D_i likewise at i sA)
struct RcPullEntry {
    const double *F, *A, *D;   // D null: no second summand
    long long sF, sA;
    double jk;
    int conj, pad;
};
struct RcPullArgs {
    RcPullEntry e[RC_PULL_ENTRIES];
    int first[RC_PULL_TERMS + 1];   // entries of term t: first[t] .. first[t + 1] - 1
    int wg0[RC_PULL_TERMS + 1];     // workgroups of term t
    double c[RC_PULL_TERMS];        // weight of term t in the sums over the terms
    const double *Rh, *wn, *jn;     // R^+, node weights w and j
    int nn, nterms;
    double* partial;                // two Dp x Dp matrices per stream of nodes
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
