// Persistent Arnoldi steps of the kinetic resolvents (arnoldi.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define RC_ARN_VALUES 256   // complex values of one workgroup's sum record; bounds the steps' basis sizes
#define RC_ARN_MAX_K (RC_ARN_VALUES - 2)

// Steps k0 .. k1 - 1 of one basis of M (classical Gram-Schmidt twice), on vectors of one block (Dp^2
// complex) or two:
//   forward  M x = L x;   M(x0, x1) = (L x0,  Qs x1 + x1 Q^+ + R x1 R^+ + v x0 + w x0 R^+)
//   adjoint  M x = L* x;  M(a1, a0) = (L* a1, Qs a0 + a0 Q  + R^+ a0 R + a1 v + R^+ a1 w)
struct RcArnProb {
    const double *Q, *Qh, *R, *Rh;   // Dp x Dp, row-major complex
    const double *Qs, *v, *w;        // two blocks only
    double* V;               // vectors at stride n = blocks Dp^2 complex; 0 .. k0 in, k0 + 1 .. k1 out
    double *h1, *h2, *hw, *hn;   // projections of the two passes, |M v|^2 and the new vector's |w|^2 before
                             // its normalisation; step j at + (j - k0) hstride doubles
    long long hstride;
    double* exch;            // rc_arn_exch_bytes, every slot empty at entry
    int adj, k0, k1, pad;    // k1 <= RC_ARN_MAX_K
};

// bytes of one basis's exchange area at Dp = 16 nb: two slots of the vector (two orders) and of the
// level-1 tiles, four of the sum records
__host__ __device__ inline size_t rc_arn_exch_bytes(int nb, int blocks) {
    const size_t nt = (size_t)nb * nb;
    return 2 * (2 * blocks + (blocks == 2 ? 3 : 1)) * nt * 4096 + 4 * (nt * blocks) * RC_ARN_VALUES * 16;
}

// bases that can be resident at once (0: not launchable); n <= that per launch
hipError_t rc_arn_capacity(int nb, int blocks, int* bases);
hipError_t rc_launch_arnoldi(int nb, int blocks, int n, const RcArnProb* probs, uint32_t* abort_flag,
                             long long wait_ticks, hipStream_t stream);

#define RC_PROJ_MAX_K 512

// Projected solves (I - z_i H_k) y_i = beta e_1 of one basis: H upper Hessenberg with its row k, column c
// (rows 0 .. c + 1) at complex offset c (c + 3) / 2; y_i at Y + i ldy complex, zero from k on; est[i]
// the Arnoldi residual estimate |z_i h_{k+1,k} y_i[k-1]| / beta, not finite when the solve is singular
struct RcProjProb {
    const double* H;
    double* Y;
    double* est;
    double beta;
    int k, ldy;   // k <= RC_PROJ_MAX_K; 0: zeros
};
// every basis at every node z_i, i < nz; maxk: the largest k among them
hipError_t rc_launch_projected(int n, int maxk, const RcProjProb* probs, int nz, const double* z, hipStream_t stream);
