// Persistent solve of the pinned Poisson-type equations by restarted GMRES (gmres.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define RC_GMRES_MAX_M 40     // Krylov vectors of one restart cycle
#define RC_GMRES_RING 16      // exchange slots, one matrix each
#define RC_GMRES_REC 64       // complex values of one workgroup's sum record

// One equation  op(x) = b,  op(x) = -L x + i sig x + c2 tr(phi x) psi, solved as op(pre(y)) = b with
// pre(y) = N y - c1 tr(phi N y) Z, N the no-jump inverse in the eigenbasis of Q:
//   N y = A2 (S o (A1 y B1)) B2,  S_ij = -1 / den_ij,  den = lam_i + conj(lam_j) - s (adjoint:
//   conj(lam_i) + lam_j - s), s = s_re + i s_im, zero outside the D x D block;
//   L u = C1 u + u C2 + C4 (u C3);  Z = N psi, c1 = ds / (1 + ds tr(phi Z)).
// b = a - tr(phi a) psi with project_b, else a.  x is projected the same way with project_x.
struct RcGmresProb {
    int D, adjoint, project_b, project_x, pin, m, maxiter, pad;   // pin: the residual includes the pin term; m <= 40
    const double *A1, *B1, *A2, *B2, *lam, *C1, *C2, *C3, *C4, *phi, *psi, *a;   // padded Dp x Dp, row-major
    double* x;               // the solution
    double* exch;            // RC_GMRES_RING Dp^2 complex, then the records: 4 (Dp/16)^2 RC_GMRES_REC complex;
                             // every slot empty at entry (unused for Dp = 16)
    double* out;             // [8]: status, converged, matvecs, GMRES residual, |b|, true residual
    double s_re, s_im, sig, c2, ds;
    double tol;              // the GMRES residual aims at tol max(1, |b|)
};
// an equation's results as the host reads them from out
struct RcGmresResult {
    int status;   // not 0: a wait failed, and the rest means nothing
    bool converged;
    int matvecs;
    double resid, nb, true_res;
};
inline RcGmresResult rc_gmres_result(const double* q) {
    return RcGmresResult{(int)q[0], q[1] != 0, (int)q[2], q[3], q[4], q[5]};
}
// what becomes of the equation, whatever became of the launch's others: 0 when its solution is accepted, its
// status, or `refused` when the residual of the physical equation is above bar max(1, |b|)
inline int rc_gmres_code(const RcGmresResult& r, double bar, int refused) {
    if (r.status != 0) return r.status;
    return r.true_res <= bar * (r.nb > 1.0 ? r.nb : 1.0) ? 0 : refused;
}

// bytes of the exchange area of one equation at Dp = 16 nb
__host__ __device__ inline size_t rc_gmres_exch_bytes(int nb) {
    return nb == 1 ? 16 : (size_t)RC_GMRES_RING * nb * nb * 4096 + (size_t)4 * nb * nb * RC_GMRES_REC * 16;
}

// equations that can be resident at once (0: not launchable); n <= that per launch
hipError_t rc_gmres_capacity(int nb, int* probs);
// n equations: `one` by value when n = 1, else the device array `many`
hipError_t rc_launch_gmres(int nb, int n, const RcGmresProb& one, const RcGmresProb* many, uint32_t* abort_flag,
                           long long wait_ticks, hipStream_t stream);
