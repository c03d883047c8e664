// Device kernels of the tangent-space excitation action: the momentum-shifted no-jump
// preconditioner, Gram-Schmidt over sets of Arnoldi bases, the fused right-hand side of the :phi^4:
// action ODEs, DOP853 stage combinations and error norms, and batched trace products.
#include <algorithm>

#include "device_common.h"
#include "exchange.h"
#include "excitation.h"
#include "trajectory.h"

// Z_ij = -Y_ij / den_ij with den = lam_i + conj(lam_j) - (s_re + i s_im) (forward) or
// conj(lam_i) + lam_j - (s_re + i s_im) (adjoint)
__global__ void rc_sylvester_diag_c(int Dp, int D, int adjoint, double s_re, double s_im, const double* lam,
                                    const double* Y, double* Z) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= Dp * Dp) return;
    const int r = i / Dp, c = i % Dp;
    cplx* z = reinterpret_cast<cplx*>(Z);
    if (r >= D || c >= D) { z[i] = cmake(0, 0); return; }
    const cplx* l = reinterpret_cast<const cplx*>(lam);
    cplx den = adjoint ? cadd(cconj(l[r]), l[c]) : cadd(l[r], cconj(l[c]));
    den.re -= s_re;
    den.im -= s_im;
    const cplx y = reinterpret_cast<const cplx*>(Y)[i];
    const double m = cabs2(den);
    const cplx q = cmake((y.re * den.re + y.im * den.im) / m, (y.im * den.re - y.re * den.im) / m);
    z[i] = cmake(-q.re, -q.im);
}

// out[b * ldo + k] = <V_{b,k}, W_b> (conjugate-linear in V); grid (nk, nbases)
__global__ void __launch_bounds__(256) rc_mdots(const double* V, long long sb, long long sv, int nk, const double* W,
                                                long long sw, int n, double* out, int ldo) {
    __shared__ double sre[256], sim[256];
    const int k = blockIdx.x, b = blockIdx.y, t = threadIdx.x;
    const cplx* v = reinterpret_cast<const cplx*>(V) + (long long)b * sb + (long long)k * sv;
    const cplx* w = reinterpret_cast<const cplx*>(W) + (long long)b * sw;
    // thread t adds elements t, t + 256, ... in increasing order, eight elements' loads in flight
    double re = 0, im = 0;
    for (int i0 = t; i0 < n; i0 += 8 * 256) {
        cplx a[8], c[8];
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (i0 + 256 * u < n) {
                a[u] = v[i0 + 256 * u];
                c[u] = w[i0 + 256 * u];
            }
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (i0 + 256 * u < n) {
                re += a[u].re * c[u].re + a[u].im * c[u].im;
                im += a[u].re * c[u].im - a[u].im * c[u].re;
            }
    }
    tree_sum_256(re, im, sre, sim, out + 2 * ((long long)b * ldo + k));
}

// W_b -= sum_{k < nk} h[b * ldh + k] V_{b,k}; grid (ceil(n / 256), nbases)
__global__ void rc_msubtract(const double* V, long long sb, long long sv, int nk, const double* h, int ldh, int n,
                             double* W, long long sw) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x, b = blockIdx.y;
    if (i >= n) return;
    const cplx* v = reinterpret_cast<const cplx*>(V) + (long long)b * sb;
    const cplx* hh = reinterpret_cast<const cplx*>(h) + (long long)b * ldh;
    cplx* w = reinterpret_cast<cplx*>(W) + (long long)b * sw;
    cplx s = w[i];
    // eight vectors' loads in flight, subtracted in increasing k
    for (int k0 = 0; k0 < nk; k0 += 8) {
        cplx x[8], c[8];
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (k0 + u < nk) {
                x[u] = v[(long long)(k0 + u) * sv + i];
                c[u] = hh[k0 + u];
            }
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (k0 + u < nk) s = csub(s, cmul(c[u], x[u]));
    }
    w[i] = s;
}

// out_b = W_b / sqrt(Re nrm2[b * ldn]) (a zero norm writes zeros); grid (ceil(n / 256), nbases)
__global__ void rc_mnormalize(int n, const double* W, long long sw, const double* nrm2, int ldn, double* out,
                              long long so) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x, b = blockIdx.y;
    if (i >= n) return;
    const double q = nrm2[2 * (long long)b * ldn];
    const double s = q > 0.0 ? 1.0 / sqrt(q) : 0.0;
    reinterpret_cast<cplx*>(out)[(long long)b * so + i] =
        cscale(s, reinterpret_cast<const cplx*>(W)[(long long)b * sw + i]);
}

// ---------------------------------------------------------------------------------------------
// The action ODE's step controller on the device (the host loop it replaces: SciPy's DOP853
// controller as the reference's action integration uses it, src/excitation_action.jl:56-123).
// ---------------------------------------------------------------------------------------------
// rc_ode_step, one workgroup of 256.  finish = 1: judge the attempt that just ran (when active): per
// tracked trajectory its tiles' E5 and E3 sums (slot ranges ranges[tr][r] = (first, count), one wave
// per trajectory, lane-strided with a fixed shuffle tree), |h| e5 / sqrt((e5 + e3 / 100) cnt), the
// worst over trajectories; accept or reject and the next step size.  Then, unless done, set up the
// next attempt: the step clipped at the next stop (a quadrature node, 0 or the window's end) and the
// source coefficients [2|t_s|, s(t_s)] of stages 1..12 (one thread each) with the step at cf[26].
// The controller step shared by rc_ode_step and the persistent launch (C: c and every operand in LDS,
// barriers that order LDS only; stops[0], stops[1] and stop_node[0] are the stop c->si, the one after
// it and its node).  No barrier after the cf writes.
template <bool C>
__device__ __forceinline__ void ode_step_body(RcOdeCtl* c, int finish, const double* partial, const int* ranges,
                                              int nranges, int ntrack, double cnt, const double* stops,
                                              const int* stop_node, const double* cheb, double* cf) {
    __shared__ double smax[4];
    __shared__ int sbad[4];
    __shared__ double s_t, s_he, s_tn;
    __shared__ int s_go;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const bool judge = finish && c->active;   // uniform
    if (judge) {
        const double he = c->he;
        double worst = 0.0;
        int bad = 0;
        for (int tr = wave; tr < ntrack; tr += 4) {
            double e5 = 0.0, e3 = 0.0;
            for (int r = 0; r < nranges; ++r) {
                const int first = ranges[2 * (tr * nranges + r)], count = ranges[2 * (tr * nranges + r) + 1];
                for (int q = lane; q < count; q += 64) {
                    e5 += partial[2 * (first + q)];
                    e3 += partial[2 * (first + q) + 1];
                }
            }
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) {
                e5 += __shfl_xor(e5, off);
                e3 += __shfl_xor(e3, off);
            }
            double et = 0.0;
            if (e5 > 0 || e3 > 0) et = fabs(he) * e5 / sqrt((e5 + 0.01 * e3) * cnt);
            if (!isfinite(et)) bad = 1;
            else worst = fmax(worst, et);
        }
        if (lane == 0) {
            smax[wave] = worst;
            sbad[wave] = bad;
        }
    }
    if constexpr (C) lds_barrier();
    else __syncthreads();
    if (tid == 0) {
        s_go = 0;
        int moved = 0;   // the step reached its stop
        if (judge) {
            const double err = fmax(fmax(smax[0], smax[1]), fmax(smax[2], smax[3]));
            const int bad = sbad[0] | sbad[1] | sbad[2] | sbad[3];
            const double he = c->he;
            c->commit = 0;
            c->sample = -1;
            if (bad) {
                c->status = RC_ST_NONFINITE;
                c->done = 1;
            } else if (err <= 1.0) {
                c->accepted += 1;
                c->commit = 1;
                c->t = c->tn;
                if (c->t == stops[C ? 0 : c->si]) {
                    const int nd = stop_node[C ? 0 : c->si];
                    if (nd >= 0) {
                        c->sample = nd;
                        c->node = nd + 1;
                    }
                    c->si += 1;
                    moved = 1;
                }
                double factor = err == 0 ? 10.0 : fmin(10.0, 0.9 / sqrt(sqrt(sqrt(err))));   // 0.9 err^(-1/8)
                if (c->last_rejected) factor = fmin(1.0, factor);
                const double hn = he * factor;
                c->h = c->clipped ? fmax(hn, c->h) : hn;
                c->last_rejected = 0;
                if (c->si >= c->nstops) {
                    c->done = 1;
                    if (c->node != c->npts) c->status = RC_ST_MISSING_SAMPLES;
                }
            } else {
                c->rejected += 1;
                c->h = he * fmax(0.2, 0.9 / sqrt(sqrt(sqrt(err))));
                c->last_rejected = 1;
            }
        }
        c->active = 0;
        if (!c->done) {
            const double t = c->t, h = c->h, stop = stops[C ? moved : c->si];
            double he = fmin(h, stop - t);
            const int clipped = he < h;
            if (stop - t - he <= 1e-14 * fmax(1.0, fabs(stop))) he = stop - t;
            if (!(he > 10 * 2.220446049250313e-16 * fmax(1.0, fabs(t)))) {
                c->status = RC_ST_STEP_UNDERFLOW;
                c->done = 1;
            } else if (++c->attempts > c->maxiters) {
                c->status = RC_ST_MAX_STEPS;
                c->done = 1;
            } else {
                const double tn = (he == stop - t) ? stop : t + he;
                c->he = he;
                c->tn = tn;
                c->clipped = clipped;
                c->active = 1;
                s_t = t;
                s_he = he;
                s_tn = tn;
                s_go = 1;
            }
        }
    }
    if constexpr (C) lds_barrier();
    else __syncthreads();
    if (s_go && tid >= 1 && tid < 13) {
        const double ts = tid < 12 ? s_t + RC_C[tid] * s_he : s_tn;
        cf[2 * tid] = 2 * fabs(ts);
        cf[2 * tid + 1] = rc_source(ts, cheb);
    }
    if (s_go && tid == 0) cf[26] = s_he;
}

__global__ void __launch_bounds__(256) rc_ode_step(RcOdeCtl* c, int finish, const double* partial,
                                                   const int* ranges, int nranges, int ntrack, double cnt,
                                                   const double* stops, const int* stop_node, const double* cheb,
                                                   double* cf) {
    ode_step_body<false>(c, finish, partial, ranges, nranges, ntrack, cnt, stops, stop_node, cheb, cf);
}

// First stage input of the attempt, U1 = y + h a10 K_0, preceded by the commit of the previous
// attempt when it was accepted (y <- y_new, K_0 <- K_12, and at a quadrature node the forward half
// of y_new as sample `sample`, the adjoint half as sample npts - 1 - sample).
__global__ void rc_ode_stage(const RcOdeCtl* c, long long N, long long half, double a10, const double* hp,
                             const double* ynew, double* y, const double* K12, double* K0, double* Sf, double* Sa,
                             double* U1) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    const int commit = c->commit, active = c->active;
    cplx yi, ki;
    if (commit) {
        yi = reinterpret_cast<const cplx*>(ynew)[i];
        ki = reinterpret_cast<const cplx*>(K12)[i];
        reinterpret_cast<cplx*>(y)[i] = yi;
        reinterpret_cast<cplx*>(K0)[i] = ki;
        const int smp = c->sample;
        if (smp >= 0) {
            if (i < half) reinterpret_cast<cplx*>(Sf)[(long long)smp * half + i] = yi;
            else reinterpret_cast<cplx*>(Sa)[(long long)(c->npts - 1 - smp) * half + (i - half)] = yi;
        }
    } else {
        if (!active) return;
        yi = reinterpret_cast<const cplx*>(y)[i];
        ki = reinterpret_cast<const cplx*>(K0)[i];
    }
    if (active) reinterpret_cast<cplx*>(U1)[i] = cfma(hp[0], cscale(a10, ki), yi);
}

// Resolvent step in the transfer's eigenbasis: out[v][k] = Y[src(v)][k] / (1 - z_i (mu_k + i s_b)) for
// vector v = b nz + i (src(v) = b when per_basis, else v), mu conjugated for the adjoint; N entries
// per vector; s null: no shift.  grid (nb nz, ceil(N / 256)).
__global__ void rc_res_scale(long long N, int nz, int per_basis, int adjoint, const double* Y, const double* mu,
                             const double* z, const double* s, double* out) {
    const long long k = (long long)blockIdx.y * blockDim.x + threadIdx.x;
    if (k >= N) return;
    const int v = blockIdx.x, b = v / nz, i = v % nz;
    const cplx y = reinterpret_cast<const cplx*>(Y)[(long long)(per_basis ? b : v) * N + k];
    cplx l = reinterpret_cast<const cplx*>(mu)[k];
    if (adjoint) l = cconj(l);
    const double zi = z[i], sb = s ? s[b] : 0.0;
    const cplx den = cmake(1.0 - zi * l.re, -zi * (l.im + sb));
    const double m = cabs2(den);
    reinterpret_cast<cplx*>(out)[(long long)v * N + k] =
        cmake((y.re * den.re + y.im * den.im) / m, (y.im * den.re - y.re * den.im) / m);
}

// The pinned Poisson operator in the transfer's eigenbasis: out_k = Y_k / (-l_k + i s + [k == k0]),
// l = mu (adjoint: conj mu), k0 the zero mode; zero on the padding of the Dp^2 space (where the
// eigenvalue is a placeholder 0).  N = Dp^2, grid ceil(N / 256).
__global__ void rc_poisson_scale(long long N, int Dp, int D, int adjoint, double s, int k0, const double* mu,
                                 const double* Y, double* out) {
    const long long k = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= N) return;
    if (k / Dp >= D || k % Dp >= D) {
        reinterpret_cast<cplx*>(out)[k] = cmake(0, 0);
        return;
    }
    cplx l = reinterpret_cast<const cplx*>(mu)[k];
    if (adjoint) l = cconj(l);
    const cplx den = cmake(-l.re + (k == k0 ? 1.0 : 0.0), -l.im + s);
    const cplx y = reinterpret_cast<const cplx*>(Y)[k];
    const double m = cabs2(den);
    reinterpret_cast<cplx*>(out)[k] = cmake((y.re * den.re + y.im * den.im) / m, (y.im * den.re - y.re * den.im) / m);
}

// ---- the pinned Poisson solves and tangent algebra of many tangents at once (blockIdx.y = tangent
// v, strides in complex elements); each kernel repeats its single-matrix counterpart's arithmetic.
// X_v -= t_v Z with t_v the device complex at t + 2 v (rc_sub_scaled with den = 1)
__global__ void rc_sub_scaled_n(int n, const double* t, const double* Z, double* X, long long sx) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x, v = blockIdx.y;
    if (i >= n) return;
    const cplx tt = cmake(t[2 * v], t[2 * v + 1]);
    const double dre = 1.0, dim = 0.0, m = dre * dre + dim * dim;
    const cplx f = cmake((tt.re * dre + tt.im * dim) / m, (tt.im * dre - tt.re * dim) / m);
    cplx* x = reinterpret_cast<cplx*>(X) + v * sx;
    x[i] = csub(x[i], cmul(f, reinterpret_cast<const cplx*>(Z)[i]));
}

// X_v += scale t_v I on the D x D block (rc_add_identity)
__global__ void rc_add_identity_n(int Dp, int D, const double* t, double scale, double* X, long long sx) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x, v = blockIdx.y;
    if (i >= D) return;
    cplx* x = reinterpret_cast<cplx*>(X) + v * sx;
    x[i * Dp + i].re += scale * t[2 * v];
    x[i * Dp + i].im += scale * t[2 * v + 1];
}

// out + so v = <X_v, X_v>, one workgroup per tangent (Xl = X: the left operand passed apart, so the
// products compile as rc_dots's do)
__global__ void __launch_bounds__(256) rc_norms_n(int n, const double* Xl, const double* X, long long sx, double* out,
                                                  long long so) {
    __shared__ double sre[256], sim[256];
    const int v = blockIdx.x;
    dot_block(reinterpret_cast<const cplx*>(Xl) + v * sx, reinterpret_cast<const cplx*>(X) + v * sx, n, sre, sim,
              out + so * v);
}

// rc_poisson_scale with the shift s_v of tangent v
__global__ void rc_poisson_scale_n(long long N, int Dp, int D, int adjoint, const double* s, int k0, const double* mu,
                                   const double* Y, long long sy, double* out, long long so) {
    const long long k = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const int v = blockIdx.y;
    if (k >= N) return;
    cplx* o = reinterpret_cast<cplx*>(out) + v * so;
    if (k / Dp >= D || k % Dp >= D) {
        o[k] = cmake(0, 0);
        return;
    }
    cplx l = reinterpret_cast<const cplx*>(mu)[k];
    if (adjoint) l = cconj(l);
    const cplx den = cmake(-l.re + (k == k0 ? 1.0 : 0.0), -l.im + s[v]);
    const cplx y = (reinterpret_cast<const cplx*>(Y) + v * sy)[k];
    const double m = cabs2(den);
    o[k] = cmake((y.re * den.re + y.im * den.im) / m, (y.im * den.re - y.re * den.im) / m);
}

// out_v = a X_v + b_v Y_v with b_v the device complex at b + 2 v (rc_axpby)
__global__ void rc_axpby_n(int n, double ar, double ai, const double* X, long long sx, const double* b, const double* Y,
                           long long sy, double* out, long long so) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x, v = blockIdx.y;
    if (i >= n) return;
    const cplx* x = reinterpret_cast<const cplx*>(X) + v * sx;
    const cplx* y = reinterpret_cast<const cplx*>(Y) + v * sy;
    cplx r = cmul(cmake(ar, ai), x[i]);
    r = cadd(r, cmul(cmake(b[2 * v], b[2 * v + 1]), y[i]));
    (reinterpret_cast<cplx*>(out) + v * so)[i] = r;
}

// X_v += c_v Z_v with c_v the device complex at c + 2 v (rc_axpy_c)
__global__ void rc_axpy_c_n(int n, const double* c, const double* Z, long long sz, double* X, long long sx) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x, v = blockIdx.y;
    if (i >= n) return;
    cplx* x = reinterpret_cast<cplx*>(X) + v * sx;
    x[i] = cadd(x[i], cmul(cmake(c[2 * v], c[2 * v + 1]), (reinterpret_cast<const cplx*>(Z) + v * sz)[i]));
}

// out[v] = src[v / nz] (N complex each): block 1 of basis b's right-hand side for each node.
// grid (nb nz, ceil(N / 256)).
__global__ void rc_bcast_rhs(long long N, int nz, const double* src, long long ss, double* out) {
    const long long k = (long long)blockIdx.y * blockDim.x + threadIdx.x;
    if (k >= N) return;
    const int v = blockIdx.x;
    reinterpret_cast<cplx*>(out)[(long long)v * N + k] = reinterpret_cast<const cplx*>(src)[(long long)(v / nz) * ss + k];
}

// out[b] = tr(A_b B_b) for Dp x Dp matrices; grid (nb)
__global__ void __launch_bounds__(256) rc_trace_prod_batched(int Dp, const double* A, long long sa, const double* B,
                                                             long long sb, double* out) {
    __shared__ double sre[256], sim[256];
    const int b = blockIdx.x, t = threadIdx.x;
    const cplx* a = reinterpret_cast<const cplx*>(A) + (long long)b * sa;
    const cplx* c = reinterpret_cast<const cplx*>(B) + (long long)b * sb;
    double re = 0, im = 0;
    for (int idx = t; idx < Dp * Dp; idx += 256) {
        const int i = idx / Dp, k = idx % Dp;
        const cplx p = cmul(a[i * Dp + k], c[k * Dp + i]);
        re += p.re;
        im += p.im;
    }
    sre[t] = re;
    sim[t] = im;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (t < s) { sre[t] += sre[t + s]; sim[t] += sim[t + s]; }
        __syncthreads();
    }
    if (t == 0) { out[2 * b] = sre[0]; out[2 * b + 1] = sim[0]; }
}

// X += (c_re + i c_im) Z elementwise over n complex (c by value)
__global__ void rc_axpy_c(int n, double c_re, double c_im, const double* Z, double* X) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    cplx* x = reinterpret_cast<cplx*>(X);
    x[i] = cadd(x[i], cmul(cmake(c_re, c_im), reinterpret_cast<const cplx*>(Z)[i]));
}

// X += c Z with c = -scale sum_j sum_k wz[k] tr[j nodes + k] over nj sets of `nodes` complex traces: the
// sums in increasing j, then k, with each product and sum rounded on its own (the host loop's
// arithmetic), made by every thread alike
__device__ __forceinline__ void trace_axpy_elem(int nj, int nodes, const double* tr, const double* wz, double scale,
                                                const double* Z, double* X, int i) {
    double sr = 0.0, si = 0.0;
    for (int j = 0; j < nj; ++j)
        for (int k = 0; k < nodes; ++k) {
            const double w = wz[k];
            const double* t = tr + 2 * ((long long)j * nodes + k);
            sr = __dadd_rn(sr, __dmul_rn(w, t[0]));
            si = __dadd_rn(si, __dmul_rn(w, t[1]));
        }
    sr = __dmul_rn(sr, scale);
    si = __dmul_rn(si, scale);
    cplx* x = reinterpret_cast<cplx*>(X);
    x[i] = cadd(x[i], cmul(cmake(-sr, -si), reinterpret_cast<const cplx*>(Z)[i]));
}

__global__ void rc_trace_axpy(int n, int nj, int nodes, const double* tr, const double* wz, double scale,
                              const double* Z, double* X) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    trace_axpy_elem(nj, nodes, tr, wz, scale, Z, X, i);
}

// rc_trace_axpy for several tangents (blockIdx.y = v): traces tr + 2 v nj nodes, Z + v sz, X + v sx
__global__ void rc_trace_axpy_n(int n, int nj, int nodes, const double* tr, const double* wz, double scale,
                                const double* Z, long long sz, double* X, long long sx) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const long long v = blockIdx.y;
    trace_axpy_elem(nj, nodes, tr + 2 * v * nj * nodes, wz, scale, Z + 2 * v * sz, X + 2 * v * sx, i);
}

// ---------------------------------------------------------------------------------------------
// One right-hand side of the :phi^4: action ODEs (forward and adjoint, every tangent and channel) in
// two launches, the graph route's (rc_quartic_ode has both levels in one persistent launch).
// Workgroup = one 16 x 16 tile of one matrix; the products of a tile accumulate in one MFMA accumulator
// (k split across the 4 waves).  rc_quartic_p forms P, the inner factor of the two-sided products and
// the neighbour channel's one-sided insertion; rc_quartic_rhs the rest.
//   forward  dx_k = jac (Q x + x Q^+ + R x R^+) + k jt (R x_{k-1} + x_{k-1} R^+)
//            dy_k = jac (Qs y + y Q^+ + R y R^+ + v x + w x R^+) + k jt (R y_{k-1} + y_{k-1} R^+ + w x_{k-1})
//   adjoint  da0_k = jac (Qhs a0 + a0 Q + R^+ (a0 R + a1 w) + a1 v) + (k+1) jt (a0 R + a1 w + R^+ a0)_{k+1}
//            da1_k = jac (Q^+ a1 + a1 Q + R^+ a1 R) + (k+1) jt (a1 R + R^+ a1)_{k+1}
// with Qs = Q - ip, Qhs = Q^+ + ip of each tangent's momentum.  grid ((Dp/16)^2, 4 * 5 na).
// ---------------------------------------------------------------------------------------------
namespace {

// Every fragment of this wave's k-steps (Dp / 16 of them, at most 4) is loaded before the first MFMA,
// so a product pays one load round trip instead of one per k-step; the MFMAs run in the same k order.
// Wave w runs k-step w + 4 i of k-tile i.  kmask (uniform) selects the k-tiles: bit i for k-tile i.
__device__ __forceinline__ void qprod(cacc& acc, const cplx* A, const cplx* B, int Dp, int bi, int bj, int wave,
                                      int lane, double scale, int kmask = 15) {
    const int nk = Dp / 16;
    cplx a[4], b[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (i < nk && ((kmask >> i) & 1)) {
            const int kk = 4 * (wave + 4 * i) + (lane >> 4);
            a[i] = A[(16 * bi + (lane & 15)) * Dp + kk];
            b[i] = B[kk * Dp + 16 * bj + (lane & 15)];
        }
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (i < nk && ((kmask >> i) & 1)) cmfma(acc, cscale(scale, a[i]), b[i]);
}

// The same beyond Dp = 64, over k-tiles first .. first + count - 1, four at a time in the k order.  (One
// function for both, with the loop, costs a right-hand side at D = 16 to 64 1 to 3%.)
struct KTiles {
    int first, count;
};
__device__ __forceinline__ void qprod_wide(cacc& acc, const cplx* A, const cplx* B, int Dp, int bi, int bj, int wave,
                                           int lane, double scale, KTiles kt) {
    for (int g = 0; g < kt.count; g += 4) {
        cplx a[4], b[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (g + i < kt.count) {
                const int kk = 16 * (kt.first + g + i) + 4 * wave + (lane >> 4);
                a[i] = A[(16 * bi + (lane & 15)) * Dp + kk];
                b[i] = B[kk * Dp + 16 * bj + (lane & 15)];
            }
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (g + i < kt.count) cmfma(acc, cscale(scale, a[i]), b[i]);
    }
}

// A[tile rows, :] T with T a Dp x 16 block in LDS
__device__ __forceinline__ void qprod_t(cacc& acc, const cplx* A, const cplx* T, int Dp, int bi, int wave, int lane,
                                        double scale) {
    const int nk = Dp / 16;
    cplx a[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (i < nk) a[i] = A[(16 * bi + (lane & 15)) * Dp + 4 * (wave + 4 * i) + (lane >> 4)];
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (i < nk) {
            const int kk = 4 * (wave + 4 * i) + (lane >> 4);
            cmfma(acc, cscale(scale, a[i]), T[kk * 16 + (lane & 15)]);
        }
}

// the same beyond Dp = 64
__device__ __forceinline__ void qprod_t_wide(cacc& acc, const cplx* A, const cplx* T, int Dp, int bi, int wave,
                                             int lane, double scale) {
    const int nk = Dp / 16;
    for (int g = 0; g < nk; g += 4) {
        cplx a[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (g + i < nk) a[i] = A[(16 * bi + (lane & 15)) * Dp + 16 * (g + i) + 4 * wave + (lane >> 4)];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (g + i < nk)
                cmfma(acc, cscale(scale, a[i]), T[(16 * (g + i) + 4 * wave + (lane >> 4)) * 16 + (lane & 15)]);
    }
}

// k-tiles of A(b, :) B(:, c) for operands of parities pa, pb under parity blocks of zt tiles (zt = 0:
// every k-tile): none unless the output tile's blocks have parity pa ^ pb, then the k-tiles of block
// blk(b) ^ pa.  The skipped k-steps multiply exact zeros, so the sums keep their bits.
__device__ __forceinline__ KTiles zrange(int zt, int nk, int b, int c, int pa, int pb) {
    if (zt == 0) return KTiles{0, nk};
    const int bb = b / zt, bc = c / zt;
    if ((bb ^ bc) != (pa ^ pb)) return KTiles{0, 0};
    return KTiles{(bb ^ pa) * zt, zt};
}
// the same as a mask, up to four k-tiles
__device__ __forceinline__ int zmask(int zt, int nk, int b, int c, int pa, int pb) {
    if (zt == 0) return 15;
    const int bb = b / zt, bc = c / zt;
    if ((bb ^ bc) != (pa ^ pb)) return 0;
    int m = 0;
    for (int t = 0; t < nk; ++t)
        if (t / zt == (bb ^ pa)) m |= 1 << t;
    return m;
}

__device__ __forceinline__ cplx qreduce(const cacc& acc, cplx* red, int wave, int lane) {
#pragma unroll
    for (int q = 0; q < 4; ++q) red[wave * 256 + (4 * q + (lane >> 4)) * 16 + (lane & 15)] = cacc_get(acc, q);
    __syncthreads();
    const int t = threadIdx.x;
    const cplx s = cadd(cadd(cadd(red[t], red[256 + t]), red[512 + t]), red[768 + t]);
    __syncthreads();
    return s;
}

// One wave's whole product A(bi, :) B(:, bj) over every k-step (no cross-wave reduction), one k-tile of
// fragments loaded ahead of its four MFMAs.
__device__ __forceinline__ void qprod_rows(cacc& acc, const cplx* A, const cplx* B, int Dp, int bi, int bj, int lane) {
    const int nk = Dp / 16;
    for (int t = 0; t < nk; ++t) {
        cplx a[4], b[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int kk = 16 * t + 4 * s + (lane >> 4);
            a[s] = A[(16 * bi + (lane & 15)) * Dp + kk];
            b[s] = B[kk * Dp + 16 * bj + (lane & 15)];
        }
#pragma unroll
        for (int s = 0; s < 4; ++s) cmfma(acc, a[s], b[s]);
    }
}

// one term X B[:, bj] of an LDS column block (X null: no term)
struct QTerm {
    const cplx* X;
    const cplx* B;
};

// Column blocks (Dp x 16, in LDS) T0 = a0 + a1 and, when T1 is given, T1 = b0 + b1.  The row tiles of
// both blocks are spread over the waves, each wave running every k-step of its row tiles and writing
// them straight to LDS; one barrier at the end.
__device__ __forceinline__ void qcolumns(cplx* T0, QTerm a0, QTerm a1, cplx* T1, QTerm b0, QTerm b1, int Dp, int bj,
                                         int wave, int lane) {
    const int nbt = Dp / 16, ntask = (T1 ? 2 : 1) * nbt;
    for (int i = wave; i < ntask; i += 4) {
        const int col = i / nbt, rt = i % nbt;
        const QTerm p = col ? b0 : a0, q = col ? b1 : a1;
        cplx* T = col ? T1 : T0;
        cacc acc;
        cacc_zero(acc);
        qprod_rows(acc, p.X, p.B, Dp, rt, bj, lane);
        if (q.X) qprod_rows(acc, q.X, q.B, Dp, rt, bj, lane);
#pragma unroll
        for (int e = 0; e < 4; ++e) T[(16 * rt + 4 * e + (lane >> 4)) * 16 + (lane & 15)] = cacc_get(acc, e);
    }
    __syncthreads();
}

}  // namespace

// block, tangent and channel of matrix mi (rc_qmat's inverse; the shared blocks 0 and 3 take a = 0)
__device__ __forceinline__ void qmat_of(int mi, int nb, int& blk, int& a, int& k) {
    if (mi < RC_QCH) { blk = 0; a = 0; k = mi; }
    else if (mi < RC_QCH + nb) { blk = 1; a = (mi - RC_QCH) / RC_QCH; k = (mi - RC_QCH) % RC_QCH; }
    else if (mi < RC_QCH + 2 * nb) { blk = 2; a = (mi - RC_QCH - nb) / RC_QCH; k = (mi - RC_QCH - nb) % RC_QCH; }
    else { blk = 3; a = 0; k = mi - RC_QCH - 2 * nb; }
}

// Operands of tile (bi, bj) of matrix mi: the constant matrices, the tangent's, the stage input's and the
// level-1 matrices' of this channel and of its neighbour, whose insertion it takes; Z2 parities and
// their k-tiles (see RcQuarticArgs).  Parities for g.zt > 0: Q, Q^+ and the shifted ones even, R, R^+
// odd, w = W of parity pw, v = -R^+ W of parity pw ^ 1; channels x_k and a1_k of parity k & 1 (x_0 =
// rho, a1 of the last channel = I), y_k and a0_k of parity (k + 1 + pw) & 1 (y_0 = R W, a0 driven by
// a1 w and a1 v).
template <bool WIDE>
struct QTile {
    int Dp, bi, bj, blk, a, k, nb, zt, nk, pw, px, py, lane, wave;
    long long m;
    const cplx *Q, *Qh, *Qs, *Qhs, *R, *Rh, *v, *w;
    __device__ __forceinline__ QTile(const RcQuarticArgs& g) {
        lane = threadIdx.x & 63;
        wave = threadIdx.x >> 6;
        Dp = g.Dp;
        nk = Dp / 16;
        bi = blockIdx.x / nk;
        bj = blockIdx.x % nk;
        nb = g.na * RC_QCH;
        qmat_of(blockIdx.y, nb, blk, a, k);
        m = (long long)Dp * Dp;
        Q = reinterpret_cast<const cplx*>(g.Q);
        Qh = reinterpret_cast<const cplx*>(g.Qh);
        Qs = reinterpret_cast<const cplx*>(g.Qs) + (long long)a * g.qstride;
        Qhs = reinterpret_cast<const cplx*>(g.Qhs) + (long long)a * g.qstride;
        R = reinterpret_cast<const cplx*>(g.R);
        Rh = reinterpret_cast<const cplx*>(g.Rh);
        v = reinterpret_cast<const cplx*>(g.Vrep) + (long long)a * 5 * m;
        w = reinterpret_cast<const cplx*>(g.Wrep) + (long long)a * 5 * m;
        zt = g.zt;
        pw = g.wpar;
        px = k & 1;
        py = (k + 1 + pw) & 1;
    }
    __device__ __forceinline__ const cplx* mat(const cplx* U, int b, int ch) const {
        return U + (long long)rc_qmat(b, a, ch, nb) * m;
    }
    // acc += scale A(bi, :) B(:, bj), operands of parities pa, pb
    __device__ __forceinline__ void add(cacc& acc, double scale, const cplx* A, int pa, const cplx* B, int pb) const {
        if constexpr (WIDE) qprod_wide(acc, A, B, Dp, bi, bj, wave, lane, scale, zrange(zt, nk, bi, bj, pa, pb));
        else qprod(acc, A, B, Dp, bi, bj, wave, lane, scale, zmask(zt, nk, bi, bj, pa, pb));
    }
    __device__ __forceinline__ long long element() const {
        return (long long)blockIdx.y * m + (16 * bi + (threadIdx.x >> 4)) * Dp + 16 * bj + (threadIdx.x & 15);
    }
};

// Level 1 of a right-hand side: the tiles of P (x R^+, y R^+, a0 R + a1 w, a1 R).
template <bool WIDE>
__global__ void __launch_bounds__(256) rc_quartic_p(RcQuarticArgs g) {
    __shared__ cplx red[1024];
    if (g.active && !*g.active) return;
    const QTile<WIDE> q(g);
    const cplx* U = reinterpret_cast<const cplx*>(g.U);
    cacc acc;
    cacc_zero(acc);
    if (q.blk == 0) q.add(acc, 1.0, q.mat(U, 0, q.k), q.px, q.Rh, 1);
    else if (q.blk == 1) q.add(acc, 1.0, q.mat(U, 1, q.k), q.py, q.Rh, 1);
    else if (q.blk == 2) {
        q.add(acc, 1.0, q.mat(U, 2, q.k), q.py, q.R, 1);
        q.add(acc, 1.0, q.mat(U, 3, q.k), q.px, q.w, q.pw);
    } else q.add(acc, 1.0, q.mat(U, 3, q.k), q.px, q.R, 1);
    reinterpret_cast<cplx*>(g.P)[q.element()] = qreduce(acc, red, q.wave, q.lane);
}

// Level 2: the one-sided products, then R P (and w P^x), then the insertion's P tile; thread t receives
// element (t/16, t%16).  The order of the sums is rc_quartic_ode's.
template <bool WIDE>
__device__ __forceinline__ cplx quartic_tile(const RcQuarticArgs& g, const QTile<WIDE>& q, double jac, double jt, cplx* red) {
    const cplx* U = reinterpret_cast<const cplx*>(g.U);
    const cplx* P = reinterpret_cast<const cplx*>(g.P);
    const int blk = q.blk, k = q.k, px = q.px, py = q.py, pw = q.pw;
    const double c = (blk < 2 ? k : k + 1) * jt;
    const bool nbr = blk < 2 ? k >= 1 : k <= 3;   // the channel has an insertion
    const int kn = blk < 2 ? k - 1 : k + 1;
    cacc acc;
    cacc_zero(acc);
    if (blk == 0) {
        const cplx* x = q.mat(U, 0, k);
        q.add(acc, jac, q.Q, 0, x, px);
        q.add(acc, jac, x, px, q.Qh, 0);
        if (nbr) q.add(acc, c, q.R, 1, q.mat(U, 0, kn), px ^ 1);
        q.add(acc, jac, q.R, 1, q.mat(P, 0, k), px ^ 1);
    } else if (blk == 1) {
        const cplx* y = q.mat(U, 1, k);
        q.add(acc, jac, q.Qs, 0, y, py);
        q.add(acc, jac, y, py, q.Qh, 0);
        q.add(acc, jac, q.v, pw ^ 1, q.mat(U, 0, k), px);
        if (nbr) {
            q.add(acc, c, q.R, 1, q.mat(U, 1, kn), py ^ 1);
            q.add(acc, c, q.w, pw, q.mat(U, 0, kn), px ^ 1);
        }
        q.add(acc, jac, q.R, 1, q.mat(P, 1, k), py ^ 1);
        q.add(acc, jac, q.w, pw, q.mat(P, 0, k), px ^ 1);
    } else if (blk == 2) {
        const cplx* a0 = q.mat(U, 2, k);
        q.add(acc, jac, q.Qhs, 0, a0, py);
        q.add(acc, jac, a0, py, q.Q, 0);
        q.add(acc, jac, q.mat(U, 3, k), px, q.v, pw ^ 1);
        if (nbr) q.add(acc, c, q.Rh, 1, q.mat(U, 2, kn), py ^ 1);
        q.add(acc, jac, q.Rh, 1, q.mat(P, 2, k), py ^ 1);
    } else {
        const cplx* a1 = q.mat(U, 3, k);
        q.add(acc, jac, q.Qh, 0, a1, px);
        q.add(acc, jac, a1, px, q.Q, 0);
        if (nbr) q.add(acc, c, q.Rh, 1, q.mat(U, 3, kn), px ^ 1);
        q.add(acc, jac, q.Rh, 1, q.mat(P, 3, k), px ^ 1);
    }
    cplx ins = cmake(0, 0);
    if (nbr) ins = q.mat(P, blk, kn)[q.element() - (long long)blockIdx.y * q.m];
    const cplx val = qreduce(acc, red, q.wave, q.lane);
    return nbr ? cfma(c, ins, val) : val;
}

// This tile's part of the error sums, |r|^2 / sc^2 of the thread's element summed over the workgroup:
// the waves' sums in order (thread 0 holds them); s: 8 doubles of LDS, `sync` a workgroup barrier
__device__ __forceinline__ void tile_error_put(cplx r5, cplx r3, double sc, double* s, int wave, int lane) {
    const double e5 = wave_sum(fma(r5.re, r5.re, r5.im * r5.im) / (sc * sc));
    const double e3 = wave_sum(fma(r3.re, r3.re, r3.im * r3.im) / (sc * sc));
    if (lane == 0) {
        s[wave] = e5;
        s[4 + wave] = e3;
    }
}
__device__ __forceinline__ cplx tile_error_sum(const double* s) {
    return cmake(((s[0] + s[1]) + s[2]) + s[3], ((s[4] + s[5]) + s[6]) + s[7]);
}

template <bool WIDE>
__global__ void __launch_bounds__(256) rc_quartic_rhs(RcQuarticArgs g) {
    __shared__ cplx red[1024];
    if (g.active && !*g.active) return;
    const int tid = threadIdx.x;
    const QTile<WIDE> q(g);
    const int nbt = q.nk, mi = blockIdx.y;
    const cplx* U = reinterpret_cast<const cplx*>(g.U);
    const double jac = g.coef ? g.coef[0] : g.jac;
    const double jt = g.coef ? g.coef[1] : g.jt;
    const cplx val = quartic_tile(g, q, jac, jt, red);
    const long long e = q.element();
    reinterpret_cast<cplx*>(g.F)[e] = val;
    if (g.epi == 0) return;
    const cplx* Kc = reinterpret_cast<const cplx*>(g.K);
    const cplx y0 = reinterpret_cast<const cplx*>(g.y)[e];
    if (g.epi == 1) {
        const double h = g.hp ? g.hp[0] : g.h;
        cplx sum = cmake(0, 0);
        for (int j = 0; j < g.stage; ++j)
            if (g.comb.a[j] != 0.0) sum = cfma(g.comb.a[j], Kc[(long long)j * g.sk + e], sum);
        reinterpret_cast<cplx*>(g.Unext)[e] = cfma(h, cfma(g.comb.a[g.stage], val, sum), y0);
        return;
    }
    cplx r5 = cmake(0, 0), r3 = cmake(0, 0);
    for (int j = 0; j < g.stage; ++j) {
        const cplx kj = Kc[(long long)j * g.sk + e];
        if (g.comb.a[j] != 0.0) r5 = cfma(g.comb.a[j], kj, r5);
        if (g.comb3.a[j] != 0.0) r3 = cfma(g.comb3.a[j], kj, r3);
    }
    r5 = cfma(g.comb.a[g.stage], val, r5);
    r3 = cfma(g.comb3.a[g.stage], val, r3);
    double* se = reinterpret_cast<double*>(red);
    tile_error_put(r5, r3, g.atol + g.rtol * fmax(cabsd(y0), cabsd(U[e])), se, tid >> 6, tid & 63);
    __syncthreads();
    if (tid == 0) {
        const long long slot = (long long)mi * nbt * nbt + blockIdx.x;
        const cplx es = tile_error_sum(se);
        g.partial[2 * slot] = es.re;
        g.partial[2 * slot + 1] = es.im;
    }
}
template __global__ void rc_quartic_p<false>(RcQuarticArgs g);
template __global__ void rc_quartic_p<true>(RcQuarticArgs g);
template __global__ void rc_quartic_rhs<false>(RcQuarticArgs g);
template __global__ void rc_quartic_rhs<true>(RcQuarticArgs g);

// ---------------------------------------------------------------------------------------------
// The whole :phi^4: action ODE integration in one persistent launch (cooperative: every workgroup
// resident), tiles exchanged between workgroups as in rc_trajectory (exchange.h): ring slots that are
// empty until the value is stored, polling loads straight into MFMA fragments, constants in
// registers, two barriers of the workgroup per right-hand side.
//
// Workgroup = one 16 x 16 tile of one matrix.  A right-hand side has two levels: level 1 forms the
// tile of P (x R^+, y R^+, a0 R + a1 w, a1 R) and publishes it; the one-sided products of the stage
// input and of the neighbour channel's follow while the P tiles travel; level 2 adds R P (and
// w P^x) and the neighbour's P tile, which is its insertion.  The order of every sum is that of
// rc_quartic_p and rc_quartic_rhs, so the two routes give the same bits.
//
// Z2 states (KT = NB / 2): the tiles that are exactly zero have no workgroup; the workgroup of tile
// (bi, bj) also forms the P tile (bi, bj') of the other parity block, and products run half the
// k-tiles.
//
// Step controller: every workgroup reads all tiles' error sums and runs ode_step_body on them, so
// all take the same decision.  Ring: 12 events between two gathers, so at event e every reader is
// done with event e - 16, which is emptied then and next used at e + 16.  Waits are bounded in wall
// time: a workgroup that outlasts the budget sets the abort word and every workgroup leaves; the host
// then reports RC_ST_WAIT_LIMIT.
//
// Up to 32 workgroups (D <= 16 with one tangent) are laid on one XCD and exchange through its L2.  With
// that and running sums of the combinations instead of a window of derivatives a right-hand side
// takes 3.1 us at D = 16 (3.35 before), 4.7 at D = 64 with parity blocks (4.9), 3.4 at D = 32 (3.4).
//
// What bounds it: the two exchanges (about 1.2 us each) around up to eight products of a tile.
// ---------------------------------------------------------------------------------------------
// What the derivative of stage s adds to the combinations still ahead of it: row s, the coefficients of
// k_s in the inputs of stages s + 2, s + 3, .. (stage 12's is the step end), then in E5 and E3.
#define RC_ODE_AHEAD 11
struct RcOdeRows {
    double c[12][RC_ODE_AHEAD + 3];
};
constexpr RcOdeRows rc_make_ode_rows() {
    RcOdeRows r{};
    for (int s = 0; s < 12; ++s) {
        for (int i = 0; s + 2 + i <= 12; ++i) r.c[s][i] = s + 2 + i == 12 ? RC_B[s] : RC_A[s + 2 + i][s];
        r.c[s][RC_ODE_AHEAD] = RC_E5[s];
        r.c[s][RC_ODE_AHEAD + 1] = RC_E3[s];
    }
    return r;
}
__constant__ const RcOdeRows rc_ode_rows = rc_make_ode_rows();

// Running sums of the combinations ahead, in stage order: each moves up by one as its multiply-add's
// destination, so a[0] is all but the last term of the input after the next stage (the sums of a window
// of derivatives, in the same order: the graph route's bits)
struct RcOdeAhead {
    cplx a[RC_ODE_AHEAD + 1], e5, e3;
    __device__ __forceinline__ void clear() {
        e5 = e3 = cmake(0, 0);
#pragma unroll
        for (int i = 0; i <= RC_ODE_AHEAD; ++i) a[i] = cmake(0, 0);
    }
    __device__ __forceinline__ void add(int s, cplx k) {
        const __attribute__((address_space(4))) double* c =
            (const __attribute__((address_space(4))) double*)&rc_ode_rows.c[s][0];
#pragma unroll
        for (int i = 0; i < RC_ODE_AHEAD; ++i) a[i] = cfma(c[i], k, a[i + 1]);
        e5 = cfma(c[RC_ODE_AHEAD], k, e5);
        e3 = cfma(c[RC_ODE_AHEAD + 1], k, e3);
    }
};

// dynamic LDS: two levels of partial tiles, every tile's error sums, the trajectories' slot ranges (two
// of two ints each)
#define RC_ODE_LDS(nslots, ntrack) (2048 * 16 + (nslots) * 16 + (ntrack) * 16)

#define RC_ODE_LDS_ALONE (84 * 1024)

template <int NB, int KT>
__global__ void __launch_bounds__(256, KT <= 2 ? 2 : 1) rc_quartic_ode(const RcOdeRun* __restrict__ pp) {
    extern __shared__ __align__(16) unsigned char ode_lds[];
    cplx* red1 = reinterpret_cast<cplx*>(ode_lds);
    cplx* red2 = red1 + 1024;
    double* s_slots = reinterpret_cast<double*>(red2 + 1024);
    __shared__ RcOdeCtl sc;
    __shared__ double s_cf[32], s_err[8], s_al[13], s_stops[2];
    __shared__ double s_cheb[RC_SOURCE_SEGMENTS * (RC_SOURCE_DEGREE + 1)];
    __shared__ int s_bad, s_stop, s_node;
    const RcOdeRun& p = *pp;
    // the slot ranges of the tracked trajectories, behind the error sums
    int* s_ranges = reinterpret_cast<int*>(s_slots + 2 * p.nslots);
    const RcQuarticArgs& g = p.g;
    constexpr int Dp = 16 * NB, NT = NB * NB;
    constexpr uint32_t TB = 4096;
    const int tid = threadIdx.x, lane = tid & 63, wave = uni(tid >> 6);
    const int ei = tid >> 4, ej = tid & 15, fi = lane & 15, fk = 4 * wave + (lane >> 4);
    const int nb = g.na * RC_QCH, nmat = rc_qmats(nb);
    // spread: only every eighth workgroup works, so that all share an XCD
    if (p.spread && (blockIdx.x & 7)) return;
    const int wg = p.spread ? blockIdx.x >> 3 : blockIdx.x, mi = wg / (NB * KT), bi = wg / KT % NB, jj = wg % KT;
    int blk, a, k;
    qmat_of(mi, nb, blk, a, k);
    // parities (all k-tiles when KT = NB): as quartic_tile
    const int pw = g.wpar, px = k & 1, py = (k + 1 + pw) & 1, po = blk == 0 || blk == 3 ? px : py;
    const int hb = KT < NB ? bi / KT : 0;                     // parity block of the row tile
    auto kt0 = [&](int pa) { return KT < NB ? KT * (hb ^ pa) : 0; };   // first k-tile of A(bi, :) of parity pa
    const int bj = kt0(po) + jj, bjp = kt0(po ^ 1) + jj;      // own tile's column and its P tile's
    const long long m = (long long)Dp * Dp;
    const double c_nbr = blk < 2 ? k : k + 1;
    const bool nbr = blk < 2 ? k >= 1 : k <= 3;
    // matrices read besides the own one: the neighbour channel's, x_k and x_{k-1} (y), a1_k (a0)
    const int mn = blk < 2 ? mi - 1 : mi + 1;
    const int mx = blk == 1 ? rc_qmat(0, 0, k, nb) : rc_qmat(3, 0, k, nb), mxn = blk == 1 ? mx - 1 : mx + 1;
    // constant panels
    cplx cQ[KT], cB[KT], cR[KT], cL[KT], cV[KT], cW[KT];
    {
        auto rows = [&](cplx* K, const double* gm, int t0) {
            const cplx* q = reinterpret_cast<const cplx*>(gm);
#pragma unroll
            for (int t = 0; t < KT; ++t) K[t] = q[(16 * bi + fi) * Dp + 16 * (t0 + t) + fk];
        };
        auto cols = [&](cplx* K, const double* gm, int t0, int col) {
            const cplx* q = reinterpret_cast<const cplx*>(gm);
#pragma unroll
            for (int t = 0; t < KT; ++t) K[t] = q[(16 * (t0 + t) + fk) * Dp + 16 * col + fi];
        };
        const double *Qs = g.Qs + 2 * (long long)a * g.qstride, *Qhs = g.Qhs + 2 * (long long)a * g.qstride;
        const double *v = g.Vrep + 2 * (long long)a * 5 * m, *w = g.Wrep + 2 * (long long)a * 5 * m;
        rows(cQ, blk == 0 ? g.Q : blk == 1 ? Qs : blk == 2 ? Qhs : g.Qh, kt0(0));
        cols(cB, blk < 2 ? g.Qh : g.Q, kt0(po), bj);
        rows(cR, blk < 2 ? g.R : g.Rh, kt0(1));
        cols(cL, blk < 2 ? g.Rh : g.R, kt0(po), bjp);
        if (blk == 1) {
            rows(cV, v, kt0(pw ^ 1));
            rows(cW, w, kt0(pw));
        } else {   // unused by x and a1
            cols(cV, v, kt0(px), bj);
            cols(cW, w, kt0(px), bjp);
        }
    }
    // exchange buffers: tile (r, c) of a matrix at (r NB + c) TB, copy A (read as row blocks) column by
    // column, copy B (read as column blocks) row by row; P as copy B
    const __amdgpu_buffer_rsrc_t rX = rc_rsrc(p.exch, p.exch_bytes);
    const uint32_t mat_bytes = NT * TB, ring_bytes = (uint32_t)nmat * mat_bytes;
    const uint32_t oB = RC_RING * ring_bytes, oP = 2 * oB, oR = 3 * oB, rec_bytes = (uint32_t)p.nslots * 16;
    const uint32_t tile = (uint32_t)(bi * NB + bj) * TB, ptile = (uint32_t)(bi * NB + bjp) * TB;
    const uint32_t a_el = tile + (uint32_t)(ej * 16 + ei) * 16, b_el = tile + (uint32_t)tid * 16;
    const uint32_t p_el = ptile + (uint32_t)tid * 16;
    // fragment offsets: row block bi from k-tile t0, column block col from k-tile t0
    auto row_at = [&](int t0) { return (uint32_t)(bi * NB + t0) * TB + (uint32_t)tid * 16; };
    auto col_at = [&](int t0) { return (uint32_t)(t0 * NB + bj) * TB + (uint32_t)tid * 16; };
    constexpr uint32_t rs = TB, cs = NB * TB;
    const uint32_t f_r1 = row_at(kt0(po)), f_r2 = row_at(kt0(px));
    const uint32_t f_c1 = col_at(kt0(0)), f_c2 = col_at(kt0(pw ^ 1)), f_c3 = col_at(kt0(1)), f_c4 = col_at(kt0(pw));
    const uint32_t sx = (uint32_t)mi * mat_bytes, sn = (uint32_t)mn * mat_bytes, sxx = (uint32_t)mx * mat_bytes,
                   sxn = (uint32_t)mxn * mat_bytes;
    const Ctl ctl{p.abort_flag, p.wait_ticks};
    const long long e = (long long)mi * m + (16 * bi + ei) * Dp + 16 * bj + ej;

    // Whether all workgroups share an XCD (they post its id as the record of attempt 0): then nothing needs
    // to leave its L2.  Only asked when they were laid out for it.
    bool loc = false;
    if (p.spread) {
        __shared__ int s_far;
        if (tid == 0) s_far = 0;
        __syncthreads();
        if (tid < (KT < NB ? 2 : 1))
            rc_put(rX, (uint32_t)(mi * NT + bi * NB + (tid ? bjp : bj)) * 16, oR, cmake(xcd_id(), 0.0));
        for (int q0 = 0; q0 < p.nslots; q0 += 256) {
            const bool use = q0 + tid < p.nslots;
            cplx v;
            rc_fetch<1>(rX, (uint32_t)(q0 + tid) * 16, oR, 0, &v, use);
            if (!rc_await<1>(ctl, rX, (uint32_t)(q0 + tid) * 16, oR, 0, &v, use) || (use && (int)v.re != xcd_id())) s_far = 1;
        }
        __syncthreads();
        loc = uni(s_far) == 0;
    }
    uint32_t ev = 0;
    auto put = [&](cplx v) {
        ++ev;
        const uint32_t so = (ev & (RC_RING - 1)) * ring_bytes + sx;
        rc_put(rX, a_el, so, v, loc);
        rc_put(rX, b_el, oB + so, v, loc);
    };
    RcOdeAhead ahead;
    ahead.clear();
    // right-hand side on the stage input of event ev
    auto rhs = [&](double jac, double jt) -> cplx {
        const uint32_t ring = (ev & (RC_RING - 1)) * ring_bytes;
        const double c = c_nbr * jt;
        cplx r1[KT], r2[KT], c1[KT], c2[KT], c3[KT], c4[KT], q1[KT], q2[KT], ins = cmake(0, 0);
        const RcWant<KT> w1{f_r1, ring + sx, rs, r1, true, true}, w2{f_r2, ring + sxx, rs, r2, blk == 2, true},
            w3{f_c1, oB + ring + sx, cs, c1, true, true}, w4{f_c2, oB + ring + sxx, cs, c2, blk == 1, true},
            w5{f_c3, oB + ring + sn, cs, c3, nbr, true}, w6{f_c4, oB + ring + sxn, cs, c4, nbr && blk == 1, true};
        w1.fetch(rX);
        w2.fetch(rX);
        w3.fetch(rX);
        w4.fetch(rX);
        w5.fetch(rX);
        w6.fetch(rX);
        bool ok = rc_await_all(ctl, rX, w1, w2, w3, w4, w5, w6);
        // level 1
        cacc acc;
        cacc_zero(acc);
        frag_product<KT>(acc, r1, cL);
        if (blk == 2) frag_product<KT>(acc, r2, cW);
        put_partial(acc, red1, wave, lane);
        lds_barrier();
        rc_put(rX, p_el, oP + ring + sx, sum_partial(red1), loc);
        if (ev > RC_RING / 2) {   // empty the slots of event ev - 16
            const uint32_t old = ((ev - RC_RING / 2) & (RC_RING - 1)) * ring_bytes + sx;
            rc_reset(rX, a_el, old, loc);
            rc_reset(rX, b_el, oB + old, loc);
            rc_reset(rX, p_el, oP + old, loc);
        }
        // one-sided products
        cacc_zero(acc);
        auto scaled = [&](double f, const cplx* A, const cplx* B) {
#pragma unroll
            for (int t = 0; t < KT; ++t) cmfma(acc, cscale(f, A[t]), B[t]);
        };
        scaled(jac, cQ, c1);
        scaled(jac, r1, cB);
        if (blk == 1) scaled(jac, cV, c2);
        if (blk == 2) scaled(jac, r2, cV);
        if (nbr) scaled(c, cR, c3);
        if (nbr && blk == 1) scaled(c, cW, c4);
        // level 2
        const RcWant<KT> p1{f_c3, oP + ring + sx, cs, q1, true, true}, p2{f_c4, oP + ring + sxx, cs, q2, blk == 1, true};
        const RcWant<1> p3{b_el, oP + ring + sn, 0, &ins, nbr, true};
        p1.fetch(rX);
        p2.fetch(rX);
        p3.fetch(rX);
        ok = rc_await_all(ctl, rX, p1, p2, p3) && ok;
        scaled(jac, cR, q1);
        if (blk == 1) scaled(jac, cW, q2);
        put_partial(acc, red2, wave, lane);
        if (!ok) s_bad = 1;
        lds_barrier();
        const cplx val = sum_partial(red2);
        return nbr ? cfma(c, ins, val) : val;
    };
    // workgroup 0's time (constant-rate clock) in the right-hand sides (exchanges included), the step
    // end's exchange and the controller
    uint64_t t_rhs = 0, t_sync = 0, t_ctl = 0, tk = __builtin_amdgcn_s_memrealtime();
    const uint64_t t_start = tk;
    auto lap = [&](uint64_t& acc) {
        const uint64_t now = __builtin_amdgcn_s_memrealtime();
        acc += now - tk;
        tk = now;
    };
    cplx yv = reinterpret_cast<const cplx*>(p.ybuf)[e], k0 = cmake(0, 0);
    if (tid == 0) {
        sc = p.c0;
        s_bad = s_stop = 0;
    }
    // what the controller reads, in LDS: each of its device loads would stand in the step's chain
    for (int i = tid; i < RC_SOURCE_SEGMENTS * (RC_SOURCE_DEGREE + 1); i += 256) s_cheb[i] = p.cheb[i];
    for (int i = tid; i < 2 * p.ntrack * p.nranges; i += 256) s_ranges[i] = p.ranges[i];
    if (tid < 2) s_stops[tid] = p.c0.si + tid < p.c0.nstops ? p.stops[p.c0.si + tid] : 0.0;
    if (tid == 0) s_node = p.stop_node[p.c0.si];
    if (tid < 13) s_al[tid] = tid == 11 ? RC_B[11] : tid < 11 ? RC_A[tid + 1][tid] : 0.0;
    __syncthreads();
    put(yv);
    k0 = rhs(p.jac0, p.jt0);   // the first right-hand side (first same as last)
    ode_step_body<true>(&sc, 0, s_slots, s_ranges, p.nranges, p.ntrack, p.cnt, s_stops, &s_node, s_cheb, s_cf);
    lds_barrier();
    while (sc.active && !s_stop) {
        const double he = s_cf[26];
        put(cfma(he, cscale(RC_A[1][0], k0), yv));
        ahead.clear();
        ahead.add(0, k0);
        cplx ynew = cmake(0, 0), F = cmake(0, 0);
        lap(t_ctl);
        // the stops the verdict of this attempt may need, behind its first publish
        if (tid < 2) s_stops[tid] = sc.si + tid < sc.nstops ? p.stops[sc.si + tid] : 0.0;
        if (tid == 2) s_node = p.stop_node[sc.si];
        for (int st = 1; st < 13; ++st) {
            F = rhs(s_cf[2 * st], s_cf[2 * st + 1]);
            if (st == 12) break;
            const cplx u = cfma(he, cfma(s_al[st], F, ahead.a[0]), yv);
            put(u);
            ynew = u;   // stage 11's is the step end
            ahead.add(st, F);
        }
        lap(t_rhs);
        // error sums of this tile, and of every other
        tile_error_put(cfma(RC_E5[12], F, ahead.e5), cfma(RC_E3[12], F, ahead.e3), p.atol + p.rtol * fmax(cabsd(yv), cabsd(ynew)),
                       s_err, wave, lane);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // every emptied slot is empty before the record is seen
        lds_barrier();
        const uint32_t att = (uint32_t)sc.attempts;
        const uint32_t so_rec = oR + (att & (RC_REC_RING - 1)) * rec_bytes;
        const uint32_t so_old = oR + ((att + 2) & (RC_REC_RING - 1)) * rec_bytes;
        if (tid < (KT < NB ? 2 : 1)) {   // Z2: the tile of the other parity block, exactly zero, has no workgroup
            const uint32_t off = (uint32_t)(mi * NT + bi * NB + (tid ? bjp : bj)) * 16;
            rc_put(rX, off, so_rec, tid ? cmake(0, 0) : tile_error_sum(s_err), loc);
            rc_reset(rX, off, so_old, loc);   // attempt - 2: all published attempt - 1 after reading it
        }
        bool ok = true;
        for (int q0 = 0; q0 < p.nslots; q0 += 256) {
            const bool use = q0 + tid < p.nslots;
            cplx v;
            rc_fetch<1>(rX, (uint32_t)(q0 + tid) * 16, so_rec, 0, &v, use);
            ok = rc_await<1>(ctl, rX, (uint32_t)(q0 + tid) * 16, so_rec, 0, &v, use) && ok;
            if (use) {
                s_slots[2 * (q0 + tid)] = v.re;
                s_slots[2 * (q0 + tid) + 1] = v.im;
            }
        }
        if (!ok) s_bad = 1;
        lds_barrier();
        if (tid == 0) s_stop = s_bad;
        lap(t_sync);
        ode_step_body<true>(&sc, 1, s_slots, s_ranges, p.nranges, p.ntrack, p.cnt, s_stops, &s_node, s_cheb, s_cf);
        lds_barrier();
        if (sc.commit) {
            yv = ynew;
            k0 = F;
            const int smp = sc.sample;
            if (smp >= 0) {
                if (e < p.half) reinterpret_cast<cplx*>(p.Sf)[(long long)smp * p.half + e] = ynew;
                else reinterpret_cast<cplx*>(p.Sa)[(long long)(p.c0.npts - 1 - smp) * p.half + (e - p.half)] = ynew;
            }
        }
    }
    reinterpret_cast<cplx*>(p.ybuf)[e] = yv;
    if (wg == 0 && tid == 0) {
        p.out[0] = (double)sc.status;   // the host looks at the abort word first (rc_launch_status)
        p.out[1] = (double)sc.attempts;
        p.out[2] = (double)sc.accepted;
        p.out[3] = (double)sc.rejected;
        p.out[4] = (double)t_rhs;
        p.out[5] = (double)t_sync;
        p.out[6] = (double)t_ctl;
        p.out[7] = (double)(__builtin_amdgcn_s_memrealtime() - t_start);
    }
}

static const void* quartic_ode_fn(int nb, int z2) {
    switch (nb) {
        case 1: return (const void*)rc_quartic_ode<1, 1>;
        case 2: return z2 ? (const void*)rc_quartic_ode<2, 1> : (const void*)rc_quartic_ode<2, 2>;
        case 3: return (const void*)rc_quartic_ode<3, 3>;
        case 4: return z2 ? (const void*)rc_quartic_ode<4, 2> : (const void*)rc_quartic_ode<4, 4>;
        default: return nullptr;
    }
}

// workgroups of rc_quartic_ode that can be resident at once on the current device (0: not launchable)
hipError_t rc_quartic_ode_capacity(int nb, int z2, int nslots, int ntrack, int* blocks) {
    int per_cu = 0, dev = 0, cus = 0, coop = 0;
    hipError_t e;
    const void* fn = quartic_ode_fn(nb, z2);
    const int lds = RC_ODE_LDS(nslots, ntrack);
    *blocks = 0;
    if (!fn || nslots > 4096) return hipSuccess;
    if ((e = hipGetDevice(&dev)) != hipSuccess) return e;
    if ((e = hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, dev)) != hipSuccess) return e;
    if ((e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, std::max(lds, RC_ODE_LDS_ALONE))) !=
        hipSuccess)
        return e;
    if ((e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, 256, lds)) != hipSuccess) return e;
    if ((e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev)) != hipSuccess) return e;
    *blocks = coop ? per_cu * cus : 0;
    return hipSuccess;
}

hipError_t rc_launch_quartic_ode(int nb, int z2, int nwg, int spread, int nslots, int ntrack, const RcOdeRun* dparams,
                                 hipStream_t stream) {
    void* args[] = {(void*)&dparams};
    const void* fn = quartic_ode_fn(nb, z2);
    if (!fn) return hipErrorInvalidValue;
    int dev = 0, cus = 0;
    hipError_t e;
    if ((e = hipGetDevice(&dev)) != hipSuccess) return e;
    if ((e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev)) != hipSuccess) return e;
    // a workgroup per CU where there are CUs for all: more LDS than half a CU's keeps two from sharing one
    // (and its matrix cores) while others idle
    const int lds = RC_ODE_LDS(nslots, ntrack);
    if (spread) nwg *= 8;
    return hipLaunchCooperativeKernel(fn, dim3(nwg), dim3(256), args, nwg <= cus ? std::max(lds, RC_ODE_LDS_ALONE) : lds,
                                      stream);
}

// ---------------------------------------------------------------------------------------------
// L(X) = Q X + X Q^+ + R X R^+ (adjoint: L*(X) = Q^+ X + X Q + R^+ X R, src/transfer.jl:2-19) of
// one Dp x Dp matrix in one launch: one workgroup per 16 x 16 output tile, the one-sided products
// k-split over the waves into one accumulator, the two-sided term through the LDS column block
// T = X R^+[:, bj] (adjoint X R[:, bj]).  Dp <= 64; out must not alias X.  grid (Dp/16)^2.
// ---------------------------------------------------------------------------------------------
__device__ __forceinline__ void lindblad_tile(int Dp, int adjoint, const double* Q, const double* Qh, const double* R,
                                              const double* Rh, const double* X, double* out, cplx* red, cplx* T) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int nbt = Dp / 16, bi = blockIdx.x / nbt, bj = blockIdx.x % nbt;
    const cplx* x = reinterpret_cast<const cplx*>(X);
    const cplx* a1 = reinterpret_cast<const cplx*>(adjoint ? Qh : Q);    // a1 X
    const cplx* b2 = reinterpret_cast<const cplx*>(adjoint ? Q : Qh);    // X b2
    const cplx* c = reinterpret_cast<const cplx*>(adjoint ? R : Rh);     // T = X c[:, bj]
    const cplx* l = reinterpret_cast<const cplx*>(adjoint ? Rh : R);     // l T
    qcolumns(T, QTerm{x, c}, QTerm{}, nullptr, QTerm{}, QTerm{}, Dp, bj, wave, lane);
    cacc acc;
    cacc_zero(acc);
    qprod(acc, a1, x, Dp, bi, bj, wave, lane, 1.0);
    qprod(acc, x, b2, Dp, bi, bj, wave, lane, 1.0);
    qprod_t(acc, l, T, Dp, bi, wave, lane, 1.0);
    const cplx v = qreduce(acc, red, wave, lane);
    reinterpret_cast<cplx*>(out)[(long long)(16 * bi + (tid >> 4)) * Dp + 16 * bj + (tid & 15)] = v;
}

__global__ void __launch_bounds__(256) rc_lindblad(int Dp, int adjoint, const double* Q, const double* Qh,
                                                   const double* R, const double* Rh, const double* X,
                                                   double* out) {
    __shared__ cplx red[1024];
    __shared__ cplx T[64 * 16];
    lindblad_tile(Dp, adjoint, Q, Qh, R, Rh, X, out, red, T);
}

// rc_lindblad on count operands X + v sx into out + v so (blockIdx.y = v), one direction
__global__ void __launch_bounds__(256) rc_lindblad_n(int Dp, int adjoint, const double* Q, const double* Qh,
                                                     const double* R, const double* Rh, const double* X, long long sx,
                                                     double* out, long long so) {
    __shared__ cplx red[1024];
    __shared__ cplx T[64 * 16];
    const long long v = blockIdx.y;
    lindblad_tile(Dp, adjoint, Q, Qh, R, Rh, X + 2 * v * sx, out + 2 * v * so, red, T);
}

// rc_lindblad on up to four operands at once (blockIdx.y = operand), each with its own direction
__global__ void __launch_bounds__(256) rc_lindblad_multi(int Dp, const double* Q, const double* Qh, const double* R,
                                                         const double* Rh, RcLindbladMulti M) {
    __shared__ cplx red[1024];
    __shared__ cplx T[64 * 16];
    const int b = blockIdx.y;
    lindblad_tile(Dp, M.adj[b], Q, Qh, R, Rh, M.X[b], M.out[b], red, T);
}

// ---------------------------------------------------------------------------------------------
// out = A X B in one launch (one workgroup per 16 x 16 output tile, X B[:, bj] as an LDS column
// block), optionally followed by the no-jump inverse's elementwise step in the eigenbasis of Q:
// out_ij <- -out_ij / den_ij, den = lam_i + conj(lam_j) - s (adjoint: conj(lam_i) + lam_j - s),
// s = s_re + i s_im, zero outside the D x D block.  Dp <= 64; out must not alias X.  grid (Dp/16)^2.
// ---------------------------------------------------------------------------------------------
__global__ void __launch_bounds__(256) rc_two_sided(int Dp, int D, const double* A, const double* X, const double* B,
                                                    double* out, int sylvester, int adjoint, const double* lam,
                                                    double s_re, double s_im) {
    __shared__ cplx red[1024];
    __shared__ cplx T[64 * 16];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int nbt = Dp / 16, bi = blockIdx.x / nbt, bj = blockIdx.x % nbt;
    qcolumns(T, QTerm{reinterpret_cast<const cplx*>(X), reinterpret_cast<const cplx*>(B)}, QTerm{}, nullptr,
             QTerm{}, QTerm{}, Dp, bj, wave, lane);
    cacc acc;
    cacc_zero(acc);
    qprod_t(acc, reinterpret_cast<const cplx*>(A), T, Dp, bi, wave, lane, 1.0);
    cplx v = qreduce(acc, red, wave, lane);
    const int r = 16 * bi + (tid >> 4), c = 16 * bj + (tid & 15);
    if (sylvester) {
        if (r >= D || c >= D) {
            v = cmake(0, 0);
        } else {
            const cplx* l = reinterpret_cast<const cplx*>(lam);
            cplx den = adjoint ? cadd(cconj(l[r]), l[c]) : cadd(l[r], cconj(l[c]));
            den.re -= s_re;
            den.im -= s_im;
            const double m = cabs2(den);
            v = cmake(-(v.re * den.re + v.im * den.im) / m, -(v.im * den.re - v.re * den.im) / m);
        }
    }
    reinterpret_cast<cplx*>(out)[(long long)r * Dp + c] = v;
}

// ---------------------------------------------------------------------------------------------
// The connected four-block transfer of a tangent pair (u, w) (blocks 00, ket, bra, ket+bra) applied
// to nch channels in one launch: output matrix (pair p, channel c, block k) =
//   jac T(x_c)_k + c jt S(x_{c-1})_k
// with T the four-block transfer (L on every block, -ip on the ket block, +ip on the bra block, the
// ket insertion v x + w x R^+ from blocks 0 -> 1 and 2 -> 3, the bra insertion x vbra^+ + R x u^+ from
// blocks 0 -> 2 and 1 -> 3, and w x0 u^+ - n x0 into block 3) and S the :phi^4: edge sources (left:
// R x_k, w x_0 -> 1, w x_2 -> 3; right: x_k R^+, x_0 u^+ -> 2, x_1 u^+ -> 3).  With nch = 1, jac = 1 and
// jt = 0 this is the transfer alone (the Krylov operator of the kinetic resolvent).  grid
// ((Dp/16)^2, npair * nch * 4).
// ---------------------------------------------------------------------------------------------
template <bool WIDE>
__global__ void __launch_bounds__(256) rc_pair_rhs(RcPairArgs g) {
    __shared__ cplx red[1024];
    // the column blocks T1 and T2, Dp x 16 each: for WIDE in dynamic LDS
    __shared__ cplx columns[WIDE ? 1 : 2 * 64 * 16];
    extern __shared__ __align__(16) unsigned char pair_lds[];
    cplx* T1 = WIDE ? reinterpret_cast<cplx*>(pair_lds) : columns;
    cplx* T2 = T1 + (WIDE ? g.Dp * 16 : 64 * 16);
    if (g.active && !*g.active) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int Dp = g.Dp, nbt = Dp / 16, bi = blockIdx.x / nbt, bj = blockIdx.x % nbt;
    const int per = 4 * g.nch, mi = blockIdx.y, p = mi / per, r = mi % per, c = r / 4, k = r % 4;
    const long long m = (long long)Dp * Dp;
    const cplx* U = reinterpret_cast<const cplx*>(g.U) + (long long)p * g.ustride;
    auto x = [&](int ch, int blk) { return U + (long long)(4 * ch + blk) * m; };
    const long long dofs = (long long)p * g.dstride;
    const cplx* Q = reinterpret_cast<const cplx*>(g.Q);
    const cplx* Qh = reinterpret_cast<const cplx*>(g.Qh);
    const cplx* R = reinterpret_cast<const cplx*>(g.R);
    const cplx* Rh = reinterpret_cast<const cplx*>(g.Rh);
    const cplx* Qs = reinterpret_cast<const cplx*>(g.Qs) + dofs;
    const cplx* Qb = reinterpret_cast<const cplx*>(g.Qb) + dofs;
    const cplx* v = reinterpret_cast<const cplx*>(g.V) + dofs;
    const cplx* w = reinterpret_cast<const cplx*>(g.W) + dofs;
    const cplx* vbh = reinterpret_cast<const cplx*>(g.Vbh) + dofs;
    const cplx* uh = reinterpret_cast<const cplx*>(g.Uh) + dofs;
    const double jac = g.coef ? g.coef[0] : g.jac;
    const double jt = g.coef ? g.coef[1] : g.jt;
    const double cj = c * jt;
    cacc acc;
    cacc_zero(acc);
    // acc += scale A(bi, :) B(:, bj); with T in LDS, of its columns
    auto mul = [&](const cplx* A, const cplx* B, double scale) {
        if constexpr (WIDE) qprod_wide(acc, A, B, Dp, bi, bj, wave, lane, scale, KTiles{0, nbt});
        else qprod(acc, A, B, Dp, bi, bj, wave, lane, scale);
    };
    auto mul_t = [&](const cplx* A, const cplx* T) {
        if constexpr (WIDE) qprod_t_wide(acc, A, T, Dp, bi, wave, lane, jac);
        else qprod_t(acc, A, T, Dp, bi, wave, lane, jac);
    };
    if (jac != 0.0) {
        const cplx* xk = x(c, k);
        mul(k == 1 ? Qs : k == 2 ? Qb : Q, xk, jac);
        mul(xk, Qh, jac);
        if (k == 0) {
            qcolumns(T1, QTerm{xk, Rh}, QTerm{}, nullptr, QTerm{}, QTerm{}, Dp, bj, wave, lane);
            mul_t(R, T1);
        } else if (k == 1) {
            mul(v, x(c, 0), jac);
            qcolumns(T1, QTerm{xk, Rh}, QTerm{}, T2, QTerm{x(c, 0), Rh}, QTerm{}, Dp, bj, wave, lane);
            mul_t(R, T1);
            mul_t(w, T2);
        } else if (k == 2) {
            mul(x(c, 0), vbh, jac);
            qcolumns(T1, QTerm{xk, Rh}, QTerm{x(c, 0), uh}, nullptr, QTerm{}, QTerm{}, Dp, bj, wave, lane);
            mul_t(R, T1);
        } else {
            mul(v, x(c, 2), jac);
            mul(x(c, 1), vbh, jac);
            qcolumns(T1, QTerm{xk, Rh}, QTerm{x(c, 1), uh}, T2, QTerm{x(c, 2), Rh},
                     QTerm{x(c, 0), uh}, Dp, bj, wave, lane);
            mul_t(R, T1);
            mul_t(w, T2);
        }
    }
    if (c >= 1 && cj != 0.0) {
        const cplx* xp = x(c - 1, k);
        mul(R, xp, cj);
        mul(xp, Rh, cj);
        if (k == 1) mul(w, x(c - 1, 0), cj);
        if (k == 2) mul(x(c - 1, 0), uh, cj);
        if (k == 3) {
            mul(w, x(c - 1, 2), cj);
            mul(x(c - 1, 1), uh, cj);
        }
    }
    cplx val = qreduce(acc, red, wave, lane);
    const long long local = (long long)(16 * bi + (tid >> 4)) * Dp + 16 * bj + (tid & 15);
    if (k == 3 && jac != 0.0) {   // - n x0
        const cplx nn = cmake(g.nov[2 * (long long)p * g.nstride], g.nov[2 * (long long)p * g.nstride + 1]);
        val = csub(val, cscale(jac, cmul(nn, x(c, 0)[local])));
    }
    const long long e = (long long)p * g.fstride + (long long)r * m + local;
    reinterpret_cast<cplx*>(g.F)[e] = val;
    if (g.epi == 0) return;
    // the ODE layout is contiguous (ustride = fstride = 4 nch Dp^2): e indexes y, K and Unext too
    const cplx* Kc = reinterpret_cast<const cplx*>(g.K);
    const cplx y0 = reinterpret_cast<const cplx*>(g.y)[e];
    if (g.epi == 1) {
        const double h = g.hp ? g.hp[0] : g.h;
        cplx sum = cscale(g.comb.a[g.stage], val);
        for (int j = 0; j < g.stage; ++j)
            if (g.comb.a[j] != 0.0) sum = cadd(sum, cscale(g.comb.a[j], Kc[(long long)j * g.sk + e]));
        reinterpret_cast<cplx*>(g.Unext)[e] = cadd(y0, cscale(h, sum));
        return;
    }
    cplx r5 = cscale(g.comb.a[g.stage], val), r3 = cscale(g.comb3.a[g.stage], val);
    for (int j = 0; j < g.stage; ++j) {
        const cplx kj = Kc[(long long)j * g.sk + e];
        if (g.comb.a[j] != 0.0) r5 = cadd(r5, cscale(g.comb.a[j], kj));
        if (g.comb3.a[j] != 0.0) r3 = cadd(r3, cscale(g.comb3.a[j], kj));
    }
    const double sc = g.atol + g.rtol * fmax(cabsd(y0), cabsd(reinterpret_cast<const cplx*>(g.U)[e]));
    double* s5 = reinterpret_cast<double*>(red);
    double* s3 = s5 + 256;
    s5[tid] = cabs2(r5) / (sc * sc);
    s3[tid] = cabs2(r3) / (sc * sc);
    __syncthreads();
    for (int hh = 128; hh > 0; hh >>= 1) {
        if (tid < hh) { s5[tid] += s5[tid + hh]; s3[tid] += s3[tid + hh]; }
        __syncthreads();
    }
    if (tid == 0) {
        const long long slot = (long long)mi * nbt * nbt + blockIdx.x;
        g.partial[2 * slot] = s5[0];
        g.partial[2 * slot + 1] = s3[0];
    }
}
template __global__ void rc_pair_rhs<false>(RcPairArgs g);
template __global__ void rc_pair_rhs<true>(RcPairArgs g);

// Which parity blocks (halves of the basis) of the tangents' matrices hold a nonzero: bit 0 of
// flags[i] an even block of W, bit 1 an odd one, bits 2 and 3 the same of v.  Matrix i at + i ts complex.
__global__ void __launch_bounds__(256) rc_parity_flags(int D, int Dp, const double* w, const double* v, long long ts,
                                                       int* flags) {
    __shared__ int s;
    if (threadIdx.x == 0) s = 0;
    __syncthreads();
    const long long off = (long long)blockIdx.x * ts;
    const cplx* a = reinterpret_cast<const cplx*>(w) + off;
    const cplx* b = reinterpret_cast<const cplx*>(v) + off;
    int f = 0;
    for (int e = threadIdx.x; e < D * D; e += 256) {
        const int i = e / D, j = e % D, odd = (i < D / 2) != (j < D / 2) ? 1 : 0;
        const cplx x = a[(long long)i * Dp + j], y = b[(long long)i * Dp + j];
        if (x.re != 0.0 || x.im != 0.0) f |= 1 << odd;
        if (y.re != 0.0 || y.im != 0.0) f |= 4 << odd;
    }
    atomicOr(&s, f);
    __syncthreads();
    if (threadIdx.x == 0) flags[blockIdx.x] = s;
}
// X_i: the blocks of the other parity set to zero
__global__ void __launch_bounds__(256) rc_parity_project(int D, int Dp, int parity, double* x, long long ts) {
    cplx* a = reinterpret_cast<cplx*>(x) + (long long)blockIdx.y * ts;
    const int e = blockIdx.x * 256 + threadIdx.x;
    if (e >= D * D) return;
    const int i = e / D, j = e % D, odd = (i < D / 2) != (j < D / 2) ? 1 : 0;
    if (odd != parity) a[(long long)i * Dp + j] = cmake(0, 0);
}
