// Node sums of the pullback (src/observables.jl:161-199): for every pair of forward and adjoint channels
// the sums over the Gauss nodes of F_i (w R^+ A_i + j k A'_i) and w F_i A_i, and the plain weighted sums of
// samples that meet constant matrices.
//
// As batched products and reductions per channel the pullback was 85 launches: 0.55 ms at D = 8, all of it
// launches, and 1.6 ms at D = 64, where the products' intermediates made two more passes over memory.
// Here a wave takes one column block of a stream of nodes and keeps its products in registers: the
// accumulator of M = w R^+ A + .. (lane: rows 4 q + lane / 16, column lane % 16) is, quad by quad, the
// right-hand fragment of k-step q, so M feeds the next product without a move.  The waves of a
// workgroup hold the column blocks of the same nodes, whose F they read together.  From three column blocks
// on R^+ and F are in LDS, and still 208 bytes a lane (NB = 3; 272 at NB = 4) are kept in scratch.  Every stream of nodes
// leaves whole partial matrices, summed in order by a second kernel.
//
// Bound by the matrix cores at D = 64 (3 products a node and pair: 0.28 ms at the peak rate for 512
// nodes), by the latency of a node's chain of loads and products below.  Measured on MI355X, the
// whole pullback: D = 8 0.55 -> 0.07 ms, D = 32 0.65 -> 0.18, D = 64 1.61 -> 0.69 (256 node pairs, window 20).
#include "device_common.h"
#include "pullback.h"

namespace {

// a record through scalar loads (the address is uniform)
template <class T>
__device__ __forceinline__ T load_uniform(const T* p) {
    static_assert(sizeof(T) % 8 == 0, "records are copied in 8-byte words");
    const __attribute__((address_space(4))) uint64_t* q =
        (const __attribute__((address_space(4))) uint64_t*)uni64(reinterpret_cast<uint64_t>(p));
    T t;
    uint64_t* w = reinterpret_cast<uint64_t*>(&t);
#pragma unroll
    for (int k = 0; k < (int)(sizeof(T) / 8); ++k) w[k] = q[k];
    return t;
}
// two accumulators a tile: re += a.re b.re - a.im b.im, im += a.re b.im + a.im b.re
struct Acc2 {
    v4d re, im;
};
__device__ __forceinline__ void zero2(Acc2& c) { c.re = c.im = v4d{0, 0, 0, 0}; }
__device__ __forceinline__ void mma2(Acc2& c, cplx a, cplx b) {
    c.re = __builtin_amdgcn_mfma_f64_16x16x4f64(a.re, b.re, c.re, 0, 0, 0);
    c.im = __builtin_amdgcn_mfma_f64_16x16x4f64(a.re, b.im, c.im, 0, 0, 0);
    c.re = __builtin_amdgcn_mfma_f64_16x16x4f64(-a.im, b.im, c.re, 0, 0, 0);
    c.im = __builtin_amdgcn_mfma_f64_16x16x4f64(a.im, b.re, c.im, 0, 0, 0);
}

}  // namespace

template <int NB>
__global__ void __launch_bounds__(NB == 3 ? 192 : 256, 1) rc_pullback(const RcPullArgs g) {
    constexpr int Dp = 16 * NB, G = NB == 1 ? 4 : NB == 2 ? 2 : 1, NF = 4 * NB;   // k-steps of a product
    // NB > 2: the fragments of R^+ and of the node's F in LDS, read by the NB waves.  In registers they
    // would not fit, and read by each wave from memory they cost three times the products.
    constexpr bool SHARED = NB > 2;
    extern __shared__ __align__(16) unsigned char pull_lds[];
    cplx* sR = reinterpret_cast<cplx*>(pull_lds);   // [row block][k-step][lane]
    cplx* sF = sR + NB * NF * 64;
    const int lane = threadIdx.x & 63, wave = uni(threadIdx.x >> 6), bj = wave % NB;
    const int fi = lane & 15, fk = lane >> 4;
    int term = 0;
    RcPullTerm tm = load_uniform(g.t);
    while ((int)blockIdx.x >= tm.wg0 + tm.nwg) tm = load_uniform(g.t + ++term);
    const int stream = ((int)blockIdx.x - tm.wg0) * G + wave / NB, nstreams = tm.nwg * G;
    // left-hand fragments of op(F)(b, :): row 16 b + fi, column 4 s + fk
    auto left = [&](cplx* f, const cplx* F, int b, bool conj) {
        if (!conj) {
#pragma unroll
            for (int s = 0; s < NF; ++s) f[s] = F[(16 * b + fi) * Dp + 4 * s + fk];
        } else {
#pragma unroll
            for (int s = 0; s < NF; ++s) f[s] = cconj(F[(4 * s + fk) * Dp + 16 * b + fi]);
        }
    };
    // right-hand fragments of op(A)(:, bj): row 4 s + fk, column 16 bj + fi
    auto right = [&](cplx* f, const cplx* A, bool conj) {
        if (!conj) {
#pragma unroll
            for (int s = 0; s < NF; ++s) f[s] = A[(4 * s + fk) * Dp + 16 * bj + fi];
        } else {
#pragma unroll
            for (int s = 0; s < NF; ++s) f[s] = cconj(A[(16 * bj + fi) * Dp + 4 * s + fk]);
        }
    };
    const cplx* rh = reinterpret_cast<const cplx*>(tm.B);
    cplx rf[SHARED ? 1 : NB][NF];
    if constexpr (SHARED) {
        cplx f[NF];
        left(f, rh, bj, false);
#pragma unroll
        for (int s = 0; s < NF; ++s) sR[(bj * NF + s) * 64 + lane] = f[s];
        __syncthreads();
    } else {
#pragma unroll
        for (int r = 0; r < NB; ++r) left(rf[r], rh, r, false);
    }
    Acc2 t1[NB], t2[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        zero2(t1[b]);
        zero2(t2[b]);
    }
    // the stream's units: pair q of node i, one after the other; the next one's A (and the share of its F)
    // is loaded ahead
    const int q0 = tm.first, q1 = tm.last;
    int i = stream, q = q0;
    cplx af[NF], na[NF], nf[SHARED ? NF : 1];
    auto load = [&](int i, int q) {
        const RcPullEntry e = load_uniform(g.e + q);
        right(na, reinterpret_cast<const cplx*>(e.A) + (long long)i * e.sA, e.conj);
        if constexpr (SHARED) left(nf, reinterpret_cast<const cplx*>(e.F) + (long long)i * e.sF, bj, e.conj);
    };
    if (i < g.nn) load(i, q);
    while (i < g.nn) {
        const RcPullEntry e = load_uniform(g.e + q);
        const double wi = ld_const(g.wn, i), ji = ld_const(g.jn, i);
        cplx mf[NF];
#pragma unroll
        for (int s = 0; s < NF; ++s) af[s] = na[s];
        if constexpr (SHARED) {
            __syncthreads();   // the last unit's F has been read
#pragma unroll
            for (int s = 0; s < NF; ++s) sF[(bj * NF + s) * 64 + lane] = nf[s];
        }
        const int ni = q + 1 < q1 ? i : i + nstreams, nq = q + 1 < q1 ? q + 1 : q0;
        if (ni < g.nn) load(ni, nq);
        cplx d[NF];
        if (e.D) right(d, reinterpret_cast<const cplx*>(e.D) + (long long)i * e.sA, false);
#pragma unroll
        for (int r = 0; r < NB; ++r) {
            Acc2 m;
            zero2(m);
#pragma unroll
            for (int s = 0; s < NF; ++s) {
                if constexpr (SHARED) mma2(m, sR[(r * NF + s) * 64 + lane], af[s]);
                else mma2(m, rf[r][s], af[s]);
            }
#pragma unroll
            for (int h = 0; h < 4; ++h) mf[4 * r + h] = cmake(wi * m.re[h], wi * m.im[h]);
        }
        if (e.D) {
            const double c = e.jk * ji;
#pragma unroll
            for (int s = 0; s < NF; ++s) mf[s] = cmake(fma(c, d[s].re, mf[s].re), fma(c, d[s].im, mf[s].im));
        }
#pragma unroll
        for (int s = 0; s < NF; ++s) af[s] = cscale(wi, af[s]);
        if constexpr (SHARED) {
            __syncthreads();
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int s = 0; s < NF; ++s) {
                    const cplx f = sF[(b * NF + s) * 64 + lane];
                    mma2(t1[b], f, mf[s]);
                    mma2(t2[b], f, af[s]);
                }
        } else {
            const cplx* F = reinterpret_cast<const cplx*>(e.F) + (long long)i * e.sF;
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                cplx f[NF];
                left(f, F, b, e.conj);
#pragma unroll
                for (int s = 0; s < NF; ++s) {
                    mma2(t1[b], f[s], mf[s]);
                    mma2(t2[b], f[s], af[s]);
                }
            }
        }
        i = ni;
        q = nq;
    }
    cplx* out = reinterpret_cast<cplx*>(g.partial) + ((long long)blockIdx.x * G + wave / NB) * 2 * Dp * Dp;
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int h = 0; h < 4; ++h) {
            const int el = (16 * b + 4 * h + fk) * Dp + 16 * bj + fi;
            out[el] = cmake(t1[b].re[h], t1[b].im[h]);
            out[Dp * Dp + el] = cmake(t2[b].re[h], t2[b].im[h]);
        }
}

// sums over the four quarters of a list, 64 elements a workgroup: quarter q in wave q
__device__ __forceinline__ cplx quarters(cplx v, cplx* red) {
    red[threadIdx.x] = v;
    __syncthreads();
    const int l = threadIdx.x & 63;
    return cadd(cadd(cadd(red[l], red[64 + l]), red[128 + l]), red[192 + l]);
}

// quarter q of the sum over matrices s0 .. s0 + ns - 1 (two matrices of n elements apart)
__device__ __forceinline__ cplx quarter_sum(const cplx* p, int s0, int ns, int q, int n) {
    const int a = s0 + ns * q / 4, b = s0 + ns * (q + 1) / 4;
    cplx s = cmake(0, 0);
#pragma unroll 8
    for (int i = a; i < b; ++i) s = cadd(s, p[(long long)i * 2 * n]);
    return s;
}

// blockIdx.y = 0: XR = W + sum_t c_t T1_t; 1: XQ = sum_t c_t T2_t, over the terms' partial matrices
__global__ void __launch_bounds__(256) rc_pull_sum(const RcPullArgs g, int n, int streams, const double* W, double* XR,
                                                   double* XQ) {
    __shared__ cplx red[256];
    const int e = blockIdx.x * 64 + (threadIdx.x & 63), q = threadIdx.x >> 6, y = blockIdx.y;
    const cplx* p = reinterpret_cast<const cplx*>(g.partial) + (long long)y * n + e;
    cplx v = cmake(0, 0);
    for (int t = 0; t < g.nterms; ++t) {
        const RcPullTerm tm = load_uniform(g.t + t);
        v = cadd(v, cscale(tm.c, quarter_sum(p, tm.wg0 * streams, tm.nwg * streams, q, n)));
    }
    v = quarters(v, red);
    if (q) return;
    if (y == 0 && W) v = cadd(v, reinterpret_cast<const cplx*>(W)[e]);
    reinterpret_cast<cplx*>(y ? XQ : XR)[e] = v;
}

// sum blockIdx.y & 1 of term blockIdx.y >> 1, into sums
__global__ void __launch_bounds__(256) rc_pull_sum_terms(const RcPullArgs g, int n, int streams, double* sums) {
    __shared__ cplx red[256];
    const int e = blockIdx.x * 64 + (threadIdx.x & 63), q = threadIdx.x >> 6, y = blockIdx.y & 1;
    const RcPullTerm tm = load_uniform(g.t + (blockIdx.y >> 1));
    const cplx* p = reinterpret_cast<const cplx*>(g.partial) + (long long)y * n + e;
    const cplx v = quarters(quarter_sum(p, tm.wg0 * streams, tm.nwg * streams, q, n), red);
    if (q == 0) reinterpret_cast<cplx*>(sums)[(long long)blockIdx.y * n + e] = v;
}

__global__ void __launch_bounds__(256) rc_action_pull(int Dp, const double* sums, double g, const double* wrho,
                                                      double* out, long long ts) {
    __shared__ cplx red[256];
    const int n = Dp * Dp, l = threadIdx.x, a = blockIdx.y;
    const cplx* s = reinterpret_cast<const cplx*>(sums) + (long long)4 * a * n;   // T1, T2 of term 2 a, then of 2 a + 1
    red[l] = l < Dp ? s[3 * n + l * Dp + l] : cmake(0, 0);
    __syncthreads();
    cplx tr = cmake(0, 0);
    for (int i = 0; i < Dp; ++i) tr = cadd(tr, red[i]);
    const int e = blockIdx.x * 256 + l;
    if (e >= n) return;
    cplx* o = reinterpret_cast<cplx*>(out) + (long long)a * ts + e;
    const cplx w = reinterpret_cast<const cplx*>(wrho)[(long long)a * ts + e];
    *o = cadd(*o, cscale(g, csub(cadd(s[e], s[2 * n + e]), cmul(tr, w))));
}

// blockIdx.y: output; sixteen waves share the nodes of 64 elements (133 us at D = 64 with 512 nodes; four took
// 199, a chain of 128 loads' latency in eights)
__global__ void __launch_bounds__(1024) rc_lin(const RcLinArgs g, int Dp) {
    constexpr int P = 16;
    __shared__ cplx red[64 * P];
    const int l = threadIdx.x & 63, e = blockIdx.x * 64 + l, q = threadIdx.x >> 6, o = blockIdx.y;
    const int et = (e % Dp) * Dp + e / Dp;
    cplx v = cmake(0, 0);
    for (int k = 0; k < g.nsrc[o]; ++k) {
        const RcLinSource& s = g.src[o][k];
        const cplx* x = reinterpret_cast<const cplx*>(s.X) + (s.conj ? et : e);
        cplx t = cmake(0, 0);
        if (s.kind == 2) {
            if (q == 0) t = x[0];
        } else {
            const double* w = s.kind ? g.jn : g.wn;
            const int a = g.nn * q / P, b = g.nn * (q + 1) / P;
#pragma unroll 8
            for (int i = a; i < b; ++i) {
                const double c = w[i];
                const cplx y = x[(long long)i * s.s];
                t = cmake(fma(c, y.re, t.re), fma(c, y.im, t.im));
            }
        }
        v = cadd(v, cscale(s.c, s.conj ? cconj(t) : t));
    }
    red[threadIdx.x] = v;
    __syncthreads();
    if (q) return;
    for (int p = 1; p < P; ++p) v = cadd(v, red[64 * p + l]);
    reinterpret_cast<cplx*>(g.out[o])[e] = v;
}

hipError_t rc_launch_lin(int Dp, const RcLinArgs& a, hipStream_t stream) {
    hipLaunchKernelGGL(rc_lin, dim3(Dp * Dp / 64, a.nouts), dim3(1024), 0, stream, a, Dp);
    return hipGetLastError();
}

static hipError_t launch_partial(int nb, const RcPullArgs& a, hipStream_t stream) {
    const dim3 grid(a.nwg);
    const int lds = nb > 2 ? 2 * nb * 4 * nb * 1024 : 0;   // B and F
    hipError_t e = hipSuccess;
    switch (nb) {
        case 1: hipLaunchKernelGGL(rc_pullback<1>, grid, dim3(256), 0, stream, a); break;
        case 2: hipLaunchKernelGGL(rc_pullback<2>, grid, dim3(256), 0, stream, a); break;
        case 3:
            e = hipFuncSetAttribute((const void*)rc_pullback<3>, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
            if (e == hipSuccess) hipLaunchKernelGGL(rc_pullback<3>, grid, dim3(192), lds, stream, a);
            break;
        case 4:
            e = hipFuncSetAttribute((const void*)rc_pullback<4>, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
            if (e == hipSuccess) hipLaunchKernelGGL(rc_pullback<4>, grid, dim3(256), lds, stream, a);
            break;
        default: return hipErrorInvalidValue;
    }
    return e != hipSuccess ? e : hipGetLastError();
}

hipError_t rc_launch_pullback(int nb, const RcPullArgs& a, const double* W, double* XR, double* XQ, hipStream_t stream) {
    const hipError_t e = launch_partial(nb, a, stream);
    if (e != hipSuccess) return e;
    const int n = 256 * nb * nb;
    hipLaunchKernelGGL(rc_pull_sum, dim3(n / 64, 2), dim3(256), 0, stream, a, n, rc_pull_streams(nb), W, XR, XQ);
    return hipGetLastError();
}

hipError_t rc_launch_pullback_terms(int nb, const RcPullArgs& a, double* sums, hipStream_t stream) {
    const hipError_t e = launch_partial(nb, a, stream);
    if (e != hipSuccess) return e;
    const int n = 256 * nb * nb;
    hipLaunchKernelGGL(rc_pull_sum_terms, dim3(n / 64, 2 * a.nterms), dim3(256), 0, stream, a, n, rc_pull_streams(nb), sums);
    return hipGetLastError();
}

hipError_t rc_launch_action_pull(int Dp, int na, const double* sums, double g, const double* wrho, double* out,
                                 long long ts, hipStream_t stream) {
    hipLaunchKernelGGL(rc_action_pull, dim3((Dp * Dp + 255) / 256, na), dim3(256), 0, stream, Dp, sums, g, wrho, out, ts);
    return hipGetLastError();
}
