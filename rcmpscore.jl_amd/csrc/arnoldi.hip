// Arnoldi steps of the kinetic resolvents (src/kinetic_krylov.jl:68-92, src/excitation_action.jl:135-179),
// as many as asked for in one launch, every basis of a set side by side.
//
// As launches a step was 18 of them for the two-block operator (eleven batched products, then dots and
// subtractions), 165 us at D = 64 with four bases; here a workgroup owns one 16 x 16 tile of one
// block of a basis, one element per thread, and the workgroups of a basis exchange tiles as the
// trajectory kernel does (exchange.h).  A step is two levels of products (the tiles of R x and of the
// insertion's x0 R^+, then everything on them) and two all-workgroup sums, one for each Gram-Schmidt pass;
// the second pass sums <w, w> beside its coefficients, |w - V h|^2 = <w, w> - |h|^2 (V orthonormal, h of
// the size of the rounding of the first pass).  Bases do not wait for one another.
//
// The thread's element of the first 40 vectors stays in registers; of the later ones it is read from
// memory, eight loads ahead of the eight in use (each thread reads only what it wrote itself).
//
// Measured on MI355X, us per step (bases of 128 vectors): two blocks at D = 64, four bases 165 -> 29;
// one block at D = 48, four bases 45 -> 26 (of 192 vectors).  What is left: two exchanges of tiles and
// two of sums (about 1.5 us each), 2.3 us of matrix instructions, and four passes over the basis.
//
// Slots: a workgroup starts step j after taking both sums of step j - 1, so everyone is done with that
// step's tiles and it empties its own; it waits for that before it posts a sum of step j, and a reader
// looks at the slot again in step j + 1, after taking both sums of step j.  Two slots suffice.
#include "device_common.h"
#include "exchange.h"
#include "arnoldi.h"

namespace {

constexpr int RC_HOT = 40;              // vectors in registers
constexpr int RC_VAL = RC_ARN_VALUES;
constexpr int RC_WW = RC_VAL - 1;       // index of <w, w> among the values of a sum

struct ArnLds {
    cplx red[2][1024];       // partial tiles, alternating
    cplx h[RC_VAL];          // the sums of the pass at hand
    cplx rows[16][RC_VAL];   // row sums of the 16 rows of lanes
    int bad;
};

// a + b c
__device__ __forceinline__ cplx caxpy(cplx b, cplx c, cplx a) {
    return cmake(fma(b.re, c.re, fma(-b.im, c.im, a.re)), fma(b.re, c.im, fma(b.im, c.re, a.im)));
}

}  // namespace

template <int NB, int BLK>
__global__ void __launch_bounds__(256, 1) rc_arnoldi(const RcArnProb* __restrict__ probs, uint32_t* abort_flag,
                                                     long long wait_ticks) {
    extern __shared__ __align__(16) unsigned char arn_lds[];
    ArnLds& s = *reinterpret_cast<ArnLds*>(arn_lds);
    constexpr int Dp = 16 * NB, NT = NB * NB, NW = NT * BLK;
    constexpr long long m = (long long)Dp * Dp, n = BLK * m;
    constexpr uint32_t TB = 4096, MB = NT * TB;
    const RcArnProb P = load_scalar<RcArnProb>(probs, blockIdx.x / NW);
    const int wg = blockIdx.x % NW, blk = wg / NT, tile = wg % NT, bi = tile / NB, bj = tile % NB;
    const int tid = threadIdx.x, lane = tid & 63, wave = uni(tid >> 6);
    const int ei = tid >> 4, ej = tid & 15, fi = lane & 15, fk = 4 * wave + (lane >> 4);
    const bool adj = P.adj != 0, two = BLK == 2 && blk == 1;
    const Ctl ctl{abort_flag, wait_ticks};
    if (tid == 0) s.bad = 0;
    if (P.k0 >= P.k1) return;   // the same for every workgroup of the basis

    // constant panels: fragments of row block bi (left factors) and column block bj (right factors).
    // K1, Kq, Kx, Kp as the trajectory kernel's; Kt: the insertion's level-1 factor (block 0), Kv, Kw:
    // its level-2 factors (block 1)
    cplx K1[NB], Kq[NB], Kx[NB], Kp[NB], Kt[NB], Kw[NB];
    {
        auto rows = [&](cplx* K, const double* g) {
            const cplx* q = reinterpret_cast<const cplx*>(g);
#pragma unroll
            for (int t = 0; t < NB; ++t) K[t] = q[(16 * bi + fi) * Dp + 16 * t + fk];
        };
        auto cols = [&](cplx* K, const double* g) {
            const cplx* q = reinterpret_cast<const cplx*>(g);
#pragma unroll
            for (int t = 0; t < NB; ++t) K[t] = q[(16 * t + fk) * Dp + 16 * bj + fi];
        };
        if (!adj) {
            rows(K1, P.R); rows(Kq, two ? P.Qs : P.Q); cols(Kx, P.Qh); cols(Kp, P.Rh);
        } else {
            cols(K1, P.R); rows(Kq, two ? P.Qs : P.Qh); cols(Kx, P.Q); rows(Kp, P.Rh);
        }
        if constexpr (BLK == 2) {
            if (!two) {
                cols(Kt, adj ? P.w : P.Rh);
            } else if (!adj) {
                rows(Kt, P.v); rows(Kw, P.w);
            } else {
                cols(Kt, P.v);
            }
        }
    }

    // ---- exchange: copy A (read as row blocks) column by column, copy B row by row
    const __amdgpu_buffer_rsrc_t rX = rc_rsrc(P.exch, (uint32_t)rc_arn_exch_bytes(NB, BLK));
    constexpr uint32_t XS = 2 * BLK * MB, PS = (BLK == 2 ? 3 : 1) * MB;   // bytes of a slot
    constexpr uint32_t oP = 2 * XS, oRec = oP + 2 * PS, REC = RC_VAL * 16;
    const uint32_t a_el = (uint32_t)tile * TB + (uint32_t)(ej * 16 + ei) * 16, b_el = (uint32_t)tile * TB + (uint32_t)tid * 16;
    const uint32_t f_row = (uint32_t)(bi * NB) * TB + (uint32_t)tid * 16, f_col = (uint32_t)bj * TB + (uint32_t)tid * 16;
    const uint32_t oX = (uint32_t)blk * 2 * MB;               // own block's copy A, copy B behind it
    const uint32_t oPt = (uint32_t)(blk == 0 ? 0 : 2) * MB;   // own P; T is matrix 1
    const uint32_t p_el = adj ? b_el : a_el;
    bool ok = true;
    uint32_t nrec = 0;
    int rb = 0;   // partial buffer of the next product
    auto reduced = [&](const cacc& acc) -> cplx {
        put_partial(acc, s.red[rb], wave, lane);
        lds_barrier();
        const cplx v = sum_partial(s.red[rb]);
        rb ^= 1;
        return v;
    };

    // ---- sums over the workgroups of the basis: value t on thread t (0 .. nv - 1, and RC_WW)
    auto sum = [&](int nv, cplx* out) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // every slot emptied so far is empty
        lds_barrier();
        const bool on = tid < nv || tid == RC_WW;
        ++nrec;
        cplx t = cmake(0, 0);
        const uint32_t slot = oRec + (nrec & 3) * NW * REC, old = oRec + ((nrec + 2) & 3) * NW * REC;
        if (__any(on)) {
            if (on) {
                t = s.rows[0][tid];
#pragma unroll
                for (int r = 1; r < 16; ++r) t = cadd(t, s.rows[r][tid]);
            }
            if (on) rc_put(rX, (uint32_t)wg * REC + (uint32_t)tid * 16, slot, t);
        }
        // the record before the last: every workgroup posted the last one after taking it
        rc_reset(rX, (uint32_t)wg * REC + (uint32_t)tid * 16, old);
        if (__any(on)) {
            t = cmake(0, 0);
            constexpr int G = NW % 8 == 0 ? 8 : NW % 9 == 0 ? 9 : NW % 4 == 0 ? 4 : NW % 2 == 0 ? 2 : 1;
#pragma unroll 1
            for (int g = 0; g < NW; g += G) {
                cplx v[G];
                const uint32_t so = slot + (uint32_t)g * REC;
                rc_fetch<G>(rX, (uint32_t)tid * 16, so, REC, v, on);
                ok = rc_await<G>(ctl, rX, (uint32_t)tid * 16, so, REC, v, on) && ok;
#pragma unroll
                for (int q = 0; q < G; ++q) t = cadd(t, v[q]);
            }
            if (on) s.h[tid] = t;
            if (on && out) {
                if (wg == 0 && tid < nv) reinterpret_cast<cplx*>(out)[tid] = t;
            }
        }
        lds_barrier();
    };

    cplx V[RC_HOT];   // indices are static
    cplx* Vm = reinterpret_cast<cplx*>(P.V) + (long long)blk * m + (16 * bi + ei) * Dp + 16 * bj + ej;
#pragma unroll
    for (int j = 0; j < RC_HOT; ++j) V[j] = j <= P.k0 ? Vm[(long long)j * n] : cmake(0, 0);
    cplx x = Vm[(long long)P.k0 * n];
    __syncthreads();

    // The sums conj(V_j) w, j < nv, of this workgroup into s.rows; eight at a time
    auto dots8 = [&](const cplx* q, cplx w, int g) {
        double p[16];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            p[2 * j] = fma(q[j].re, w.re, q[j].im * w.im);
            p[2 * j + 1] = fma(q[j].re, w.im, -(q[j].im * w.re));
        }
        reinterpret_cast<double*>(&s.rows[4 * wave + (lane >> 4)][8 * g])[lane & 15] = row_sums16(p, lane);
    };
    auto load8 = [&](cplx* q, int g, int nv) {   // vectors beyond the basis: zero
#pragma unroll
        for (int j = 0; j < 8; ++j) q[j] = 8 * g + j < nv ? Vm[(long long)(8 * g + j) * n] : cmake(0, 0);
    };
    auto dots = [&](cplx w, int nv) {
        cplx q[8], nx[8];
        const int ng = (nv + 7) >> 3;
        if (ng > RC_HOT / 8) load8(nx, RC_HOT / 8, nv);
#pragma unroll
        for (int g = 0; g < RC_HOT / 8; ++g) {
            if (8 * g >= nv) continue;
            dots8(V + 8 * g, w, g);
        }
#pragma unroll 1
        for (int g = RC_HOT / 8; g < ng; ++g) {
#pragma unroll
            for (int j = 0; j < 8; ++j) q[j] = nx[j];
            if (g + 1 < ng) load8(nx, g + 1, nv);
            dots8(q, w, g);
        }
        double wv = row_sum(fma(w.re, w.re, w.im * w.im));
        if ((lane & 15) == 0) s.rows[4 * wave + (lane >> 4)][RC_WW] = cmake(wv, 0.0);
    };
    auto subtract = [&](cplx w, int nv) -> cplx {
        cplx q[8], nx[8];
        const int ng = (nv + 7) >> 3;
        if (ng > RC_HOT / 8) load8(nx, RC_HOT / 8, nv);
#pragma unroll
        for (int g = 0; g < RC_HOT / 8; ++g) {
            if (8 * g >= nv) continue;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const cplx h = 8 * g + j < nv ? s.h[8 * g + j] : cmake(0, 0);
                w = caxpy(cmake(-h.re, -h.im), V[8 * g + j], w);
            }
        }
#pragma unroll 1
        for (int g = RC_HOT / 8; g < ng; ++g) {
#pragma unroll
            for (int j = 0; j < 8; ++j) q[j] = nx[j];
            if (g + 1 < ng) load8(nx, g + 1, nv);
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const cplx h = 8 * g + j < nv ? s.h[8 * g + j] : cmake(0, 0);
                w = caxpy(cmake(-h.re, -h.im), q[j], w);
            }
        }
        return w;
    };

#pragma unroll 1
    for (int j = P.k0; j < P.k1; ++j) {
        const uint32_t sx = (j & 1) * XS, sp = oP + (j & 1) * PS;
        // the vector, and the last step's slots (everyone is done with them)
        rc_put(rX, a_el, sx + oX, x);
        rc_put(rX, b_el, sx + oX + MB, x);
        if (j > P.k0) {
            const uint32_t ox = ((j - 1) & 1) * XS, op = oP + ((j - 1) & 1) * PS;
            rc_reset(rX, a_el, ox + oX);
            rc_reset(rX, b_el, ox + oX + MB);
            rc_reset(rX, p_el, op + oPt);
            if (BLK == 2 && blk == 0) rc_reset(rX, b_el, op + MB);
        }
        cplx xr[NB], xc[NB], x0[NB];
        {
            const RcWant<NB> wr{f_row, sx + oX, TB, xr, true, true}, wc{f_col, sx + oX + MB, NB * TB, xc, true, true};
            const RcWant<NB> w0{adj ? f_row : f_col, adj ? sx : sx + MB, adj ? TB : NB * TB, x0, two, true};
            wr.fetch(rX);
            wc.fetch(rX);
            w0.fetch(rX);
            ok = rc_await_all(ctl, rX, wr, wc, w0) && ok;
        }
        // level 1
        cacc acc;
        cacc_zero(acc);
        if (!adj) frag_product<NB>(acc, K1, xc);
        else frag_product<NB>(acc, xr, K1);
        rc_put(rX, p_el, sp + oPt, reduced(acc));
        if (BLK == 2 && blk == 0) {
            cacc_zero(acc);
            frag_product<NB>(acc, xr, Kt);
            rc_put(rX, b_el, sp + MB, reduced(acc));
        }
        // level 2
        cacc_zero(acc);
        frag_product<NB>(acc, Kq, xc);
        frag_product<NB>(acc, xr, Kx);
        if constexpr (BLK == 2) {
            if (two) {
                if (!adj) frag_product<NB>(acc, Kt, x0);
                else frag_product<NB>(acc, x0, Kt);
            }
        }
        {
            const uint32_t pf = adj ? f_col : f_row, ps = adj ? NB * TB : TB;
            const RcWant<NB> wp{pf, sp + oPt, ps, xr, true, true}, wt{f_col, sp + MB, NB * TB, xc, two, true};
            wp.fetch(rX);
            wt.fetch(rX);
            ok = rc_await_all(ctl, rX, wp, wt) && ok;
        }
        if (!adj) frag_product<NB>(acc, xr, Kp);
        else frag_product<NB>(acc, Kp, xr);
        if constexpr (BLK == 2) {
            if (two) {
                if (!adj) frag_product<NB>(acc, Kw, xc);
                else frag_product<NB>(acc, Kp, xc);
            }
        }
        cplx w = reduced(acc);
        // classical Gram-Schmidt twice
        const int nv = j + 1;
        const long long ho = (long long)(j - P.k0) * P.hstride;
        dots(w, nv);
        sum(nv, reinterpret_cast<cplx*>(P.h1 + ho));
        if (wg == 0 && tid == 0) P.hw[ho] = s.h[RC_WW].re;
        w = subtract(w, nv);
        dots(w, nv);
        sum(nv, reinterpret_cast<cplx*>(P.h2 + ho));
        // |w|^2 of the new direction: every wave adds the same numbers in the same order
        double hh = 0.0;
        for (int i = lane; i < nv; i += 64) hh += fma(s.h[i].re, s.h[i].re, s.h[i].im * s.h[i].im);
        const double ww = s.h[RC_WW].re - wave_sum(hh);
        const double norm2 = isnan(ww) ? ww : fmax(ww, 0.0);
        if (wg == 0 && tid == 0) P.hn[ho] = norm2;
        w = subtract(w, nv);
        const double inv = norm2 > 0.0 ? 1.0 / sqrt(norm2) : 0.0;
        x = cscale(inv, w);
        Vm[(long long)(j + 1) * n] = x;
#pragma unroll
        for (int i = 0; i < RC_HOT; ++i) {   // selects, not branches: those become one store at a computed index
            V[i].re = i == j + 1 ? x.re : V[i].re;
            V[i].im = i == j + 1 ? x.im : V[i].im;
        }
        if (!ok) s.bad = 1;
        lds_barrier();   // every thread has read s.h
        if (s.bad) break;   // a wait failed: the abort word is set and the host sees it
    }
}

static const void* arn_fn(int nb, int blocks) {
    switch (nb * 2 + blocks - 1) {
        case 2: return (const void*)rc_arnoldi<1, 1>;
        case 3: return (const void*)rc_arnoldi<1, 2>;
        case 4: return (const void*)rc_arnoldi<2, 1>;
        case 5: return (const void*)rc_arnoldi<2, 2>;
        case 6: return (const void*)rc_arnoldi<3, 1>;
        case 7: return (const void*)rc_arnoldi<3, 2>;
        case 8: return (const void*)rc_arnoldi<4, 1>;
        case 9: return (const void*)rc_arnoldi<4, 2>;
        default: return nullptr;
    }
}

hipError_t rc_arn_capacity(int nb, int blocks, int* bases) {
    const void* fn = nb >= 1 && nb <= 4 ? arn_fn(nb, blocks) : nullptr;
    *bases = 0;
    if (!fn) return hipSuccess;
    hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)sizeof(ArnLds));
    if (e != hipSuccess) return e;
    int per_cu = 0, dev = 0, cus = 0, coop = 0;
    if ((e = hipGetDevice(&dev)) != hipSuccess) return e;
    if ((e = hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, dev)) != hipSuccess) return e;
    if ((e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, 256, sizeof(ArnLds))) != hipSuccess) return e;
    if ((e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev)) != hipSuccess) return e;
    *bases = coop ? per_cu * cus / (nb * nb * blocks) : 0;
    return hipSuccess;
}

hipError_t rc_launch_arnoldi(int nb, int blocks, int n, const RcArnProb* probs, uint32_t* abort_flag,
                             long long wait_ticks, hipStream_t stream) {
    const void* fn = nb >= 1 && nb <= 4 ? arn_fn(nb, blocks) : nullptr;
    if (!fn) return hipErrorInvalidValue;
    void* args[] = {(void*)&probs, (void*)&abort_flag, (void*)&wait_ticks};
    return hipLaunchCooperativeKernel(fn, dim3(n * nb * nb * blocks), dim3(256), args, sizeof(ArnLds), stream);
}

// Projected solves, one wave per basis and node (src/kinetic_krylov.jl:95-113).
//
// I - z H is upper Hessenberg and the right-hand side a multiple of e_1, so it is reduced to upper
// triangular form from the right, rotations of the columns (i - 1, i) from the last row up: the
// triangular system's solution is then e_1 beta / r_11, and y the rotations applied to it, a chain of
// products.  Only the column at hand is kept (row r on lane r % 64), the rotations in LDS, and H, shared by
// the nodes, is read once a column ahead.  Rotations throughout, as a QR factorization.
//
// On sixteen host threads by Givens QR, with the basis's matrix in memory per node, the solves of four
// bases of 128 vectors at 112 nodes took 4 ms; here 60 us with the upload of H.
template <int KR>
__global__ void __launch_bounds__(64) rc_projected(const RcProjProb* __restrict__ probs, const double* __restrict__ zs) {
    __shared__ cplx pa[RC_PROJ_MAX_K], pg[RC_PROJ_MAX_K];   // rotation i; then pa[i]: y[i]
    const RcProjProb P = load_scalar<RcProjProb>(probs, blockIdx.y);
    const int lane = threadIdx.x, node = blockIdx.x, k = P.k;
    const double z = ld_const(zs, node);
    cplx* Y = reinterpret_cast<cplx*>(P.Y) + (long long)node * P.ldy;
    double est = 0.0;
    if (k > 0) {
        const cplx* H = reinterpret_cast<const cplx*>(P.H);
        auto column = [&](cplx* v, int c) {   // column c of H, rows 0 .. min(c + 1, k - 1)
            const long long off = (long long)c * (c + 3) / 2;
#pragma unroll
            for (int q = 0; q < KR; ++q) {
                const int r = 64 * q + lane;
                v[q] = r <= c + 1 && r < k ? H[off + r] : cmake(0, 0);
            }
        };
        auto shift = [&](cplx* v, int c) {
#pragma unroll
            for (int q = 0; q < KR; ++q) v[q] = cmake((64 * q + lane == c ? 1.0 : 0.0) - z * v[q].re, -z * v[q].im);
        };
        auto at = [&](const cplx* v, int r) -> cplx {   // r uniform
            cplx x = v[0];
#pragma unroll
            for (int q = 1; q < KR; ++q) {
                x.re = q == (r >> 6) ? v[q].re : x.re;
                x.im = q == (r >> 6) ? v[q].im : x.im;
            }
            return cmake(read_lane(x.re, r & 63), read_lane(x.im, r & 63));
        };
        cplx cur[KR], a[KR], nx[KR];
        column(cur, k - 1);
        shift(cur, k - 1);
        if (k > 1) column(nx, k - 2);
        bool singular = false;
        for (int i = k - 1; i >= 1; --i) {
#pragma unroll
            for (int q = 0; q < KR; ++q) a[q] = nx[q];
            if (i >= 2) column(nx, i - 2);
            shift(a, i - 1);
            const cplx al = at(cur, i), ga = at(a, i);
            const double r2 = fma(al.re, al.re, fma(al.im, al.im, fma(ga.re, ga.re, ga.im * ga.im)));
            singular |= !(r2 > 0.0);
            const double inv = 1.0 / sqrt(r2);
            const cplx ca = cscale(inv, al), cg = cscale(-inv, ga);
            if (lane == 0) {
                pa[i] = ca;
                pg[i] = cg;
            }
#pragma unroll
            for (int q = 0; q < KR; ++q)
                cur[q] = cmake(fma(a[q].re, ca.re, fma(-a[q].im, ca.im, fma(cur[q].re, cg.re, -(cur[q].im * cg.im)))),
                               fma(a[q].re, ca.im, fma(a[q].im, ca.re, fma(cur[q].re, cg.im, cur[q].im * cg.re))));
        }
        __syncthreads();
        const cplx r11 = at(cur, 0);
        const double d2 = fma(r11.re, r11.re, r11.im * r11.im);
        singular |= !(d2 > 0.0);
        cplx c = cmake(P.beta * r11.re / d2, -(P.beta * r11.im / d2));
#pragma unroll 4
        for (int i = 1; i < k; ++i) {
            const cplx y = cmul(pa[i], c);
            c = cmul(pg[i], c);
            if (lane == 0) pa[i - 1] = y;
        }
        if (lane == 0) pa[k - 1] = c;
        const double hk = H[(long long)(k - 1) * (k + 2) / 2 + k].re;
        est = singular ? __longlong_as_double(0x7ff8000000000000LL) : hypot(c.re, c.im) * fabs(z * hk) / P.beta;
        __syncthreads();
    }
    for (int i = lane; i < P.ldy; i += 64) Y[i] = i < k ? pa[i] : cmake(0, 0);
    if (lane == 0) P.est[node] = est;
}

hipError_t rc_launch_projected(int n, int maxk, const RcProjProb* probs, int nz, const double* z, hipStream_t stream) {
    if (maxk > RC_PROJ_MAX_K) return hipErrorInvalidValue;
    const dim3 g(nz, n), b(64);
    if (maxk <= 64) hipLaunchKernelGGL(rc_projected<1>, g, b, 0, stream, probs, z);
    else if (maxk <= 128) hipLaunchKernelGGL(rc_projected<2>, g, b, 0, stream, probs, z);
    else if (maxk <= 256) hipLaunchKernelGGL(rc_projected<4>, g, b, 0, stream, probs, z);
    else hipLaunchKernelGGL(rc_projected<8>, g, b, 0, stream, probs, z);
    return hipGetLastError();
}
