// Pinned Poisson-type equations (the stationary state, the boundary environment, the excitation's
// Poisson solves; src/transfer.jl:74-153, src/excitation_environments.jl:75-85) by restarted GMRES, a
// whole solve in one launch.
//
// As a sequence of launches a step of the solve was twelve of them (63 us at D = 64, of which the
// products are 2.6 us): all of it launch and memory latency.  Here a workgroup owns one 16 x 16 tile of
// every vector, one element per thread, and the workgroups of an equation exchange tiles as the
// trajectory kernel does (exchange.h).  A step is eight exchanges: each two-sided product A X B is two
// levels (X B published, then A (X B)), three of them (two for the no-jump inverse, one for L), then
// the two passes of classical Gram-Schmidt as all-workgroup sums.  The rank-one terms of the
// preconditioner and of the pin fold into one matrix M: op(pre(y)) = -L u + i sig u + tr(phi u) M
// with u = N y, so that they need one sum, whose records travel beside the P tiles of L.  The second
// pass sums <w, w> beside its coefficients: |w - V h|^2 = <w, w> - |h|^2 (V orthonormal, h of the size
// of the rounding of the first pass), which spares a third sum.  Every workgroup runs the rotations
// and the triangular solve on the same numbers, behind the publish of the next vector.
//
// A ring of 16 matrix slots: at most 7 events between two sums, so at event e every reader is done
// with event e - 8, which is emptied then and next used at e + 8.  With one tile (Dp = 16) nothing is
// exchanged: the tiles stay in LDS and a launch may hold any number of equations.  Otherwise the
// launch is cooperative.  Waits are bounded in wall time.
//
// The basis stays in registers (one element of 40 vectors per thread: 160 of the 512 a wave has with one
// workgroup per CU), the inner products of eight vectors are summed together by halving, and the
// rotations run with one rotation per lane: with the basis in memory, a sum tree per vector and the
// rotations in one lane, a step took 33% longer at D = 5 to 16 and 10% longer at D = 64.
//
// Measured on MI355X, a boundary solve as the caller sees it: D = 5 (17 steps) 246 us, as launches
// 1083; D = 16 (42) 680; D = 32 (48) 1190; D = 64 (54) 1570, as launches 2800.  At D = 64 a step is
// 26 us: 13 for the three two-sided products, 10 for the Gram-Schmidt passes and their sums, 2 for the
// rotations; all of it latency of the exchanges and of LDS, the matrix cores are busy for 2.6 us.
#include "device_common.h"
#include "exchange.h"
#include "gmres.h"

namespace {

constexpr int RC_M = RC_GMRES_MAX_M;
constexpr int RC_WW = RC_M;          // index of <w, w> among the values of a sum
constexpr int RC_ROWS = RC_M + 1;    // complex values of a sum
static_assert(RC_M % 8 == 0 && RC_ROWS <= 64, "groups of eight inner products, one lane per value");

__device__ __forceinline__ cplx cdiv(cplx a, cplx b) {
    const double m = fma(b.re, b.re, b.im * b.im);
    return cmake(fma(a.re, b.re, a.im * b.im) / m, fma(a.im, b.re, -(a.re * b.im)) / m);
}
// a + b c
__device__ __forceinline__ cplx caxpy(cplx b, cplx c, cplx a) {
    return cmake(fma(b.re, c.re, fma(-b.im, c.im, a.re)), fma(b.re, c.im, fma(b.im, c.re, a.im)));
}
__device__ __forceinline__ cplx cneg(cplx a) { return cmake(-a.re, -a.im); }

struct GmresLds {
    cplx red[2][1024];                                        // partial tiles, alternating
    cplx tile[16 * 17];                                       // the exchanged tile itself (Dp = 16)
    cplx H[RC_M][RC_M];                                       // column k of the triangular factor: H[k]
    cplx y[RC_M];
    cplx h[2][RC_ROWS];                                       // sums of the two Gram-Schmidt passes
    cplx rows[16][RC_ROWS];                                   // row sums of the 16 rows of lanes
    double hn;
    int bad, flag;
};

}  // namespace

template <int NB>
__global__ void __launch_bounds__(256, 1) rc_gmres(RcGmresProb one, const RcGmresProb* __restrict__ many,
                                                   uint32_t* abort_flag, long long wait_ticks) {
    extern __shared__ __align__(16) unsigned char gmres_lds[];
    GmresLds& s = *reinterpret_cast<GmresLds*>(gmres_lds);
    constexpr int Dp = 16 * NB, NT = NB * NB;
    constexpr uint32_t TB = 4096, MB = NT * TB;
    const RcGmresProb P = many ? load_scalar<RcGmresProb>(many, blockIdx.x / NT) : one;
    const int wg = blockIdx.x % NT, bi = wg / NB, bj = wg % NB;
    const int tid = threadIdx.x, lane = tid & 63, wave = uni(tid >> 6);
    const int ei = tid >> 4, ej = tid & 15, fi = lane & 15, fk = 4 * wave + (lane >> 4);
    const int row = 16 * bi + ei, col = 16 * bj + ej;
    const bool real_el = row < P.D && col < P.D;
    const Ctl ctl{abort_flag, wait_ticks};
    const size_t el = (size_t)row * Dp + col;
    if (tid == 0) s.bad = 0;

    // constant panels: fragments of row block bi (left factors) and column block bj (right factors)
    cplx a1[NB], b1[NB], a2[NB], b2[NB], c1[NB], c2[NB], c3[NB], c4[NB];
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
        rows(a1, P.A1); cols(b1, P.B1); rows(a2, P.A2); cols(b2, P.B2);
        rows(c1, P.C1); cols(c2, P.C2); cols(c3, P.C3); rows(c4, P.C4);
    }
    cplx sinv = cmake(0, 0);   // this element of S
    if (real_el) {
        const cplx* l = reinterpret_cast<const cplx*>(P.lam);
        cplx den = P.adjoint ? cadd(cconj(l[row]), l[col]) : cadd(l[row], cconj(l[col]));
        den.re -= P.s_re;
        den.im -= P.s_im;
        sinv = cdiv(cmake(-1, 0), den);
    }
    const cplx phi_t = reinterpret_cast<const cplx*>(P.phi)[(size_t)col * Dp + row];   // tr(phi u) = sum phi_ji u_ij
    const cplx psi = reinterpret_cast<const cplx*>(P.psi)[el];
    cplx b = reinterpret_cast<const cplx*>(P.a)[el];
    __syncthreads();

    // ---- exchange of tiles: copy A (read as row blocks) column by column, copy B row by row
    const __amdgpu_buffer_rsrc_t rX = rc_rsrc(P.exch, (uint32_t)rc_gmres_exch_bytes(NB));
    const uint32_t my_tile = (uint32_t)wg * TB;
    const uint32_t a_el = my_tile + (uint32_t)(ej * 16 + ei) * 16, b_el = my_tile + (uint32_t)tid * 16;
    const uint32_t f_row = (uint32_t)(bi * NB) * TB + (uint32_t)tid * 16, f_col = (uint32_t)bj * TB + (uint32_t)tid * 16;
    constexpr uint32_t oRec = RC_GMRES_RING * MB;
    uint32_t ev = 0, nrec = 0;
    bool ok = true;
    auto publish = [&](cplx v, bool copy_a) -> uint32_t {   // the slot's offset
        if constexpr (NB == 1) {
            s.tile[ei * 17 + ej] = v;
            return 0;
        } else {
            ++ev;
            const uint32_t so = (ev & (RC_GMRES_RING - 1)) * MB;
            rc_put(rX, copy_a ? a_el : b_el, so, v);
            // the slot of event ev - 8: its whole tile, whichever order it was written in
            if (ev > RC_GMRES_RING / 2) rc_reset(rX, b_el, ((ev - RC_GMRES_RING / 2) & (RC_GMRES_RING - 1)) * MB);
            return so;
        }
    };
    auto read_row = [&](cplx* f, uint32_t so) {
        if constexpr (NB == 1) {
            f[0] = s.tile[fi * 17 + fk];
        } else {
            rc_fetch<NB>(rX, f_row, so, TB, f);
            ok = rc_await<NB>(ctl, rX, f_row, so, TB, f) && ok;
        }
    };
    auto read_col = [&](cplx* f, uint32_t so) {
        if constexpr (NB == 1) {
            f[0] = s.tile[fk * 17 + fi];
        } else {
            rc_fetch<NB>(rX, f_col, so, NB * TB, f);
            ok = rc_await<NB>(ctl, rX, f_col, so, NB * TB, f) && ok;
        }
    };
    int rb = 0;   // partial buffer of the next product
    auto reduced = [&](const cacc& acc) -> cplx {
        put_partial(acc, s.red[rb], wave, lane);
        lds_barrier();
        const cplx v = sum_partial(s.red[rb]);
        rb ^= 1;
        return v;
    };
    auto product = [&](const cplx* A, const cplx* B) -> cplx {
        cacc acc;
        cacc_zero(acc);
        frag_product<NB>(acc, A, B);
        return reduced(acc);
    };
    // this element of A X B
    auto two_sided = [&](const cplx* A, cplx x, const cplx* B) -> cplx {
        cplx f[NB];
        uint32_t so = publish(x, true);
        if (NB == 1) lds_barrier();
        read_row(f, so);
        const cplx t = product(f, B);
        so = publish(t, false);
        if (NB == 1) lds_barrier();
        read_col(f, so);
        return product(A, f);
    };
    auto nojump = [&](cplx x) -> cplx { return two_sided(a2, cmul(two_sided(a1, x, b1), sinv), b2); };

    // ---- sums over all threads of the equation: sum_post after a barrier that follows the row sums,
    // sum_take into h (LDS) ending with a barrier; sum = both with the barrier before
    auto row_put = [&](int j, cplx p) {
        p.re = row_sum(p.re);
        p.im = row_sum(p.im);
        if ((lane & 15) == 0) s.rows[4 * wave + (lane >> 4)][j] = p;
    };
    cplx posted = cmake(0, 0);
    // the values of a sum: the first n and, with ww, <w, w>; lane j of wave 0 holds value j
    auto sum_post = [&](int n, bool ww) {
        if (wave != 0) return;
        const bool on = lane < n || (ww && lane == RC_WW);
        ++nrec;
        posted = cmake(0, 0);
        if (on) {
            posted = s.rows[0][lane];
#pragma unroll
            for (int r = 1; r < 16; ++r) posted = cadd(posted, s.rows[r][lane]);
        }
        if constexpr (NB > 1) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the record slot emptied before the last one is empty
            const uint32_t off = (uint32_t)(wg * RC_GMRES_REC + lane) * 16;
            if (on) rc_put(rX, off, oRec + (nrec & 3) * NT * RC_GMRES_REC * 16, posted);
            // the record before the last: every workgroup posted the last one after taking it
            rc_reset(rX, off, oRec + ((nrec + 2) & 3) * NT * RC_GMRES_REC * 16);
        }
    };
    auto sum_take = [&](int n, bool ww, cplx* h) {
        if (wave == 0) {
            const bool on = lane < n || (ww && lane == RC_WW);
            if constexpr (NB > 1) {
                cplx v[NT];
                const uint32_t so = oRec + (nrec & 3) * NT * RC_GMRES_REC * 16;
                rc_fetch<NT>(rX, (uint32_t)lane * 16, so, RC_GMRES_REC * 16, v, on);
                ok = rc_await<NT>(ctl, rX, (uint32_t)lane * 16, so, RC_GMRES_REC * 16, v, on) && ok;
                posted = v[0];
#pragma unroll
                for (int t = 1; t < NT; ++t) posted = cadd(posted, v[t]);
            }
            if (on) h[lane] = posted;
        }
        lds_barrier();
    };
    auto sum = [&](int n, bool ww, cplx* h) {
        if constexpr (NB > 1) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // every slot emptied so far is empty
        lds_barrier();
        sum_post(n, ww);
        sum_take(n, ww, h);
    };
    auto sum1 = [&](cplx p) -> cplx {
        row_put(0, p);
        sum(1, false, s.h[0]);
        const cplx v = s.h[0][0];
        lds_barrier();   // the sum's place is free again
        return v;
    };
    auto norm2 = [](cplx p) { return cmake(fma(p.re, p.re, p.im * p.im), 0.0); };
    auto dnorm = [](double v) { return isnan(v) ? v : sqrt(fmax(0.0, v)); };

    // -L u + i sig u; when `t` is given, t = tr(phi u) summed beside
    auto lin = [&](cplx u, cplx* t) -> cplx {
        cplx r[NB], c[NB], p[NB];
        if (t) row_put(0, cmul(phi_t, u));
        const uint32_t sa = publish(u, true);
        const uint32_t sb = NB == 1 ? 0 : publish(u, false);
        if constexpr (NB == 1) {
            lds_barrier();
            read_row(r, sa);
            read_col(c, sb);
        } else {
            const RcWant<NB> wr{f_row, sa, TB, r, true, true}, wc{f_col, sb, NB * TB, c, true, true};
            wr.fetch(rX);
            wc.fetch(rX);
            ok = rc_await_all(ctl, rX, wr, wc) && ok;
        }
        const cplx q = product(r, c3);
        if (t) sum_post(1, false);
        const uint32_t sp = publish(q, false);
        cacc acc;
        cacc_zero(acc);
        frag_product<NB>(acc, c1, c);
        frag_product<NB>(acc, r, c2);
        if (NB == 1) lds_barrier();
        read_col(p, sp);
        frag_product<NB>(acc, c4, p);
        const cplx v = reduced(acc);
        if (t) {
            sum_take(1, false, s.h[0]);
            *t = s.h[0][0];
        }
        return cmake(fma(-P.sig, u.im, -v.re), fma(P.sig, u.re, -v.im));
    };
    // one uniform decision from wave 0's lane 0
    auto decide = [&](int f) -> int {
        if (!ok) s.bad = 1;
        lds_barrier();
        if (tid == 0) s.flag = s.bad ? 2 : f;
        lds_barrier();
        return uni(s.flag);
    };

    // ---- right-hand side, preconditioner's rank-one term, M
    if (P.project_b) b = caxpy(cneg(sum1(cmul(phi_t, b))), psi, b);
    const double nb = dnorm(sum1(norm2(b)).re);
    const cplx z = nojump(psi);
    const cplx tz = sum1(cmul(phi_t, z));
    const cplx k1 = cdiv(cmake(P.ds, 0), cmake(fma(P.ds, tz.re, 1.0), P.ds * tz.im));   // c1
    const cplx lz = lin(z, nullptr);
    // M = -c1 (-L Z + i sig Z) + c2 (1 - c1 tr(phi Z)) psi
    const cplx f1 = caxpy(cneg(k1), tz, cmake(1, 0));
    const cplx M = caxpy(cneg(k1), lz, cmul(cscale(P.c2, f1), psi));
    (void)sum1(norm2(M));   // a sum between Z's seven events and the first step's
    const double tol_abs = P.tol * fmax(1.0, nb);
    // The Krylov basis: this thread's element of every vector, in registers (from memory, the four
    // passes over the basis cost a step 8 us of load latency).  Indices are static, groups of eight.
    cplx V[RC_M];
#pragma unroll
    for (int j = 0; j < RC_M; ++j) V[j] = cmake(0, 0);
    auto set_V = [&](int i, cplx v) {   // selects, not branches: those become one store at a computed index
#pragma unroll
        for (int j = 0; j < RC_M; ++j) {
            V[j].re = i == j ? v.re : V[j].re;
            V[j].im = i == j ? v.im : V[j].im;
        }
    };
    // wave 0, lane l: rotation l, the right-hand side's entry l
    double cs = 1.0;
    cplx sn = cmake(0, 0), gl = cmake(0, 0);
    auto bcast = [&](cplx v, int l) { return cmake(read_lane(v.re, l), read_lane(v.im, l)); };

    // ---- restarted GMRES on op(pre(y)) = b from y = 0
    cplx x = cmake(0, 0), r = b;
    double beta = nb, beta_prev = INFINITY;
    int matvecs = 1, status = 0;
    bool converged = false;
    for (int outer = 0; outer < P.maxiter && !converged; ++outer) {
        if (beta <= tol_abs) { converged = true; break; }
        if (!(beta <= 0.9 * beta_prev)) break;   // a restart cycle that gains under 10%: stagnation
        beta_prev = beta;
        cplx v = cscale(1.0 / beta, r);
        set_V(0, v);
        gl = cmake(lane == 0 ? beta : 0.0, 0);
        int kk = 0;
        for (int k = 0;; ++k) {
            // w = op(pre(v))
            const cplx u = nojump(v);
            cplx t;
            cplx w = lin(u, &t);
            w = caxpy(t, M, w);
            ++matvecs;
            // classical Gram-Schmidt twice
#pragma unroll 1
            for (int pass = 0; pass < 2; ++pass) {
#pragma unroll
                for (int g = 0; g < RC_M / 8; ++g) {
                    if (8 * g > k) continue;
                    double p[16];
#pragma unroll
                    for (int j = 0; j < 8; ++j) {
                        const cplx q = V[8 * g + j];
                        p[2 * j] = fma(q.re, w.re, q.im * w.im);
                        p[2 * j + 1] = fma(q.re, w.im, -(q.im * w.re));
                    }
                    const double r16 = row_sums16(p, lane);
                    reinterpret_cast<double*>(&s.rows[4 * wave + (lane >> 4)][8 * g])[lane & 15] = r16;
                }
                if (pass) row_put(RC_WW, norm2(w));
                cplx* h = s.h[pass];
                sum(k + 1, pass != 0, h);
#pragma unroll
                for (int g = 0; g < RC_M / 8; ++g) {
                    if (8 * g > k) continue;
                    cplx hq[8];
#pragma unroll
                    for (int j = 0; j < 8; ++j) hq[j] = 8 * g + j <= k ? h[8 * g + j] : cmake(0, 0);
#pragma unroll
                    for (int j = 0; j < 8; ++j) w = caxpy(cneg(hq[j]), V[8 * g + j], w);
                }
            }
            if (wave == 0) {
                const double hh = lane <= k ? norm2(s.h[1][lane]).re : 0.0;
                const double nn = s.h[1][RC_WW].re - wave_sum(hh);
                if (lane == 0) s.hn = dnorm(nn);
            }
            lds_barrier();
            const double hn = s.hn;
            v = cscale(hn > 0.0 ? 1.0 / hn : 0.0, w);
            if (k + 1 < P.m) set_V(k + 1, v);
            // rotations of the new column (wave 0, one rotation per lane), and the verdict
            int f = 0;
            if (wave == 0) {
                const cplx hl = lane <= k ? cadd(s.h[0][lane], s.h[1][lane]) : cmake(0, 0);
                cplx cur = bcast(hl, 0);
                for (int i = 0; i < k; ++i) {
                    const cplx nx = bcast(hl, i + 1), si = bcast(sn, i);
                    const double ci = read_lane(cs, i);
                    const cplx hi = caxpy(si, nx, cscale(ci, cur));
                    if (lane == 0) s.H[k][i] = hi;
                    cur = caxpy(cneg(cconj(si)), cur, cscale(ci, nx));
                }
                const double ax = hypot(cur.re, cur.im), ay = hn;
                double c = 0;
                cplx sk = cmake(1, 0);
                if (ay == 0) {
                    c = 1;
                    sk = cmake(0, 0);
                } else if (ax != 0) {
                    const double rr = hypot(ax, ay);
                    c = ax / rr;
                    sk = cscale(ay / rr, cmake(cur.re / ax, cur.im / ax));
                }
                if (lane == k) {
                    cs = c;
                    sn = sk;
                }
                if (lane == 0) s.H[k][k] = caxpy(sk, cmake(hn, 0), cscale(c, cur));
                const cplx gk = bcast(gl, k), gn = cneg(cmul(cconj(sk), gk));
                if (lane == k) gl = cscale(c, gk);
                if (lane == k + 1) gl = gn;
                const double res = hypot(gn.re, gn.im);
                f = (res <= tol_abs || hn == 0 || k + 1 >= P.m || !isfinite(res)) ? 1 : 0;
            }
            kk = k + 1;
            const int dec = decide(f);
            if (dec == 2) { status = RC_ST_WAIT_LIMIT; break; }
            if (dec) break;
        }
        if (status) break;
        // y from the triangular system: lane l keeps g_l, the columns from the last one on
        if (wave == 0) {
            for (int i = kk - 1; i >= 0; --i) {
                const cplx yi = bcast(cdiv(gl, s.H[i][i]), i);
                if (lane == 0) s.y[i] = yi;
                if (lane < i) gl = caxpy(cneg(yi), s.H[i][lane], gl);
            }
        }
        lds_barrier();
#pragma unroll
        for (int g = 0; g < RC_M / 8; ++g) {
            if (8 * g >= kk) continue;
#pragma unroll
            for (int j = 0; j < 8; ++j)
                if (8 * g + j < kk) x = caxpy(s.y[8 * g + j], V[8 * g + j], x);
        }
        // true residual of the preconditioned system
        const cplx u = nojump(x);
        cplx t;
        const cplx w = lin(u, &t);
        r = csub(b, caxpy(t, M, w));
        ++matvecs;
        beta = dnorm(sum1(norm2(r)).re);
        if (beta <= tol_abs) converged = true;
        if (!isfinite(beta)) break;
    }
    // ---- the solution, its projection and the residual of the physical equation
    double true_res = 0.0;
    if (!status) {
        const cplx u = nojump(x);
        cplx h = caxpy(cneg(cmul(k1, sum1(cmul(phi_t, u)))), z, u);
        if (P.project_x) h = caxpy(cneg(sum1(cmul(phi_t, h))), psi, h);
        cplx t;
        cplx w = lin(h, &t);
        if (P.pin) w = caxpy(cscale(P.c2, t), psi, w);
        true_res = dnorm(sum1(norm2(csub(w, b))).re);
        reinterpret_cast<cplx*>(P.x)[el] = real_el ? h : cmake(0, 0);
        if (decide(0) == 2) status = RC_ST_WAIT_LIMIT;
    }
    if (wg == 0 && tid == 0) {
        P.out[0] = status;
        P.out[1] = converged ? 1.0 : 0.0;
        P.out[2] = matvecs;
        P.out[3] = beta;
        P.out[4] = nb;
        P.out[5] = true_res;
    }
}

static const void* gmres_fn(int nb) {
    switch (nb) {
        case 1: return (const void*)rc_gmres<1>;
        case 2: return (const void*)rc_gmres<2>;
        case 3: return (const void*)rc_gmres<3>;
        case 4: return (const void*)rc_gmres<4>;
        default: return nullptr;
    }
}

hipError_t rc_gmres_capacity(int nb, int* probs) {
    const void* fn = gmres_fn(nb);
    *probs = 0;
    if (!fn) return hipSuccess;
    hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)sizeof(GmresLds));
    if (e != hipSuccess) return e;
    if (nb == 1) {   // no workgroup waits for another
        *probs = 1 << 16;
        return hipSuccess;
    }
    int per_cu = 0, dev = 0, cus = 0, coop = 0;
    if ((e = hipGetDevice(&dev)) != hipSuccess) return e;
    if ((e = hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, dev)) != hipSuccess) return e;
    if ((e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, 256, sizeof(GmresLds))) != hipSuccess) return e;
    if ((e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev)) != hipSuccess) return e;
    *probs = coop ? per_cu * cus / (nb * nb) : 0;
    return hipSuccess;
}

hipError_t rc_launch_gmres(int nb, int n, const RcGmresProb& one, const RcGmresProb* many, uint32_t* abort_flag,
                           long long wait_ticks, hipStream_t stream) {
    const void* fn = gmres_fn(nb);
    if (!fn || (n > 1 && !many)) return hipErrorInvalidValue;
    RcGmresProb p = one;
    if (n == 1) many = nullptr;
    void* args[] = {(void*)&p, (void*)&many, (void*)&abort_flag, (void*)&wait_ticks};
    if (nb == 1) return hipLaunchKernel(fn, dim3(n), dim3(256), args, sizeof(GmresLds), stream);
    return hipLaunchCooperativeKernel(fn, dim3(n * nb * nb), dim3(256), args, sizeof(GmresLds), stream);
}
