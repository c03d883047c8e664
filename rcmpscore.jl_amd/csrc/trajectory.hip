// Persistent dataflow DOP853 for the six reduced transfer-ODE systems of fg_phi4
// (kinetic, kinetic commutator, phi^4) x (forward, adjoint), FP64 on MFMA.
//
// Equations (reduced channels of src/observables.jl:37-63; Lindblad maps src/transfer.jl:2-19):
//   forward  k(X) = jac(t) [Q X + X Q^+ + (R X) R^+] + s(t) [insertions + fixed]
//   adjoint  k(X) = jac(t) [Q^+ X + X Q + R^+ (X R)] + s(t) [insertions + fixed]
// with jac = 2|t| and s(t) = 2|t| J(t^2).  Integrator and controller: adaptive DOP853 with the
// error norm h e5 / sqrt((e5 + 0.01 e3) N), factor min(10, 0.9 err^-1/8), rejection factor
// max(0.2, .), no step across t = 0, 7th-order dense output at the Gauss nodes, as the reference
// GPU package (gpu/src/rcmps_gpu/optimizer/runtime/ode_backend.py:500-586,
// device_control_backend.py:30-47).  The FSAL stage counts as evaluated only after acceptance.
//
// Work decomposition: one workgroup per (system, live channel, 16x16 output tile), plus, for the
// kinetic commutator's adjoint system, one E task per tile forming E = X [Q,R] of channel 1, which
// channel 0's insertion reads (so no channel forms two level-1 products).  A stage is
// two levels: level 1 forms the tile of P = R X (forward) or X R (adjoint) and publishes it;
// level 2 forms Q X + X Q^+ (resp. Q^+ X + X Q) while neighbours' P tiles arrive, then adds
// P R^+ (resp. R^+ P), the insertion terms and the next stage input.
//
// Exchange between workgroups: the data are their own arrival flags.  Every stage input Y, level-1
// tile P, E tile and error record goes into a ring of slots whose words hold a NaN pattern no
// computation produces (RC_EMPTY_WORD) until the value is stored; a consumer loads the elements it needs
// with device-coherent loads straight into its MFMA fragments and repeats those that are still
// empty.  An exchange is then one store and one load of device scope, with no wait for the store's
// completion, no flag and no barrier of the workgroup; the products were a third of a stage and
// these round trips most of the rest.  Ring of RC_RING events: an attempt's error records are posted
// after stage 11 and taken within the next event (the FSAL stage), so between two takes lie at most
// 16 events from post to take (stages 12..15 and 1..11, and the FSAL stage again).  At event e every
// reader is done with event e - 16, whose slot the producer empties again; the slot is used next at
// event e + 16, and a post lies between, before which the producer waited for its stores.
// The gather is deterministic (every workgroup adds the same records in the same order), so every
// workgroup of a system takes the same controller decision.  Every wait is bounded by a time
// budget and watches an abort word; a workgroup whose wait failed leaves a mark in its system's results
// (rc_system_status), which the host takes before the status.
//
// Places: the launch lays a system on one XCD where it fits, and a channel's tiles are then kept in
// that XCD's L2 (rc_put).  At D = 64 that is 10% of a stage of a system of one or two channels; the
// longest systems span two XCDs and gain 4%, at D = 32 to 48 it is within the noise, at D = 8 (only
// insertions are exchanged) 9%.
//
// FP64 products read no LDS: each wave runs one k-step of every k-tile, so the operands of its
// products are fragments it alone needs, loaded from the exchange buffers into registers (the
// constant panels R, Q, .. once per task).  LDS holds only the four waves' partial tiles, in one
// buffer per level, which leaves two barriers per stage.  Split precision stages digit planes in
// LDS (every wave needs every row of a panel's digits).  With one tile per channel (Dp = 16) the
// stage input and P stay in LDS and only what another channel reads is exchanged.
//
// What bounds it: a chain of two exchanges, 1.7 us of matrix instructions (64 a wave, 64 cycles each) and
// two sums of partial tiles per stage at D = 64, and the wave's own instructions: a check of the arrived
// words by one running maximum instead of two compares an element is worth 5% of a stage, running sums
// of the combinations ahead instead of a window of derivatives, the wide gather of records and the FSAL
// stage ahead of the verdict another 5%.  Measured on MI355X, the launch's time over the right-hand sides of the
// system that has most of them, against one flag per tile, a wait for the store and LDS panels, in one run:
// D = 8 6.1 -> 2.7 us, D = 32 with Z2 blocks 7.1 -> 3.0, D = 40 9.0 -> 4.2, D = 64 9.2 -> 4.5 (split 9.3 ->
// 5.8); six trajectories at D = 64, window 30, 1e-13/1e-12: 60.6 -> 29.8 ms.
#include "device_common.h"
#include "exchange.h"
#include "split.h"
#include "trajectory.h"

namespace {

template <int NB>
struct Lay {
    static constexpr int Dp = 16 * NB;
    // partial tiles of the two levels, then (Dp = 16 only) the stage input and P tiles, rows of 17
    static constexpr int RED1 = 0, RED2 = 1024, YT = 2048, PT = YT + 16 * 17;
    static constexpr int NCPLX = NB == 1 ? PT + 16 * 17 : 2048;
    static constexpr int NDOUBLE_SCRATCH = 64;
    static constexpr int BYTES = NCPLX * 16 + NDOUBLE_SCRATCH * 8;
};

// ---------------------------------------------------------------------------------------
// split precision: LDS layout, panel loads into digit planes, wave-split real products
// ---------------------------------------------------------------------------------------
struct LaySplit {
    static constexpr int P = RC_PANEL_BYTES;
    static constexpr int XR = 0, XC = P, PB = 2 * P, K0 = 3 * P, K1 = 4 * P, K2 = 5 * P, K3 = 6 * P;
    static constexpr int RED = 7 * P;                  // two levels of 4 x 256 doubles
    static constexpr int SCR = RED + 2 * 4 * 256 * 8;  // 64 doubles
    static constexpr int BYTES = SCR + 64 * 8;
};

__device__ __forceinline__ double wave_max(double v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = fmax(v, __shfl_xor(v, off));
    return v;
}

__device__ __forceinline__ double max4(const cplx* v) {
    double m = 0.0;
#pragma unroll
    for (int q = 0; q < 4; ++q) m = fmax(m, fmax(fabs(v[q].re), fabs(v[q].im)));
    return m;
}

// Block maxima of N panels (one value per thread each) -> uniform panel scales S[n].
template <int N>
__device__ __forceinline__ void block_scales(const double* m, int* S, double* scr) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int n = 0; n < N; ++n) {
        const double v = wave_max(m[n]);
        if (lane == 0) scr[8 + 4 * n + wave] = v;
    }
    __syncthreads();
#pragma unroll
    for (int n = 0; n < N; ++n) {
        const double* q = scr + 8 + 4 * n;
        S[n] = uni(rc_split_scale(fmax(fmax(q[0], q[1]), fmax(q[2], q[3]))));
    }
}

// Thread t holds four consecutive k of one row (row t / 16, k = 4 (t % 16) + q) of a row block,
// or of one column (column t / 16, k = 4 (t % 16) + q) of a column block; zero beyond Dp.  The 16
// lanes of one row or column are consecutive, so its largest entry is a 16-lane reduction.
template <int NB>
__device__ __forceinline__ void fetch_row4(cplx* v, const double* g, int b) {
    constexpr int Dp = 16 * NB;
    const int t = threadIdx.x, i = t >> 4, k0 = 4 * (t & 15);
    const cplx* gc = reinterpret_cast<const cplx*>(g);
#pragma unroll
    for (int q = 0; q < 4; ++q) v[q] = k0 < Dp ? gc[(16 * b + i) * Dp + k0 + q] : cmake(0, 0);
}
template <int NB>
__device__ __forceinline__ void fetch_col4(cplx* v, const double* g, int c) {
    constexpr int Dp = 16 * NB;
    const int t = threadIdx.x, j = t >> 4, k0 = 4 * (t & 15);
    const cplx* gc = reinterpret_cast<const cplx*>(g);
#pragma unroll
    for (int q = 0; q < 4; ++q) v[q] = k0 < Dp ? gc[(k0 + q) * Dp + 16 * c + j] : cmake(0, 0);
}
template <int NB>
__device__ __forceinline__ void store_row4(unsigned char* panel, const cplx* v, int S) {
    const int t = threadIdx.x, k0 = 4 * (t & 15);
    if (k0 < 16 * NB) rc_store_digits4(panel, t >> 4, k0, v, ldexp(1.0, S));
}
template <int NB>
__device__ __forceinline__ void store_col4(unsigned char* panel, const cplx* v, int S) {
    const int t = threadIdx.x, k0 = 4 * (t & 15);
    if (k0 < 16 * NB) rc_store_digits4(panel, t >> 4, k0, v, ldexp(1.0, S));
}

// biased FP64 exponent of the largest |re|, |im| of v[0..3] (0 for zeros and subnormals)
__device__ __forceinline__ int max_exp4(const cplx* v) {
    int e = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        e = max(e, (int)((uint32_t)__double2hiint(v[q].re) >> 20) & 0x7ff);
        e = max(e, (int)((uint32_t)__double2hiint(v[q].im) >> 20) & 0x7ff);
    }
    return e;
}
// scale of this thread's row (or column) of a row (column) block: the maximum over its 16 lanes.
// The lane holding k = 0 writes it to sg[row or column].
__device__ __forceinline__ int line_scale(const cplx* v, int* sg) {
    int e = max_exp4(v);
    // 16-lane maximum by DPP moves within each row of 16 lanes: quad_perm [1,0,3,2] and [2,3,0,1]
    // give the quad's maximum, row_half_mirror joins quads 0-1 and 2-3, row_mirror the two halves
    e = max(e, __builtin_amdgcn_update_dpp(0, e, 0xB1, 0xF, 0xF, false));
    e = max(e, __builtin_amdgcn_update_dpp(0, e, 0x4E, 0xF, 0xF, false));
    e = max(e, __builtin_amdgcn_update_dpp(0, e, 0x141, 0xF, 0xF, false));
    e = max(e, __builtin_amdgcn_update_dpp(0, e, 0x140, 0xF, 0xF, false));
    const int S = rc_split_scale_e(e);
    if ((threadIdx.x & 15) == 0) sg[threadIdx.x >> 4] = S;
    return S;
}

// one constant panel (row block b or column block c of a fixed matrix) at kernel start
template <int NB>
__device__ __forceinline__ int const_panel(unsigned char* panel, const double* g, bool row, int blk, double* scr) {
    cplx v[4];
    if (row) fetch_row4<NB>(v, g, blk);
    else fetch_col4<NB>(v, g, blk);
    const double m = max4(v);
    int S;
    block_scales<1>(&m, &S, scr);
    if (row) store_row4<NB>(panel, v, S);
    else store_col4<NB>(panel, v, S);
    __syncthreads();
    return S;
}

// Waves 0..3 hold the real products re.re, im.im, re.im, im.re of the same complex tile product;
// thread t receives element (t/16, t%16) of the complex result.
__device__ __forceinline__ void put_partial_split(const double* part, double* red, int wave, int lane) {
#pragma unroll
    for (int q = 0; q < 4; ++q) red[wave * 256 + (4 * (lane >> 4) + q) * 16 + (lane & 15)] = part[q];
}
__device__ __forceinline__ cplx sum_partial_split(const double* red) {
    const int t = threadIdx.x;
    return cmake(red[t] - red[256 + t], red[512 + t] + red[768 + t]);
}

// What the derivative of stage s adds to the combinations that still lie ahead of it.  Row s: the
// coefficients of k_s in the next RC_AHEAD combinations after stage s + 1 (the input of stage s + 2 first;
// the one after stage 11 is the solution, the FSAL stage's input), then in the error estimators E5 and
// E3 and the dense output's four rows.
#define RC_AHEAD 14
struct RcRows {
    double c[RC_NSTAGES_EXT][24];
};
constexpr RcRows rc_make_rows() {
    RcRows r{};
    for (int s = 0; s < RC_NSTAGES_EXT - 1; ++s) {
        for (int i = 0; s + 2 + i < RC_NSTAGES_EXT; ++i)
            r.c[s][i] = s + 2 + i == RC_NSTAGES ? (s < RC_NSTAGES ? RC_B[s] : 0.0) : RC_A[s + 2 + i][s];
        if (s < RC_NSTAGES) {
            r.c[s][RC_AHEAD] = RC_E5[s];
            r.c[s][RC_AHEAD + 1] = RC_E3[s];
        }
        for (int q = 0; q < 4; ++q) r.c[s][RC_AHEAD + 2 + q] = RC_D[q][s];
    }
    return r;
}
__constant__ const RcRows rc_rows = rc_make_rows();
// coefficients of the trace's derivatives k_j in the solution and the error estimators
struct RcScalarRows {
    double c[RC_NSTAGES][4];
};
constexpr RcScalarRows rc_make_scalar_rows() {
    RcScalarRows r{};
    for (int j = 0; j < RC_NSTAGES; ++j) {
        r.c[j][0] = RC_B[j];
        r.c[j][1] = RC_E5[j];
        r.c[j][2] = RC_E3[j];
    }
    return r;
}
__constant__ const RcScalarRows rc_scalar_rows = rc_make_scalar_rows();

// The combinations ahead, as running sums in stage order: add(s, k) adds k_s to each and moves them up by
// one, so that a[0] is all but the last term of the combination after the next stage.  A sum's move is
// the destination of its multiply-add: no register array is indexed at run time and nothing is shifted
// (a window of the k_s themselves costs 60 moves a stage for the shift).  The coefficients come through the
// scalar cache.
struct RcAhead {
    cplx a[RC_AHEAD + 1], e5, e3, d[4];
    __device__ __forceinline__ void clear() {
        e5 = e3 = cmake(0, 0);
#pragma unroll
        for (int i = 0; i <= RC_AHEAD; ++i) a[i] = cmake(0, 0);
#pragma unroll
        for (int q = 0; q < 4; ++q) d[q] = cmake(0, 0);
    }
    __device__ __forceinline__ void add(int s, cplx k) {
        const __attribute__((address_space(4))) double* c =
            (const __attribute__((address_space(4))) double*)&rc_rows.c[s][0];
#pragma unroll
        for (int i = 0; i < RC_AHEAD; ++i) a[i] = cfma(c[i], k, a[i + 1]);
        e5 = cfma(c[RC_AHEAD], k, e5);
        e3 = cfma(c[RC_AHEAD + 1], k, e3);
#pragma unroll
        for (int q = 0; q < 4; ++q) d[q] = cfma(c[RC_AHEAD + 2 + q], k, d[q]);
    }
};

// One attempt's records of every workgroup of the system, for wave 0: lane 8 q + i takes pair q of the
// records of tasks i, i + 8, .. (those beyond the last repeat it and count nothing).
struct RcRecords {
    uint32_t so, pair;
    int part, ntasks;
    cplx* v;
    __device__ __forceinline__ void fetch(__amdgpu_buffer_rsrc_t r) const {
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (8 * i < ntasks) v[i] = ld_coh_s(r, (uint32_t)(min(part + 8 * i, ntasks - 1) * RC_REC * 8) + pair, so);
    }
    __device__ __forceinline__ bool late() const {
        uint32_t m = 0;
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (8 * i < ntasks) m = rc_max_word(m, v[i]);
        return __any(m == RC_EMPTY_WORD);
    }
    __device__ __forceinline__ void settle() const {}
    // the pair's sums over the tasks, on each of the pair's eight lanes
    __device__ __forceinline__ cplx sum() const {
        cplx t = cmake(0, 0);
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (8 * i < ntasks && part + 8 * i < ntasks) t = cadd(t, v[i]);
        t = cadd(t, cmake(dpp_move<0xB1>(t.re), dpp_move<0xB1>(t.im)));
        t = cadd(t, cmake(dpp_move<0x4E>(t.re), dpp_move<0x4E>(t.im)));
        return cadd(t, cmake(dpp_move<0x141>(t.re), dpp_move<0x141>(t.im)));
    }
};

}  // namespace

template <int NB, int KT, bool SPLIT, bool TIMED>
__device__ void run_task(const TrajParams& p, int task, unsigned char* smem_raw) {
    using L = Lay<NB>;
    constexpr int Dp = L::Dp;
    constexpr bool LOCAL = NB == 1 && !SPLIT;   // one tile per channel: its stage input and P stay in LDS
    cplx* sm = reinterpret_cast<cplx*>(smem_raw);
    cplx* red1 = sm + L::RED1;
    cplx* red2 = sm + L::RED2;
    cplx* Yt = sm + L::YT;
    cplx* Pt = sm + L::PT;
    // split precision: digit planes of the stage input's row and column block, of the P block and of
    // the constant panels, and the partial real products
    unsigned char* pXr = smem_raw + LaySplit::XR;
    unsigned char* pXc = smem_raw + LaySplit::XC;
    unsigned char* pPb = smem_raw + LaySplit::PB;
    unsigned char* pK1 = smem_raw + LaySplit::K0;
    unsigned char* pKq = smem_raw + LaySplit::K1;
    unsigned char* pKx = smem_raw + LaySplit::K2;
    unsigned char* pKp = smem_raw + LaySplit::K3;
    double* redd1 = reinterpret_cast<double*>(smem_raw + LaySplit::RED);
    double* redd2 = redd1 + 4 * 256;
    double* scratch = SPLIT ? reinterpret_cast<double*>(smem_raw + LaySplit::SCR)
                            : reinterpret_cast<double*>(sm + L::NCPLX);
    __shared__ int s_bad;   // a wait of this attempt failed (read at the step's end only)
    __shared__ int s_loc;   // which of this workgroup's stores stay on the XCD
    __shared__ double s_verdict[4];   // an attempt's error, step factor, scalar solution; whether a wait failed
    __shared__ double s_err[8];
    __shared__ double s_trp[RC_NSTAGES_EXT][4], s_trs[RC_NSTAGES_EXT];   // trace: wave sums, coefficient
    __shared__ double s_src[2][RC_NSTAGES_EXT];                         // source values, by attempt parity
    __shared__ double s_cheb[RC_SOURCE_SEGMENTS * (RC_SOURCE_DEGREE + 1)];
    __shared__ double s_cnode[RC_NSTAGES_EXT], s_alast[RC_NSTAGES_EXT];

    const int tid = threadIdx.x, lane = tid & 63, wave = uni(tid >> 6);
    const int spa = (wave == 1 || wave == 3), spb = (wave == 1 || wave == 2);   // this wave's real product
    const int ei = tid >> 4, ej = tid & 15;
    const TrajTask tk = load_scalar<TrajTask>(p.tasks, task);
    const TrajSys S = load_scalar<TrajSys>(p.sys, tk.sys);
    const int b = tk.b, c = tk.c, ch = tk.ch, adj = tk.adj;
    // k-tile masks of the tile products (uniform): level 1, the two of level 2a, level 2b, E.  KT = NB:
    // every k-tile of every product.  KT = NB / 2 (Z2 states, FP64): a product has the k-tiles of one
    // parity block or none, and a tile either forms level 1 (do1) or level 2 (do2), since the
    // stage input and P = R X have opposite parities.  Split precision skips whole products.
    const int m1 = tk.kmask & 15, m2a = (tk.kmask >> 4) & 15, m2b = (tk.kmask >> 8) & 15,
              m3 = (tk.kmask >> 12) & 15, mE = (tk.kmask >> 16) & 15;
    const bool do1 = (KT == NB && !SPLIT) || m1 != 0, do2 = (KT == NB && !SPLIT) || m2a != 0;
    const bool doE = (KT == NB && !SPLIT) || mE != 0;
    auto first = [](int m) { return KT == NB || m == 0 ? 0 : __builtin_ctz(m); };
    // first k-tile of the column block's and the row block's fragments, and of P's
    const int tc = first(m2a ? m2a : adj ? 0 : m1), tr = first(tk.e_only ? mE : m2b ? m2b : adj ? m1 : 0), tp = first(m3);
    const int row = 16 * b + ei, col = 16 * c + ej;
    const bool e_only = tk.e_only != 0;                  // uniform over the workgroup
    const bool real_el = !e_only && row < S.D && col < S.D;
    const Ctl ctl{p.abort_flag, p.wait_ticks};
    const uint32_t mat_bytes = (uint32_t)(Dp * Dp * 16);
    const uint32_t stage_stride = (uint32_t)S.nlive * mat_bytes;
    // the system's exchange buffers: rings of stage inputs Y (copies A and B), of level-1 tiles P and of
    // E tiles, then the error records
    const __amdgpu_buffer_rsrc_t rX = rc_rsrc(S.exch, S.exch_bytes);
    const uint32_t oB = RC_RING * stage_stride, oP = 2 * oB, oP2 = 3 * oB, oE = 4 * oB, oR = oE + (S.has_E ? RC_RING * mat_bytes : 0);
    const uint32_t el_off = (uint32_t)((row * Dp + col) * 16);
    // The exchange buffers hold whole tiles (tile (r, c) at (r NB + c) TB), each in the order in which
    // its readers' waves take it, so that one load instruction of a wave reads one contiguous 1 KB
    // (split: four of 256 B): copy A for the readers of row blocks (FP64: column by column), copy B
    // for those of column blocks (row by row).  A stage input has both, P the one its readers need.
    // Element (r, c) of a tile at byte at_a / at_b.
    constexpr uint32_t TB = 4096;
    auto at_a = [](int r, int c) { return (uint32_t)((SPLIT ? (c & 3) * 64 + r * 4 + (c >> 2) : c * 16 + r) * 16); };
    auto at_b = [](int r, int c) { return (uint32_t)((SPLIT ? (r & 3) * 64 + c * 4 + (r >> 2) : r * 16 + c) * 16); };
    const uint32_t my_tile = (uint32_t)(b * NB + c) * TB, mirror_tile = (uint32_t)(c * NB + b) * TB;
    const uint32_t ya_off = my_tile + at_a(ei, ej), yb_off = my_tile + at_b(ei, ej);   // own element of Y
    const uint32_t pub_off = adj ? yb_off : ya_off;                                   // and of P
    // own and mirrored element of the insertion source (E is held as copy B)
    const bool ins_b = adj || tk.edge_from_E;
    const uint32_t ins_off = ins_b ? yb_off : ya_off;
    const uint32_t ins_off_t = mirror_tile + (ins_b ? at_b(ej, ei) : at_a(ej, ei));
    // this lane's element of k-tile 0's fragment in row block b and in column block c, and the
    // distance to the next k-tile's; split: this thread's four consecutive k of a row or column
    const int fi = lane & 15, fk = 4 * wave + (lane >> 4);
    const uint32_t in_tile = (uint32_t)(SPLIT ? (ei * 4 + (ej & 3)) * 16 : tid * 16);
    constexpr uint32_t row_step = SPLIT ? 1024 : TB, col_step = SPLIT ? 1024 : NB * TB;
    const uint32_t row_off0 = (uint32_t)(b * NB + (SPLIT ? ej >> 2 : 0)) * TB + in_tile;
    const uint32_t col_off0 = (uint32_t)((SPLIT ? (ej >> 2) * NB : 0) + c) * TB + in_tile;
    const uint32_t row_off = row_off0 + (SPLIT ? 0 : tr * row_step), col_off = col_off0 + (SPLIT ? 0 : tc * col_step);
    const uint32_t p_off = (adj ? col_off0 : row_off0) + (SPLIT ? 0 : tp * (adj ? col_step : row_step));
    const uint32_t p_step = adj ? col_step : row_step;
    constexpr int NF = SPLIT ? 4 : KT;
    // split: the lanes whose k lies in a k-tile that can be nonzero (the others' tiles are never written)
    auto lanes = [&](int m) { return !SPLIT || (((m >> (ej >> 2)) & 1) && 4 * ej < Dp); };
    const bool use_r = lanes(tk.e_only ? mE : m2b | (adj ? m1 : 0)), use_c = lanes(m2a | (adj ? 0 : m1)), use_p = lanes(m3);

    // constant panels: fragments in registers (split: digit planes).  K1 level 1 (R; an E task's C),
    // Kq and Kx the one-sided products, Kp level 2
    cplx K1[KT], Kq[KT], Kx[KT], Kp[KT];
    int sK1 = 0, sKq = 0, sKx = 0, sKp = 0;   // split-precision panel scales
    // per-row / per-column scales of the stage input's row block [0, 16) and column block
    // [16, 32), and of the P block (split precision)
    int* sgX = reinterpret_cast<int*>(scratch + 16);
    int* sgP = sgX + 32;
    if constexpr (SPLIT) {
        // zero every digit plane once: k beyond Dp stays zero
        for (int i = tid; i < 7 * RC_PANEL_BYTES / 16; i += 256) reinterpret_cast<v4i*>(smem_raw)[i] = v4i{0, 0, 0, 0};
        __syncthreads();
        if (e_only) {
            sK1 = const_panel<NB>(pK1, S.C, false, c, scratch);
        } else if (!adj) {
            sK1 = const_panel<NB>(pK1, S.R, true, b, scratch);
            sKq = const_panel<NB>(pKq, S.Q, true, b, scratch);
            sKx = const_panel<NB>(pKx, S.Qh, false, c, scratch);
            sKp = const_panel<NB>(pKp, S.Rh, false, c, scratch);
        } else {
            sK1 = const_panel<NB>(pK1, S.R, false, c, scratch);
            sKq = const_panel<NB>(pKq, S.Qh, true, b, scratch);
            sKx = const_panel<NB>(pKx, S.Q, false, c, scratch);
            sKp = const_panel<NB>(pKp, S.Rh, true, b, scratch);
        }
    } else {
        auto rows = [&](cplx* K, const double* g, int m) {
            const cplx* gc = reinterpret_cast<const cplx*>(g);
#pragma unroll
            for (int t = 0; t < KT; ++t) K[t] = gc[(16 * b + fi) * Dp + 16 * (first(m) + t) + fk];
        };
        auto cols = [&](cplx* K, const double* g, int m) {
            const cplx* gc = reinterpret_cast<const cplx*>(g);
#pragma unroll
            for (int t = 0; t < KT; ++t) K[t] = gc[(16 * (first(m) + t) + fk) * Dp + 16 * c + fi];
        };
        if (!adj) {
            rows(K1, S.R, m1); rows(Kq, S.Q, m2a); cols(Kx, S.Qh, m2b); cols(Kp, S.Rh, m3);
        } else {
            cols(K1, e_only ? S.C : S.R, e_only ? mE : m1); rows(Kq, S.Qh, m2a); cols(Kx, S.Q, m2b); rows(Kp, S.Rh, m3);
        }
    }
    cplx fixed_e = cmake(0, 0), trop_e = cmake(0, 0);
    if (tk.fixed) fixed_e = reinterpret_cast<const cplx*>(tk.fixed)[row * Dp + col];
    if (tk.trace_kind == 1) trop_e = reinterpret_cast<const cplx*>(tk.trace_op)[row * Dp + col];
    for (int i = tid; i < RC_SOURCE_SEGMENTS * (RC_SOURCE_DEGREE + 1); i += 256) s_cheb[i] = p.cheb[i];
    if (tid < RC_NSTAGES_EXT) {
        s_cnode[tid] = RC_C[tid];
        // coefficient of the newest derivative k_s in the stage input after stage s
        s_alast[tid] = tid == RC_NSTAGES - 1 ? RC_B[tid] : tid + 1 < RC_NSTAGES_EXT ? RC_A[tid + 1][tid] : 0.0;
    }
    if (tid == 0) {
        s_bad = 0;
        s_verdict[3] = 0.0;
    }
    __syncthreads();

    // phase timers (constant-rate clock ticks): wait for the stage input, (split) slice it, level 1 +
    // publish P, level 2a, wait for P, (split) slice it, level 2b + epilogue, integrator bookkeeping,
    // step end (error norm, record, all-gather), total, publish Y.
    // The timers are an instantiation of their own (TIMED): each reading of the clock waits for the
    // scalar memory counter and the sums take registers, which the untimed kernel does not pay.
    uint64_t tacc[RC_NTIMERS];
#pragma unroll
    for (int q = 0; q < RC_NTIMERS; ++q) tacc[q] = 0;
    uint64_t tmark = TIMED ? __builtin_amdgcn_s_memrealtime() : 0;
    const uint64_t tstart = tmark;
    auto lap = [&](int q) {
        if constexpr (TIMED) {
            uint64_t now = __builtin_amdgcn_s_memrealtime();
            tacc[q] += now - tmark;
            tmark = now;
        }
    };

    // ------------------------------------------------------------------------------------
    // integrator state.  All of a combination (next stage input, solution, error estimators) but its last
    // term is summed while the stages before it wait for their neighbours, so one multiply-add stands
    // between a stage's derivative and the next stage input.
    // ------------------------------------------------------------------------------------
    const double a = p.a;
    RcAhead ahead;
    ahead.clear();
    cplx y = cmake(0, 0), ynew = cmake(0, 0), k0 = cmake(0, 0), k12 = cmake(0, 0);
    double ysc = 0.0, ysc_new = 0.0;
    double t = -a, h = fmin(p.h0, 2.0 * a), t_new = t, endpoint = 0.0, factor = 1.0;
    uint32_t ev = 0;
    uint32_t attempts = 0, accepted = 0, rejected = 0, dense = 0, rhs = 0;
    int next_point = 0, rej = 0, status = RC_ST_OK;
    const __amdgpu_buffer_rsrc_t rS = rc_rsrc(S.samples, (uint32_t)((size_t)p.npoints * S.nlive * mat_bytes));
    const int my_rank = task - S.first_task;

    // Who shares an XCD: every workgroup posts the id of its own (the record of attempt 0) and looks at
    // those of its partners, so the verdicts agree.  A channel's tiles stay in the L2 when all its tasks
    // (with the E tasks that read it) run on one XCD; when its insertions' readers do not, they get a
    // copy of P through memory.
    if (tid == 0) s_loc = 0;
    if (wave == 0) {
        const uint32_t rec0 = (uint32_t)(lane * RC_REC * 8);
        if (lane == 0) rc_put(rX, (uint32_t)(my_rank * RC_REC * 8), oR, cmake(xcd_id(), 0.0));
        const bool in = lane < S.ntasks;
        cplx v;
        rc_fetch<1>(rX, rec0, oR, 16, &v, in);
        const bool ok = rc_await<1>(ctl, rX, rec0, oR, 16, &v, in);
        const int id = (int)v.re;
        const TrajTask& t = p.tasks[S.first_task + (in ? lane : 0)];
        const int t_ch = t.ch, t_src = t.edge_from_E || !in ? -1 : t.edge_src;
        auto tiles = [&](int x) { return rc_same(__ballot(in && t_ch == x), id); };
        auto inserts = [&](int x) { return rc_same(__ballot(in && (t_ch == x || t_src == x)), id); };
        int f = 0;
        if (tiles(ch)) f |= 1;
        if (inserts(ch)) f |= 2;
        if (tk.edge_src >= 0 && !tk.edge_from_E && tiles(tk.edge_src) && !inserts(tk.edge_src)) f |= 4;
        if (rc_same(__ballot(in && (t.e_only || t.edge_from_E)), id)) f |= 8;
        if (rc_same(__ballot(in), id)) f |= 16;
        if (__ballot(in && t_src == ch) != 0) f |= 32;
        if (lane == 0) {
            s_loc = f;
            if (!ok) s_bad = 1;
        }
    }
    __syncthreads();
    const int loc = uni(s_loc);
    const bool loc_Y = loc & 1, loc_P = LOCAL ? (loc & 2) != 0 : (loc & 1) != 0;   // Dp = 16: P is for insertions only
    const bool copy_P = !LOCAL && (loc & 35) == 33;           // tiles together, an insertion's reader elsewhere
    const bool ins_copy = !LOCAL && (loc & 4);                // this task's insertion reads the copy
    const bool loc_E = loc & 8, loc_R = loc & 16;

    // stage input of the next event
    auto publish_Y = [&](cplx v) {
        ++ev;
        if (e_only) return;   // an E task reads channel ch's stage input; the channel's own task writes it
        if constexpr (LOCAL) Yt[ei * 17 + ej] = v;
        const uint32_t so = (ev & (RC_RING - 1)) * stage_stride + (uint32_t)ch * mat_bytes;
        if (LOCAL ? tk.pub_y : do2) {
            rc_put(rX, ya_off, so, v, loc_Y);
            if constexpr (!LOCAL) rc_put(rX, yb_off, oB + so, v, loc_Y);
        }
    };

    // empty this workgroup's slots of event ev - 16 (once for every event, also one that is skipped)
    auto empty_old = [&] {
        if (ev <= RC_RING / 2) return;
        const uint32_t old = (ev - RC_RING / 2) & (RC_RING - 1), so = old * stage_stride + (uint32_t)ch * mat_bytes;
        if (e_only) {
            rc_reset(rX, yb_off, oE + old * mat_bytes, loc_E);
            return;
        }
        if (LOCAL ? tk.pub_y : do2) {
            rc_reset(rX, ya_off, so, loc_Y);
            if constexpr (!LOCAL) rc_reset(rX, yb_off, oB + so, loc_Y);
        }
        if (LOCAL ? tk.pub_p : do1) {
            rc_reset(rX, pub_off, oP + so, loc_P);
            if (copy_P) rc_reset(rX, pub_off, oP2 + so);
        }
    };

    // wave 0: the current attempt's records, and from their sums the attempt's verdict (every workgroup adds
    // the same records in the same order)
    const uint32_t rec_bytes = (uint32_t)(S.ntasks * RC_REC * 8);
    constexpr int NREC = (2 + RC_NSTAGES) / 2;   // pairs of a record: (e5, e3), the trace partials of k_0..k_11
    auto records = [&](cplx* v) {
        const int q = lane >> 3;
        return RcRecords{oR + (attempts & (RC_REC_RING - 1)) * rec_bytes,
                         (uint32_t)(16 * (q < (S.has_scalar ? NREC : 1) ? q : 0)), lane & 7, S.ntasks, v};
    };
    auto judge = [&](const RcRecords& recs) {
        const bool ok = rc_await_all(ctl, rX, recs);
        const cplx t = recs.sum();
        double e5 = read_lane(t.re, 0), e3 = read_lane(t.im, 0), sc_new = ysc;
        if (S.has_scalar) {
            const int q = lane >> 3, j = min(max(2 * q - 2, 0), RC_NSTAGES - 2);
            const double *c0 = rc_scalar_rows.c[j], *c1 = rc_scalar_rows.c[j + 1];
            const bool on = (lane & 7) == 0 && q >= 1 && q < NREC;
            const double sb = wave_sum(on ? fma(c0[0], t.re, c1[0] * t.im) : 0.0);
            const double s5 = wave_sum(on ? fma(c0[1], t.re, c1[1] * t.im) : 0.0);
            const double s3 = wave_sum(on ? fma(c0[2], t.re, c1[2] * t.im) : 0.0);
            sc_new = fma(h, sb, ysc);
            const double sc = 1.0 / (p.atol + p.rtol * fmax(fabs(ysc), fabs(sc_new)));
            e5 = fma(s5 * sc, s5 * sc, e5);
            e3 = fma(s3 * sc, s3 * sc, e3);
        }
        const double den = e5 + 0.01 * e3;
        const double error = den > 0.0 ? h * e5 / sqrt(den * S.n_elems) : 0.0;
        // 0.9 error^(-1/8)
        const double grow = error > 0.0 ? fmin(10.0, 0.9 / sqrt(sqrt(sqrt(error)))) : 10.0;
        if (lane == 0) {
            s_verdict[0] = error;
            s_verdict[1] = grow;
            s_verdict[2] = sc_new;
            s_verdict[3] = ok && !s_bad ? 0.0 : 1.0;
        }
    };

    // ------------------------------------------------------------------------------------
    // one right-hand-side evaluation on the stage input of event ev (own element `own`); al: the
    // coefficient of its derivative in the combination that follows, which is the next stage input
    // and published at once when `chain`
    // ------------------------------------------------------------------------------------
    auto stage = [&](int slot, double ts, cplx own, double al, bool chain, cplx& k_out, cplx& comb_out) {
        const double jac = 2.0 * fabs(ts);
        const uint32_t ring = ev & (RC_RING - 1);
        const uint32_t so = ring * stage_stride + (uint32_t)ch * mat_bytes;
        cplx xr[NF], xc[NF];
        if (e_only) {
            // E = X C of channel ch: its row block b times C's column block c
            if (doE) {
                cplx Ee;
                rc_fetch<NF>(rX, row_off, so, row_step, xr, use_r);
                if (!rc_await<NF>(ctl, rX, row_off, so, row_step, xr, use_r)) s_bad = 1;
                lap(0);
                // the two partial buffers alternate: one barrier a stage
                if constexpr (SPLIT) {
                    store_row4<NB>(pXr, xr, line_scale(xr, sgX));
                    lds_barrier();
                    lap(1);
                    int s2[4];
#pragma unroll
                    for (int q = 0; q < 4; ++q) s2[q] = -(sgX[4 * (lane >> 4) + q] + sK1);
                    double pe[4] = {0.0, 0.0, 0.0, 0.0};
                    rc_split_product(pe, pXr, spa, pK1, spb, s2, lane);
                    double* redd = (rhs & 1) ? redd2 : redd1;
                    put_partial_split(pe, redd, wave, lane);
                    lds_barrier();
                    Ee = sum_partial_split(redd);
                } else {
                    cacc ae;
                    cacc_zero(ae);
                    frag_product<KT>(ae, xr, K1);
                    cplx* red = (rhs & 1) ? red2 : red1;
                    put_partial(ae, red, wave, lane);
                    lds_barrier();
                    Ee = sum_partial(red);
                }
                rc_put(rX, yb_off, oE + ring * mat_bytes, Ee, loc_E);
            }
            empty_old();
            if (slot == RC_NSTAGES) {
                if (wave == 0) {
                    cplx rec[8];
                    RcRecords recs = records(rec);
                    recs.fetch(rX);
                    judge(recs);
                }
                lds_barrier();
            }
            k_out = comb_out = cmake(0, 0);
            if (chain) publish_Y(comb_out);
            lap(2);
            return;
        }
        // stage input
        bool ok = true;
        const bool get_c = do2 || !adj, get_r = do2 || adj;   // what the tile's products read
        if constexpr (LOCAL) {
            lds_barrier();
            xr[0] = Yt[fi * 17 + fk];
            xc[0] = Yt[fk * 17 + fi];
        } else {
            const RcWant<NF> wc{col_off, oB + so, col_step, xc, get_c, use_c};
            const RcWant<NF> wr{row_off, so, row_step, xr, get_r, use_r};
            wc.fetch(rX);
            wr.fetch(rX);
            ok = rc_await_all(ctl, rX, wc, wr);
        }
        lap(0);
        cacc acc;
        double part[4] = {0.0, 0.0, 0.0, 0.0};
        int sXr[4], sXc = 0;
        cplx Pe = cmake(0, 0);
        if constexpr (SPLIT) {
            if (get_r) store_row4<NB>(pXr, xr, line_scale(xr, sgX));
            if (get_c) store_col4<NB>(pXc, xc, line_scale(xc, sgX + 16));
            lds_barrier();
            lap(1);
            // per-element product scales: this lane's output rows 4 (lane/16) + q and column lane%16
#pragma unroll
            for (int q = 0; q < 4; ++q) sXr[q] = sgX[4 * (lane >> 4) + q];
            sXc = sgX[16 + (lane & 15)];
        }
        if (do1) {
            if constexpr (SPLIT) {
                if (!adj) {
                    const int s2[4] = {-(sK1 + sXc), -(sK1 + sXc), -(sK1 + sXc), -(sK1 + sXc)};
                    rc_split_product(part, pK1, spa, pXc, spb, s2, lane);
                } else {
                    const int s2[4] = {-(sXr[0] + sK1), -(sXr[1] + sK1), -(sXr[2] + sK1), -(sXr[3] + sK1)};
                    rc_split_product(part, pXr, spa, pK1, spb, s2, lane);
                }
                put_partial_split(part, redd1, wave, lane);
            } else {
                cacc_zero(acc);
                if (!adj) frag_product<KT>(acc, K1, xc);
                else frag_product<KT>(acc, xr, K1);
                put_partial(acc, red1, wave, lane);
            }
            lds_barrier();
            Pe = SPLIT ? sum_partial_split(redd1) : sum_partial(red1);
            if constexpr (LOCAL) Pt[ei * 17 + ej] = Pe;
            if (!LOCAL || tk.pub_p) rc_put(rX, pub_off, oP + so, Pe, loc_P);
            if (copy_P) rc_put(rX, pub_off, oP2 + so, Pe);
        } else {
            lds_barrier();   // two level-2 sums in a row need a barrier between them
        }
        lap(2);
        // the slots of event ev - 16 (ahead of the P loads: a wait for those does not include a younger store)
        empty_old();
        // level 2a
        if (do2) {
            if constexpr (SPLIT) {
                part[0] = part[1] = part[2] = part[3] = 0.0;
                const int s2a[4] = {-(sKq + sXc), -(sKq + sXc), -(sKq + sXc), -(sKq + sXc)};
                const int s2b[4] = {-(sXr[0] + sKx), -(sXr[1] + sKx), -(sXr[2] + sKx), -(sXr[3] + sKx)};
                rc_split_product(part, pKq, spa, pXc, spb, s2a, lane);
                rc_split_product(part, pXr, spa, pKx, spb, s2b, lane);
            } else {
                cacc_zero(acc);
                frag_product<KT>(acc, Kq, xc);
                frag_product<KT>(acc, xr, Kx);
            }
        }
        // the P tiles of this channel (row block forward, column block adjoint) and the insertion source
        cplx vp[NF], s1 = cmake(0, 0), s2 = cmake(0, 0);
        const bool insert = do2 && tk.edge_src >= 0;
        const uint32_t so_i = tk.edge_from_E ? oE + ring * mat_bytes
                                             : (ins_copy ? oP2 : oP) + ring * stage_stride + (uint32_t)tk.edge_src * mat_bytes;
        if (!LOCAL && do2) rc_fetch<NF>(rX, p_off, oP + so, p_step, vp, use_p);
        if (insert) {
            s1 = ld_coh_s(rX, ins_off, so_i);
            s2 = ld_coh_s(rX, ins_off_t, so_i);
        }
        // while they arrive: the trace of this stage, the records of the attempt at its FSAL stage
        if (tk.trace_kind) {
            double trv = 0.0;
            if (tk.trace_kind == 2 && b == c && ei == ej && real_el) trv = Pe.re;
            if (tk.trace_kind == 1 && real_el) trv = fma(own.re, trop_e.re, own.im * trop_e.im);   // Re(x conj(o))
            trv = wave_sum(trv);
            if (lane == 0) s_trp[slot][wave] = trv;
        }
        const double src = slot == 0 ? rc_source(ts, s_cheb) : unid(s_src[attempts & 1][slot]);
        if (tk.trace_kind && tid == 0) s_trs[slot] = tk.trace_coef * src;
        cplx rec[8];
        RcRecords recs = records(rec);
        if (slot == RC_NSTAGES && wave == 0) recs.fetch(rX);
        lap(3);
        cplx Le = cmake(0, 0);
        if (do2) {
            if constexpr (LOCAL) {
                lds_barrier();
                vp[0] = adj ? Pt[fk * 17 + fi] : Pt[fi * 17 + fk];
            } else {
                ok = rc_await<NF>(ctl, rX, p_off, oP + so, p_step, vp, use_p) && ok;
            }
            lap(4);
            if constexpr (SPLIT) {
                if (!adj) store_row4<NB>(pPb, vp, line_scale(vp, sgP));
                else store_col4<NB>(pPb, vp, line_scale(vp, sgP));
                lds_barrier();
                lap(5);
                if (!adj) {
                    const int s2[4] = {-(sgP[4 * (lane >> 4)] + sKp), -(sgP[4 * (lane >> 4) + 1] + sKp),
                                       -(sgP[4 * (lane >> 4) + 2] + sKp), -(sgP[4 * (lane >> 4) + 3] + sKp)};
                    rc_split_product(part, pPb, spa, pKp, spb, s2, lane);
                } else {
                    const int sc = -(sKp + sgP[lane & 15]);
                    const int s2[4] = {sc, sc, sc, sc};
                    rc_split_product(part, pKp, spa, pPb, spb, s2, lane);
                }
            } else {
                if (!adj) frag_product<KT>(acc, vp, Kp);
                else frag_product<KT>(acc, Kp, vp);
            }
        }
        if (slot == RC_NSTAGES && wave == 0) judge(recs);   // in the shadow of the products
        if (do2) {
            if constexpr (SPLIT) put_partial_split(part, redd2, wave, lane);
            else put_partial(acc, red2, wave, lane);
            if (insert) {
                ok = rc_await_all(ctl, rX, RcWant<1>{ins_off, so_i, 0, &s1, true, true},
                                  RcWant<1>{ins_off_t, so_i, 0, &s2, true, true}) && ok;
            }
        }
        lds_barrier();   // without level 2: two level-1 sums in a row likewise
        if (do2) Le = SPLIT ? sum_partial_split(redd2) : sum_partial(red2);
        if (!ok) s_bad = 1;
        const cplx ins = cfma(insert ? tk.edge_coef : 0.0, cadd(s1, cconj(s2)), fixed_e);
        cplx k = cfma(jac, Le, cscale(src, ins));
        if (!real_el) k = cmake(0, 0);
        k_out = k;
        comb_out = cfma(h, cfma(al, k, ahead.a[0]), y);
        lap(6);
        if (chain) publish_Y(comb_out);
        lap(10);
    };

    // ------------------------------------------------------------------------------------
    // a state machine over stage slots with a single stage call site; the stage input of the event
    // at hand is published before the stage is entered
    // ------------------------------------------------------------------------------------
    int slot = 0;
    cplx Yin = y;
    double ts = t;
    publish_Y(Yin);
    while (true) {
        cplx kn, comb;
        ++rhs;
        // stages 1..10 chain to the next one, and 13..14 of the dense output's
        const bool chain = (slot > 0 && slot < RC_NSTAGES - 1) || (slot > RC_NSTAGES && slot < RC_NSTAGES_EXT - 1);
        stage(slot, ts, Yin, s_alast[slot], chain, kn, comb);
        int next = -1;       // -1: start a new step attempt
        bool published = chain, interpolate = false;
        const double t_old = t, h_old = h;
        const cplx y_old = y, k0_old = k0;
        if (slot == 0) {
            k0 = kn;
        } else if (slot < RC_NSTAGES - 1) {
            next = slot + 1;
        } else if (slot == RC_NSTAGES - 1) {
            lap(7);
            ynew = comb;
            const cplx acc5 = cfma(RC_E5[RC_NSTAGES - 1], kn, ahead.e5);
            const cplx acc3 = cfma(RC_E3[RC_NSTAGES - 1], kn, ahead.e3);
            double e5p = 0.0, e3p = 0.0;
            if (real_el) {
                const double sc = 1.0 / (p.atol + p.rtol * fmax(cabsd(y), cabsd(ynew)));
                const cplx r5 = cscale(sc, acc5), r3 = cscale(sc, acc3);
                e5p = fma(r5.re, r5.re, r5.im * r5.im);
                e3p = fma(r3.re, r3.re, r3.im * r3.im);
            }
            e5p = wave_sum(e5p);
            e3p = wave_sum(e3p);
            if (lane == 0) {
                s_err[wave] = e5p;
                s_err[4 + wave] = e3p;
            }
            // every emptied slot is empty at its scope before the record can be seen
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            lds_barrier();
            // the record, and behind it the FSAL stage on the solution, ahead of the verdict: the records
            // arrive during that stage (a rejected step's is not counted and its derivative not used)
            if (wave == 0 && lane < (S.has_scalar ? NREC : 1)) {
                cplx v;
                if (lane == 0) {
                    v = cmake(((s_err[0] + s_err[1]) + s_err[2]) + s_err[3], ((s_err[4] + s_err[5]) + s_err[6]) + s_err[7]);
                } else {
                    const int q = 2 * lane - 2;
                    v = tk.trace_kind ? cmake(s_trs[q] * (((s_trp[q][0] + s_trp[q][1]) + s_trp[q][2]) + s_trp[q][3]),
                                              s_trs[q + 1] * (((s_trp[q + 1][0] + s_trp[q + 1][1]) + s_trp[q + 1][2]) +
                                                              s_trp[q + 1][3]))
                                      : cmake(0, 0);
                }
                const uint32_t off = (uint32_t)(my_rank * RC_REC * 8 + 16 * lane);
                rc_put(rX, off, oR + (attempts & (RC_REC_RING - 1)) * rec_bytes, v, loc_R);
                // the record of attempt - 2: every workgroup published that of attempt - 1, so all read it
                rc_reset(rX, off, oR + ((attempts + 2) & (RC_REC_RING - 1)) * rec_bytes, loc_R);
            }
            lap(8);
            next = RC_NSTAGES;
        } else if (slot == RC_NSTAGES) {
            if (unid(s_verdict[3]) != 0.0) break;
            const double error = unid(s_verdict[0]);
            factor = unid(s_verdict[1]);
            ysc_new = unid(s_verdict[2]);
            if (!isfinite(error)) { --rhs; status = RC_ST_NONFINITE; break; }
            if (error > 1.0) {
                --rhs;
                ++rejected;
                rej = 1;
                h *= fmax(0.2, factor);
            } else {
                ++accepted;
                t_new = (h == endpoint - t) ? endpoint : t + h;
                k12 = kn;
                next = -2;   // finish the accepted step, unless a quadrature node lies in it
                if (next_point < p.npoints && ld_const(p.points, next_point) <= t_new) {
                    ++dense;
                    next = RC_NSTAGES + 1;
                }
            }
        } else if (slot < RC_NSTAGES_EXT - 1) {
            next = slot + 1;
        } else {
            interpolate = true;
            next = -2;
        }
        if (next == -2) {
            // accepted step complete: FSAL and state update
            y = ynew;
            k0 = k12;
            if (tk.trace_kind && tid == 0) {
#pragma unroll
                for (int q = 0; q < 4; ++q) s_trp[0][q] = s_trp[RC_NSTAGES][q];
                s_trs[0] = s_trs[RC_NSTAGES];
            }
            t = t_new;
            ysc = ysc_new;
            h *= rej ? fmin(1.0, factor) : factor;
            rej = 0;
            next = -1;
        }
        bool done = false;
        if (next == -1) {
            // start an attempt from (t, y, k0) with step h
            if (!(t < a)) {
                done = true;
            } else {
                endpoint = t < 0.0 ? 0.0 : a;
                h = fmin(h, endpoint - t);
                if (!(h > 10.0 * fabs(nextafter(t, INFINITY) - t))) { status = RC_ST_STEP_UNDERFLOW; done = true; }
                else if ((long long)attempts >= p.max_steps) { status = RC_ST_MAX_STEPS; done = true; }
                else ++attempts;
            }
            next = 1;
        }
        t = unid(t);
        h = unid(h);
        if (!done) {
            if (next == 1) {
                Yin = cfma(h, cscale(RC_A[1][0], k0), y);
                ts = t + RC_C[1] * h;
            } else {
                Yin = comb;   // also the solution, the FSAL stage's input
                ts = t + s_cnode[next] * h;
            }
            lap(7);
            if (!published) publish_Y(Yin);
        }
        // behind the publish: the source values of the attempt's stages (one lane each), the dense
        // output, the combinations ahead
        if (next == 1 && !done && tid >= 1 && tid < RC_NSTAGES_EXT)
            s_src[attempts & 1][tid] = rc_source(t + s_cnode[tid] * h, s_cheb);
        if (interpolate) {
            cplx dd[4];
#pragma unroll
            for (int q = 0; q < 4; ++q)
                dd[q] = cscale(h_old, cfma(RC_D[q][RC_NSTAGES_EXT - 1], kn, ahead.d[q]));
            const cplx d0 = csub(ynew, y_old);
            const cplx d1 = cfma(h_old, k0_old, cmake(-d0.re, -d0.im));
            const cplx d2 = cfma(-h_old, cadd(k12, k0_old), cscale(2.0, d0));
            while (next_point < p.npoints && ld_const(p.points, next_point) <= t_new) {
                const double pt = ld_const(p.points, next_point);
                cplx v;
                if (pt == t_new) {
                    v = ynew;
                } else {
                    const double x = (pt - t_old) / h_old, xm = 1.0 - x;
                    cplx r = cfma(x, dd[3], dd[2]);
                    r = cfma(xm, r, dd[1]);
                    r = cfma(x, r, dd[0]);
                    r = cfma(xm, r, d2);
                    r = cfma(x, r, d1);
                    r = cfma(xm, r, d0);
                    v = cfma(x, r, y_old);
                }
                if (!e_only) st_coh(rS, (uint32_t)next_point * stage_stride + (uint32_t)ch * mat_bytes + el_off, v);
                ++next_point;
            }
            next_point = uni(next_point);
        }
        if (done) break;
        if (next == 1) ahead.clear();
        ahead.add(next - 1, next == 1 ? k0 : kn);
        slot = uni(next);
    }
    // every workgroup reports a wait of its own that failed, in whatever stage (rc_system_status)
    lds_barrier();
    if (tid == 0 && (s_bad || s_verdict[3] != 0.0))
        __hip_atomic_store(&S.out[RC_OUT_WAIT_FAILED], 1.0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (status == RC_ST_OK && next_point != p.npoints) status = RC_ST_MISSING_SAMPLES;
    __builtin_amdgcn_s_waitcnt(0);
    if (my_rank == 0 && tid == 0) {
        S.out[RC_OUT_STATUS] = status;
        S.out[RC_OUT_ATTEMPTS] = (double)attempts;
        S.out[RC_OUT_ACCEPTED] = (double)accepted;
        S.out[RC_OUT_REJECTED] = (double)rejected;
        S.out[RC_OUT_DENSE] = (double)dense;
        S.out[RC_OUT_RHS] = (double)rhs;
        S.out[RC_OUT_SCALAR] = ysc;
        S.out[RC_OUT_T] = t;
        S.out[RC_OUT_NEXTPOINT] = next_point;
        lap(7);
        if constexpr (TIMED) tacc[9] = __builtin_amdgcn_s_memrealtime() - tstart;
#pragma unroll
        for (int q = 0; q < RC_NTIMERS; ++q) S.out[RC_OUT_TIMERS + q] = (double)tacc[q];
    }
}

template <int NB, int KT, bool SPLIT, bool TIMED>
__global__ void __launch_bounds__(256, 1) rc_trajectory(const TrajParams* __restrict__ pp) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const TrajParams& p = *pp;
    const __attribute__((address_space(4))) int* sched = (const __attribute__((address_space(4))) int*)p.schedule;
    for (int r = 0; r < p.nrounds; ++r) {
        const int task = __builtin_amdgcn_readfirstlane(sched[r * (int)gridDim.x + (int)blockIdx.x]);
        if (task < 0) continue;
        run_task<NB, KT, SPLIT, TIMED>(p, task, smem_raw);
        __syncthreads();
    }
}

// Empty every slot of a launch's exchange buffers (n 16-byte words).
__global__ void __launch_bounds__(256) rc_fill_empty(v4u* w, long long n) {
    const v4u e = {RC_EMPTY_WORD, RC_EMPTY_WORD, RC_EMPTY_WORD, RC_EMPTY_WORD};
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long long)gridDim.x * 256) w[i] = e;
}

// ---------------------------------------------------------------------------------------
// host launcher
// ---------------------------------------------------------------------------------------
int rc_trajectory_smem_bytes(int nb, int split) {
    if (nb < 1 || nb > 4) return -1;
    if (split) return LaySplit::BYTES;
    switch (nb) {
        case 1: return Lay<1>::BYTES;
        case 2: return Lay<2>::BYTES;
        case 3: return Lay<3>::BYTES;
        default: return Lay<4>::BYTES;
    }
}

template <bool TIMED>
static const void* trajectory_fn(int nb, int split, int z2) {
    if (z2 && !split && nb == 2) return (const void*)rc_trajectory<2, 1, false, TIMED>;
    if (z2 && !split && nb == 4) return (const void*)rc_trajectory<4, 2, false, TIMED>;
    switch (nb * 2 + (split ? 1 : 0)) {
        case 2: return (const void*)rc_trajectory<1, 1, false, TIMED>;
        case 3: return (const void*)rc_trajectory<1, 1, true, TIMED>;
        case 4: return (const void*)rc_trajectory<2, 2, false, TIMED>;
        case 5: return (const void*)rc_trajectory<2, 2, true, TIMED>;
        case 6: return (const void*)rc_trajectory<3, 3, false, TIMED>;
        case 7: return (const void*)rc_trajectory<3, 3, true, TIMED>;
        case 8: return (const void*)rc_trajectory<4, 4, false, TIMED>;
        case 9: return (const void*)rc_trajectory<4, 4, true, TIMED>;
        default: return nullptr;
    }
}
// z2: every state of the launch is Z2-symmetric with whole-tile parity blocks
static const void* trajectory_fn(int nb, int split, int z2, int timed) {
    return timed ? trajectory_fn<true>(nb, split, z2) : trajectory_fn<false>(nb, split, z2);
}

// workgroups of the trajectory kernel that can be resident at once on the current device
hipError_t rc_trajectory_capacity(int nb, int split, int z2, int timed, int* blocks) {
    const void* fn = trajectory_fn(nb, split, z2, timed);
    if (!fn) return hipErrorInvalidValue;
    const int bytes = rc_trajectory_smem_bytes(nb, split);
    hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e != hipSuccess) return e;
    int per_cu = 0, dev = 0, cus = 0;
    if ((e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, 256, bytes)) != hipSuccess) return e;
    if ((e = hipGetDevice(&dev)) != hipSuccess) return e;
    if ((e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev)) != hipSuccess) return e;
    *blocks = per_cu * cus;
    return hipSuccess;
}

hipError_t rc_launch_trajectory(int nb, int split, int z2, int timed, int nblocks, const TrajParams* dparams, hipStream_t stream) {
    void* args[] = {(void*)&dparams};
    const void* fn = trajectory_fn(nb, split, z2, timed);
    const int bytes = rc_trajectory_smem_bytes(nb, split);
    if (!fn) return hipErrorInvalidValue;
    hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e != hipSuccess) return e;
    return hipLaunchCooperativeKernel(fn, dim3(nblocks), dim3(256), args, (unsigned)bytes, stream);
}

hipError_t rc_launch_fill_empty(void* dst, size_t bytes, hipStream_t stream) {
    const long long n = (long long)(bytes / 16);
    const long long blocks = (n + 1023) / 1024;
    hipLaunchKernelGGL(rc_fill_empty, dim3((unsigned)(blocks < 2048 ? blocks : 2048)), dim3(256), 0, stream,
                       static_cast<v4u*>(dst), n);
    return hipGetLastError();
}
