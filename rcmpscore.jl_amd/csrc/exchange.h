// Exchange of tiles between the workgroups of a persistent launch, and the wave-level pieces both
// persistent integrators use (rc_trajectory, rc_quartic_ode): ring slots that hold a NaN pattern until
// their value is stored, polling loads straight into MFMA fragments, partial tiles in LDS, wave sums.
#pragma once
#include "device_common.h"
#include "trajectory.h"

namespace {

// c k + a, each part one fused multiply-add: the instantiations of the kernel (Z2 blocks or every
// k-tile, timed or not) round alike whatever the compiler would contract
__device__ __forceinline__ cplx cfma(double c, cplx k, cplx a) { return cmake(fma(c, k.re, a.re), fma(c, k.im, a.im)); }

struct Ctl {
    uint32_t* abort_flag;
    long long wait_ticks;   // longest single wait, in ticks of the constant-rate clock (s_memrealtime)
};

// Barrier of the workgroup that orders LDS accesses only: device-coherent stores and polling loads
// in flight stay in flight (__syncthreads would wait for them).
__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// The empty slot's word is all ones: a quiet NaN no arithmetic here produces (the hardware's own NaN has
// payload zero, the state's matrices are finite) and the largest unsigned number, so that one maximum
// over the high words of many elements tells whether any is still empty.
__device__ __forceinline__ uint32_t rc_max_word(uint32_t m, cplx v) {
    return max(m, max((uint32_t)__double2hiint(v.re), (uint32_t)__double2hiint(v.im)));
}
__device__ __forceinline__ double rc_not_empty(double x) {
    return (uint32_t)__double2hiint(x) == RC_EMPTY_WORD ? __longlong_as_double(0x7ff8000000000000LL) : x;
}
// Publish a value / empty a slot again; every aligned 8-byte half is written whole, and a reader checks
// both.  `local` (uniform): every reader of the slot runs on this workgroup's XCD, so the value need not
// leave its L2, where a device-coherent load finds it: 275 ns from store to seen on MI355X, against 495
// through memory on one XCD and 560 to 635 between two, and no traffic beyond the L2.
__device__ __forceinline__ void rc_store(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff, cplx z, bool local) {
    if (local) st_xcd_s(r, voff, soff, z);
    else st_coh_s(r, voff, soff, z);
}
__device__ __forceinline__ void rc_put(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff, cplx z, bool local = false) {
    rc_store(r, voff, soff, cmake(rc_not_empty(z.re), rc_not_empty(z.im)), local);
}
__device__ __forceinline__ void rc_reset(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff, bool local = false) {
    const double e = __hiloint2double((int)RC_EMPTY_WORD, (int)RC_EMPTY_WORD);
    rc_store(r, voff, soff, cmake(e, e), local);
}
// whether the lanes of `mask` (bit i: lane i) all hold the same id; an empty mask does
__device__ __forceinline__ bool rc_same(uint64_t mask, int id) {
    if (mask == 0) return true;
    const int id0 = __builtin_amdgcn_readlane(id, __builtin_ctzll(mask));
    return (mask & ~__ballot(id == id0)) == 0;
}

// Elements voff + soff + t stride, t < N, of the lanes that `use` them: the loads alone; rc_await then
// repeats them until every element of the wave has arrived.  False when the abort word is set or
// the wait outlasts its time budget (then the abort word is set).  The budget is wall-clock time: in
// a batched launch every workgroup runs a list of tasks, and one that starts a system early waits while its
// partners still run the systems before it in theirs.
template <int N>
__device__ __forceinline__ void rc_fetch(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff, uint32_t stride,
                                         cplx* v, bool use = true) {
    if (use) {
#pragma unroll
        for (int t = 0; t < N; ++t) v[t] = ld_coh_s(r, voff, soff + t * stride);
    } else {
#pragma unroll
        for (int t = 0; t < N; ++t) v[t] = cmake(0, 0);
    }
}
// Hide the values from the compiler's count of outstanding loads: they have arrived, and their later
// uses must not wait for whatever store or load was issued since.
template <int N>
__device__ __forceinline__ void rc_settle(cplx* v) {
#pragma unroll
    for (int t = 0; t < N; ++t) asm volatile("" : "+v"(v[t].re), "+v"(v[t].im));
}
// one group of fragments to wait for: N elements voff + soff + t stride of the lanes that use them
template <int N>
struct RcWant {
    uint32_t voff, soff, stride;
    cplx* v;
    bool on, use;   // on (uniform): the group is wanted at all
    __device__ __forceinline__ void fetch(__amdgpu_buffer_rsrc_t r) const {
        if (on) rc_fetch<N>(r, voff, soff, stride, v, use);
    }
    __device__ __forceinline__ bool late() const {
        uint32_t m = 0;
#pragma unroll
        for (int t = 0; t < N; ++t) m = rc_max_word(m, v[t]);
        return on && __any(m == RC_EMPTY_WORD);
    }
    __device__ __forceinline__ void settle() const { rc_settle<N>(v); }
};
// Wait for every group: a round looks at all of them and repeats the loads of all late ones together (one
// after the other, each group's early loads would cost a round trip of their own; looking at every element
// by itself, to repeat only those that are late, costs more instructions than it spares loads).
template <class... W>
__device__ __forceinline__ bool rc_await_all(const Ctl& ctl, __amdgpu_buffer_rsrc_t r, const W&... w) {
    uint64_t t0 = 0;
    bool ok = true;
    for (uint32_t polls = 1;; ++polls) {
        int late = 0, bit = 1;
        (((late |= w.late() ? bit : 0), bit <<= 1), ...);
        if (late == 0) break;
        asm volatile("" ::: "memory");
        bit = 1;
        (((late & bit) ? w.fetch(r) : (void)0, bit <<= 1), ...);
        if ((polls & 63) == 0) {   // the clock and the abort word are read every 64th poll only
            const uint64_t now = __builtin_amdgcn_s_memrealtime();
            if (t0 == 0) t0 = now;
            const bool over = (long long)(now - t0) > ctl.wait_ticks;
            if (over) st_flag(ctl.abort_flag, 1u);
            if (over || uni((int)ld_flag(ctl.abort_flag))) {
                ok = false;
                break;
            }
        }
    }
    (w.settle(), ...);
    return ok;
}
template <int N>
__device__ __forceinline__ bool rc_await(const Ctl& ctl, __amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff,
                                         uint32_t stride, cplx* v, bool use = true) {
    return rc_await_all(ctl, r, RcWant<N>{voff, soff, stride, v, true, use});
}

// acc += A B over this wave's k-steps (fragment t: its k-step of the t-th k-tile)
template <int KT>
__device__ __forceinline__ void frag_product(cacc& acc, const cplx* A, const cplx* B) {
#pragma unroll
    for (int t = 0; t < KT; ++t) cmfma(acc, A[t], B[t]);
}

// Sum of the four waves' partial tiles; thread t receives element (t/16, t%16).  The barrier also
// orders the other level's buffer: its readers pass here before anyone writes it again.
__device__ __forceinline__ void put_partial(const cacc& acc, cplx* red, int wave, int lane) {
#pragma unroll
    for (int q = 0; q < 4; ++q) red[wave * 256 + (4 * q + (lane >> 4)) * 16 + (lane & 15)] = cacc_get(acc, q);
}
__device__ __forceinline__ cplx sum_partial(const cplx* red) {
    const int t = threadIdx.x;
    return cadd(cadd(cadd(red[t], red[256 + t]), red[512 + t]), red[768 + t]);
}

// a DPP move of a double within each row of 16 lanes (CTRL a compile-time DPP control)
template <int CTRL>
__device__ __forceinline__ double dpp_move(double x) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), CTRL, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), CTRL, 0xF, 0xF, false);
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double read_lane(double x, int l) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(x), l),
                            __builtin_amdgcn_readlane(__double2loint(x), l));
}
// Wave sum in a fixed order: pairs, quads (quad_perm), halves (row_half_mirror) and rows
// (row_mirror) by DPP moves, every lane of a row holding the same row sum (addition commutes),
// then the four row sums in order.
__device__ __forceinline__ double wave_sum(double v) {
    v += dpp_move<0xB1>(v);
    v += dpp_move<0x4E>(v);
    v += dpp_move<0x141>(v);
    v += dpp_move<0x140>(v);
    return ((read_lane(v, 0) + read_lane(v, 16)) + read_lane(v, 32)) + read_lane(v, 48);
}

// sum over each row of 16 lanes (every lane of the row holds it)
__device__ __forceinline__ double row_sum(double v) {
    v += dpp_move<0xB1>(v);
    v += dpp_move<0x4E>(v);
    v += dpp_move<0x141>(v);
    v += dpp_move<0x140>(v);
    return v;
}

// The sums of sixteen values over each row of 16 lanes: lane l of the row gets the sum of v[l].  Each
// step halves the values a lane still carries (it keeps those whose index shares its own next bit and
// hands over the others), 15 additions and exchanges instead of the 64 of sixteen separate sums.
template <int CTRL>
__device__ __forceinline__ double xchg(double x) {   // the value of the lane across the step
    if constexpr (CTRL == 4) {   // lane ^ 4: rotations of the row by 4 and by 12, by banks of four lanes
        int lo = __double2loint(x), hi = __double2hiint(x);
        int l4 = __builtin_amdgcn_update_dpp(0, lo, 0x124, 0xF, 0xA, false);
        int h4 = __builtin_amdgcn_update_dpp(0, hi, 0x124, 0xF, 0xA, false);
        l4 = __builtin_amdgcn_update_dpp(l4, lo, 0x12C, 0xF, 0x5, false);
        h4 = __builtin_amdgcn_update_dpp(h4, hi, 0x12C, 0xF, 0x5, false);
        return __hiloint2double(h4, l4);
    } else {
        return dpp_move<CTRL == 1 ? 0xB1 : CTRL == 2 ? 0x4E : 0x128>(x);
    }
}
template <int CTRL, int N>
__device__ __forceinline__ void halve(double* v, bool up) {
#pragma unroll
    for (int i = 0; i < N / 2; ++i) {
        const double keep = up ? v[2 * i + 1] : v[2 * i], give = up ? v[2 * i] : v[2 * i + 1];
        v[i] = keep + xchg<CTRL>(give);
    }
}
__device__ __forceinline__ double row_sums16(double* v, int lane) {
    halve<1, 16>(v, lane & 1);
    halve<2, 8>(v, lane & 2);
    halve<4, 4>(v, lane & 4);
    halve<8, 2>(v, lane & 8);
    return v[0];
}

// Record i of a read-only array through scalar loads, so that every field is known wave-uniform.
template <typename T>
__device__ __forceinline__ T load_scalar(const T* arr, int i) {
    static_assert(sizeof(T) % 8 == 0, "records are copied in 8-byte words");
    const __attribute__((address_space(4))) uint64_t* q =
        (const __attribute__((address_space(4))) uint64_t*)(arr + __builtin_amdgcn_readfirstlane(i));
    T t;
    uint64_t* w = reinterpret_cast<uint64_t*>(&t);
#pragma unroll
    for (int k = 0; k < (int)(sizeof(T) / 8); ++k) w[k] = q[k];
    return t;
}

}  // namespace
