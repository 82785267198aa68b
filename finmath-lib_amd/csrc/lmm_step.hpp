// Definitions shared by the path kernels (lmm_spot.hpp: the spot-measure Euler kernel,
// lmm_general.hpp: the other measures and schemes, lmm_spot_adjoint.hpp: the reverse sweep):
// the model records, the increments, the state-space transform and the wavefront reductions
// of the per-path payoffs.
//
// Model data layout: one record of rec_size_of(FCAP) reals per (time step,
// component): the factor loadings padded with zeros to FCAP, then variance*(-0.5),
// d/d and 1/d. A zero loading adds exact zeros, so the padding changes no value;
// a record is one aligned scalar load.
#pragma once

#include <hip/hip_runtime.h>
#include <type_traits>
#include "fm_internal.hpp"
#include "fm_math.hpp"

namespace fm {

constexpr int kStepThreads = 256;

template <int I, int N, typename Fn>
__device__ __forceinline__ void static_for(Fn&& fn) {
    if constexpr (I < N) {
        fn(std::integral_constant<int, I>{});
        static_for<I + 1, N>(fn);
    }
}

// Wavefront sum by DPP row operations (quad_perm [1,0,3,2], [2,3,0,1], row_ror 4 and 8,
// row_bcast 15 and 31): the total is valid in lane 63 only. Each step moves the two
// 32-bit halves of the double; lanes without a source read 0. Call with every lane of the
// wavefront active.
template <int CTRL>
__device__ __forceinline__ double dpp_move(double x) {
    const long long b = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)(b & 0xffffffffll), CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, true);
    return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}

__device__ __forceinline__ double wave_sum_dpp(double v) {
    v = v + dpp_move<0xb1>(v);
    v = v + dpp_move<0x4e>(v);
    v = v + dpp_move<0x124>(v);
    v = v + dpp_move<0x128>(v);
    v = v + dpp_move<0x142>(v);
    v = v + dpp_move<0x143>(v);
    return v;
}

// Wavefront sum, returned in every lane: the DPP sum read from lane 63. Unlike a butterfly of
// lane permutes it keeps no per-lane permute addresses live across the kernel.
__device__ __forceinline__ double wave_reduce_sum(double v) {
    const long long b = __double_as_longlong(wave_sum_dpp(v));
    const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffll), 63);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), 63);
    return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}

// The hardware base-2 exponential and logarithm (about 1 ulp each). FP32 only: the FP64 kernels carry base-2 states.
template <typename real> __device__ __forceinline__ real dev_exp(real x);
template <typename real> __device__ __forceinline__ real dev_log(real x);
template <> __device__ __forceinline__ float dev_exp<float>(float x) { return __builtin_amdgcn_exp2f(x * 1.44269504088896341f); }
template <> __device__ __forceinline__ float dev_log<float>(float x) { return __builtin_amdgcn_logf(x) * 0.693147180559945309f; }

// Java Math.max(x, 0.0) / Math.min(x, c): NaN propagates.
template <typename real> __device__ __forceinline__ real jmax0(real x) { return (x != x) ? x : (x >= (real)0 ? x : (real)0); }
template <typename real> __device__ __forceinline__ real jmin(real x, real c) { return (x > c) ? c : x; }

// Reduce one per-path value into the wave partial of `slot`.
__device__ __forceinline__ void reduce_slot(double x, bool active, int cnt, int lane, int64_t wave,
                                            double* __restrict__ wave_sum, double* __restrict__ wave_m2,
                                            int stride, int slot) {
    const double s = wave_reduce_sum(active ? x : 0.0);
    const double mean = (cnt > 0) ? s / (double)cnt : 0.0;
    const double d = active ? (x - mean) : 0.0;
    const double m2 = wave_reduce_sum(d * d);
    if (lane == 0 && cnt > 0) {
        wave_sum[(size_t)wave * stride + slot] = s;
        wave_m2[(size_t)wave * stride + slot] = m2;
    }
}

// Sum of a double over the wavefront's four rows of sixteen lanes, in every lane: the halves and
// then the row pairs exchanged by the lane-swap instructions (both swapped copies of one value add
// up to the sum over the pair).
__device__ __forceinline__ double rows_sum(double a) {
    auto swapped = [](double x, auto swap) -> double {
        const long long b = __double_as_longlong(x);
        const auto lo = swap((unsigned)(b & 0xffffffffll));
        const auto hi = swap((unsigned)((unsigned long long)b >> 32));
        return __longlong_as_double((long long)(((unsigned long long)hi[0] << 32) | lo[0])) +
               __longlong_as_double((long long)(((unsigned long long)hi[1] << 32) | lo[1]));
    };
    a = swapped(a, [](unsigned x) { return __builtin_amdgcn_permlane16_swap(x, x, false, false); });
    return swapped(a, [](unsigned x) { return __builtin_amdgcn_permlane32_swap(x, x, false, false); });
}

// Wavefront sums of four per-lane values at once, lane l returning the total of value
// 2 (l & 1) + ((l >> 1) & 1): two exchange steps within each quad halve the values a lane carries,
// two row rotations and the exchanges across the rows sum the lanes that carry the same value
// (11 adds and 20 moves for four values; one value alone takes 6 and 12).
__device__ __forceinline__ double wave_sum4_all(const double (&v)[4], int lane) {
    const bool b0 = (lane & 1) != 0, b1 = (lane & 2) != 0;
    double a2[2];
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const double send = b0 ? v[i] : v[i + 2];
        const double keep = b0 ? v[i + 2] : v[i];
        a2[i] = keep + dpp_move<0xb1>(send);      // quad_perm [1,0,3,2]: lane ^ 1
    }
    const double send = b1 ? a2[0] : a2[1];
    const double keep = b1 ? a2[1] : a2[0];
    double a = keep + dpp_move<0x4e>(send);       // quad_perm [2,3,0,1]: lane ^ 2
    a = a + dpp_move<0x124>(a);                   // row_ror:4
    a = a + dpp_move<0x128>(a);                   // row_ror:8
    return rows_sum(a);
}

__device__ __forceinline__ double read_lane(double v, int lane) {
    const long long b = __double_as_longlong(v);
    const unsigned lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffll), lane);
    const unsigned hi = __builtin_amdgcn_readlane((int)((unsigned long long)b >> 32), lane);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// Reduce up to four per-path values into the wave partials of their slots (value g to slot[g],
// g < m): reduce_slot for a group, inv_cnt = 1 / (active lanes).
__device__ __forceinline__ void reduce_slots4(const double (&x)[4], int m, bool active, int cnt, double inv_cnt,
                                              int lane, int64_t wave, double* __restrict__ wave_sum,
                                              double* __restrict__ wave_m2, int stride, const int (&slot)[4]) {
    constexpr int lane_of[4] = {0, 2, 1, 3};
    double v[4];
#pragma unroll
    for (int g = 0; g < 4; g++) v[g] = active ? x[g] : 0.0;
    const double s = wave_sum4_all(v, lane);
    const double mean = s * inv_cnt;
#pragma unroll
    for (int g = 0; g < 4; g++) {
        const double d = active ? x[g] - read_lane(mean, lane_of[g]) : 0.0;
        v[g] = d * d;
    }
    const double m2 = wave_sum4_all(v, lane);
    const int g = 2 * (lane & 1) + ((lane >> 1) & 1);
    if (lane < 4 && g < m && cnt > 0) {
        const int to = g == 0 ? slot[0] : g == 1 ? slot[1] : g == 2 ? slot[2] : slot[3];
        wave_sum[(size_t)wave * stride + to] = s;
        wave_m2[(size_t)wave * stride + to] = m2;
    }
}

// An array that the launch only reads, at an index uniform over the wavefront: read through the
// constant address space, so the reads are scalar loads wherever the pointer came from (a pointer
// read from a structure is not known to be free of the kernel's stores otherwise).
template <typename T>
struct ConstArray {
    const T* p;
    __device__ __forceinline__ T operator[](int64_t i) const {
        typedef const uint32_t __attribute__((address_space(4)))* Words;
        static_assert(sizeof(T) % 4 == 0, "whole words");
        struct { uint32_t w[sizeof(T) / 4]; } v;
        const Words q = (Words)(uintptr_t)(p + i);
#pragma unroll
        for (int k = 0; k < (int)(sizeof(T) / 4); k++) v.w[k] = q[k];
        return __builtin_bit_cast(T, v);
    }
};

// The kernel's arguments where they lie. A pointer made opaque once per time step keeps the compiler
// from holding every argument in scalar registers across the step (where they would be spilled
// into vector registers and read back lane by lane); what a step needs is a scalar load.
typedef const StepArgs __attribute__((address_space(4)))* ArgPtr;
__device__ __forceinline__ ArgPtr kernel_arguments() {
    ArgPtr a = (ArgPtr)__builtin_amdgcn_kernarg_segment_ptr();
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+s"(a));
#endif
    return a;
}

// A uniform value whose origin the compiler does not see: comparisons with it are made where they are
// used, instead of being hoisted out of a loop as one mask per unrolled component and spilled.
__device__ __forceinline__ int opaque(int x) {
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+s"(x));
#endif
    return x;
}

// Record of one (time step, component).
template <int FCAP, typename real>
struct Rec {
    static constexpr int size = rec_size_of(FCAP);
    const real* __restrict__ r;
    __device__ __forceinline__ real lam(int k) const { return r[k]; }
    __device__ __forceinline__ real hv() const { return r[FCAP]; }
    __device__ __forceinline__ real c1() const { return r[FCAP + 1]; }
    __device__ __forceinline__ real c2() const { return r[FCAP + 2]; }
};

template <int FCAP, typename real>
__device__ __forceinline__ Rec<FCAP, real> rec_at(const real* __restrict__ rec, int n, int i, int j) {
    const real* r = rec + ((size_t)i * n + j) * Rec<FCAP, real>::size;
    return Rec<FCAP, real>{(const real*)__builtin_assume_aligned(r, Rec<FCAP, real>::size * sizeof(real))};
}

// Value of a state: applyStateSpaceTransform (LMM:1200-1212), exp in the log-normal
// state space, then the cap.
template <typename real>
__device__ __forceinline__ real to_value(real y, bool lognormal, bool capped, real cap) {
    const real v = lognormal ? dev_exp<real>(y) : y;
    return capped ? jmin(v, cap) : v;
}

// The increments dW_k(t_i) of one path, zero above the F factors (path-major layout
// [path][time index][factor]).
template <int FCAP, typename real>
__device__ __forceinline__ void load_increments(real (&dW)[FCAP], const real* __restrict__ dw, int64_t pc, int nT,
                                                int i, int F) {
#pragma unroll
    for (int k = 0; k < FCAP; k++) dW[k] = (k < F) ? dw[((size_t)pc * nT + i) * F + k] : (real)0;
}

} // namespace fm
