// The Euler step and the swaption walk of the FP32-mixed spot kernel (lmm_spot.hpp), also run by its
// reverse sweep.
//
// The state of a forward is its value; the step takes its logarithm with the hardware log2. Every
// operation is written with the contraction it has always been compiled with, since the adjoint
// differentiates these float paths and prices are compared in their last places:
//   w    = L / (L c1 + c2)                      1 / (L c1 + c2) in the normal state space
//   S_k  = S_k + w lambda_jk                    ascending j
//   mu_j = sum_k S_k lambda_jk + h_j
//   y    = ln 2 log2(L) + mu dt + sum_k dW_k lambda_jk
//   L    = min(2^(y log2 e), cap)
// Components are unrolled over the register array in pairs, as in lmm_spot64.hpp: a constant register
// index needs no indexed move, and two independent chains cover the latency of the transcendental
// unit and of the record loads. Where the alive range starts or ends at an odd index, the pair's other
// forward has a record without loadings, which adds exact zeros to the sums, and keeps its value (a fixed one
// that has overflowed is set aside first).
//
// The kernel is bound by vector issue: 40 forwards x 5 factors x 4,000,000 paths with 30 swaptions 3.7 ms
// at 1.0 vector ALU busy (5.53 ms and 0.72 with rolled loops and one record read per component), 80 x 10 x
// 1,000,000 paths 4.7 ms (7.20 ms, 0.60).
#pragma once

#include "lmm_chunks.hpp"

namespace fm {

typedef const float __attribute__((address_space(4)))* RecPtr32;

// The two records of a pair of components, read whole into scalar registers.
template <int FCAP>
struct PairRec32 {
    static constexpr int size = rec_size_of(FCAP);
    typedef float V __attribute__((ext_vector_type(2 * size)));
    V v;
    // records j and j + 1 of a time step whose first record is at rec. The read is volatile so that it
    // is issued here and not where its values are first used.
    __device__ __forceinline__ void read(RecPtr32 rec, int j) {
        typedef const volatile V __attribute__((address_space(4)))* P;
        v = *(P)(rec + j * size);
    }
    // wait for the read
    __device__ __forceinline__ void arrive() const {
#if defined(__HIP_DEVICE_COMPILE__)
        asm volatile("" :: "s"(v));
#endif
    }
    __device__ __forceinline__ float lam(int c, int k) const { return v[c * size + k]; }
    __device__ __forceinline__ float h(int c) const { return v[c * size + FCAP]; }
    __device__ __forceinline__ float c1(int c) const { return v[c * size + FCAP + 1]; }
    __device__ __forceinline__ float c2(int c) const { return v[c * size + FCAP + 2]; }
};

// A record read whole into scalar registers.
template <int FCAP>
struct RecVec32 {
    static constexpr int size = rec_size_of(FCAP);
    typedef float V __attribute__((ext_vector_type(size)));
    V v;
    __device__ __forceinline__ RecVec32(RecPtr32 rec, int j) {
        typedef const V __attribute__((address_space(4)))* P;
        v = *(P)(rec + j * size);
    }
    __device__ __forceinline__ float lam(int k) const { return v[k]; }
};

// One Euler step of the alive components [first, n), in place.
template <int NCH, int FCAP, bool lognormal, typename Chunks>
__device__ __forceinline__ void spot32_step(Chunks& Y, int n, int rec_n, int i, int first, float dt, const float (&dW)[FCAP],
                                            const float* rec, float cap) {
    RecPtr32 recs = (RecPtr32)(uintptr_t)(rec + (size_t)i * rec_n * rec_size_of(FCAP));
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+s"(recs));      // one base address for the step's records
#endif
    float S[FCAP];
#pragma unroll
    for (int k = 0; k < FCAP; k++) S[k] = 0.0f;
    auto component = [&](auto C, float L, float l2, float w, const PairRec32<FCAP>& R) -> float {
        constexpr int c = decltype(C)::value;
#pragma unroll
        for (int k = 0; k < FCAP; k++) S[k] = fmaf(w, R.lam(c, k), S[k]);
        float mu;
        if constexpr (FCAP == 1) {
            mu = fmaf(S[0], R.lam(c, 0), R.h(c));
        } else {
            mu = fmaf(S[0], R.lam(c, 0), S[1] * R.lam(c, 1));
#pragma unroll
            for (int k = 2; k < FCAP; k++) mu = fmaf(S[k], R.lam(c, k), mu);
            mu = mu + R.h(c);
        }
        float y;
        if constexpr (lognormal) y = fmaf(l2, 0.693147180559945309f, mu * dt);
        else y = fmaf(mu, dt, L);
#pragma unroll
        for (int k = 0; k < FCAP; k++) y = fmaf(dW[k], R.lam(c, k), y);
        return lognormal ? dev_exp<float>(y) : y;
    };
    n = opaque(n);
    const unsigned alive = (unsigned)(n - first + 1);
    // a pair's records are read while the pair before it runs: two sets of scalar registers, even pairs
    // in A and odd pairs in B (the pair after the last reads the table's padding)
    PairRec32<FCAP> A, B;
    if (first & 2) B.read(recs, first & ~1);
    else A.read(recs, first & ~1);
    static_for<0, 8 * NCH>([&](auto Q) {
        constexpr int j = 2 * decltype(Q)::value;
        if ((unsigned)(j + 1 - first) < alive) {        // j + 1 >= first and j < n
            PairRec32<FCAP>& R = (j & 2) ? B : A;
            R.arrive();
            if (__builtin_expect(j < first, 0)) {
                // the fixed one of the pair: its weight times no loading is zero unless it is NaN (an infinite forward,
                // log-normal) or infinite (one of -1/d, normal): then the path's value, used no more, is set to zero
                const float x = Y.template at<j>();
                const bool lost = lognormal ? !(x < HUGE_VALF) : fmaf(x, R.c1(0), R.c2(0)) == 0.0f;
                if (__builtin_amdgcn_ballot_w64(lost) != 0) {
                    asm volatile("");       // hardly ever
                    Y.template put<j>(lost ? 0.0f : x);
                }
            }
            ((j & 2) ? A : B).read(recs, j + 2);
            __builtin_amdgcn_sched_barrier(0);
            const float L0 = Y.template at<j>(), L1 = Y.template at<j + 1>();
            const float l0 = lognormal ? __builtin_amdgcn_logf(L0) : 0.0f;
            const float l1 = lognormal ? __builtin_amdgcn_logf(L1) : 0.0f;
            const float r0 = __builtin_amdgcn_rcpf(fmaf(L0, R.c1(0), R.c2(0)));
            const float r1 = __builtin_amdgcn_rcpf(fmaf(L1, R.c1(1), R.c2(1)));
            float v0 = component(std::integral_constant<int, 0>{}, L0, l0, lognormal ? L0 * r0 : r0, R);
            float v1 = component(std::integral_constant<int, 1>{}, L1, l1, lognormal ? L1 * r1 : r1, R);
            // the cap seldom binds: one comparison each (min(v, cap) keeps NaN, as a comparison does)
            if (__builtin_amdgcn_ballot_w64(v0 > cap || v1 > cap) != 0) {
                asm volatile("");
                v0 = jmin(v0, cap);
                v1 = jmin(v1, cap);
            }
            if (j < first || j + 1 >= n) {              // one of the pair is fixed or absent
                asm volatile("");
                v0 = j < first ? L0 : v0;
                v1 = j + 1 >= n ? 0.0f : v1;
            }
            Y.template put<j>(v0);
            Y.template put<j + 1>(v1);
        }
    });
}

// A group of up to four swaptions over the same periods, valued backwards as Swaption.java:150-190 does,
// V = ((V + payoff) / (1 + L tau)) adj, with the reciprocal shared by the group. One table row
// {tau, period length, adjustment, -, strikes} per period.
template <int NCH, typename Chunks>
__device__ __forceinline__ void swaption_walk32(Chunks& Y, const float* table, int j0, int periods, int m,
                                                const float (&notional)[kSwaptionGroup], float (&V)[kSwaptionGroup]) {
    typedef float Row __attribute__((ext_vector_type(8)));
    typedef const Row __attribute__((address_space(4)))* RowPtr;
    RowPtr rows = (RowPtr)(uintptr_t)table - j0;
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+s"(rows));
#endif
#pragma unroll
    for (int g = 0; g < kSwaptionGroup; g++) V[g] = 0.0f;
    static_for<0, 16 * NCH>([&](auto Q) {
        constexpr int j = 16 * NCH - 1 - decltype(Q)::value;
        if ((unsigned)(j - j0) < (unsigned)periods) {
            const Row row = rows[j];
            const float L = Y.template at<j>();
            const float r = __builtin_amdgcn_rcpf(fmaf(L, row[0], 1.0f));
            auto member = [&](int g) {
                V[g] = fmaf((L - row[4 + g]) * row[1], notional[g], V[g]);
                V[g] = V[g] * r;
                V[g] = V[g] * row[2];
            };
            member(0);
            if (m > 1) {
                member(1);
                if (m > 2) {
                    member(2);
                    if (m > 3) member(3);
                }
            }
        }
    });
}

} // namespace fm
