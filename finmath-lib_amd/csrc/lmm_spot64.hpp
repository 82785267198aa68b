// The Euler step of the FP64 spot kernel (lmm_spot.hpp), also run by its reverse sweep.
//
// The state of a forward is z_j = log2(L_j / s_j) with the scale s_j its initial value (1 where that
// is not positive; in the normal state space the state is the forward itself and s_j = 1): the
// exponential of a step needs no scaling of its argument, and a state near zero is rounded more
// finely than a logarithm of the forward. With E_j = L_j / s_j and c = 1/ln 2 (E_j = z_j and c = 1 in
// the normal state space) the step of an alive component is
//   E_j = 2^z_j
//   w   = c dt E_j / (E_j + e_j)               e_j = 1/(d_j s_j); c dt / (E_j + e_j) in the normal
//   T_k = T_k + w lambda_jk                    ascending j, from T_k = c dW_k
//   z_j = z_j + (h_j + sum_k T_k lambda_jk)    h_j = -1/2 variance_j c dt, 0
//   z_j = min(z_j, log2(cap / s_j))
// which is the drift and the diffusion of lmm_spot.hpp taken together: sum_k (c dt S_k + c dW_k)
// lambda_jk, with S_k the reference's factor sums. One pair of multiply-adds per factor replaces two
// products and two sums in the drift and one of each in the diffusion, and the state takes one
// rounding per step instead of one per factor. The record of (t_i, j) holds lambda_jk, h_j, the cap
// of z_j and e_j.
//
// The components are processed in pairs, unrolled over the register array: a pair's two exponentials
// and reciprocals are independent, which hides the latency of the FP64 pipeline and of the scalar
// loads of the two records, and a constant register index needs no indexed moves. A pair holds a
// fixed or absent forward beside an alive one where the alive range starts or ends at an odd
// index: its record has no loadings, so it adds an exact zero to every sum and to its state (a fixed
// forward that has overflowed is set aside first).
//
// Swaptions that exercise at t_i over consecutive tenor periods are valued by the same walk
// (SwaptionWalk): it has E_j and the reciprocal at hand, so a period of a swaption costs two
// operations and three more that its group shares, where a walk of its own needs another
// exponential and another reciprocal.
//
// The kernel is bound by the FP64 vector pipeline. At 40 forwards x 5 factors x 1,000,000 paths with 30
// swaptions it issues 38,600 vector instructions per wavefront (80,400 with rolled component loops,
// a general exponential and separate products and sums) and takes 1.55 ms (3.46 ms), the vector ALUs
// 0.78 busy (0.67) at four wavefronts per SIMD (three): the registers are held to 128 by reading the
// kernel's arguments where they are used and the increments when the step begins. Bringing the next
// pair's records into the scalar cache took it from 1.88 to 1.79 ms at three wavefronts; two sets of
// scalar registers for them instead spilled.
#pragma once

#include "lmm_chunks.hpp"

namespace fm {

typedef const double __attribute__((address_space(4)))* RecPtr;

// A record read whole into scalar registers (pieces of at most 64 bytes; a record is aligned to its size, or to 64).
template <int FCAP>
struct RecVec {
    static constexpr int size = rec_size_of(FCAP);
    static constexpr int W = size < 8 ? size : 8, N = size / W;
    typedef double V __attribute__((ext_vector_type(W)));
    V v[N];
    // record j of a time step whose first record is at rec
    __device__ __forceinline__ RecVec(RecPtr rec, int j) {
        typedef const V __attribute__((address_space(4)))* P;
#pragma unroll
        for (int q = 0; q < N; q++) v[q] = *(P)(rec + j * size + W * q);
    }
    __device__ __forceinline__ double at(int e) const { return v[e / W][e % W]; }
    __device__ __forceinline__ double lam(int k) const { return at(k); }
    __device__ __forceinline__ double h() const { return at(FCAP); }
    __device__ __forceinline__ double zcap() const { return at(FCAP + 1); }
    __device__ __forceinline__ double e() const { return at(FCAP + 2); }
};

// Up to kSwaptionGroup swaptions exercised at one time index over the periods [j0, j0 + periods):
//   V_g = sum_j P_j a_j (E_j - k_gj),   P_j = prod_{l <= j} 1/(1 + L_l d_l) = prod_{l <= j} e_l / (E_l + e_l)
// with a_j = s_j x period length x the discounting adjustments up to j and k_gj = strike / s_j, one
// table row {a, k_0 .. k_3, -, -, -} per period. V_g is the value of Swaption.java:150-190 for a
// notional of 1, its backward recursion written out as a sum.
struct SwaptionWalk {
    RecPtr table;
    int j0 = 0, periods = 0;
    double P = 1.0, V[kSwaptionGroup] = {0.0, 0.0, 0.0, 0.0};
    // brings component j's row (the nearest one where it has none) into the scalar cache
    __device__ __forceinline__ uint32_t touch(int j) const {
        typedef const volatile uint32_t __attribute__((address_space(4)))* WordPtr;
        const int i = j < j0 ? 0 : j - j0 < periods ? j - j0 : periods - 1;
        return *(WordPtr)(table + 8 * i);
    }
    __device__ __forceinline__ void period(int j, double E, double e, double r) {
        if ((unsigned)(j - j0) >= (unsigned)periods) return;
        typedef double Row __attribute__((ext_vector_type(8)));
        typedef const Row __attribute__((address_space(4)))* RowPtr;
        const Row row = *(RowPtr)(table + 8 * (j - j0));
        P = P * (e * r);
        const double Pa = P * row[0];
#pragma unroll
        for (int g = 0; g < kSwaptionGroup; g++) V[g] = fma(E - row[1 + g], Pa, V[g]);
    }
};

// Brings the tables of the launch into the L2 of each die, the workgroups of a die (consecutive ones lie on
// different dies) touching a share of the lines each. The tables have just been written, and wavefronts
// that walk them in step would all wait for each line as it first comes up: 100,000 paths, new tables of
// 102 KB and 30 swaptions, 265 us against 312 without this and SwaptionWalk::touch.
__device__ __forceinline__ void touch_tables(ArgPtr a) {
    const int part = blockIdx.x >> 3, parts = (gridDim.x + 7) >> 3, width = blockDim.x;
    uint32_t touched = 0;
    for (int l = part * width + (int)threadIdx.x; l < a->model_lines; l += parts * width)
        touched |= *(const volatile uint32_t*)((const char*)a->model + 128 * (size_t)l);
    for (int l = part * width + (int)threadIdx.x; l < a->table_lines; l += parts * width)
        touched |= *(const volatile uint32_t*)((const char*)a->tables + 128 * (size_t)l);
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" :: "v"(touched));
#endif
}

// The fixed forward J, which shares a pair with the first alive one: its record has no loadings, so a finite weight
// adds exact zeros, but an infinite one times zero is NaN. Where a path's weight may not be finite, in the log-normal state
// space where 2^z overflows and in the normal one where L or 1/(L + 1/d) does, the state is set to zero (a fixed
// forward is used no more). At the start of a pair this splits none of its work; a test of the weight in
// its midst cost the spot kernel 1 % and the kernels with a corrector 5 to 25 %. BRANCH: without a lost path the
// state is left alone; the general kernel spills hundreds of scalar registers with that branch, the reverse
// sweep without it.
template <bool lognormal, int FCAP, int J, bool BRANCH, typename Chunks>
__device__ __forceinline__ void set_aside_fixed64(Chunks& Y, RecPtr recs) {
    const double x = Y.template at<J>();
    const bool lost = lognormal ? !(x < 1000.0) : !(fabs(x) < 1e300) || x + recs[J * RecVec<FCAP>::size + FCAP + 2] == 0.0;
    if (BRANCH && __builtin_amdgcn_ballot_w64(lost) == 0) return;
    if constexpr (BRANCH) asm volatile("");         // hardly ever
    Y.template put<J>(lost ? 0.0 : x);
}

// The walk of the fixed forwards [sw.j0, first) before a step; value(x, j) is E_j.
template <int FCAP, typename Chunks, typename Value, typename Reciprocal>
__device__ __forceinline__ void walk_fixed64(Chunks& Y, RecPtr recs, int first, SwaptionWalk& sw, Value&& value,
                                             Reciprocal&& reciprocal) {
    if (sw.periods == 0) return;
#pragma unroll 1
    for (int j = sw.j0; j < first; j++) {
        const double E = value(Y.get(j), j), e = recs[j * RecVec<FCAP>::size + FCAP + 2];
        sw.period(j, E, e, reciprocal(E + e));
    }
}

// One Euler step of the alive components [first, n), in place. WALK: the walk's swaptions are valued
// on the states before the step, their forwards that are fixed at t_i ahead of it.
template <int NCH, int FCAP, bool lognormal, bool WALK, typename Chunks>
__device__ __forceinline__ void spot64_step(Chunks& Y, int n, int rec_n, int i, int first, double dt,
                                            const double (&dW)[FCAP], const double* rec, const Exp2Coef& ke,
                                            SwaptionWalk* sw) {
    RecPtr recs = (RecPtr)(uintptr_t)(rec + (size_t)i * rec_n * RecVec<FCAP>::size);
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+s"(recs));      // one base address for the step's records
#endif
    const double cdt = lognormal ? dt * kLog2E : dt;
    double T[FCAP];
#pragma unroll
    for (int k = 0; k < FCAP; k++) T[k] = lognormal ? dW[k] * kLog2E : dW[k];
    // 1 / b by the hardware reciprocal r0 corrected to third order: with e = 1 - b r0,
    // 1/b = r0 (1 + e + e^2 + ...); |e| < 2^-20, so the terms left out are below rounding
    auto reciprocal = [&](double b) -> double {
        const double r0 = __builtin_amdgcn_rcp(b);
        const double e = fma(-b, r0, 1.0);
        return fma(r0, fma(e, e, e), r0);
    };
    auto increment = [&](double w, const RecVec<FCAP>& R) -> double {
#pragma unroll
        for (int k = 0; k < FCAP; k++) T[k] = fma(w, R.lam(k), T[k]);
        double inc = R.h();
#pragma unroll
        for (int k = 0; k < FCAP; k++) inc = fma(T[k], R.lam(k), inc);
        return inc;
    };
    if constexpr (WALK)
        walk_fixed64<FCAP>(Y, recs, first, *sw, [&](double x, int) -> double { return lognormal ? fm_exp2(x, ke) : x; }, reciprocal);
    n = opaque(n);
    first = opaque(first);
    const unsigned alive = (unsigned)(n - first + 1);
    static_for<0, 4 * NCH>([&](auto Q) {
        constexpr int j = 2 * decltype(Q)::value;
        if ((unsigned)(j + 1 - first) < alive) {        // j + 1 >= first and j < n
            if (__builtin_expect(j < opaque(first), 0)) set_aside_fixed64<lognormal, FCAP, j, true>(Y, recs);
            const RecVec<FCAP> R0(recs, j), R1(recs, j + 1);
            __builtin_amdgcn_sched_barrier(0);          // both records are requested before the exponentials
            const double x0 = Y.template at<j>(), x1 = Y.template at<j + 1>();
            const double E0 = lognormal ? fm_exp2(x0, ke) : x0;
            const double E1 = lognormal ? fm_exp2(x1, ke) : x1;
            const double b0 = E0 + R0.e(), b1 = E1 + R1.e();
            // the next pair's records are brought into the scalar cache while this one runs (the table
            // of a model is several times that cache); a pair beyond the last reads its last record
            __builtin_amdgcn_sched_barrier(0);
            typedef const volatile uint32_t __attribute__((address_space(4)))* WordPtr;
            constexpr int step = RecVec<FCAP>::size;
            uint32_t t0 = *(WordPtr)(recs + (j + 2) * step), t1 = *(WordPtr)(recs + (j + 3) * step);
            const double r0 = reciprocal(b0), r1 = reciprocal(b1);
            if constexpr (WALK) {
                if (sw->periods > 0) {
                    const uint32_t t2 = sw->touch(j + 2), t3 = sw->touch(j + 3);
                    if (j >= opaque(first)) sw->period(j, E0, R0.e(), r0);
                    sw->period(j + 1, E1, R1.e(), r1);
#if defined(__HIP_DEVICE_COMPILE__)
                    asm volatile("" :: "s"(t2), "s"(t3));
#endif
                }
            }
            double y0 = x0 + increment((lognormal ? cdt * E0 : cdt) * r0, R0);
            double y1 = x1 + increment((lognormal ? cdt * E1 : cdt) * r1, R1);
            // the cap seldom binds: one comparison each (min(y, cap) keeps NaN, as a comparison does)
            if (__builtin_amdgcn_ballot_w64(y0 > R0.zcap() || y1 > R1.zcap()) != 0) {
                asm volatile("");       // a branch, not selects
                y0 = jmin(y0, R0.zcap());
                y1 = jmin(y1, R1.zcap());
            }
            Y.template put<j>(y0);
            Y.template put<j + 1>(y1);
#if defined(__HIP_DEVICE_COMPILE__)
            asm volatile("" :: "s"(t0), "s"(t1));
#endif
        }
    });
}

// The values of a walk's swaptions over Nsel, reduced into their slots.
__device__ __forceinline__ void reduce_walk(ConstArray<KProduct> products, int head,
                                            const double (&V)[kSwaptionGroup], double Nsel, bool active, int cnt,
                                            int lane, int64_t wave, double* wave_sum, double* wave_m2, int stride) {
    const int m = 1 + products[head].pad2;
    double x[kSwaptionGroup];
    int slot[kSwaptionGroup];
#pragma unroll
    for (int g = 0; g < kSwaptionGroup; g++) {
        const KProduct pg = products[head + (g < m ? g : 0)];
        x[g] = jmax0(V[g] * pg.notional) / Nsel;
        slot[g] = pg.out_slot;
    }
    reduce_slots4(x, m, active, cnt, cnt > 0 ? 1.0 / (double)cnt : 0.0, lane, wave, wave_sum, wave_m2, stride, slot);
}

} // namespace fm
