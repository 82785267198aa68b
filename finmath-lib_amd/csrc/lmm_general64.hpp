// General path kernel in FP64: the terminal or spot measure, the carried-state EULER and
// PREDICTOR_CORRECTOR schemes and their functional forms, both state spaces, and the local-volatility
// and stochastic-volatility wrappers of the covariance model. (FP32-mixed: lmm_general.hpp.)
//
// The states and the step are those of lmm_spot64.hpp: z_j = log2(L_j / s_j) (the forward itself in the
// normal state space), E_j = L_j / s_j, c = 1/ln 2 (1 in the normal state space), components in unrolled
// pairs. In the measure's order of components (spot ascending, terminal descending):
//   loadings   g_j lambda_jk, g_j = (a_j E_j + b_ij) S(t_i) with the local-volatility factor
//              (L - L alpha) + b_ij (a_j = s_j (1 - alpha)) and the stochastic volatility scaling
//              S(t_i); 1 without wrappers
//   w_j        c dt E_j/(E_j + e_j) (c dt/(E_j + e_j) normal), negative under the terminal measure
//   T_k        c dW_k plus w_l g_l lambda_lk of the components before j, and of j itself (spot)
//   z'_j       z_j + h_j + g_j sum_k T_k lambda_jk
//   h_j        -1/2 c dt variance_j; with wrappers -1/2 c dt g_j^2 sum_k lambda_jk^2
//              (AbstractLIBORCovarianceModel.getCovariance, covariance/AbstractLIBORCovarianceModel.java:79-92)
// PREDICTOR_CORRECTOR (EulerSchemeFromProcessModel.java:292-314): w'_j, g'_j and h'_j from the predicted
// value of z'_j, and half the difference of the two drifts is added. Component j's two drifts depend
// only on the components before it in the measure's order, so one pass computes the predictor's drift
// and state, the corrector's drift on the predicted value and the corrected state.
// Carried schemes cap the value min(2^z, cap/s_j) where it is read; functional ones cap the state.
//
// The FP64 vector pipeline bounds it, as it does the spot kernel. 200,000 paths, 40 forwards,
// 5 factors, 40 steps, terminal measure, PREDICTOR_CORRECTOR: 0.86 ms
// (1.86 ms for the kernel with natural exponentials, divisions and rolled components that this one replaces);
// 150,000 paths, spot measure, normal, stochastic volatility: 0.31 ms (1.50 ms).
#pragma once

#include "lmm_spot64.hpp"

namespace fm {

// The step's arguments that do not change with the component.
struct General64 {
    int n, first;
    bool carry;
    double dt, sv;              // sv: the path's stochastic volatility scaling at t_i
    RecPtr recs;                // records of t_i: lambda, h (sum of squares of lambda for the wrappers), cap, e
    RecPtr lv;                  // wrappers: pairs {a_j, b_ij} of t_i
};

template <int NCH, int FCAP, bool TERMINAL, bool PC, bool LV, bool lognormal, typename Chunks>
__device__ __forceinline__ void general64_step(Chunks& Y, const General64& s, const double (&dW)[FCAP],
                                               const Exp2Coef& ke, SwaptionWalk* sw) {
    constexpr bool WALK = !TERMINAL;
    const int n = opaque(s.n);
    int first = s.first;
    const double cdt = lognormal ? s.dt * kLog2E : s.dt;
    // T: diffusion and drift sums. PC: D, the corrector's less the predictor's drift sums; with wrappers
    // the two have their own loadings, so Sc holds the corrector's sums and the predictor's drift is
    // taken out of T.
    double T[FCAP], D[PC ? FCAP : 1];
#pragma unroll
    for (int k = 0; k < FCAP; k++) {
        T[k] = lognormal ? dW[k] * kLog2E : dW[k];
        if constexpr (PC) D[k] = 0.0;
    }
    auto reciprocal = [&](double b) -> double {
        const double r0 = __builtin_amdgcn_rcp(b);
        const double e = fma(-b, r0, 1.0);
        return fma(r0, fma(e, e, e), r0);
    };
    auto value = [&](double z, double cap) -> double {
        double E = lognormal ? fm_exp2(z, ke) : z;
        if (s.carry) E = jmin(E, cap);
        return E;
    };
    auto weight = [&](double E, double r) -> double {
        const double w = lognormal ? cdt * E : cdt;
        return TERMINAL ? -w * r : w * r;
    };
    auto dot = [&](const double (&V)[FCAP], const RecVec<FCAP>& R, double x) -> double {
#pragma unroll
        for (int k = 0; k < FCAP; k++) x = fma(V[k], R.lam(k), x);
        return x;
    };
    // drift and diffusion of one component from its value E and reciprocal r; returns the new state
    auto component = [&](double z, double E, double r, const RecVec<FCAP>& R, double a, double b) -> double {
        const double w = weight(E, r);
        double g = 1.0, h = R.h();
        if constexpr (LV) {
            g = fma(a, E, b) * s.sv;
            h = lognormal ? (-0.5 * cdt) * (g * g) * R.h() : 0.0;
        }
        const double wg = LV ? w * g : w;
        double zn;
        if constexpr (!TERMINAL) {
#pragma unroll
            for (int k = 0; k < FCAP; k++) T[k] = fma(wg, R.lam(k), T[k]);
        }
        if constexpr (LV) zn = z + fma(g, dot(T, R, 0.0), h);
        else zn = z + dot(T, R, h);
        if constexpr (PC) {
            double zc = zn;
            if (!s.carry) zc = jmin(zn, R.zcap());      // the predicted value is capped in either form
            const double Ep = value(zc, R.zcap());
            const double wp = weight(Ep, reciprocal(Ep + R.e()));
            if constexpr (LV) {
                const double gp = fma(a, Ep, b) * s.sv;
                const double hp = lognormal ? (-0.5 * cdt) * (gp * gp) * R.h() : 0.0;
                // the predictor's drift alone: T without the increments
                double m = dot(T, R, 0.0);
#pragma unroll
                for (int k = 0; k < FCAP; k++) m = fma(lognormal ? dW[k] * -kLog2E : -dW[k], R.lam(k), m);
                const double wgp = wp * gp;
                if constexpr (!TERMINAL) {
#pragma unroll
                    for (int k = 0; k < FCAP; k++) D[k] = fma(wgp, R.lam(k), D[k]);
                }
                const double mp = dot(D, R, 0.0);
                zn = fma(0.5, (fma(gp, mp, hp) - fma(g, m, h)), zn);
                if constexpr (TERMINAL) {
#pragma unroll
                    for (int k = 0; k < FCAP; k++) D[k] = fma(wgp, R.lam(k), D[k]);
                }
            } else {
                const double dw = wp - w;
                if constexpr (!TERMINAL) {
#pragma unroll
                    for (int k = 0; k < FCAP; k++) D[k] = fma(dw, R.lam(k), D[k]);
                }
                zn = fma(0.5, dot(D, R, 0.0), zn);
                if constexpr (TERMINAL) {
#pragma unroll
                    for (int k = 0; k < FCAP; k++) D[k] = fma(dw, R.lam(k), D[k]);
                }
            }
        }
        if constexpr (TERMINAL) {
#pragma unroll
            for (int k = 0; k < FCAP; k++) T[k] = fma(wg, R.lam(k), T[k]);
        }
        return zn;
    };
    if constexpr (WALK)
        walk_fixed64<FCAP>(Y, s.recs, first, *sw, [&](double x, int j) -> double {
            return value(x, s.recs[j * RecVec<FCAP>::size + FCAP + 1]);
        }, reciprocal);
    first = opaque(first);
    const unsigned alive = (unsigned)(n - first + 1);
    static_for<0, 4 * NCH>([&](auto Q) {
        constexpr int q = decltype(Q)::value;
        constexpr int j = 2 * (TERMINAL ? 4 * NCH - 1 - q : q);
        if ((unsigned)(j + 1 - first) < alive) {        // j + 1 >= first and j < n
            // (under the terminal measure the fixed forward comes last)
            if (WALK && __builtin_expect(j < first, 0)) set_aside_fixed64<lognormal, FCAP, j, false>(Y, s.recs);
            const RecVec<FCAP> R0(s.recs, j), R1(s.recs, j + 1);
            typedef double V4 __attribute__((ext_vector_type(4)));
            typedef const V4 __attribute__((address_space(4)))* P4;
            V4 l = {0.0, 1.0, 0.0, 1.0};
            if constexpr (LV) l = *(P4)(s.lv + 2 * j);
            __builtin_amdgcn_sched_barrier(0);          // the records are requested before the exponentials
            const double x0 = Y.template at<j>(), x1 = Y.template at<j + 1>();
            const double E0 = value(x0, R0.zcap()), E1 = value(x1, R1.zcap());
            const double r0 = reciprocal(E0 + R0.e()), r1 = reciprocal(E1 + R1.e());
            if constexpr (WALK) {
                if (sw->periods > 0) {
                    if (j >= first) sw->period(j, E0, R0.e(), r0);
                    sw->period(j + 1, E1, R1.e(), r1);
                }
            }
            double y0, y1;
            if constexpr (TERMINAL) {
                y1 = component(x1, E1, r1, R1, l[2], l[3]);
                y0 = component(x0, E0, r0, R0, l[0], l[1]);
            } else {
                y0 = component(x0, E0, r0, R0, l[0], l[1]);
                y1 = component(x1, E1, r1, R1, l[2], l[3]);
            }
            // the cap seldom binds: one comparison each (min(y, cap) keeps NaN, as a comparison does)
            if (!s.carry && __builtin_amdgcn_ballot_w64(y0 > R0.zcap() || y1 > R1.zcap()) != 0) {
                asm volatile("");       // a branch, not selects
                y0 = jmin(y0, R0.zcap());
                y1 = jmin(y1, R1.zcap());
            }
            Y.template put<j>(y0);
            Y.template put<j + 1>(y1);
        }
    });
}

// One thread per path, as lmm_spot_kernel. Under the terminal measure N(T_k) = prod_{l >= k} 1/(1 + L_l(T_k)
// d_l) (LMM:1020-1042) is the reciprocal of the product of 1 + L_l d_l, formed at the time index of T_k.
//
// Four waves per SIMD where the registers allow them without scratch memory (the spot measure's corrector and
// the wrappers need up to 167, three waves): at 200,000 paths three are one pass and a nearly empty
// second one, 1.00 ms against 0.93 (before the model's tables were touched ahead, which took the four to 0.86).
template <int NCH, int FCAP, bool TERMINAL, bool PC, bool LV, bool lognormal>
__global__ void __launch_bounds__(kStepThreads) __attribute__((amdgpu_waves_per_eu(NCH <= 5 && FCAP <= 5 ? (LV || (PC && !TERMINAL) ? 3 : 4) : 1)))
lmm_general64_kernel(const StepArgs) {
    constexpr int W = chunk_width<double>();
    ArgPtr a = kernel_arguments();
    const uint32_t p0 = blockIdx.x * (uint32_t)kStepThreads + threadIdx.x;      // P < 2^31
    const int lane = threadIdx.x & 63;
    const int64_t wave = (int64_t)blockIdx.x * (kStepThreads / 64) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const Exp2Coef ke;
    touch_tables(a);
    ChunkedForwards<NCH, double> Y;
    {
        const ConstArray<double> z0{a->Y0};
        static_for<0, W * NCH>([&](auto J) {
            constexpr int j = decltype(J)::value;
            Y.template put<j>(z0[j]);           // zeros beyond the n forwards
            if constexpr (j % 8 == 7) __builtin_amdgcn_sched_barrier(0);
        });
    }
    double N = 1.0, Nprev = 1.0;   // unadjusted numeraire N(T_knum) and the one before it
    double N0 = 1.0;               // N(T_0) (terminal measure)
    int kcur = 0, knum = 0;
    int qp = 0;

    for (int ti = 0;; ti++) {
        a = kernel_arguments();
        const int P = a->P, n = a->n;
        const int64_t p = p0;
        const bool active = p < P, carry = a->carry != 0;
        const int64_t pc = active ? p : (int64_t)P - 1;
        const int cnt = (int)((int64_t)P - wave * 64 > 64 ? 64 : ((int64_t)P - wave * 64));
        const ConstArray<double> lead{a->lead};
        const double cap = a->cap;
        auto val = [&](double z, int j) -> double {
            const double L = lognormal ? lead[j] * fm_exp2(z, ke) : z;
            return carry ? jmin(L, cap) : L;
        };
        const int num_slots = a->num_slots, stride = num_slots + n + 1;
        const ConstArray<int32_t> tenor_ti{a->tenor_time_index};
        if constexpr (TERMINAL) {
            while (kcur <= n && tenor_ti[kcur] <= ti) {
                double prod = 1.0;
                const int from = kcur;
                const unsigned left = (unsigned)(n - from);
                static_for<0, W * NCH>([&](auto J) {
                    constexpr int j = decltype(J)::value;
                    if ((unsigned)(j - from) < left) {
                        double z = Y.template at<j>();
#if defined(__HIP_DEVICE_COMPILE__)
                        asm volatile("" : "+v"(z));     // the powers are not to be formed ahead of the loop
#endif
                        prod = prod * fma(val(z, j), ConstArray<double>{a->delta}[j], 1.0);
                    }
                });
                const double Nn = 1.0 / prod;
                if (kcur == 0) N0 = Nn;
                Nprev = N; N = Nn; knum = kcur; kcur++;
                // sum of N(T_0)/N(T_k) over paths (numeraire adjustment average)
                const double s = wave_reduce_sum(active ? prod * N0 : 0.0);
                if (lane == 0 && cnt > 0) a->wave_sum[(size_t)wave * stride + num_slots + knum] = s;
                if (a->numeraire && active) a->numeraire[(size_t)knum * P + p] = N;
            }
        } else {
            // ---- N(T_{k+1}) = N(T_k).accrue(L_k(T_k), d_k) once L_k is final (LMM:1050-1066)
            while (kcur < n && tenor_ti[kcur] <= ti) {
                const double Lk = val(Y.get(kcur), kcur);
                const double dk = ConstArray<double>{a->delta}[kcur];
                double Nn;
                if (kcur == 0)      Nn = Lk * (dk * 1.0) + 1.0;      // Scalar.accrue of Scalar 1.0
                else if (kcur == 1) Nn = Lk * (dk * N) + N;          // Scalar.accrue of a stochastic rate
                else                Nn = N * (1 + Lk * dk);          // RandomVariableFromDoubleArray.accrue
                Nprev = N; N = Nn; kcur++; knum = kcur;
                // sum of 1/N(T_k) over paths (numeraire adjustment average)
                const double s = wave_reduce_sum(active ? (1.0 / N) * 1.0 : 0.0);
                if (lane == 0 && cnt > 0) a->wave_sum[(size_t)wave * stride + num_slots + kcur] = s;
                if (a->numeraire && active) a->numeraire[(size_t)kcur * P + p] = N;
            }
        }
        // ---- products evaluated at this time index; under the spot measure a swaption group with a walk
        // table is left to the step
        const ConstArray<KProduct> products{a->products};
        int walk = -1;
        auto walk_group = [&](int i, const KProduct& pr) -> bool {
            if (TERMINAL || pr.walk < 0) return false;
            walk = i;
            return true;
        };
        eval_products_at<true, double>(ti, qp, a->num_products, products, ConstArray<KPeriod>{a->periods},
                                       ConstArray<double>{a->delta}, N, Nprev, knum, Y, val, active, a->contrib, p, P,
                                       [&](double x, int slot) {
                                           reduce_slot(x, active, cnt, lane, wave, a->wave_sum, a->wave_m2, stride, slot);
                                       }, walk_group);
        const int nT = a->nT;
        if (ti == nT) break;

        // ---- step ti -> ti+1
        const ConstArray<double> times{a->times};
        const int F = opaque(a->F), rec_n = a->rec_n;
        const double* dwp = (const double*)a->dw + ((size_t)pc * nT + ti) * F;
        double dW[FCAP];
        if (F == FCAP) {
#pragma unroll
            for (int k = 0; k < FCAP; k++) dW[k] = dwp[k];
        } else {
#pragma unroll
            for (int k = 0; k < FCAP; k++) dW[k] = k < F ? dwp[k] : 0.0;
        }
        General64 s;
        s.n = n;
        s.first = ConstArray<int32_t>{a->first_alive}[ti];
        s.carry = carry;
        s.dt = times[ti + 1] - times[ti];
        s.sv = (LV && a->svs) ? ((const double*)a->svs)[(size_t)ti * P + pc] : 1.0;
        s.recs = (RecPtr)(uintptr_t)((const double*)a->rec + (size_t)ti * rec_n * rec_size_of(FCAP));
        s.lv = LV ? (RecPtr)(uintptr_t)((const double*)a->lvb + (size_t)ti * rec_n * 2) : s.recs;
#if defined(__HIP_DEVICE_COMPILE__)
        asm volatile("" : "+s"(s.recs), "+s"(s.lv));
#endif
        SwaptionWalk sw;
        sw.table = (RecPtr)(uintptr_t)a->walk;
        if (walk >= 0) {
            const KProduct pr = products[walk];
            sw.table += 8 * pr.walk;
            sw.j0 = pr.first_j;
            sw.periods = pr.num_periods;
        }
        general64_step<NCH, FCAP, TERMINAL, PC, LV, lognormal>(Y, s, dW, ke, &sw);
        if (walk >= 0)
            reduce_walk(products, walk, sw.V, products[walk].num_k == knum ? N : Nprev, active, cnt, lane, wave,
                        a->wave_sum, a->wave_m2, stride);
        if (a->paths) {
            const ConstArray<int32_t> row{a->row_of + (size_t)(ti + 1) * n};
            double* paths = (double*)a->paths + pc;
            static_for<0, NCH>([&](auto Q) {
                constexpr int q = decltype(Q)::value;
                const int j1 = n < W * q + W ? n : W * q + W;
#pragma unroll 1
                for (int j = s.first > W * q ? s.first : W * q; j < j1; j++) {
                    const double v = val(Y.template ch<q>()[j - W * q], j);
                    if (active) paths[(size_t)row[j] * P] = v;
                }
            });
        }
    }
}

template <int NCH, int FCAP, bool TERMINAL, bool PC, bool LV>
void launch_general64_m(const StepArgs& a, hipStream_t stream) {
    const dim3 grid((unsigned)(((int64_t)a.P + kStepThreads - 1) / kStepThreads));
    if (a.lognormal)
        hipLaunchKernelGGL((lmm_general64_kernel<NCH, FCAP, TERMINAL, PC, LV, true>), grid, dim3(kStepThreads), 0, stream, a);
    else
        hipLaunchKernelGGL((lmm_general64_kernel<NCH, FCAP, TERMINAL, PC, LV, false>), grid, dim3(kStepThreads), 0, stream, a);
    HIP_CHECK(hipGetLastError());
}

template <int NCH, bool PC, bool LV>
void launch_general64_n(const StepArgs& a, hipStream_t stream) {
    auto with = [&](auto fcap) {
        constexpr int FCAP = decltype(fcap)::value;
        if (a.terminal) launch_general64_m<NCH, FCAP, true, PC, LV>(a, stream);
        else launch_general64_m<NCH, FCAP, false, PC, LV>(a, stream);
    };
    if (a.F <= 3) with(std::integral_constant<int, 3>{});
    else if (a.F <= 5) with(std::integral_constant<int, 5>{});
    else if (a.F <= 10) with(std::integral_constant<int, 10>{});
    else throw FmError(FM_ERR_UNSUPPORTED, "number of factors above 10 is not supported by the path kernel");
}

// Capacities 24, 40 and 80 forwards and 3, 5, 10 factors: fewer instantiations than the spot kernel.
template <bool PC, bool LV>
void launch_general64(const StepArgs& a, hipStream_t stream) {
    if (a.n <= 24) launch_general64_n<3, PC, LV>(a, stream);
    else if (a.n <= 40) launch_general64_n<5, PC, LV>(a, stream);
    else if (a.n <= 80) launch_general64_n<10, PC, LV>(a, stream);
    else throw FmError(FM_ERR_UNSUPPORTED, "more than 80 forward rates are not supported by the path kernel");
}

} // namespace fm
