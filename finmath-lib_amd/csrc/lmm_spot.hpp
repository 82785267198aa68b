// Spot-measure Euler path kernel (EULER_FUNCTIONAL, and EULER where it is the same scheme):
// the pricing and simulation pass of the plain model, FP64 or FP32-mixed.
//
// Per time step t_i -> t_{i+1} and alive component j (T_j > t_i), in the order of
// LIBORMarketModelFromCovarianceModel.getDrift
// (montecarlo/interestrate/models/LIBORMarketModelFromCovarianceModel.java:1144-1160,1183-1189)
// and EulerSchemeFromProcessModel (montecarlo/process/EulerSchemeFromProcessModel.java:232-256):
//   w    = 1 / (L_j * (d_j/d_j) + 1/d_j)        Scalar.discount (stochastic/Scalar.java:320-328)
//   w    = w * L_j                               (log-normal state space)
//   S_k  = S_k + w * lambda_jk                   ascending j
//   mu_j = sum_k S_k * lambda_jk + variance_j * (-0.5)
//   Y_j  = Y_j + mu_j * dt + sum_k dW_k * lambda_jk
//   L_j  = min(exp(Y_j), cap)
// FP64 (lmm_spot64.hpp): the state, a base-2 log-forward, is carried from step to step.
// EULER_FUNCTIONAL re-derives it from the value as log(min(exp(Y), cap)), which gives back Y up to one
// rounding (exactly whenever the log-forward is at least 2 in magnitude, that is for forwards below
// 13.5 %); the cap is applied to the state. Products read L_j where they are evaluated.
// FP32-mixed (lmm_spot32.hpp): the value is carried and the state re-derived each step with the
// hardware logarithm. The adjoint's forward pass is this kernel, so it sees the priced float paths.
//
// Layout: the forwards of a path live in registers as chunks of sixteen VGPRs (eight FP64 or sixteen
// FP32 forwards). The step is unrolled over them; products at run-time indices read them with an
// indexed register move (s_set_gpr_idx_on). The step's model records are read through the scalar
// cache.
#pragma once

#include "lmm_chunks.hpp"
#include "lmm_spot32.hpp"
#include "lmm_spot64.hpp"

namespace fm {

// One thread per path, its states in NCH chunks of sixteen registers. Per time index: checkpoints (the
// adjoint's forward pass), numeraire updates, the products evaluated there, the Euler step with its
// swaption walk, and the new forwards when the process is stored.
template <int NCH, int FCAP, typename real, bool lognormal>
__global__ void __launch_bounds__(kStepThreads)
__attribute__((amdgpu_waves_per_eu(FCAP > 5 ? 1 : sizeof(real) == 4 && NCH <= 3 ? 5 : NCH <= 5 ? 4 : 1)))
lmm_spot_kernel(const StepArgs) {
    constexpr int W = chunk_width<real>();
    constexpr bool D = sizeof(real) == 8;
    ArgPtr a = kernel_arguments();
    const uint32_t p0 = blockIdx.x * (uint32_t)kStepThreads + threadIdx.x;      // P < 2^31
    const int lane = threadIdx.x & 63;
    // the wavefront index, uniform: kept in a scalar register
    const int64_t wave = (int64_t)blockIdx.x * (kStepThreads / 64) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const Exp2Coef ke;
    if constexpr (D) touch_tables(a);

    ChunkedForwards<NCH, real> Y;
    {
        const ConstArray<double> z0{a->Y0};
        static_for<0, W * NCH>([&](auto J) {
            constexpr int j = decltype(J)::value;
            Y.template put<j>((real)z0[j]);     // zeros beyond the n forwards
            if constexpr (j % 8 == 7) __builtin_amdgcn_sched_barrier(0);    // a chunk's scalar loads at a time
        });
    }
    double N = 1.0, Nprev = 1.0;   // unadjusted numeraire N(T_knum) and the one before it
    int kcur = 0, knum = 0;
    int qp = 0;
    for (int ti = 0;; ti++) {
        a = kernel_arguments();
        const int P = a->P, n = a->n;
        const int64_t p = p0;
        const bool active = p < P;
        const int64_t pc = active ? p : (int64_t)P - 1;
        const int cnt = (int)((int64_t)P - wave * 64 > 64 ? 64 : ((int64_t)P - wave * 64));
        const ConstArray<double> lead{a->lead};
        auto val = [&](real z, int j) -> real {
            if constexpr (D && lognormal) return lead[j] * fm_exp2(z, ke);
            else return z;
        };
        // ---- the carried states every ckpt_stride steps, for the adjoint's reverse sweep:
        // [ti / stride][j][P], stored non-temporal (read back only by the sweep, after this pass)
        if (a->ckpt && (ti % a->ckpt_stride) == 0) {
            const int c = ti / a->ckpt_stride, cfirst = ConstArray<int32_t>{a->ckpt_first}[c];
            real* to = (real*)a->ckpt + (size_t)c * n * P + pc;
            static_for<0, W * NCH>([&](auto J) {
                constexpr int j = decltype(J)::value;
                if ((unsigned)(j - cfirst) < (unsigned)(n - cfirst) && active)
                    __builtin_nontemporal_store(Y.template at<j>(), to);
                to += P;
            });
        }
        // ---- N(T_{k+1}) = N(T_k).accrue(L_k(T_k), d_k) once L_k is final (LMM:1050-1066)
        const int num_slots = a->num_slots, stride = num_slots + n + 1;
        while (kcur < n && ConstArray<int32_t>{a->tenor_time_index}[kcur] <= ti) {
            const double Lk = (double)val(Y.get(kcur), kcur);
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
        // ---- products evaluated at this time index. A swaption group with a walk table is left to the
        // Euler step (FP64), or valued by an unrolled walk (FP32).
        const ConstArray<KProduct> products{a->products};
        int walk = -1;
        auto walk_group = [&](int i, const KProduct& pr) -> bool {
            if (pr.walk < 0) return false;
            if constexpr (D) {
                walk = i;
            } else {
                float V[kSwaptionGroup], notional[kSwaptionGroup];
#pragma unroll
                for (int g = 0; g < kSwaptionGroup; g++)
                    notional[g] = (float)products[i + (g <= pr.pad2 ? g : 0)].notional;
                swaption_walk32<NCH>(Y, (const float*)a->walk + 8 * pr.walk, pr.first_j, pr.num_periods, 1 + pr.pad2,
                                     notional, V);
                double x[kSwaptionGroup];
                int slot[kSwaptionGroup];
#pragma unroll
                for (int g = 0; g < kSwaptionGroup; g++) {
                    x[g] = (double)jmax0(V[g]) / (pr.num_k == knum ? N : Nprev);
                    slot[g] = products[i + (g <= pr.pad2 ? g : 0)].out_slot;
                }
                reduce_slots4(x, 1 + pr.pad2, active, cnt, cnt > 0 ? 1.0 / (double)cnt : 0.0, lane, wave, a->wave_sum,
                              a->wave_m2, stride, slot);
            }
            return true;
        };
        eval_products_at<D, real>(ti, qp, a->num_products, products, ConstArray<KPeriod>{a->periods},
                                       ConstArray<double>{a->delta}, N, Nprev, knum, Y, val, active, a->contrib, p, P,
                                       [&](double x, int slot) {
                                           reduce_slot(x, active, cnt, lane, wave, a->wave_sum, a->wave_m2, stride, slot);
                                       }, walk_group);
        const int nT = a->nT;
        if (ti == nT) break;

        // ---- Euler step ti -> ti+1
        const ConstArray<double> times{a->times};
        const real dt = (real)(times[ti + 1] - times[ti]);
        const int first = ConstArray<int32_t>{a->first_alive}[ti];
        // the step's increments. Each lane reads its own line every third step or so, and the lines in flight are
        // the whole L2: a touch of the next step's element made it fetch them once more (1.61 ms against 1.54 at
        // 1,000,000 FP64 paths, 40 x 5; 3.9 against 3.7 at 4,000,000 FP32 paths; 5.0 against 4.7 at 80 x 10).
        const int F = a->F;
        const real* dwp = (const real*)a->dw + ((size_t)pc * nT + ti) * F;
        real dW[FCAP];
        if (F == FCAP) {
#pragma unroll
            for (int k = 0; k < FCAP; k++) dW[k] = dwp[k];
        } else {
#pragma unroll
            for (int k = 0; k < FCAP; k++) dW[k] = k < F ? dwp[k] : (real)0;
        }
        if constexpr (D) {
            SwaptionWalk sw;
            sw.table = (RecPtr)(uintptr_t)a->walk;
            if (walk >= 0) {
                const KProduct pr = products[walk];
                sw.table += 8 * pr.walk;
                sw.j0 = pr.first_j;
                sw.periods = pr.num_periods;
            }
            spot64_step<NCH, FCAP, lognormal, true>(Y, n, a->rec_n, ti, first, dt, dW, (const double*)a->rec, ke, &sw);
            if (walk >= 0)
                reduce_walk(products, walk, sw.V, products[walk].num_k == knum ? N : Nprev, active, cnt, lane, wave,
                            a->wave_sum, a->wave_m2, stride);
        } else {
            spot32_step<NCH, FCAP, lognormal>(Y, n, a->rec_n, ti, first, dt, dW, (const float*)a->rec, (float)a->cap);
        }
        if (a->paths) {
            const ConstArray<int32_t> row{a->row_of + (size_t)(ti + 1) * n};
            real* paths = (real*)a->paths + pc;
            static_for<0, NCH>([&](auto Q) {
                constexpr int q = decltype(Q)::value;
                const int j1 = n < W * q + W ? n : W * q + W;
#pragma unroll 1
                for (int j = first > W * q ? first : W * q; j < j1; j++) {
                    const real v = val(Y.template ch<q>()[j - W * q], j);
                    if (active) paths[(size_t)row[j] * P] = v;
                }
            });
        }
    }
}

template <int NCH, int FCAP, typename real>
void launch_spot_cap(const StepArgs& a, hipStream_t stream) {
    const dim3 grid((unsigned)(((int64_t)a.P + kStepThreads - 1) / kStepThreads));
    if (a.lognormal)
        hipLaunchKernelGGL((lmm_spot_kernel<NCH, FCAP, real, true>), grid, dim3(kStepThreads), 0, stream, a);
    else
        hipLaunchKernelGGL((lmm_spot_kernel<NCH, FCAP, real, false>), grid, dim3(kStepThreads), 0, stream, a);
    HIP_CHECK(hipGetLastError());
}

template <int NCH, typename real>
void launch_spot_n(const StepArgs& a, hipStream_t stream) {
    if (a.F <= 1) launch_spot_cap<NCH, 1, real>(a, stream);
    else if (a.F <= 3) launch_spot_cap<NCH, 3, real>(a, stream);
    else if (a.F <= 5) launch_spot_cap<NCH, 5, real>(a, stream);
    else if (a.F <= 10) launch_spot_cap<NCH, 10, real>(a, stream);
    else throw FmError(FM_ERR_UNSUPPORTED, "number of factors above 10 is not supported by the path kernel");
}

} // namespace fm
