// Pathwise adjoint (reverse sweep) of the spot Euler pricing pass.
//
// The pricing pass (lmm_spot_kernel) stores the carried state of every path every `stride`
// time steps and the numeraire N(T_k). The reverse sweep walks the segments between
// checkpoints backwards. At the top index of a segment it reloads the segment's checkpoint and
// rebuilds the state with the pricing pass's own step, so the sweep differentiates the paths that
// were priced; the states in between go to a per-path segment buffer ([stride-2][n][P]), so each
// step is recomputed once. For each index t it then
//   1. reverses the Euler step t -> t+1,
//   2. adds the direct sensitivities of the products evaluated at t,
//   3. reverses the numeraire updates N(T_{k+1}) = N(T_k)(1 + L_k d_k) made at t,
//   4. turns the adjoint of the state at t into that of the state the step t-1 -> t computed (before
//      the cap).
// Per alive forward-step it reduces dV/dsigma_j(t_i) over the wavefront, where the factor
// loading is lambda_jk = sigma_j f_jk and the variance sigma_j^2 c_j
// (LIBORCovarianceModelFromVolatilityAndCorrelation.java:48-93); at the end it reduces dV/dL_j(0).
//
// Per path the sweep holds two register arrays, the state at t and the adjoint B. In FP64 and the
// log-normal state space B_j is the adjoint of ln L_j, into which the step's adjoint of its new state
// goes unchanged and every sensitivity to L_j enters times L_j: no exponential or division is spent on
// converting it. In FP32, in the normal state space, and for the forwards that are fixed when the simulation
// starts, B_j is the adjoint of L_j: the float arithmetic is kept operation by operation, as in
// lmm_spot32.hpp, and a forward that no step moves may be zero, where ln L_j has no adjoint.
// Components are unrolled over the register arrays in pairs, like the pricing pass's steps, except where
// a component's code is long (reverse_step).
//
// The two register arrays leave two wavefronts per SIMD at 80 FP32 or 40 FP64 forwards, so the sweep
// waits on scalar loads and on the vector pipeline in turn. 80 forwards x 10 factors x 1,000,000 FP32
// paths: 21.2 ms (22.2 ms at 0.61 vector ALU busy while the bounds of the unrolled loops were hoisted as masks and
// spilled; 29.3 ms at 0.49 with rolled loops and every kernel argument held in spilled scalar registers); 40 x 5 x 100,001 FP64 paths with 30 swaptions: 1.16 ms (2.82 ms).
//
// Conventions of the reference's AAD (RandomVariableDifferentiableAAD.java:165-219): averages
// over paths (the numeraire-adjustment factor) are constants, the floor of the swaption payoff
// has derivative 1 at and above zero and 0 below. A Bermudan period's payoff enters with a
// per-path weight: 1 or 0 by the recorded exercise (the exercise decisions held fixed), or the
// weights of the induction's own adjoint (lmm_bermudan.hip) when given.
#pragma once

#include "lmm_spot32.hpp"
#include "lmm_spot64.hpp"

namespace fm {

// The forwards below this are moved by no step: the simulation and the tenor both start at time 0, which is the
// fixing date of the first forward alone.
constexpr int kFixedAtStart = 1;

struct AdjKernelArgs {
    StepArgs a;
    AdjArgs g;
};
typedef const AdjKernelArgs __attribute__((address_space(4)))* AdjArgPtr;
__device__ __forceinline__ AdjArgPtr adjoint_arguments() {
    AdjArgPtr a = (AdjArgPtr)__builtin_amdgcn_kernarg_segment_ptr();
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+s"(a));
#endif
    return a;
}

// Wavefront sums of dV/dsigma of components j .. j+3, written to this wavefront's row for the alive ones.
__device__ __forceinline__ void gradient_sums(const double (&v)[4], int j, int first, int n, int lane, double* row) {
    const double s = wave_sum4_all(v, lane);
    const int jw = j + 2 * (lane & 1) + ((lane >> 1) & 1);
    if (lane < 4 && jw < n && jw >= first) row[jw] = s;
}

// One component's record and factor row f_jk, read whole into scalar registers (volatile: issued here
// and not where the values are first used).
template <int FCAP, typename real>
struct AdjRec {
    static constexpr int size = rec_size_of(FCAP);
    static constexpr int N = sizeof(real) * size > 64 ? 2 : 1;      // pieces of at most 64 bytes
    typedef real V __attribute__((ext_vector_type(size / N)));
    typedef const real __attribute__((address_space(4)))* Ptr;
    V r[N], f[N];
    __device__ __forceinline__ void read(Ptr rec, Ptr fsig) {
        typedef const volatile V __attribute__((address_space(4)))* P;
#pragma unroll
        for (int i = 0; i < N; i++) {
            r[i] = *(P)(rec + i * (size / N));
            f[i] = *(P)(fsig + i * (size / N));
        }
    }
    __device__ __forceinline__ void arrive() const {
#if defined(__HIP_DEVICE_COMPILE__)
        if constexpr (N == 1) asm volatile("" :: "s"(r[0]), "s"(f[0]));
        else asm volatile("" :: "s"(r[0]), "s"(f[0]), "s"(r[1]), "s"(f[1]));
#endif
    }
    __device__ __forceinline__ real at(int k) const { return r[k / (size / N)][k % (size / N)]; }
    __device__ __forceinline__ real fac(int k) const { return f[k / (size / N)][k % (size / N)]; }
};

// Step 1 of the sweep: B holds the adjoint of the new state of the moved components and gets the adjoint of
// the state at t (FP32: of L_j(t)).
//   Sb_k = sum_j mb_j lambda_jk, mb_j = Yb_j dt: the adjoint of the step's factor sums before any
//   component's share is taken off; then ascending j the factor sums S as the step built them, and Sb
//   with the shares of the components below taken off. dV/dsigma_j(t) on this path is
//   sum_k lambda-bar_jk f_jk with lambda-bar_jk = Yb dW_k + mb S_k + w Sb_k, gathered as
//   Yb (dW.f) + mb (S.f) + w (Sb.f).
// The second pass has six independent sums over the factors per component, so it takes components one
// at a time, four to a rolled iteration (unrolled over the whole array it outgrows the instruction
// cache); a component's record and factor row are read while the one before it runs.
template <int NCH, int FCAP, typename real, bool lognormal, typename Chunks>
__device__ __forceinline__ void reverse_step(Chunks& X, Chunks& B, int n, int rec_n, int t, int first, real dt,
                                             const real (&dW)[FCAP], const real* rec, const real* fsig, const real* vterm,
                                             const Exp2Coef& ke, bool active, int lane, double* row) {
    constexpr bool D = sizeof(real) == 8;
    constexpr int RS = rec_size_of(FCAP), W = chunk_width<real>();
    typedef typename AdjRec<FCAP, real>::Ptr Ptr;
    Ptr recs = (Ptr)(uintptr_t)(rec + (size_t)t * rec_n * RS);
    Ptr fs = (Ptr)(uintptr_t)fsig, vt = (Ptr)(uintptr_t)(vterm + (size_t)t * rec_n);
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+s"(recs), "+s"(fs), "+s"(vt));
#endif
    auto mad = [](real x, real y, real z) -> real {
        if constexpr (D) return fma(x, y, z);
        else return fmaf(x, y, z);
    };
    real S[FCAP], Sb[FCAP];
#pragma unroll
    for (int k = 0; k < FCAP; k++) { S[k] = (real)0; Sb[k] = (real)0; }
    const unsigned alive = (unsigned)(n - first);
    static_for<0, W * NCH / 2>([&](auto Q) {
        constexpr int j = 2 * decltype(Q)::value;
        if ((unsigned)(j + 1 - first) < alive + 1) {
            typedef typename std::conditional<D, RecVec<FCAP>, RecVec32<FCAP>>::type Vec;
            const Vec R0(recs, j), R1(recs, j + 1);
            const real m0 = B.template at<j>() * dt, m1 = B.template at<j + 1>() * dt;
#pragma unroll
            for (int k = 0; k < FCAP; k++) Sb[k] = mad(m1, R1.lam(k), mad(m0, R0.lam(k), Sb[k]));
        }
    });
    AdjRec<FCAP, real> R[2];
    const int begin = first & ~3;
    R[0].read(recs + begin * RS, fs + begin * RS);
    static_for<0, NCH>([&](auto Q) {
        constexpr int q = decltype(Q)::value;
        const int e0 = begin > W * q ? begin - W * q : 0, e1 = n < W * q + W ? n - W * q : W;
#pragma unroll 1
        for (int e = e0; e < e1; e += 4) {
            const int j4 = W * q + e;
            Ptr r4 = recs + j4 * RS, f4 = fs + j4 * RS;
            real gs[4] = {(real)0, (real)0, (real)0, (real)0};
            static_for<0, 4>([&](auto H) {
                constexpr int h = decltype(H)::value;
                const AdjRec<FCAP, real>& A = R[h & 1];
                A.arrive();
                R[(h + 1) & 1].read(r4 + (h + 1) * RS, f4 + (h + 1) * RS);
                if ((unsigned)(j4 + h - first) >= alive) return;
                const real vj = vt[j4 + h];
                const real x = X.template ch<q>()[e + h], Yb = B.template ch<q>()[e + h];
                real L, r, w;
                if constexpr (D) {
                    L = lognormal ? fm_exp2(x, ke) : x;         // L_j / s_j
                    r = fm_rcp_nr(L + A.at(FCAP + 2));
                    w = lognormal ? L * r : r;
                } else {
                    L = x;
                    r = __builtin_amdgcn_rcpf(fmaf(L, A.at(FCAP + 1), A.at(FCAP + 2)));
                    w = lognormal ? r * L : r;
                }
                const real mb = Yb * dt;
                real wb = (real)0, dwf = (real)0, sf = (real)0, sbf = (real)0;
#pragma unroll
                for (int k = 0; k < FCAP; k++) {
                    const real f = A.fac(k), lam = A.at(k);
                    S[k] = mad(w, lam, S[k]);               // S^(j-1) -> S^(j)
                    wb = mad(Sb[k], lam, wb);
                    dwf = mad(dW[k], f, dwf);
                    sf = mad(S[k], f, sf);
                    sbf = mad(Sb[k], f, sbf);
                    Sb[k] = mad(-mb, lam, Sb[k]);           // Sb^(j) -> Sb^(j+1)
                }
                real g = mad(w, sbf, mad(Yb, dwf, mb * sf));
                // variance sigma^2 c in the drift: d(-var/2)/dsigma = -sigma c
                if constexpr (lognormal) g = mad(mb, vj, g);
                gs[h] = active ? g : (real)0;
                // the new state is the old one plus the step's terms, and w_j depends on L_j(t)
                real b;
                if constexpr (D) {
                    // dw/d(ln L) = w e/(E + e), dw/dL = -1/(L + 1/d)^2
                    b = fma(wb, lognormal ? w * (A.at(FCAP + 2) * r) : -r * r, Yb);
                } else if constexpr (lognormal) {
                    const float dwdL = A.at(FCAP + 2) * r * r;
                    b = fmaf(Yb, __builtin_amdgcn_rcpf(L), wb * dwdL);
                } else {
                    const float dwdL = -A.at(FCAP + 1) * r * r;
                    b = fmaf(wb, dwdL, Yb);
                }
                B.template ch<q>()[e + h] = b;
            });
            const double v4[4] = {(double)gs[0], (double)gs[1], (double)gs[2], (double)gs[3]};
            gradient_sums(v4, j4, first, n, lane, row);
        }
    });
}

// The sensitivities of a swaption group with a walk table in FP64 (SwaptionWalk, lmm_spot64.hpp). With c_g
// the adjoint of V_g, C = sum_g c_g and G_j = P_j a_j (C E_j - sum_g c_g k_gj),
//   dV/dE_j = P_j a_j C - r_j sum_{m >= j} G_m,   r_j = 1/(E_j + e_j),
// in two ascending passes: the values, then the sensitivities. weight(V, c) turns the values into c;
// dB_dE(E, j) is what B_j gets for a sensitivity to E_j.
template <int NCH, int FCAP, bool lognormal, typename Chunks, typename Weight, typename ToB>
__device__ __forceinline__ void walk_adjoint64(Chunks& X, Chunks& B, const double* rec, int rec_n, int t,
                                               const double* table, int j0, int periods, const Exp2Coef& ke,
                                               Weight&& weight, ToB&& dB_dE) {
    constexpr int RS = rec_size_of(FCAP);
    RecPtr recs = (RecPtr)(uintptr_t)(rec + (size_t)t * rec_n * RS);
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+s"(recs));
#endif
    SwaptionWalk sw;
    sw.table = (RecPtr)(uintptr_t)table;
    sw.j0 = j0;
    sw.periods = periods;
    constexpr int W = 8;
    static_for<0, NCH>([&](auto Q) {
        constexpr int q = decltype(Q)::value;
        const int a = j0 > W * q ? j0 : W * q, b = j0 + periods < W * q + W ? j0 + periods : W * q + W;
#pragma unroll 1
        for (int j = a; j < b; j++) {
            const double x = X.template ch<q>()[j - W * q], e = recs[j * RS + FCAP + 2];
            const double E = lognormal ? fm_exp2(x, ke) : x;
            sw.period(j, E, e, fm_rcp_nr(E + e));
        }
    });
    double c[kSwaptionGroup];
    weight(sw.V, c);
    double C = 0.0, rest = 0.0;
#pragma unroll
    for (int g = 0; g < kSwaptionGroup; g++) {
        C += c[g];
        rest = fma(c[g], sw.V[g], rest);        // sum of G_m, m >= j
    }
    double P = 1.0;
    static_for<0, NCH>([&](auto Q) {
        constexpr int q = decltype(Q)::value;
        const int a = j0 > W * q ? j0 : W * q, b = j0 + periods < W * q + W ? j0 + periods : W * q + W;
#pragma unroll 1
        for (int j = a; j < b; j++) {
            const double x = X.template ch<q>()[j - W * q], e = recs[j * RS + FCAP + 2];
            const double E = lognormal ? fm_exp2(x, ke) : x;
            const double r = fm_rcp_nr(E + e);
            RecPtr row = sw.table + 8 * (j - j0);
            P = P * (e * r);
            const double Pa = P * row[0];
            double kc = 0.0;
#pragma unroll
            for (int g = 0; g < kSwaptionGroup; g++) kc = fma(c[g], row[1 + g], kc);
            const double dE = fma(Pa, C, -(r * rest));
            rest = fma(-Pa, fma(C, E, -kc), rest);
            B.template ch<q>()[j - W * q] = fma(dB_dE(E, j), dE, B.template ch<q>()[j - W * q]);
        }
    });
}

template <int NCH, int FCAP, typename real, bool lognormal>
__global__ void __launch_bounds__(kStepThreads)
__attribute__((amdgpu_waves_per_eu((sizeof(real) == 4 || NCH <= 5) ? 2 : 1)))
lmm_spot_adjoint_kernel(const AdjKernelArgs)
{
    constexpr bool D = sizeof(real) == 8;
    constexpr int W = chunk_width<real>();
    AdjArgPtr k = adjoint_arguments();
    const uint32_t p0 = blockIdx.x * (uint32_t)kStepThreads + threadIdx.x;      // P < 2^31
    const int lane = threadIdx.x & 63;
    // the wavefront index, uniform: kept in a scalar register
    const int64_t wave = (int64_t)blockIdx.x * (kStepThreads / 64) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (wave * 64 >= k->a.P) return;        // a wavefront without paths writes nothing
    const Exp2Coef ke;
    ChunkedForwards<NCH, real> X;     // state at t
    ChunkedForwards<NCH, real> B;     // adjoint
    static_for<0, W * NCH>([&](auto J) {
        constexpr int j = decltype(J)::value;
        X.template put<j>((real)0);
        B.template put<j>((real)0);
    });
    double Nb_top = 0.0, Nb_low = 0.0;      // adjoints of N(T_K) and N(T_{K-1})
    int K = ConstArray<int32_t>{k->g.kcur_at}[k->a.nT];
    int qp = k->a.num_products - 1;         // products sorted by evaluation index
    const int stride = k->g.stride;

    for (int c = (k->a.nT / stride) * stride; c >= 0; c -= stride) {
        const int hi = (c + stride - 1 < k->a.nT) ? c + stride - 1 : k->a.nT;
        for (int t = hi; t >= c; t--) {
            k = adjoint_arguments();
            const int P = k->a.P, n = k->a.n, nT = k->a.nT, rec_n = k->a.rec_n;
            const bool active = p0 < (uint32_t)P;
            const uint32_t pc = active ? p0 : (uint32_t)P - 1;
            const ConstArray<double> times{k->a.times};
            const ConstArray<int32_t> first_alive{k->a.first_alive};
            const real* rec = (const real*)k->a.rec;
            // ---- the state at t: the checkpoint at c for t = c and t = hi, the segment's stored
            // states in between. At t = hi the pricing pass's steps c .. hi-1 rebuild the state
            // and store the states c+1 .. hi-1 for the later t of the segment. Components below
            // cfirst are dead and read by nothing in this segment. Checkpoints and segment states are
            // read and written non-temporal: a wavefront's segment (two states of n components at
            // stride 4) outgrows its share of the L2 before it is read back.
            const int cfirst = ConstArray<int32_t>{k->a.ckpt_first}[c / stride];
            const unsigned held = (unsigned)(n - cfirst);
            {
                const real* src = (t > c && t < hi) ? (const real*)k->g.seg + (size_t)(t - c - 1) * n * P
                                                    : (const real*)k->a.ckpt + (size_t)(c / stride) * n * P;
                const int cf = opaque(cfirst);
                static_for<0, W * NCH>([&](auto J) {
                    constexpr int j = decltype(J)::value;
                    if ((unsigned)(j - cf) < held) X.template put<j>(__builtin_nontemporal_load(src + pc));
                    src += P;
                });
            }
            auto increments = [&](real (&dW)[FCAP], int s) {
                const int F = opaque(k->a.F);
                const real* dwp = (const real*)k->a.dw + ((size_t)pc * nT + s) * F;
                if (F == FCAP) {
#pragma unroll
                    for (int q = 0; q < FCAP; q++) dW[q] = dwp[q];
                } else {
#pragma unroll
                    for (int q = 0; q < FCAP; q++) dW[q] = q < F ? dwp[q] : (real)0;
                }
            };
            if (t == hi) {
                for (int s = c; s < t; s++) {
                    real dWs[FCAP];
                    increments(dWs, s);
                    const real dts = (real)(times[s + 1] - times[s]);
                    if constexpr (D)
                        spot64_step<NCH, FCAP, lognormal, false>(X, n, rec_n, s, first_alive[s], dts, dWs, rec, ke,
                                                                 nullptr);
                    else
                        spot32_step<NCH, FCAP, lognormal>(X, n, rec_n, s, first_alive[s], dts, dWs, rec,
                                                          (float)k->a.cap);
                    if (s + 1 < hi) {
                        real* to = (real*)k->g.seg + (size_t)(s - c) * n * P;
                        const int cf = opaque(cfirst);
                        static_for<0, W * NCH>([&](auto J) {
                            constexpr int j = decltype(J)::value;
                            if ((unsigned)(j - cf) < held && active)
                                __builtin_nontemporal_store(X.template at<j>(), to + pc);
                            to += P;
                        });
                    }
                }
            }
            const ConstArray<double> lead{k->a.lead};
            auto val = [&](real x, int j) -> real {
                if constexpr (D && lognormal) return lead[j] * fm_exp2(x, ke);
                else return x;
            };
            // a sensitivity to L_j as a part of B_j; 1/s_0 is read here, since a read within the walk spilled 90
            // scalar registers more (40 x 5 x 100,001 FP64 paths: 1.76 ms a call against 1.72)
            const double inv_scale0 = D ? lead[n] : 0.0;
            auto scale = [&](real Lj, int j) -> real { return D && lognormal && j >= kFixedAtStart ? Lj : (real)1; };

            // ---- 1. reverse the Euler step t -> t+1
            if (t < nT) {
                const int first = first_alive[t];
                real dW[FCAP];
                increments(dW, t);
                double* row = k->g.wave_grad + (size_t)wave * (nT * n + n) + (size_t)t * n;
                const real dt = (real)(times[t + 1] - times[t]);
                reverse_step<NCH, FCAP, real, lognormal>(X, B, n, rec_n, t, first, dt, dW, rec, (const real*)k->g.fsig,
                                                         (const real*)k->g.vterm, ke, active, lane, row);
                // the components the step does not move have dV/dsigma_j(t) = 0: this row of the
                // wavefront's gradient is then written in full and needs no clearing beforehand
                for (int j = lane; j < first; j += 64) row[j] = 0.0;
            }

            // ---- 2. products evaluated at t (reverse order of evaluation). The per-path conditions
            // (in the money, exercised) scale the contributions instead of branching around them.
            const int Kt = ConstArray<int32_t>{k->g.kcur_at}[t];
            const ConstArray<KProduct> products{k->a.products};
            const ConstArray<KPeriod> periods{k->a.periods};
            const double* numeraire = k->a.numeraire;
            while (qp >= 0 && products[qp].eval_index == t) {
                KProduct pr = products[qp];
#if defined(__HIP_DEVICE_COMPILE__)
                // the fields one by one: as one piece of sixteen scalar registers, live through the products, the record
                // had 400 other scalar registers spilled (40 x 5 x 100,001 FP64 paths: 1.82 ms a call against 1.73); with
                // ten factors, where the records take more, it is the fields that spill (40 x 10: 2.49 ms against 1.98)
                if constexpr (FCAP <= 5) {
                    asm volatile("" : "+s"(pr.type), "+s"(pr.first_j), "+s"(pr.num_periods), "+s"(pr.out_slot),
                                 "+s"(pr.is_floorlet), "+s"(pr.flags), "+s"(pr.num_k));
                    asm volatile("" : "+s"(pr.notional), "+s"(pr.weight), "+s"(pr.param_off), "+s"(pr.pad2), "+s"(pr.pad3));
                }
#endif
                const bool top = (pr.num_k == Kt);
                const double Nsel = (pr.num_k == 0) ? 1.0 : numeraire[(size_t)pr.num_k * P + pc];
                double nb = 0.0;            // adjoint of the selected numeraire
                real xadd = (real)0;        // adjoint of L_{first_j}(t) (caplets and swap periods)
                const int m = pr.type == FM_PRODUCT_SWAPTION ? pr.pad3 + 1 : 1;     // the last of its group of m
                const int head = qp - (m - 1);
                bool walked = false;
                if constexpr (D) {
                    if (pr.type == FM_PRODUCT_SWAPTION && products[head].walk >= 0) {
                        walked = true;
                        {
                            walk_adjoint64<NCH, FCAP, lognormal>(
                                X, B, rec, rec_n, t, (const double*)k->a.walk + 8 * products[head].walk, pr.first_j,
                                pr.num_periods, ke, [&](const double (&V)[kSwaptionGroup], double (&cg)[kSwaptionGroup]) {
#pragma unroll
                                    for (int g = 0; g < kSwaptionGroup; g++) {
                                        const KProduct pg = products[head + (g < m ? g : 0)];
                                        const double v = V[g] * pg.notional;
                                        // floor(0.0): derivative 1 at and above the floor, 0 below
                                        const bool itm = g < m && v >= 0.0;
                                        cg[g] = itm ? pg.weight * pg.notional / Nsel : 0.0;
                                        nb += itm ? -pg.weight * v / (Nsel * Nsel) : 0.0;
                                    }
                                },
                                [&](double E, int j) -> double {        // L_j = s_j E_j
                                    return !lognormal ? 1.0 : j >= kFixedAtStart ? E : inv_scale0;
                                });
                        }
                        qp -= m - 1;
                    }
                }
                if (walked) {
                } else if (pr.type == FM_PRODUCT_SWAPTION) {
                    // V = sum_j p_j prod_{l<=j} D_l, D_l = adj_l / (1 + L_l tau_l), walked backwards
                    const int j0 = pr.first_j, j1 = pr.first_j + pr.num_periods;
                    real V = (real)0, Pc = (real)1;
                    static_for<0, NCH>([&](auto QR) {
                        constexpr int q = NCH - 1 - decltype(QR)::value;
                        const int ja = j0 > W * q ? j0 : W * q;
                        const int jb = j1 < W * q + W ? j1 : W * q + W;
#pragma unroll 1
                        for (int j = jb - 1; j >= ja; j--) {
                            const KPeriod pe = periods[pr.param_off + (j - j0)];
                            const real Lj = val(X.template ch<q>()[j - W * q], j);
                            const real Dl = (real)pe.adj * spot_rcp<real>((real)1.0 + Lj * (real)pe.tau);
                            V = (V + ((Lj - (real)pe.strike) * (real)pe.period_length) * (real)pr.notional) * Dl;
                            Pc = Pc * Dl;
                        }
                    });
                    const double Vb = (V >= (real)0) ? pr.weight / Nsel : 0.0;
                    nb = (V >= (real)0) ? -pr.weight * (double)V / (Nsel * Nsel) : 0.0;
                    // descending over j: P_j = prod_{l<=j} D_l, U_j = sum_{m>=j} p_m P_m
                    real U = (real)0;
                    static_for<0, NCH>([&](auto QR) {
                        constexpr int q = NCH - 1 - decltype(QR)::value;
                        const int ja = j0 > W * q ? j0 : W * q;
                        const int jb = j1 < W * q + W ? j1 : W * q + W;
#pragma unroll 1
                        for (int j = jb - 1; j >= ja; j--) {
                            const KPeriod pe = periods[pr.param_off + (j - j0)];
                            const real Lj = val(X.template ch<q>()[j - W * q], j);
                            const real one = (real)1.0 + Lj * (real)pe.tau;
                            const real inv = spot_rcp<real>(one);
                            const real pj = ((Lj - (real)pe.strike) * (real)pe.period_length) * (real)pr.notional;
                            U = U + pj * Pc;
                            const real dV = (real)pe.period_length * (real)pr.notional * Pc - ((real)pe.tau * inv) * U;
                            if constexpr (D && lognormal)
                                B.template ch<q>()[j - W * q] = fma(Vb * scale(Lj, j), dV, B.template ch<q>()[j - W * q]);
                            else
                                B.template ch<q>()[j - W * q] = B.template ch<q>()[j - W * q] + (real)Vb * dV;
                            Pc = Pc * (one * (real)pe.inv_adj);      // P_{j-1} = P_j / D_j
                        }
                    });
                } else if (pr.type == FM_PRODUCT_CAPLET) {
                    const KPeriod pe = periods[pr.param_off];
                    const real Lj = val(X.get(pr.first_j), pr.first_j);
                    const real v = Lj - (real)pe.strike;
                    // floor(0.0) has derivative 1 for v >= 0, cap(0.0) has derivative 1 for v < 0
                    // (RandomVariableDifferentiableAAD.java:333-348)
                    const bool itm = pr.is_floorlet ? (v < (real)0) : (v >= (real)0);
                    const double dcf = pe.notional;
                    const double x = pr.is_floorlet ? -(double)v * dcf : (double)v * dcf;
                    xadd = itm ? (real)((pr.is_floorlet ? -dcf : dcf) * pr.weight / Nsel) * scale(Lj, pr.first_j) : (real)0;
                    nb = itm ? -pr.weight * x / (Nsel * Nsel) : 0.0;
                } else if (pr.type == K_BERM_BASIS) {
                    // regression basis: not differentiated (the reference's conditional
                    // expectation treats its basis functions as constants)
                } else {
                    double pw = 1.0;       // the payoff's weight on this path
                    if (pr.type == K_BERM_PERIOD) {
                        if (k->g.berm_weight) {
                            pw = k->g.berm_weight[(size_t)pr.out_slot * P + pc];
                        } else {
                            // the period pays on this path if the exercise (callable: entered at or
                            // before it; cancelable: terminated after it) keeps it in the value
                            const int ex = k->g.berm_ex[(size_t)pr.pad2 * P + pc];
                            pw = ((pr.flags & 2) ? (ex >= 0 && pr.is_floorlet >= ex)
                                                 : (ex < 0 || pr.is_floorlet < ex)) ? 1.0 : 0.0;
                        }
                    }
                    const KPeriod pe = periods[pr.param_off];
                    const real Lj = val(X.get(pr.first_j), pr.first_j);
                    const double sgn = (pr.flags & 1) ? 1.0 : -1.0;
                    const double pay = sgn * (double)(((Lj - (real)pe.strike) * (real)pe.period_length) * (real)pe.notional);
                    xadd = (real)(pw * sgn * pe.period_length * pe.notional * pr.weight / Nsel) * scale(Lj, pr.first_j);
                    nb = -pw * pr.weight * pay / (Nsel * Nsel);
                }
                qp--;
                if (top) Nb_top += nb; else Nb_low += nb;
                B.add(pr.first_j, xadd);
            }

            // ---- 3. numeraire updates made at t: N_{k+1} = N_k (1 + L_k d_k), k = K-1 down to kcur_at[t-1]
            const int Kprev = (t > 0) ? ConstArray<int32_t>{k->g.kcur_at}[t - 1] : 0;
            while (K > Kprev) {
                const int i = K - 1;
                const double Nk = (i == 0) ? 1.0 : numeraire[(size_t)i * P + pc];
                const real Lr = val(X.get(i), i);
                const double Lk = (double)Lr;
                const double dk = ConstArray<double>{k->a.delta}[i];
                B.add(i, (real)(Nb_top * dk * Nk) * scale(Lr, i));
                Nb_low += Nb_top * (1.0 + Lk * dk);
                Nb_top = Nb_low;
                Nb_low = 0.0;
                K--;
            }

            // ---- 4. the adjoint of the state the step t-1 -> t computed: in FP32 the adjoint of L(t)
            // times L_j(t) (log-normal), and zero where the cap binds (cap(x, c) has derivative 0 for
            // x >= c, RandomVariableDifferentiableAAD.java:316-323; x >= c exactly where the capped
            // state equals the cap).
            if (t > 0) {
                const int first = first_alive[t - 1];
                const unsigned moved = (unsigned)(n - first);
                const bool capped = k->a.capped != 0;
                if constexpr (D) {
                    if (capped) {
                        RecPtr recs = (RecPtr)(uintptr_t)((const double*)rec + (size_t)(t - 1) * rec_n * rec_size_of(FCAP));
                        static_for<0, W * NCH>([&](auto J) {
                            constexpr int j = decltype(J)::value;
                            if ((unsigned)(j - first) < moved) {
                                const double xcap = recs[j * rec_size_of(FCAP) + FCAP + 1];
                                if (__builtin_amdgcn_ballot_w64(X.template at<j>() >= xcap) != 0) {
                                    asm volatile("");
                                    B.template put<j>(X.template at<j>() >= xcap ? 0.0 : B.template at<j>());
                                }
                            }
                        });
                    }
                } else {
                    const float cap = (float)k->a.cap;
                    static_for<0, W * NCH>([&](auto J) {
                        constexpr int j = decltype(J)::value;
                        if ((unsigned)(j - first) < moved) {
                            const float x = X.template at<j>(), lb = B.template at<j>();
                            float yb = lognormal ? lb * x : lb;
                            if (__builtin_amdgcn_ballot_w64(x >= cap) != 0) {
                                asm volatile("");
                                yb = (capped && x >= cap) ? 0.0f : yb;
                            }
                            B.template put<j>(yb);
                        }
                    });
                }
            }
        }
    }
    // ---- dV/dL_j(0)
    k = adjoint_arguments();
    const int n = k->a.n;
    const bool active = p0 < (uint32_t)k->a.P;
    double* row = k->g.wave_grad + (size_t)wave * (k->a.nT * n + n) + (size_t)k->a.nT * n;
    static_for<0, W * NCH>([&](auto J) {
        constexpr int j = decltype(J)::value;
        if (j < n) {
            double b = (double)B.template at<j>();
            if constexpr (D && lognormal && j >= kFixedAtStart)
                b = b / (ConstArray<double>{k->a.lead}[j] * fm_exp2(X.template at<j>(), ke));
            const double s = wave_sum_dpp(active ? b : 0.0);
            if (lane == 63) row[j] = s;
        }
    });
}

template <int NCH, int FCAP, typename real>
void launch_spot_adjoint_cap(const StepArgs& a, const AdjArgs& g, hipStream_t stream) {
    const dim3 grid((unsigned)(((int64_t)a.P + kStepThreads - 1) / kStepThreads));
    const AdjKernelArgs args{a, g};
    if (a.lognormal)
        hipLaunchKernelGGL((lmm_spot_adjoint_kernel<NCH, FCAP, real, true>), grid, dim3(kStepThreads), 0, stream, args);
    else
        hipLaunchKernelGGL((lmm_spot_adjoint_kernel<NCH, FCAP, real, false>), grid, dim3(kStepThreads), 0, stream, args);
    HIP_CHECK(hipGetLastError());
}

template <int NCH, typename real>
void launch_spot_adjoint_n(const StepArgs& a, const AdjArgs& g, hipStream_t stream) {
    if (a.F <= 1) launch_spot_adjoint_cap<NCH, 1, real>(a, g, stream);
    else if (a.F <= 3) launch_spot_adjoint_cap<NCH, 3, real>(a, g, stream);
    else if (a.F <= 5) launch_spot_adjoint_cap<NCH, 5, real>(a, g, stream);
    else if (a.F <= 10) launch_spot_adjoint_cap<NCH, 10, real>(a, g, stream);
    else throw FmError(FM_ERR_UNSUPPORTED, "number of factors above 10 is not supported by the adjoint kernel");
}

} // namespace fm
