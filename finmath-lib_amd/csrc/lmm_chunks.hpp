// The register layout of a path's forwards and the valuation of products on it, shared by the path
// kernels (lmm_spot.hpp, lmm_general.hpp) and the reverse sweep (lmm_spot_adjoint.hpp).
#pragma once

#include "lmm_step.hpp"
#include "hip_check.hpp"

namespace fm {

// Forwards per chunk: a chunk is sixteen VGPRs, eight FP64 or sixteen FP32 forwards. At this
// width the compiler reads and writes an element at a uniform run-time index with one indexed
// move (s_set_gpr_idx_on); narrower FP32 chunks are lowered to chains of compares and selects.
template <typename real> constexpr int chunk_width() { return 64 / (int)sizeof(real); }
template <typename real> struct VecCh;
template <> struct VecCh<double> { typedef double t __attribute__((ext_vector_type(8))); };
template <> struct VecCh<float> { typedef float t __attribute__((ext_vector_type(16))); };

// NCH chunks of forwards in registers (NCH <= 10).
template <int NCH, typename real>
struct ChunkedForwards {
    using V = typename VecCh<real>::t;
    static constexpr int W = chunk_width<real>(), chunks = NCH;
    static_assert(NCH >= 1 && NCH <= 10, "one to ten chunks of forwards");
    V c0, c1, c2, c3, c4, c5, c6, c7, c8, c9;
    template <int Q> __device__ __forceinline__ V& ch() {
        if constexpr (Q == 0) return c0; else if constexpr (Q == 1) return c1; else if constexpr (Q == 2) return c2;
        else if constexpr (Q == 3) return c3; else if constexpr (Q == 4) return c4; else if constexpr (Q == 5) return c5;
        else if constexpr (Q == 6) return c6; else if constexpr (Q == 7) return c7; else if constexpr (Q == 8) return c8;
        else return c9;
    }
    template <int J> __device__ __forceinline__ real at() { return ch<J / W>()[J % W]; }
    template <int J> __device__ __forceinline__ void put(real v) { ch<J / W>()[J % W] = v; }
    template <int Q> __device__ __forceinline__ real element(int e) { return ch<Q>()[e]; }
    // Element j for a uniform run-time j: one indexed register read in the chunk of j. The
    // empty asm keeps each chunk a register value, so the per-chunk reads are not merged into
    // a load from a memory copy of the forwards.
    __device__ __forceinline__ real get(int j) {
        const int e = j % W, qj = j / W;
        real r = (real)0;
        static_for<0, NCH>([&](auto Q) {
            constexpr int q = decltype(Q)::value;
            if (qj == q) {
                const V v = ch<q>();
#if defined(__HIP_DEVICE_COMPILE__)
                asm volatile("" :: "v"(v));
#endif
                r = v[e];
            }
        });
        return r;
    }
    // Element j += x for a uniform run-time j: one indexed register write in the chunk of j. The
    // asm takes the chunk as an input and output, which keeps it a register value.
    __device__ __forceinline__ void add(int j, real x) {
        const int e = j % W, qj = j / W;
        static_for<0, NCH>([&](auto Q) {
            constexpr int q = decltype(Q)::value;
            if (qj == q) {
                V v = ch<q>();
#if defined(__HIP_DEVICE_COMPILE__)
                asm volatile("" : "+v"(v));
#endif
                v[e] = v[e] + x;
                ch<q>() = v;
            }
        });
    }
};

// a / b by the reciprocal of b, which numerators with one divisor share
template <typename real> __device__ __forceinline__ real spot_rcp(real b);
template <> __device__ __forceinline__ double spot_rcp<double>(double b) { return fm_rcp_nr(b); }
template <> __device__ __forceinline__ float spot_rcp<float>(float b) { return __builtin_amdgcn_rcpf(b); }
template <typename real> __device__ __forceinline__ real spot_div_r(real a, real b, real r);
template <> __device__ __forceinline__ double spot_div_r<double>(double a, double b, double r) { return fm_div_nr_r(a, b, r); }
template <> __device__ __forceinline__ float spot_div_r<float>(float a, float, float r) { return a * r; }

// Products evaluated at time index ti, in the order they were lowered (qp advances over them):
// swaptions and caplets are reduced into their wave partials, swap periods and Bermudan
// regression bases go to per-path contribution columns. Y holds the path's states and val(y, j)
// gives the forward L_j(t_ti) of state y; N and Nprev are the numeraires N(T_knum) and the one
// before it. GROUP values a swaption group in one walk; without it every member walks its own
// copy of the periods (the FP32 kernels: the shared walk measured slower there).
// walk_group(i) takes over the swaption group at product i when it has a walk table of its own
// (the spot kernels: valued by the Euler step or by an unrolled walk); it returns whether it did.
// emit(x, slot) takes a per-path value for its reduction slot.
template <bool GROUP, typename real, typename Chunks, typename Val, typename Products, typename Periods,
          typename Doubles, typename Emit, typename Walk>
__device__ __forceinline__ void eval_products_at(int ti, int& qp, int num_products, Products products,
                                                 Periods periods, Doubles delta, double N, double Nprev, int knum,
                                                 Chunks& Y, Val&& val, bool active, double* __restrict__ contrib,
                                                 int64_t p, int P, Emit&& emit, Walk&& walk_group) {
    constexpr int W = Chunks::W, NCH = Chunks::chunks;
    auto value_of = [&](int j) -> real { return val(Y.get(j), j); };
    while (qp < num_products && products[qp].eval_index == ti) {
        const KProduct pr = products[qp];
        qp++;
        if (pr.type == FM_PRODUCT_SWAPTION && walk_group(qp - 1, pr)) {
            qp += pr.pad2;
            continue;
        }
        const double Nsel = (pr.num_k == knum) ? N : Nprev;
        if (pr.type == FM_PRODUCT_SWAPTION) {
            // Swaption.java:150-190: the periods backwards, value = (value + payoff) / (1 + L tau) * adj.
            // The periods are walked chunk by chunk, each element read with one indexed move. With
            // GROUP, the pr.pad2 swaptions that follow differ from this one only in strike and
            // notional: the walk values them too, sharing L_j and the reciprocal of 1 + L_j tau;
            // member s's periods follow this one's at s * num_periods and carry its notional.
            constexpr int G = GROUP ? kSwaptionGroup : 1;
            const int m = GROUP ? 1 + pr.pad2 : 1;
            real V[G];
#pragma unroll
            for (int g = 0; g < G; g++) V[g] = (real)0;
            const int j0 = pr.first_j, j1 = pr.first_j + pr.num_periods;
            static_for<0, NCH>([&](auto QR) {
                constexpr int q = NCH - 1 - decltype(QR)::value;
                const int ja = j0 > W * q ? j0 : W * q;
                const int jb = j1 < W * q + W ? j1 : W * q + W;
#pragma unroll 1
                for (int j = jb - 1; j >= ja; j--) {
                    const KPeriod pe = periods[pr.param_off + (j - j0)];
                    const real Lj = val(Y.template element<q>(j - W * q), j);
                    const real b = (real)1.0 + Lj * (real)pe.tau;
                    const real r = spot_rcp<real>(b);
                    // every member's strike and notional are read up front (indices clamped to the
                    // group) so their scalar loads issue together
                    real Kg[G], Ng[G];
#pragma unroll
                    for (int g = 0; g < G; g++) {
                        const KPeriod& pg = periods[pr.param_off + (g < m ? g : 0) * pr.num_periods + (j - j0)];
                        Kg[g] = (real)pg.strike;
                        Ng[g] = GROUP ? (real)pg.notional : (real)pr.notional;
                    }
#pragma unroll
                    for (int g = 0; g < G; g++) {
                        if (g < m) {
                            const real payoff = ((Lj - Kg[g]) * (real)pe.period_length) * Ng[g];
                            V[g] = V[g] + payoff;
                            V[g] = spot_div_r<real>(V[g], b, r);
                            V[g] = V[g] * (real)pe.adj;
                        }
                    }
                }
            });
#pragma unroll
            for (int g = 0; g < G; g++)
                if (g < m)
                    emit((double)jmax0(V[g]) / Nsel, products[qp - 1 + g].out_slot);
            qp += m - 1;
        } else if (pr.type == FM_PRODUCT_CAPLET) {
            const KPeriod pe = periods[pr.param_off];
            const real Lj = value_of(pr.first_j);
            real v = Lj - (real)pe.strike;
            if (!pr.is_floorlet) v = jmax0(v) * (real)pe.notional;
            else v = ((v != v) ? v : (v > (real)0 ? (real)0 : v)) * ((real)(-1.0) * (real)pe.notional);
            emit((double)v / Nsel, pr.out_slot);
        } else if (pr.type == K_BERM_BASIS) {
            // raw regression basis of a Bermudan exercise date T_e (BermudanSwaption.java:215-252)
            if (pr.flags == FM_BASIS_REFERENCE) {
                // L_short over tenor periods [first_j, pe.j), L_long over [first_j, pe.pay_k):
                // a single period is the forward itself, several accrue (LMM:1290-1305)
                const KPeriod pe = periods[pr.param_off];
                real accS = (real)0, accL = (real)0, rs = (real)0, rl = (real)0;
#pragma unroll 1
                for (int j = pr.first_j; j < pe.pay_k; j++) {
                    const real Lj = value_of(j);
                    const real d = (real)delta[j];
                    if (j == pr.first_j) { rs = Lj; rl = Lj; }
                    accL = (j == pr.first_j) ? Lj * d + (real)1.0 : accL * ((real)1 + Lj * d);
                    if (j < pe.j) accS = (j == pr.first_j) ? Lj * d + (real)1.0 : accS * ((real)1 + Lj * d);
                }
                if (pe.j > pr.first_j + 1) rs = (accS - (real)1.0) / (real)pe.tau;
                if (pe.pay_k > pr.first_j + 1) rl = (accL - (real)1.0) / (real)pe.period_length;
                const real ds = (real)1.0 / (rs * (real)pe.tau + (real)1.0);
                const real dl = (real)1.0 / (rl * (real)pe.period_length + (real)1.0);
                if (active) {
                    contrib[(size_t)pr.out_slot * P + p] = (double)ds;
                    contrib[(size_t)(pr.out_slot + 1) * P + p] = (double)dl;
                    contrib[(size_t)(pr.out_slot + 2) * P + p] = Nsel;
                }
            } else {
                // par rate of the remaining periods: P = 1/(L pl + 1), A = P pl, then
                // P = P/(L pl + 1), A = A + P pl; S = (1 - P)/A
                real Pd = (real)1, A = (real)0;
#pragma unroll 1
                for (int j = pr.first_j; j < pr.first_j + pr.num_periods; j++) {
                    const real pl = (real)periods[pr.param_off + (j - pr.first_j)].period_length;
                    const real Lj = value_of(j);
                    if (j == pr.first_j) { Pd = (real)1.0 / (Lj * pl + (real)1.0); A = Pd * pl; }
                    else { Pd = Pd / (Lj * pl + (real)1.0); A = A + Pd * pl; }
                }
                const real S = (Pd * (real)(-1.0) + (real)1.0) / A;
                if (active) {
                    contrib[(size_t)pr.out_slot * P + p] = (double)S;
                    contrib[(size_t)(pr.out_slot + 1) * P + p] = Nsel;
                }
            }
        } else {   // one period of a swap: contribution column, combined after the adjustment is known
            const KPeriod pe = periods[pr.param_off];
            const real Lj = value_of(pr.first_j);
            double payoff = (double)(((Lj - (real)pe.strike) * (real)pe.period_length) * (real)pe.notional);
            if (!(pr.flags & 1)) payoff = payoff * -1.0;
            if (active) contrib[(size_t)pr.out_slot * P + p] = payoff / Nsel;
        }
    }
}

} // namespace fm
