// The FP64 spot kernel for few paths: a path on a row of sixteen lanes.
//
// One path per lane leaves most of the chip idle below some 60,000 paths (1,024 SIMDs, 64 paths each), and
// the time is then that of one wavefront's chain of instructions, whatever the number of paths. Here
// lane g of a path's row holds the components g, 16 + g, ...: their exponentials, reciprocals, weights and
// new states are formed side by side, sixteen components in the instructions of one. What is
// sequential in the step keeps its order, so every state is lmm_spot_kernel's bit for bit (a path's values
// do not depend on how many are simulated with it):
//   factor sums   lane k holds T_k and adds the row's weights one after the other, T_k = T_k + w_l lambda_lk
//                 with w_l broadcast over the row (row_newbcast). The sums after each component go through
//                 the LDS to the lane of that component, which needs all of them:
//                 z_j + (h_j + sum_k T_k lambda_jk).
//   swaptions     lane g < 4 holds V_g of a group's walk and takes the row's E_l and discount factors in order.
// Products read a forward from its lane by a permute and are otherwise valued by every lane of the row alike.
//
// A lane's records of the next step (its own, and column k of the row's sixteen) are requested as soon
// as this step's are used: with one or two wavefronts per SIMD nothing else hides their latency.
// It is bound by latency: of a wavefront's time about 0.4 are waits for loads and the LDS and 0.25 vector
// instructions. 2,000 paths, 40 forwards x 5 factors, 30 swaptions: 117 us (187 us for lmm_spot_kernel); 80 x 10 and 4,000
// paths: 400 us (815 us).
//
// Values to be averaged go to a table [column][P], and rows64_partials_kernel forms from it the partials
// of 64 paths, in the operations of lmm_spot_kernel.
#pragma once

#include "lmm_chunks.hpp"
#include "lmm_spot64.hpp"

namespace fm {

constexpr int kRowPaths = 4;        // paths per wavefront, and per workgroup

// x of lane L of each row of sixteen lanes.
template <int L>
__device__ __forceinline__ double row_broadcast(double x) {
    return __builtin_amdgcn_update_dpp(x, x, 0x150 + L, 0xf, 0xf, false);
}

// R components per lane: component 16 q + g in element q of lane g.
template <int R>
struct RowForwards {
    static constexpr int W = 16 * R, chunks = 1;
    double z[R];
    // Component j for a uniform run-time j, in every lane of the row.
    __device__ __forceinline__ double get(int j) {
        double r = z[0];
        static_for<1, R>([&](auto Q) { r = j / 16 == decltype(Q)::value ? z[decltype(Q)::value] : r; });
        return __shfl(r, j % 16, 16);
    }
    template <int Q> __device__ __forceinline__ double element(int e) { return get(e); }
};

// A lane's record of one round and column k = g of the round's sixteen.
template <int FCAP>
struct RowRecord {
    double own[FCAP + 3], col[16];
    __device__ __forceinline__ void load(const double* rec, int rec_n, int q, int g) {
        constexpr int size = rec_size_of(FCAP);
        // components beyond the table's last repeat it (their weights are zero)
        const double* o = rec + (16 * q + g < rec_n ? 16 * q + g : rec_n - 1) * size;
#pragma unroll
        for (int k = 0; k < FCAP + 3; k++) own[k] = o[k];
        const double* c = rec + (g < FCAP ? g : FCAP - 1);
#pragma unroll
        for (int l = 0; l < 16; l++) col[l] = c[(16 * q + l < rec_n ? 16 * q + l : rec_n - 1) * size];
    }
};

template <int R, int FCAP, bool lognormal>
__global__ void __launch_bounds__(64) lmm_rows64_kernel(const StepArgs) {
    constexpr int pitch = 17;       // odd: the sixteen components of a row lie on different banks
    __shared__ double sums[4][16][pitch];
    ArgPtr a = kernel_arguments();
    const int lane = threadIdx.x, g = lane & 15, row = lane >> 4;
    const Exp2Coef ke;
    constexpr int size = rec_size_of(FCAP);
    const uint32_t p0 = blockIdx.x * (uint32_t)kRowPaths + row;     // P < 2^31
    RowForwards<R> Y;
    double scale[R];                // s_j of the lane's components
    RowRecord<FCAP> recs[R];
    double dW;
    {
        const int P = a->P, n = a->n, nT = a->nT, F = a->F, rec_n = a->rec_n;
        const double* dw = (const double*)a->dw + (size_t)(p0 < (uint32_t)P ? p0 : P - 1) * nT * F;
        touch_tables(a);
        uint32_t touched = 0;       // and the increments of these paths
        for (int l = 16 * g; l < nT * F; l += 256) touched |= *(const volatile uint32_t*)(dw + l);
#if defined(__HIP_DEVICE_COMPILE__)
        asm volatile("" :: "v"(touched));
#endif
#pragma unroll
        for (int q = 0; q < R; q++) {
            const int j = 16 * q + g;
            Y.z[q] = j < n ? a->Y0[j] : 0.0;
            scale[q] = j < n ? a->lead[j] : 1.0;
            recs[q].load((const double*)a->rec, rec_n, q, g);
        }
        dW = dw[g < F ? g : F - 1];
    }
    double N = 1.0, Nprev = 1.0;
    int kcur = 0, knum = 0, qp = 0;
    // what the next step asks of the scalar cache first, requested a step ahead
    int first = ConstArray<int32_t>{a->first_alive}[0], tenor_at = ConstArray<int32_t>{a->tenor_time_index}[0];
    int eval_at = a->num_products > 0 ? ConstArray<KProduct>{a->products}[0].eval_index : -1;
    double t0 = ConstArray<double>{a->times}[0], t1 = ConstArray<double>{a->times}[1];
    double dk = ConstArray<double>{a->delta}[0], sk = ConstArray<double>{a->lead}[0];
    for (int ti = 0;; ti++) {
        a = kernel_arguments();
        const int P = a->P, n = a->n, nT = a->nT, F = a->F, rec_n = a->rec_n, num_slots = a->num_slots;
        const int64_t p = p0, pc = p < P ? p : (int64_t)P - 1;
        const bool active = p < P && g == 0;
        const ConstArray<double> lead{a->lead};
        const double* rec = (const double*)a->rec;
        double* const vals = a->values;
        auto val = [&](double z, int j) -> double { return lognormal ? lead[j] * fm_exp2(z, ke) : z; };
        while (kcur < n && tenor_at <= ti) {
            const double z = Y.get(kcur);
            const double Lk = lognormal ? sk * fm_exp2(z, ke) : z;
            double Nn;
            if (kcur == 0)      Nn = Lk * (dk * 1.0) + 1.0;
            else if (kcur == 1) Nn = Lk * (dk * N) + N;
            else                Nn = N * (1 + Lk * dk);
            Nprev = N; N = Nn; kcur++; knum = kcur;
            tenor_at = ConstArray<int32_t>{a->tenor_time_index}[kcur];      // n + 1 of them
            const int kn = kcur < n ? kcur : n - 1;
            dk = ConstArray<double>{a->delta}[kn];
            sk = lead[kn];
            if (active) {
                vals[(size_t)(num_slots + kcur) * P + p] = (1.0 / N) * 1.0;
                if (a->numeraire) a->numeraire[(size_t)kcur * P + p] = N;
            }
        }
        const ConstArray<KProduct> products{a->products};
        int walk = -1;
        auto walk_group = [&](int i, const KProduct& pr) -> bool {
            if (pr.walk < 0) return false;
            walk = i;
            return true;
        };
        if (eval_at == ti) {
            eval_products_at<true, double>(ti, qp, a->num_products, products, ConstArray<KPeriod>{a->periods},
                                           ConstArray<double>{a->delta}, N, Nprev, knum, Y, val, active, a->contrib, p, P,
                                           [&](double x, int slot) { if (active) vals[(size_t)slot * P + p] = x; }, walk_group);
            eval_at = qp < a->num_products ? products[qp].eval_index : -1;
        }
        if (ti == nT) break;

        const double dt = t1 - t0;
        const double cdt = lognormal ? dt * kLog2E : dt;
        const int next = ti + 1 < nT ? ti + 1 : ti;
        const int first_next = ConstArray<int32_t>{a->first_alive}[next];
        t0 = t1;
        t1 = ConstArray<double>{a->times}[next + 1];
        const double* rec_next = rec + (size_t)next * rec_n * size;
        double T = lognormal ? dW * kLog2E : dW;        // of factor g
        dW = ((const double*)a->dw)[((size_t)pc * nT + next) * F + (g < F ? g : F - 1)];
        int j0 = first, jw = 0, mw = 0;                 // the walk's first component, periods and swaptions
        const double* table = (const double*)a->walk;
        double Pw = 1.0, V = 0.0;
        int head = 0;
        if (walk >= 0) {
            const KProduct pr = products[walk];
            table += 8 * pr.walk;
            j0 = pr.first_j; jw = pr.num_periods; mw = 1 + pr.pad2; head = walk;
        }
        const int from = j0 < first ? j0 : first;
        static_for<0, R>([&](auto Q) {
            constexpr int q = decltype(Q)::value;
            if (16 * q + 15 >= from && 16 * q < n) {
                RowRecord<FCAP>& rc = recs[q];
                const int j = 16 * q + g;
                const bool walked = jw > 0 && 16 * q + 15 >= j0 && 16 * q < j0 + jw;
                const int i0 = 16 * q - j0;
                double aj = 0.0, strike[16];
                if (walked) {
                    auto at = [&](int i) { return i < 0 ? 0 : i < jw ? i : jw - 1; };
                    aj = table[8 * at(i0 + g)];
                    const double* st = table + 1 + (g < kSwaptionGroup ? g : 0);
#pragma unroll
                    for (int l = 0; l < 16; l++) strike[l] = st[8 * at(i0 + l)];
                }
                const double z = Y.z[q], e = rc.own[FCAP + 2];
                const double E = lognormal ? fm_exp2(z, ke) : z;
                const double b = E + e;
                const double r0 = __builtin_amdgcn_rcp(b);
                const double x = fma(-b, r0, 1.0);
                const double r = fma(r0, fma(x, x, x), r0);
                if (walked) {
                    const double f = e * r;
                    static_for<0, 16>([&](auto L) {
                        constexpr int l = decltype(L)::value;
                        if ((unsigned)(i0 + l) < (unsigned)jw) {
                            Pw = Pw * row_broadcast<l>(f);
                            const double Pa = Pw * row_broadcast<l>(aj);
                            V = fma(row_broadcast<l>(E) - strike[l], Pa, V);
                        }
                    });
                }
                if (16 * q + 15 >= first) {
                    double w = (lognormal ? cdt * E : cdt) * r;
                    w = j >= first && j < n ? w : 0.0;
                    static_for<0, 16>([&](auto L) {
                        constexpr int l = decltype(L)::value;
                        T = fma(row_broadcast<l>(w), rc.col[l], T);
                        sums[row][l][g] = T;
                    });
                    // the LDS works off a wavefront's accesses in order
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                    __builtin_amdgcn_wave_barrier();
                    double inc = rc.own[FCAP];
#pragma unroll
                    for (int k = 0; k < FCAP; k++) inc = fma(sums[row][g][k], rc.own[k], inc);
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                    __builtin_amdgcn_wave_barrier();
                    Y.z[q] = jmin(z + inc, rc.own[FCAP + 1]);
                    rc.load(rec_next, rec_n, q, g);
                }
            }
        });
        if (jw > 0 && g < mw && p < P) {
            const KProduct pg = a->products[head + g];
            vals[(size_t)pg.out_slot * P + p] = jmax0(V * pg.notional) / (pg.num_k == knum ? N : Nprev);
        }
        if (a->paths) {
            double* paths = (double*)a->paths + pc;
            const int32_t* row_of = a->row_of + (size_t)(ti + 1) * n;
#pragma unroll
            for (int q = 0; q < R; q++) {
                const int j = 16 * q + g;
                const double L = lognormal ? scale[q] * fm_exp2(Y.z[q], ke) : Y.z[q];
                if (j >= first && j < n && p < P) paths[(size_t)row_of[j] * P] = L;
            }
        }
        first = first_next;
    }
}

// Partials of 64 paths per wavefront from the table of values: of product i (a swaption group's at its first
// member) or, beyond the products, of a numeraire.
__device__ __forceinline__ void rows64_partials(const StepArgs& a, int i) {
    const int lane = threadIdx.x & 63;
    const int64_t p = (int64_t)blockIdx.x * kStepThreads + threadIdx.x;
    const int64_t wave = (int64_t)blockIdx.x * (kStepThreads / 64) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t left = (int64_t)a.P - wave * 64;
    if (left <= 0) return;
    const bool active = p < a.P;
    const int64_t pc = active ? p : (int64_t)a.P - 1;
    const int cnt = left > 64 ? 64 : (int)left;
    const int stride = a.num_slots + a.n + 1;
    if (i >= a.num_products) {
        const int k = i - a.num_products, col = a.num_slots + 1 + k;
        if (a.tenor_time_index[k] > a.nT) return;       // beyond the simulation: no such numeraire
        const double s = wave_reduce_sum(active ? a.values[(size_t)col * a.P + pc] : 0.0);
        if (lane == 0) a.wave_sum[(size_t)wave * stride + col] = s;
        return;
    }
    const KProduct pr = a.products[i];
    if ((unsigned)pr.eval_index > (unsigned)a.nT) return;
    if (pr.type == FM_PRODUCT_SWAPTION && a.products[i - pr.pad3].walk >= 0) {      // the first member's
        if (pr.pad3 != 0) return;
        double x[kSwaptionGroup];
        int slot[kSwaptionGroup];
#pragma unroll
        for (int g = 0; g < kSwaptionGroup; g++) {
            slot[g] = a.products[i + (g <= pr.pad2 ? g : 0)].out_slot;
            x[g] = a.values[(size_t)slot[g] * a.P + pc];
        }
        reduce_slots4(x, 1 + pr.pad2, active, cnt, 1.0 / (double)cnt, lane, wave, a.wave_sum, a.wave_m2, stride, slot);
    } else if (pr.type == FM_PRODUCT_SWAPTION || pr.type == FM_PRODUCT_CAPLET) {
        reduce_slot(a.values[(size_t)pr.out_slot * a.P + pc], active, cnt, lane, wave, a.wave_sum, a.wave_m2, stride,
                    pr.out_slot);
    }
}

static __global__ void __launch_bounds__(kStepThreads) rows64_partials_kernel(const StepArgs a) {
    for (int64_t i = blockIdx.y; i < (int64_t)a.num_products + a.n; i += gridDim.y) rows64_partials(a, (int)i);
}

template <int R, int FCAP>
void launch_rows64_cap(const StepArgs& a, hipStream_t stream) {
    const dim3 grid((unsigned)(((int64_t)a.P + kRowPaths - 1) / kRowPaths));
    if (a.lognormal) hipLaunchKernelGGL((lmm_rows64_kernel<R, FCAP, true>), grid, dim3(64), 0, stream, a);
    else hipLaunchKernelGGL((lmm_rows64_kernel<R, FCAP, false>), grid, dim3(64), 0, stream, a);
    HIP_CHECK(hipGetLastError());
}

template <int R>
void launch_rows64_n(const StepArgs& a, hipStream_t stream) {
    if (a.F <= 1) launch_rows64_cap<R, 1>(a, stream);
    else if (a.F <= 3) launch_rows64_cap<R, 3>(a, stream);
    else if (a.F <= 5) launch_rows64_cap<R, 5>(a, stream);
    else if (a.F <= 10) launch_rows64_cap<R, 10>(a, stream);
    else throw FmError(FM_ERR_UNSUPPORTED, "number of factors above 10 is not supported by the path kernel");
}

} // namespace fm
