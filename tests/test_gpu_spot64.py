"""The FP64 spot kernel (csrc/lmm_spot64.hpp) at the sizes where its layout changes: components in
pairs, register chunks of eight, factor capacities 1, 3, 5, 10, swaption groups valued by the Euler
step's walk or by a walk of their own.

Bars: process values within 1e-12 and prices within 1e-10 relative of the oracle, those of
test_gpu_parity.py. The two ways to value a swaption group differ in the rounding of at most 20 periods
(six operations each): 1e-13 relative."""
import numpy as np
import pytest

import _oracle as O
from finmath_hip import _abi
from finmath_hip import workloads as W
from test_gpu_parity import make_context, say, to_products

pytestmark = pytest.mark.gpu


def workload(n, F, strikes=(0.02, 0.03, 0.035, 0.04, 0.05)):
    wl = W.Workload(f"n{n}F{F}", n, 0.5, F, 0, 0.08, 0.02 + 0.0004 * np.arange(n))
    m = max(1, n // 2)
    for i in sorted({0, 1, n // 3, n - m} - {n}):
        if i + m <= n:
            wl.products += [W.swaption_spec(0.5 * i, 0.5 * m, 0.5, k) for k in strikes]
    wl.products.append(W.swap_spec(0.0, 0.5 * n, 0.5, 0.03))
    return wl


@pytest.mark.parametrize("n,F,P", [(1, 1, 65), (2, 2, 64), (3, 1, 1), (7, 3, 300), (8, 4, 257), (9, 5, 63), (16, 6, 130),
                                   (23, 10, 129), (24, 2, 256), (25, 5, 255), (39, 10, 191), (40, 3, 321), (41, 1, 70),
                                   (79, 5, 100), (80, 10, 90)])
def test_sizes_against_the_oracle(n, F, P):
    say(f"case spot64 n={n} F={F} P={P}")
    F = min(F, n)
    wl = workload(n, F)
    t = O.ModelTables(wl)
    ctx = make_context(wl, t, P, store_paths=True)
    ctx.simulate()
    om = O.OracleModel(t, P)
    for ti in {1, n // 2, n - 1, n} - {0}:
        for j in range(n):
            g, r = ctx.process_value(ti, j), om.process_value(ti, j)
            assert np.max(np.abs(g - r) / np.abs(r)) < 1e-12
    vals, errs = ctx.value_products(to_products(wl.products))
    for s, v, e in zip(wl.products, vals, errs):
        ov, oe = om.value(s)
        assert v == pytest.approx(ov, rel=1e-10, abs=1e-16)
        assert e == pytest.approx(oe, rel=1e-9, abs=1e-16)


@pytest.mark.parametrize("state", ["LOGNORMAL", "NORMAL"])
def test_cap_and_zero_forward(state):
    wl = workload(11, 3)
    t = O.ModelTables(wl, vol_params=(0.2, 0.0, 0.25, 0.1) if state == "LOGNORMAL" else (0.01, 0.0, 0.25, 0.004))
    t.L0 = t.L0.copy()
    t.L0[5] = 0.0
    say(f"case spot64 binding cap {state}")
    P, cap = 2001, 0.03
    ctx = _abi.LmmContext(t.times, t.tenor, 3, P, wl.seed, store_paths=True, libor_cap=cap, state_space=state)
    ctx.set_initial_forwards(t.L0)
    ctx.set_covariance(t.lam, t.var)
    ctx.simulate()
    om = O.OracleModel(t, P, cap=cap, with_discount=False, state_space=1 if state == "LOGNORMAL" else 0)
    capped = 0
    for ti in range(1, 12):
        for j in range(11):
            g, r = ctx.process_value(ti, j), om.process_value(ti, j)
            assert np.max(np.abs(g - r) / np.maximum(np.abs(r), 1e-3)) < 1e-12
            capped += int(np.sum(r == cap))
    assert capped > P


@pytest.mark.parametrize("members", [1, 3, 4, 5, 9])
def test_walk_in_the_step_and_walk_of_its_own(members):
    # periods whose discounting length is not the tenor period take a walk of their own, and so does a
    # second group of one date; a relative shift of 1e-12 in the payment dates keeps the value
    say(f"case spot64 swaption walks, {members} strikes")
    wl = workload(24, 5)
    t = O.ModelTables(wl)
    ctx = make_context(wl, t, 777)
    fix = t.tenor[6:18]
    pay = t.tenor[7:19]
    strikes = np.linspace(0.02, 0.05, members)
    near = [_abi.Product.swaption(fix[0], fix, pay, [k] * 12, period_lengths=pay - fix, notional=2.5) for k in strikes]
    far = [_abi.Product.swaption(fix[0], fix, pay * (1 + 1e-12), [k] * 12, period_lengths=pay - fix, notional=2.5)
           for k in strikes]
    a, ea = ctx.value_products(near)
    b, eb = ctx.value_products(far)
    # the shifted discounting lengths move a value by at most 12 periods x 1e-11 x L tau
    assert np.allclose(a, b, rtol=1e-11, atol=0)
    assert np.allclose(ea, eb, rtol=1e-10, atol=0)
    single = [ctx.value_products([p])[0][0] for p in near]
    assert np.allclose(a, single, rtol=1e-13, atol=0)
