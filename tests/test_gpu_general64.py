"""The FP64 general kernel (csrc/lmm_general64.hpp) at the sizes where its layout changes: pairs of
components and an odd last one, capacities of 24, 40 and 80 forwards and of 3, 5 and 10 factors, one
path more or less than a wavefront; every scheme under both measures, with and without the wrappers, and
a binding cap.

Bars: process values within 1e-12 (of the larger of the value and 1 %, as normal forwards cross zero) and
prices within 1e-10 relative of the oracle, those of test_gpu_variants.py."""
import numpy as np
import pytest

import _oracle as O
from finmath_hip import _abi
from test_gpu_parity import say, to_products
from test_gpu_spot64 import workload
from test_gpu_variants import MEASURES, SCHEMES

pytestmark = pytest.mark.gpu

SIZES = [(1, 1, 65), (2, 2, 64), (3, 3, 1), (8, 1, 257), (9, 4, 63), (23, 5, 130), (24, 10, 129), (25, 3, 70), (39, 6, 90),
         (40, 5, 200), (41, 2, 66), (79, 10, 64), (80, 5, 70)]


def case(n, F, P, measure, scheme, state, wrapper, cap=1e5):
    say(f"case general64 n={n} F={F} P={P} {measure} {scheme} {state} {wrapper} cap={cap}")
    wl = workload(n, min(F, n))
    lv = (0.4, 0.01) if "lv" in wrapper else None
    scale = 15.0 if lv and state == "LOGNORMAL" else 1.0
    vol = (0.2, 0.0, 0.25, 0.1) if state == "LOGNORMAL" or lv else (0.006, 0.0, 0.25, 0.002)
    t = O.ModelTables(wl, vol_params=tuple(v * (scale if i in (0, 1, 3) else 1.0) for i, v in enumerate(vol)))
    ctx = _abi.LmmContext(t.times, t.tenor, wl.num_factors, P, wl.seed, measure=measure, scheme=scheme, state_space=state,
                          store_paths=True, libor_cap=cap)
    ctx.set_initial_forwards(t.L0)
    ctx.set_covariance(t.lam, t.var)
    ctx.set_discount_curve(t.pd)
    if lv:
        ctx.set_local_volatility(lv[0], np.full((wl.num_time_steps, n), lv[1]))
    sv = None
    if "sv" in wrapper:
        driver = _abi.LmmContext(t.times, t.tenor, 2, P, 31415)
        ctx.set_stochastic_volatility(0.3, -0.3, driver, 0, 1)
        sv = (0.3, -0.3, 31415, 2, 0, 1)
    om = O.OracleModel(t, P, measure=MEASURES.index(measure), scheme=SCHEMES.index(scheme),
                       state_space=1 if state == "LOGNORMAL" else 0, local_vol=lv, stochastic_vol=sv, cap=cap)
    ctx.simulate()
    for ti in {1, n // 2, n - 1, n} - {0}:
        for j in range(n):
            g, r = ctx.process_value(ti, j), om.process_value(ti, j)
            assert np.max(np.abs(g - r) / np.maximum(np.abs(r), 0.01)) < 1e-12
    vals, errs = ctx.value_products(to_products(wl.products))
    for s, v, e in zip(wl.products, vals, errs):
        ov, oe = om.value(s)
        assert v == pytest.approx(ov, rel=1e-10, abs=1e-15)
        assert e == pytest.approx(oe, rel=1e-9, abs=1e-15)


@pytest.mark.parametrize("n,F,P", SIZES)
@pytest.mark.parametrize("measure", ["SPOT", "TERMINAL"])
def test_sizes(n, F, P, measure):
    i = SIZES.index((n, F, P)) + (measure == "TERMINAL")
    state = ["LOGNORMAL", "NORMAL"][i % 2]
    case(n, F, P, measure, "PREDICTOR_CORRECTOR", state, "")
    case(n, F, P, measure, "EULER" if measure == "SPOT" else "EULER_FUNCTIONAL", state, "")
    case(n, F, P, measure, ["EULER_FUNCTIONAL", "PREDICTOR_CORRECTOR"][i // 2 % 2], state, ["lv", "sv", "lv+sv"][i % 3])


@pytest.mark.parametrize("measure", ["SPOT", "TERMINAL"])
@pytest.mark.parametrize("state", ["LOGNORMAL", "NORMAL"])
@pytest.mark.parametrize("scheme", SCHEMES)
@pytest.mark.parametrize("wrapper", ["", "lv", "sv"])
def test_binding_cap(measure, state, scheme, wrapper):
    case(11, 3, 301, measure, scheme, state, wrapper, cap=0.031)
