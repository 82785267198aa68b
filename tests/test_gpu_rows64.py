"""The FP64 spot kernel for few paths (csrc/lmm_rows64.hpp) against the kernel for many (csrc/lmm_spot.hpp), which
does the same operations in the same order: prices, errors and process values are equal bit for bit. The
sizes are those where the layout changes: rounds of sixteen components, factor capacities, four paths
per wavefront, 64 per partial. A pricing call without device allocation always takes the kernel for many."""
import numpy as np
import pytest

import _oracle as O
from finmath_hip import _abi
from test_gpu_parity import say, to_products
from test_gpu_spot64 import workload

pytestmark = pytest.mark.gpu

SIZES = [(1, 1, 1), (2, 2, 3), (3, 3, 64), (8, 1, 65), (15, 4, 61), (16, 5, 129), (17, 3, 5), (31, 10, 200), (32, 2, 127),
         (33, 5, 70), (47, 7, 33), (48, 10, 258), (49, 1, 66), (64, 3, 90), (65, 5, 4), (79, 10, 63), (80, 6, 1001)]


def context(wl, t, P, state, cap=1e5, **kw):
    ctx = _abi.LmmContext(t.times, t.tenor, wl.num_factors, P, wl.seed, state_space=state, libor_cap=cap, **kw)
    ctx.set_initial_forwards(t.L0)
    ctx.set_covariance(t.lam, t.var)
    ctx.set_discount_curve(t.pd)
    return ctx


def tables(wl, state):
    return O.ModelTables(wl, vol_params=(0.2, 0.0, 0.25, 0.1) if state == "LOGNORMAL" else (0.01, 0.0, 0.25, 0.004))


@pytest.mark.parametrize("state,cap", [("LOGNORMAL", 1e5), ("NORMAL", 1e5), ("LOGNORMAL", 0.031)])
@pytest.mark.parametrize("n,F,P", SIZES)
def test_prices_are_those_of_the_other_kernel(n, F, P, state, cap):
    say(f"case rows64 n={n} F={F} P={P} {state} cap={cap}")
    wl = workload(n, min(F, n))
    ctx = context(wl, tables(wl, state), P, state, cap)
    products = to_products([s for s in wl.products if s["type"] == "swaption"])
    products += [_abi.Product.caplet(0.5 * i, 0.5, 0.025) for i in range(0, n, 3)]
    v, e = ctx.value_products(products)
    w, f = ctx.value_products_noalloc(products)
    assert np.array_equal(v, w) and np.array_equal(e, f, equal_nan=True)


@pytest.mark.parametrize("n,F", [(11, 3), (40, 5)])
def test_process_values_are_those_of_a_larger_run(n, F):
    P, p0, m = 70_000, 65_432, 301
    say(f"case rows64 process n={n} F={F}")
    wl = workload(n, F)
    t = tables(wl, "LOGNORMAL")
    full = context(wl, t, P, "LOGNORMAL", store_paths=True)
    part = context(wl, t, m, "LOGNORMAL", store_paths=True, path_offset=p0)
    full.simulate()
    part.simulate()
    for ti in (1, n // 2, n):
        for j in range(n):
            assert np.array_equal(part.process_value(ti, j), full.process_value(ti, j)[p0:p0 + m])
