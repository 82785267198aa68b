"""Models and calls at the edge of what the entry points take. Each is compared with the oracle, with the same call
in another form, or with a value worked out by hand; the bars are stated with each test."""
import ctypes

import numpy as np
import pytest

import _oracle as O
from finmath_hip import _abi
from test_gpu_aad_oracle import gpu_context, swaptions
from test_gpu_parity import make_context, say, to_products
from test_gpu_spot64 import workload

pytestmark = pytest.mark.gpu


# ---- a first forward at or below zero: fixed at time 0, moved by no step ----------------------------

@pytest.mark.parametrize("precision,tol", [("FP64", 1e-9), ("FP32_MIXED", 1e-5)])
def test_gradient_of_a_fixed_forward_at_zero(precision, tol):
    """A negative first forward of the log-normal model is held at zero. The gradient is a smooth function of that forward,
    so at zero it is the one at 1e-11 up to 1e-11 times a bounded second derivative (at most a few times
    the number of periods): 1e-9 of its largest entry in FP64. In FP32 the paths are those of L = 1e-11 f: float rounding, 1e-5."""
    say(f"case adjoint fixed forward at zero {precision}")
    wl = workload(9, 3)
    t = O.ModelTables(wl)
    products = to_products([s for s in wl.products if s["type"] == "swaption"])
    products += [_abi.Product.caplet(0.0, 0.5, -0.01), _abi.Product.caplet(0.0, 0.5, 0.02, is_floorlet=True),
                 _abi.Product.caplet(1.0, 0.5, 0.02), to_products([wl.products[-1]])[0]]
    got = {}
    for first in (1e-11, 0.0, -0.01):
        t.L0 = t.L0.copy()
        t.L0[0] = first
        got[first] = gpu_context(wl, t, 500, precision=precision, with_discount=False).adjoint(products)
    v, dL, dsig = got[1e-11]
    for first in (0.0, -0.01):
        w, eL, esig = got[first]
        assert w == pytest.approx(v, rel=tol)
        assert np.max(np.abs(eL - dL)) <= tol * np.max(np.abs(dL))
        assert np.max(np.abs(esig - dsig)) <= tol * np.max(np.abs(dsig))
    assert abs(dL[0]) > 0.1 * np.max(np.abs(dL))


# ---- a cap at zero: every log-normal forward is zero ------------------------------------------------

@pytest.mark.parametrize("P", [300, 9000])
@pytest.mark.parametrize("measure,scheme", [("SPOT", "EULER_FUNCTIONAL"), ("SPOT", "PREDICTOR_CORRECTOR_FUNCTIONAL"),
                                            ("TERMINAL", "EULER_FUNCTIONAL"), ("SPOT", "EULER")])
@pytest.mark.parametrize("precision", ["FP64", "FP64_LOGSTATE"])
def test_cap_at_zero(precision, measure, scheme, P):
    """Every forward and every rate is zero and every numeraire one: a floorlet pays its strike times its daycount
    fraction on every path, exactly."""
    say(f"case cap at zero {precision} {measure} {scheme} P={P}")
    wl = workload(9, 3)
    t = O.ModelTables(wl)
    ctx = _abi.LmmContext(t.times, t.tenor, 3, P, wl.seed, precision=precision, measure=measure, scheme=scheme, libor_cap=0.0)
    ctx.set_initial_forwards(t.L0)
    ctx.set_covariance(t.lam, t.var)
    products = [_abi.Product.caplet(T, 0.5, 0.03125, is_floorlet=True) for T in (0.5, 2.0, 4.0)]
    products += to_products([s for s in wl.products if s["type"] == "swaption" and s["exercise"] > 0])
    v, e = ctx.value_products(products)
    assert np.array_equal(v[:3], np.full(3, 0.5 * 0.03125)) and np.array_equal(v[3:], np.zeros(len(v) - 3))
    assert np.array_equal(e, np.zeros(len(e)))
