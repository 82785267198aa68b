"""The FP32-mixed spot kernel (csrc/lmm_spot32.hpp) and the reverse sweep (csrc/lmm_spot_adjoint.hpp) at
the sizes where their layout changes: pairs and groups of four components, register chunks, factor
capacities, swaption groups of one to four members and more.

Bars: FP32-mixed prices within 0.1 bp of the oracle (test_gpu_parity.py); FP64 gradients within 1e-10 and
FP32-mixed ones within 2e-3 of the tape's largest entry (test_gpu_aad_oracle.py)."""
import numpy as np
import pytest

import _oracle as O
from finmath_hip import workloads as W
from test_gpu_aad_oracle import close, gpu_context, swaptions
from test_gpu_parity import make_context, say, to_products
from test_gpu_spot64 import workload

pytestmark = pytest.mark.gpu

SIZES = [(1, 1, 65), (2, 2, 64), (3, 3, 200), (7, 3, 300), (8, 4, 257), (9, 5, 63), (15, 10, 130), (17, 1, 129), (25, 5, 255),
         (32, 2, 190), (33, 3, 321), (41, 6, 130), (48, 5, 100), (49, 1, 70), (79, 10, 90), (80, 5, 66)]


@pytest.mark.parametrize("n,F,P", SIZES)
def test_fp32_prices(n, F, P):
    say(f"case spot32 n={n} F={F} P={P}")
    wl = workload(n, min(F, n))
    t = O.ModelTables(wl)
    vals, errs = make_context(wl, t, P, precision="FP32_MIXED").value_products(to_products(wl.products))
    om = O.OracleModel(t, P)
    for s, v, e in zip(wl.products, vals, errs):
        ov, oe = om.value(s)
        assert abs(v - ov) < 1e-5 and abs(e - oe) < 1e-5


@pytest.mark.parametrize("precision,tol", [("FP64", 1e-10), ("FP32_MIXED", 2e-3)])
@pytest.mark.parametrize("n,F,P", SIZES[1:])
def test_gradients(n, F, P, precision, tol):
    state = "NORMAL" if n % 3 == 0 else "LOGNORMAL"
    stride = 1 + n % 5
    say(f"case adjoint n={n} F={F} P={P} {precision} {state} stride={stride}")
    wl = workload(n, min(F, n))
    t = O.ModelTables(wl, vol_params=(0.2, 0.0, 0.25, 0.1) if state == "LOGNORMAL" else (0.01, 0.0, 0.25, 0.004))
    specs = [s for s in wl.products if s["type"] == "swaption"]
    ctx = gpu_context(wl, t, P, precision=precision, stride=stride, state_space=state)
    v, dL, dsig = ctx.adjoint(swaptions(specs))
    vt, dY, dvol, _ = O.aad_swaptions(t, P, specs, state_space=1 if state == "LOGNORMAL" else 0)
    assert v == pytest.approx(vt, rel=1e-12 if precision == "FP64" else 1e-4)
    close(dL * t.L0 if state == "LOGNORMAL" else dL, dY, tol, "deltas")
    close(dsig, dvol, tol, "volatility entries")


@pytest.mark.parametrize("precision,tol", [("FP64", 1e-10), ("FP32_MIXED", 2e-3)])
def test_gradients_under_a_binding_cap(precision, tol):
    say(f"case adjoint binding cap {precision}")
    wl = workload(13, 3)
    t = O.ModelTables(wl)
    specs = [s for s in wl.products if s["type"] == "swaption"]
    v, dL, dsig = gpu_context(wl, t, 1500, precision=precision, cap=0.031).adjoint(swaptions(specs))
    vt, dY, dvol, _ = O.aad_swaptions(t, 1500, specs, cap=0.031)
    assert v == pytest.approx(vt, rel=1e-12 if precision == "FP64" else 1e-4)
    close(dL * t.L0, dY, tol, "deltas")
    close(dsig, dvol, tol, "volatility entries")
