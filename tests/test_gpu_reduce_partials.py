"""Averages over more wavefronts than one workgroup per column merges by itself (csrc/lmm_reduce.hip: rows of
partials are merged 128 at a time first), at one wavefront and one path more than the limit and with a
ragged last group, swaps and numeraires included. Bars: prices within 1e-10 and errors within 1e-9 relative of
the oracle, those of test_gpu_parity.py."""
import pytest

import _oracle as O
from test_gpu_parity import make_context, say, to_products
from test_gpu_spot64 import workload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P", [131_072, 131_073, 139_329, 200_001])
def test_averages(P):
    say(f"case reduce partials P={P}")
    wl = workload(4, 2)
    t = O.ModelTables(wl)
    vals, errs = make_context(wl, t, P).value_products(to_products(wl.products))
    om = O.OracleModel(t, P)
    for s, v, e in zip(wl.products, vals, errs):
        ov, oe = om.value(s)
        assert v == pytest.approx(ov, rel=1e-10, abs=1e-16)
        assert e == pytest.approx(oe, rel=1e-9, abs=1e-16)
