"""Models and calls at the edge of what the entry points take. Each is compared with the oracle, with the same call
in another form, or with a value worked out by hand; the bars are stated with each test."""
import ctypes

import numpy as np
import pytest

import _oracle as O
from finmath_hip import _abi
from finmath_hip.randomvariable import RandomVariable
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


# ---- a forward that overflows as it is fixed ---------------------------------------------------------

@pytest.mark.parametrize("P", [300, 9001])
@pytest.mark.parametrize("precision,scheme", [("FP64", "EULER_FUNCTIONAL"), ("FP32_MIXED", "EULER_FUNCTIONAL"), ("FP64", "EULER")])
def test_overflow_of_a_fixed_forward(precision, scheme, P):
    """L_2 starts at 1e6 with a volatility in the step that ends at its fixing, on a factor of its own, that takes its
    logarithm to the overflow: on about half of the paths it is infinite from then on, and so are the later numeraires.
    Products on other forwards are worth nothing there and must not become NaN. Bars: those of test_gpu_parity.py
    (FP64) and 0.1 bp (FP32-mixed)."""
    say(f"case overflow of a fixed forward {precision} {scheme} P={P}")
    n = 6
    wl = workload(n, 2)
    t = O.ModelTables(wl)
    t.L0 = t.L0.copy()
    t.L0[2] = 1.0e6
    t.vol = np.full_like(t.vol, 0.2)
    t.vol[:, 2] = 0.0
    # the drift of the logarithm is sigma^2 dt / 2 at L d >> 1: to ln(1.8e308), or ln(3.4e38), from ln(1e6)
    t.vol[1, 2] = (4 * ((709.8 if precision == "FP64" else 88.7) - 13.8)) ** 0.5
    t.factors = np.zeros_like(t.factors)
    t.factors[:, 0] = 1.0
    t.factors[2] = [0.0, 1.0]
    t.lam = t.vol[:, :, None] * t.factors[None]
    t.var = t.vol * t.vol
    ctx = _abi.LmmContext(t.times, t.tenor, 2, P, wl.seed, precision=precision, scheme=scheme, libor_cap=np.inf)
    ctx.set_initial_forwards(t.L0)
    ctx.set_covariance(t.lam, t.var)
    v, e = ctx.value_products([_abi.Product.caplet(0.5 * j, 0.5, 0.02) for j in (1, 3, 4, 5)])
    om = O.OracleModel(t, P, cap=None, with_discount=False, scheme={"EULER": 0, "EULER_FUNCTIONAL": 2}[scheme])
    over = om.process_value(2, 2) > np.finfo(np.float64 if precision == "FP64" else np.float32).max
    assert 0.2 < np.mean(over) < 0.8
    for j, x, y in zip((1, 3, 4, 5), v, e):
        ov, oe = om.caplet(0.5 * j, 0.5, 0.02)
        if precision == "FP64":
            assert x == pytest.approx(ov, rel=1e-10, abs=1e-16) and y == pytest.approx(oe, rel=1e-9, abs=1e-16)
        else:
            assert abs(x - ov) < 1e-5 and abs(y - oe) < 1e-5


# ---- calls without device allocation after a change of the model ------------------------------------

def _sv_driver(t, P):
    return _abi.LmmContext(t.times, t.tenor, 2, P, 31415)


@pytest.mark.parametrize("n,F,precision,state,scheme", [
    (9, 1, "FP64", "LOGNORMAL", "EULER_FUNCTIONAL"), (9, 3, "FP64", "NORMAL", "EULER_FUNCTIONAL"),
    (8, 2, "FP64", "LOGNORMAL", "PREDICTOR_CORRECTOR"), (9, 1, "FP32_MIXED", "LOGNORMAL", "EULER_FUNCTIONAL"),
    (9, 3, "FP32_MIXED", "NORMAL", "EULER_FUNCTIONAL"), (7, 1, "FP64_LOGSTATE", "LOGNORMAL", "EULER_FUNCTIONAL")])
@pytest.mark.parametrize("first", ["plain", "scaled"])
def test_noalloc_after_a_stochastic_volatility_comes_or_goes(n, F, precision, state, scheme, first):
    """A stochastic volatility scaling brings no table of its own, so a call without allocation goes on working after
    it is set or removed, whichever model the context was first priced with; values and errors are those of the
    allocating call, bit for bit. A first local-volatility table is still refused."""
    say(f"case noalloc after a change n={n} F={F} {precision} {state} {scheme} {first}")
    P = 500
    wl = workload(n, F)
    t = O.ModelTables(wl, vol_params=(0.2, 0.0, 0.25, 0.1) if state == "LOGNORMAL" else (0.01, 0.0, 0.25, 0.004))
    ctx = _abi.LmmContext(t.times, t.tenor, F, P, wl.seed, precision=precision, state_space=state, scheme=scheme)
    ctx.set_initial_forwards(t.L0)
    ctx.set_covariance(t.lam, t.var)
    ctx.set_discount_curve(t.pd)
    products = to_products([s for s in wl.products if s["type"] == "swaption"])
    driver = _sv_driver(t, P)
    order = [False, True, False] if first == "plain" else [True, False, True]
    for i, scaled in enumerate(order):
        ctx.set_stochastic_volatility(0.3, -0.3, driver if scaled else None)
        if i == 0:
            ctx.value_products(products)
        v, e = ctx.value_products_noalloc(products)
        w, f = ctx.value_products(products)
        assert np.array_equal(v, w) and np.array_equal(e, f)
    ctx.set_local_volatility(0.5, 0.5 * t.L0[None, :] + 0.0 * t.vol)
    with pytest.raises(_abi.IllegalStateException):
        ctx.value_products_noalloc(products)
    w, f = ctx.value_products(products)
    v, e = ctx.value_products_noalloc(products)
    assert np.array_equal(v, w) and np.array_equal(e, f)


@pytest.mark.parametrize("precision", ["FP64", "FP32_MIXED"])
def test_noalloc_up_to_its_documented_scratch(precision):
    """Two partials of 8 bytes per slot, forward and 64 paths, a product table of 64 bytes and periods of 56 bytes (every
    swaption of a group has a second copy of its own), the averages, all rounded up to 256 bytes: what fits 64 MiB
    by that count is valued."""
    n, strikes = 10, np.linspace(0.01, 0.06, 40)
    wl = workload(n, 1, strikes=strikes)
    specs = [s for s in wl.products if s["type"] == "swaption"]
    t = O.ModelTables(wl)
    def up(b):
        return (b + 255) // 256 * 256
    m = len(specs)
    columns = m + n + 1
    periods = sum(len(s["fixing"]) for s in specs)
    fixed = up(64 * m) + up(56 * 2 * periods) + up(16 * columns)
    waves = ((64 << 20) - fixed) // 2 // 256 * 256 // (8 * columns)
    assert 2 * up(waves * columns * 8) + fixed <= 64 << 20
    P = waves * 64
    say(f"case noalloc at its limit {precision} P={P} products={m}")
    ctx = make_context(wl, t, P, precision=precision)
    w, f = ctx.value_products(to_products(specs))
    v, e = ctx.value_products_noalloc(to_products(specs))
    assert np.array_equal(v, w) and np.array_equal(e, f)


def test_noalloc_beyond_its_derived_tables():
    """3,400 swaptions of 79 periods that share no walk need 8.6 MB of FP32 walk tables; without them each is valued by
    a walk over its periods, as one whose group has none. Bar: that of FP32-mixed prices, 0.1 bp."""
    say("case noalloc beyond its derived tables")
    n, m = 80, 3400
    wl = workload(n, 1)
    t = O.ModelTables(wl)
    fix, pay = t.tenor[1:n], t.tenor[2:n + 1]
    products = [_abi.Product.swaption(fix[0], fix, pay, np.full(n - 1, 0.03), period_lengths=(pay - fix) * (1 + 1e-6 * i))
                for i in range(m)]
    ctx = make_context(wl, t, 100, precision="FP32_MIXED")
    w, f = ctx.value_products(products)
    v, e = ctx.value_products_noalloc(products)
    assert np.max(np.abs(v - w)) < 1e-5 and np.max(np.abs(e - f)) < 1e-5
    assert np.all(np.isfinite(w)) and np.min(w) > 1e-4


# ---- grid dimensions --------------------------------------------------------------------------------

@pytest.mark.parametrize("count,P", [(66_000, 64), (4_000, 8192), (4_200, 8192), (70_000, 200)])
def test_many_products_on_few_paths(count, P):
    """More lowered products than 65,536, and tables of values on both sides of the size up to which the kernel for few
    paths runs: values and errors are those of the kernel for many paths, bit for bit."""
    say(f"case many products {count} P={P}")
    wl = workload(28, 2)
    t = O.ModelTables(wl)
    ctx = make_context(wl, t, P)
    products = [_abi.Product.caplet(0.5 * (i % 4), 0.5, 0.01 + 1e-7 * i) for i in range(count)]
    v, e = ctx.value_products(products)
    w, f = ctx.value_products_noalloc(products)
    assert np.array_equal(v, w) and np.array_equal(e, f)


def test_swaps_of_many_periods_on_few_paths():
    """67,200 periods of 2,400 swaps: each is worth the same swap's alone."""
    say("case many swap periods")
    wl = workload(28, 2)
    t = O.ModelTables(wl)
    ctx = make_context(wl, t, 70)
    products = to_products([wl.products[-1]])
    v, e = ctx.value_products(products)
    w, f = ctx.value_products(products * 2_400)
    assert np.array_equal(w, np.full(2_400, v[0])) and np.array_equal(f, np.full(2_400, e[0]))


def test_more_partials_than_a_grid_dimension():
    """8,388,610 wavefronts, 65,537 groups of them: every path of a forward fixed at time 0 pays the same, so the average
    is that payoff over 1 + L d, exactly (a sum of 2^29 + 130 equal numbers rounds once), and its error is rounding."""
    P = (1 << 29) + 130
    say(f"case partials beyond a grid dimension P={P}")
    ctx = _abi.LmmContext([0.0, 0.5], [0.0, 0.5], 1, P, 3141, precision="FP32_MIXED")
    ctx.set_initial_forwards([0.25])
    ctx.set_covariance(np.full((1, 1, 1), 0.2), np.full((1, 1), 0.04))
    v, e = ctx.value_products([_abi.Product.caplet(0.0, 0.5, 0.125)])
    assert v[0] == pytest.approx(0.5 * 0.125 / 1.125, rel=4e-16)
    assert e[0] < 1e-15
    ctx.close()


# ---- reductions -------------------------------------------------------------------------------------

def test_merged_partials_keep_their_compensation():
    """Partials whose sum needs more than 53 bits, in rows that are merged 128 at a time first: the compensation of a merged
    row counts like its sum. Every column holds 2^53 in its first row, -2^53 in a row of another group and ones in
    between, so its sum is the number of ones, exactly."""
    say("case compensated merge of partials")
    lib = _abi.load()
    launch = lib._ZN2fm22launch_reduce_partialsEPdS0_iiiiiS0_S0_Pv
    launch.restype = None
    p, i = ctypes.c_void_p, ctypes.c_int
    launch.argtypes = [p, p, i, i, i, i, i, p, p, p]

    def pointer(rv):
        out = ctypes.c_void_p()
        _abi.check(lib.fm_rv_device_ptr(ctypes.c_void_p(rv.devicePointer()), ctypes.byref(out)))
        return out

    for rows, slots, sums in ((2049, 3, 2), (2049, 32, 0), (2176, 31, 2), (4100, 64, 5), (2050, 60, 41)):
        say(f"  rows={rows} slots={slots} sums={sums}")
        cols = slots + sums
        part = np.ones((rows, cols))
        part[0] = 2.0 ** 53
        part[rows - 1] = -2.0 ** 53
        P = rows * 64 - 7
        count = np.full(rows, 64.0)
        count[-1] = 57.0
        exact = float(rows + np.sum(count * (part[:, 0] / count - (rows - 2) / P) ** 2))
        d_part, d_m2, d_sum, d_var = (RandomVariable.from_array(x) for x in (part.ravel(), np.ones(rows * cols), np.zeros(cols + 2),
                                                                             np.zeros(cols + 2)))
        launch(pointer(d_part), pointer(d_m2), rows, cols, slots, sums, P, pointer(d_sum), pointer(d_var), None)
        lib.hipDeviceSynchronize()      # the launch is on the null stream, which the copies below do not wait for
        assert np.array_equal(d_sum.getRealizations()[:cols], np.full(cols, rows - 2.0))
        assert np.allclose(d_var.getRealizations()[:slots], exact, rtol=1e-12, atol=0)


# ---- timings ----------------------------------------------------------------------------------------

def test_the_whole_call_includes_its_product_tables():
    """30,000 caplets are 4 MB of tables: at the 64 GB/s of the host link they take 60 us, which belong to the whole call and
    to none of its stages."""
    say("case timings with large product tables")
    wl = workload(4, 1)
    t = O.ModelTables(wl)
    ctx = make_context(wl, t, 64)
    products = [_abi.Product.caplet(0.5, 0.5, 0.01 + 1e-6 * i) for i in range(30_000)]
    ctx.value_products(products)
    ctx.value_products(products)
    ms = ctx.timings()
    assert ms[0] == 0.0 and ms[4] - ms[1] - ms[2] > 0.02


# ---- few paths: the line between the two FP64 spot kernels -----------------------------------------

@pytest.mark.parametrize("n,F", [(7, 7), (8, 6), (8, 8), (13, 10), (14, 8), (15, 5), (16, 1), (16, 3), (16, 5), (16, 10), (27, 2),
                                 (28, 4), (48, 5), (49, 5), (80, 8)])
@pytest.mark.parametrize("P", [63, 4096, 4097, 8193])
def test_few_paths_are_priced_as_many(n, F, P):
    """Values and errors of either kernel are equal bit for bit: a call without allocation takes the one for many paths."""
    say(f"case few paths n={n} F={F} P={P}")
    wl = workload(n, F)
    t = O.ModelTables(wl)
    ctx = make_context(wl, t, P)
    products = to_products([s for s in wl.products if s["type"] == "swaption"]) + [_abi.Product.caplet(0.5 * (n // 2), 0.5, 0.025)]
    v, e = ctx.value_products(products)
    w, f = ctx.value_products_noalloc(products)
    assert np.array_equal(v, w) and np.array_equal(e, f)
