"""Random-variable programs on eight registers (csrc/rv.hip: rv_compact_kernel) against the general
interpreter: the same operations in the same order, so realisations, averages and variances are equal bit for
bit. A program with an unused power in it always takes the general interpreter. Sizes: one realisation,
a ragged workgroup, one trip of the grid, and more than one (four elements per thread)."""
import ctypes
from ctypes import c_double, c_void_p

import numpy as np
import pytest

from finmath_hip import _abi
from finmath_hip.randomvariable import OP, RandomVariable
from test_gpu_parity import say

pytestmark = pytest.mark.gpu

UNARY = ["EXP", "LOG", "SQRT", "ABS", "INVERT", "SQUARED", "ISNAN"]
BINARY = ["ADD", "SUB", "MULT", "DIV", "CAP", "FLOOR", "ACCRUE", "DISCOUNT"]
TERNARY = ["ADD_PRODUCT", "ADD_RATIO", "SUB_RATIO", "CHOOSE"]


def program(rng, inputs, registers, length):
    """LOADs, CONSTs and operations over `registers` registers, some of them read before they are written."""
    prog = [(OP["LOAD"], int(rng.integers(registers)), i, 0, 0, 0.0) for i in range(inputs)]
    prog.append((OP["CONST"], int(rng.integers(registers)), 0, 0, 0, 0.75))
    for _ in range(length):
        name = str(rng.choice(UNARY + 2 * BINARY + 2 * TERNARY + ["LOAD"]))
        a, b, c = (int(x) for x in rng.integers(registers, size=3))
        if name == "LOAD":
            a = int(rng.integers(inputs))
        prog.append((OP[name], int(rng.integers(registers)), a, b, c, float(rng.choice([0.5, 0.25, 2.0]))))
    return prog


def run(variables, prog, result, probabilities=None):
    lib = _abi.load()
    arr = (c_void_p * len(variables))(*[v._leaf().handle.ptr for v in variables])
    ins = (_abi.FmRvInstr * len(prog))()
    for k, (op, dst, a, b, c, imm) in enumerate(prog):
        ins[k].op, ins[k].dst, ins[k].a, ins[k].b, ins[k].c, ins[k].imm = op, dst, a, b, c, imm
    out = c_void_p()
    _abi.check(lib.fm_rv_evaluate(len(variables), arr, len(prog), ins, result, 0.0, ctypes.byref(out)))
    avg, var = c_double(), c_double()
    p = c_void_p(probabilities._leaf().handle.ptr) if probabilities is not None else None
    _abi.check(lib.fm_rv_evaluate_average(len(variables), arr, len(prog), ins, result, p, ctypes.byref(avg),
                                          ctypes.byref(var)))
    return RandomVariable._from_ptr(out.value).getRealizations(), avg.value, var.value


@pytest.mark.parametrize("size", [1, 300, 70_001, 4_194_305 + 600])
@pytest.mark.parametrize("seed", range(12))
def test_equal_to_the_general_interpreter(size, seed):
    say(f"case rv compact size={size} seed={seed}")
    rng = np.random.default_rng(seed)
    inputs = 1 + seed % 5
    values = [rng.standard_normal(size) for _ in range(inputs)]
    if size > 100 and seed % 2:
        values[0][[3, 17, 40, 77]] = [np.nan, np.inf, -0.0, 0.0]
    variables = [RandomVariable.from_array(v) for v in values]
    registers = [2, 5, 8, 13][seed % 4]
    length = [0, 1, 4, 9, 20][seed % 5]
    prog = program(rng, inputs, registers, length)
    result = int(rng.integers(registers))
    weights = RandomVariable.from_array(rng.uniform(0.5, 1.5, size) / size) if seed % 3 == 0 else None
    v, avg, var = run(variables, prog, result, weights)
    w, avg2, var2 = run(variables, prog + [(OP["POW"], 15, 0, 0, 0, 0.0)], result, weights)
    assert np.array_equal(v.view(np.int64)[~np.isnan(v)], w.view(np.int64)[~np.isnan(v)])
    assert np.array_equal(np.isnan(v), np.isnan(w))
    assert np.array_equal([avg, var], [avg2, var2], equal_nan=True)
