"""The short forms that the sweeps use for ordinary cells, one operation and one
edge at a time: every quotient and root correctly rounded, every edge the
oracle's, bit for bit.  (swe_hip_solve_edges runs the general form.)"""
import ctypes as C
from pathlib import Path

import numpy as np
import pytest

from helpers import random_edges, same_bits

pytestmark = pytest.mark.gpu
LIB = Path(__file__).resolve().parent.parent / "swe-ppm_amd" / "libswe_hip_check.so"
RCP, DIV, SQRT, SQRT0 = range(4)
FP = C.POINTER(C.c_float)
MANTISSAS = np.arange(1 << 23, dtype=np.uint32)


@pytest.fixture(scope="module")
def check(swe):  # (the product library first: one HIP runtime)
    lib = C.CDLL(str(LIB))
    for f in (lib.swe_check_edges, lib.swe_check_arith):
        f.argtypes = [C.c_int, C.c_int64, FP, FP]

    def call(f, which, arrays, outs):
        ins = np.ascontiguousarray(np.stack(arrays), np.float32)
        out = np.empty((outs, ins.shape[1]), np.float32)
        assert f(which, ins.shape[1], ins.ctypes.data_as(FP), out.ctypes.data_as(FP)) == 0
        return out

    class Check:
        arith = staticmethod(lambda op, a, b: call(lib.swe_check_arith, op, [a, b], 1)[0])
        edges = staticmethod(lambda solver, ins: call(lib.swe_check_edges, solver, ins, 5))

    return Check


def _all_at(exponent):
    """Every float32 in [2^exponent, 2^(exponent + 1))."""
    return (MANTISSAS | np.uint32((exponent + 127) << 23)).view(np.float32)


@pytest.mark.parametrize("exponent", [-126, -61, 0, 64, 125])
def test_reciprocals(check, exponent):
    b = _all_at(exponent)
    assert same_bits(check.arith(RCP, b, b), np.float32(1) / b)


@pytest.mark.parametrize("exponent", [-102, -101, 0, 1, 126, 127])
def test_roots(check, exponent):
    x = _all_at(exponent)
    for op in (SQRT, SQRT0):
        got = check.arith(op, x, x)
        if op == SQRT0 and exponent < -100:  # promised from 2^-100 on, and for 0
            continue
        assert same_bits(got, np.sqrt(x))
    assert same_bits(check.arith(SQRT0, np.zeros(1), np.zeros(1)), np.zeros(1, np.float32))


@pytest.mark.parametrize("seed", range(4))
def test_quotients(check, seed):
    """Random operands, and numerators next to a divisor times a number halfway
    between two floats: the quotients hardest to round."""
    rng = np.random.default_rng(seed)
    n = 1 << 22
    mantissa = lambda: 1.0 + rng.integers(0, 1 << 23, n) * 2.0**-23  # noqa: E731
    b = np.ldexp(mantissa(), rng.integers(-60, 60, n))
    q = np.ldexp(mantissa(), rng.integers(-40, 40, n)) * rng.choice([-1.0, 1.0], n)
    for a in (q * b, q * (1.0 + 2.0**-24) * b, np.ldexp(mantissa(), rng.integers(-60, 60, n))):
        a, d = a.astype(np.float32), b.astype(np.float32)
        for step in (-np.inf, None, np.inf):
            num = a if step is None else np.nextafter(a, np.float32(step))
            assert same_bits(check.arith(DIV, num, d), num / d)


def _ordinary(ins):
    """The edges whose cells are in in_normal_range (edge_solver.hpp)."""
    keep = np.ones(ins[0].size, bool)
    with np.errstate(all="ignore"):
        for h, hu, b in zip(ins[0:2], ins[2:4], ins[4:6]):
            keep &= (np.abs(h) + np.abs(b) <= 2.0**40) & ((h < 0.01) | (np.abs(hu / h) <= 2.0**19))
    return [a[keep] for a in ins]


def _states():
    from test_oracle_solvers import still_edges

    rng = np.random.default_rng(3)
    n = 100_000
    calm = rng.uniform(0.5, 30.0, n)  # depths and Froude numbers around calm_edge's limit
    ratio, fl, fr = rng.uniform(0.44, 2.3, n), rng.uniform(-1.1, 1.1, n), rng.uniform(-1.1, 1.1, n)
    calm = [calm, calm * ratio, calm * fl * np.sqrt(9.81 * calm),
            calm * ratio * fr * np.sqrt(9.81 * calm * ratio), rng.normal(0, 1, n), rng.normal(0, 1, n)]
    fast = random_edges(n, 5)
    fast[2], fast[3] = fast[2] * 40, fast[3] * 40  # supercritical, strong shocks and vacuum
    return {"random": random_edges(200_000, 4), "still": still_edges(20_000, 6), "calm": calm, "fast": fast}


@pytest.mark.parametrize("solver", [0, 1, 2, 3])
@pytest.mark.parametrize("name", ["random", "still", "calm", "fast"])
def test_edges(check, oracle, solver, name):
    ins = _ordinary([np.asarray(a, np.float32) for a in _states()[name]])
    assert ins[0].size > 10_000
    dry = (ins[0] < 0.01).astype(int) * 2 + (ins[1] < 0.01)
    with np.errstate(all="ignore"):
        froude = np.nan_to_num(np.abs(ins[2] / ins[0]) / np.sqrt(9.81 * ins[0]))
    # mixed waves, and waves whose lanes are of one kind (the uniform short cuts)
    for order in (np.arange(dry.size), np.lexsort((froude, dry))):
        edges = [a[order] for a in ins]
        for k, (a, c) in enumerate(zip(check.edges(solver, edges), oracle.solve_edges(solver, *edges))):
            assert same_bits(a, c), (k, int(np.count_nonzero(a.view(np.uint32) != c.view(np.uint32))))
