"""Rounding error of one sweep in precision modes 1 and 2 against the FP64 sweep
from the same amplitudes.  Each bound is the root mean square difference that
the sweep had when every product was a launch of its own (grouped and chained
launches, FP64 exactly in the register-direct products): level launches may not
compute with less."""

import numpy as np
import pytest

from ccq_amd import engine as E
from ccq_amd import synth
from ccq_amd.inputs import build_integrals

pytestmark = pytest.mark.gpu


def _error(method, n, o, mode, block):
    s = synth.make_system(n, o, 2 * n, 1, sigma=min(0.05, synth.regime_sigma(n, o, 2 * n)))
    ints = build_integrals(s.h, s.e2int(), 0.0, 0, o, o)
    eng = E.Engine(0, o, o, n, method, rhf=True)
    eng.set_ints(ints.f_a, ints.f_b, ints.v_aa, ints.v_ab, ints.v_bb)
    out = []
    for m in (0, mode):
        eng.set_precision(0)
        eng.guess("mp2")
        for _ in range(3):
            eng.update()
        eng.set_precision(m)
        eng.update()
        out.append(eng.debug_read(*block) if block else eng.get_t())
    eng.close()
    return float(np.sqrt(np.mean((out[1] - out[0]) ** 2)))


@pytest.mark.parametrize("n,o,bound", [(20, 5, 4.550e-11)])
def test_partial_accumulators_of_fp32_storage(n, o, bound):
    """Terms that go to a partial accumulator are rounded to FP32 once, with their sum."""
    print(f"case FP32-storage partial accumulators CCSDT n={n} o={o}", flush=True)
    err = _error("CCSDT", n, o, 2, None)
    assert 0.0 < err <= bound


T2AB = ("T2.oovv.abab", (5, 5, 19, 19))


@pytest.mark.parametrize("method,n,o,block,bound", [("CCSD", 24, 5, T2AB, 2.080e-10), ("CCSDT", 12, 3, None, 2.048e-11)])
def test_arithmetic_of_small_products(method, n, o, block, bound):
    """Small and narrow products are computed in FP64 in the FP32 modes, whatever
    the planner's cost model or a timing says of them."""
    print(f"case FP64 products of FP32 sweeps {method} n={n} o={o}", flush=True)
    assert 0.0 < _error(method, n, o, 1, block) <= bound


@pytest.mark.parametrize("n,o,bound", [(80, 8, 4.037e-11)])
def test_length_of_fp32_sums(n, o, bound):
    """FP32 sums end after a bounded number of summed indices, however few K splits a level takes."""
    print(f"case FP32 sums CCSD n={n} o={o}", flush=True)
    assert 0.0 < _error("CCSD", n, o, 1, ("T2.oovv.abab", (o, o, n - o, n - o))) <= bound
