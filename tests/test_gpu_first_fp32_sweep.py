"""The first FP32-storage sweep of a context (which allocates, zeroes and fills
the float shadows) equals a later one from the same amplitudes bit for bit, at
sizes where zeroing the shadows takes longer than the casts into them."""

import numpy as np
import pytest

from ccq_amd import engine as E
from gpu_helpers import Case, antisym_random
from oracle import solver as osolver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("method,n,o,ob", [("CCSD", 72, 9, 8), ("CCSDT", 30, 6, 5)])
def test_first_sweep_equals_a_later_one(method, n, o, ob):
    print(f"case first FP32-storage sweep {method} n={n} o={o} ob={ob}", flush=True)
    c = Case(n, o, 2 * n, 23, occ_b=ob)
    rng = np.random.default_rng(5)
    t = osolver.zero_amplitudes("CCSD", c.ca, c.cb, c.va, c.vb)
    for k in t:
        if osolver.BLOCKS[k][0] <= 2:
            t[k] = antisym_random(rng, k, c.ca, c.cb, c.va, c.vb, 0.02)
    vec = E.join_tvec(t, c.ca, c.cb, c.va, c.vb)
    eng = E.Engine(0, c.oa, c.ob, c.n, method, shift=0.02)
    eng.set_ints(c.fa, c.fb, c.vaa, c.vab, c.vbb)
    eng.set_precision(2)
    out = []
    for _ in range(2):
        eng.set_t(vec)
        eng.update()
        out.append(eng.get_t())
    eng.close()
    assert np.isfinite(out[0]).all()
    np.testing.assert_array_equal(out[0], out[1])
