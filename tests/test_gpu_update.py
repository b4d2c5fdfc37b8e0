"""One amplitude step with the lanes of a tuple that its sizes choose: sweeps of
systems on both sides of each bound (1, 4, 16 lanes and a wave a tuple; a block
with a single tuple) repeat bit for bit and leave exactly antisymmetric blocks
(their values are compared with the oracle in the tests of each method)."""

import numpy as np
import pytest

from oracle import solver as osolver
from ccq_amd import engine as E
from gpu_helpers import Case, antisym_random

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("method,n,o,ob", [("CCSDT", 6, 3, 3), ("CCSDT", 9, 3, 2), ("CCSDT", 12, 4, 3),
                                           ("CCSDTQ", 8, 4, 4)])
def test_step_is_antisymmetric_and_repeats(method, n, o, ob):
    print(f"case step {method} n={n} o={o} ob={ob}", flush=True)
    c = Case(n, o, 2 * n, 7, occ_b=ob)
    rng = np.random.default_rng(3)
    t = osolver.zero_amplitudes("CCSDT", c.ca, c.cb, c.va, c.vb)
    for k in t:
        t[k] = antisym_random(rng, k, c.ca, c.cb, c.va, c.vb, 0.02)
    vec = E.join_tvec(t, c.ca, c.cb, c.va, c.vb)
    out = []
    for _ in range(2):
        eng = E.Engine(0, c.oa, c.ob, c.n, method, shift=0.02)
        eng.set_ints(c.fa, c.fb, c.vaa, c.vab, c.vbb)
        eng.set_t(vec)
        eng.update()
        out.append(eng.get_t())
        if method == "CCSDTQ":
            out[-1] = np.concatenate([out[-1], eng.get_t4()])
        eng.close()
    np.testing.assert_array_equal(out[0], out[1])
    assert np.isfinite(out[0]).all() and not np.array_equal(out[0][:vec.size], vec)
    # every image of a tuple (distinct indices) holds the same value
    t3 = E.split_tvec(out[0][:vec.size], c.ca, c.cb, c.va, c.vb)["t3aaa"]
    i, j, k, x, y, z = np.indices(t3.shape)
    tuples = (i != j) & (j != k) & (i != k) & (x != y) & (y != z) & (x != z)
    for p, s in (((1, 0, 2, 3, 4, 5), -1), ((0, 2, 1, 3, 4, 5), -1), ((0, 1, 2, 4, 3, 5), -1), ((1, 2, 0, 3, 4, 5), 1)):
        np.testing.assert_array_equal(t3.transpose(p)[tuples], s * t3[tuples])
