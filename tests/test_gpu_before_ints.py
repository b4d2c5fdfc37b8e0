"""Calls that need the integrals before they are uploaded: each is an error, and
the context works as a fresh one afterwards, in every precision mode."""

import numpy as np
import pytest

from ccq_amd import engine as E
from gpu_helpers import Case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [0, 1, 2])
def test_errors_before_set_ints(prec):
    print(f"case calls before set_ints, precision {prec}", flush=True)
    c = Case(14, 4, 28, 7, occ_b=3)
    vec = c.tvec(c.random_t(3))
    out = []
    for early in (True, False):
        eng = E.Engine(0, c.oa, c.ob, c.n, "CCSD", shift=0.05)
        eng.set_precision(prec)
        if early:
            for call in (eng.update, eng.energy, lambda: eng.debug_sweep(-1), lambda: eng.debug_sweep(2),
                         lambda: eng.guess("mp2")):
                with pytest.raises(E.EngineError, match="integrals"):
                    call()
        eng.set_ints(c.fa, c.fb, c.vaa, c.vab, c.vbb)
        eng.set_t(vec)
        eng.update()
        out.append((eng.energy(), eng.get_t()))
        eng.close()
    assert out[0][0] == out[1][0]
    np.testing.assert_array_equal(out[0][1], out[1][1])
