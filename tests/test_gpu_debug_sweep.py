"""A whole sweep through ccq_hip_debug_sweep(-1) as the first call of a context
(the level tables are built by whichever sweep comes first)."""

import numpy as np
import pytest

from gpu_helpers import Case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [0, 1, 2])
def test_whole_debug_sweep_is_an_update(prec):
    print(f"case whole debug sweep, precision {prec}", flush=True)
    c = Case(12, 3, 24, 7, occ_b=2)
    vec = c.tvec(c.random_t(3))
    out = []
    for call in (lambda e: e.debug_sweep(-1), lambda e: e.update()):
        eng = c.engine(shift=0.05)
        eng.set_t(vec)
        eng.set_precision(prec)
        call(eng)
        out.append(eng.get_t())
        eng.close()
    assert not np.array_equal(out[0], vec)
    np.testing.assert_array_equal(out[0], out[1])
