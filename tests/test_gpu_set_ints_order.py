"""New integrals uploaded right after a sweep was queued: that sweep still uses the
old ones, as with a wait in between."""

import numpy as np
import pytest

from ccq_amd import engine as E
from gpu_helpers import Case

pytestmark = pytest.mark.gpu


def test_upload_waits_for_the_sweep():
    print("case integrals uploaded behind a sweep, CCSDT n=26", flush=True)
    a, b = Case(26, 4, 52, 3), Case(26, 4, 52, 4)
    out = []
    for wait in (True, False):
        eng = E.Engine(0, a.oa, a.ob, a.n, "CCSDT", shift=0.1)
        eng.set_ints(a.fa, a.fb, a.vaa, a.vab, a.vbb)
        eng.guess("mp2")
        for _ in range(2):
            eng.update()
        if wait:
            eng.sync()
        eng.set_ints(b.fa, b.fb, b.vaa, b.vab, b.vbb)
        out.append(eng.get_t())
        eng.update()
        out.append(eng.get_t())
        eng.close()
    np.testing.assert_array_equal(out[0], out[2])
    np.testing.assert_array_equal(out[1], out[3])
