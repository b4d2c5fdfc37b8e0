"""A null destination is an error of the call at every vector length (the
runtime's copy below 2 MB, the threaded read-back above it)."""

import ctypes

import numpy as np
import pytest

from ccq_amd import engine as E

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,o", [(9, 2), (26, 4)])   # t vectors of 0.1 and 22 MB
def test_null_destination_is_an_error(n, o):
    print(f"case null destination CCSDT n={n} o={o}", flush=True)
    eng = E.Engine(0, o, o, n, "CCSDT")
    vec = np.random.default_rng(n).standard_normal(eng.t_size)
    eng.set_t(vec)
    assert eng.lib.ccq_hip_get_t(eng.h, ctypes.c_void_p(None), eng.t_size) != 0
    np.testing.assert_array_equal(eng.get_t(), vec)
    eng.close()
