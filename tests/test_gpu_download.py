"""Amplitude vectors read back through the runtime's copy (small) and through
the threaded pinned chunks (2 MB and more): every value that was set comes back,
into pageable and into pinned memory."""

import ctypes

import numpy as np
import pytest
import torch

from ccq_amd import engine as E

pytestmark = pytest.mark.gpu


# t vectors of 0.1 and 1.5 MB (the runtime's copy), 2.4 MB (a short second
# chunk) and 22 MB (more chunks than threads)
@pytest.mark.parametrize("n,o", [(9, 2), (15, 3), (17, 3), (26, 4)])
def test_vector_round_trip(n, o):
    print(f"case round trip CCSDT n={n} o={o}", flush=True)
    eng = E.Engine(0, o, o, n, "CCSDT")
    rng = np.random.default_rng(n)
    eng.set_ints(*(np.zeros((n,) * r) for r in (2, 2, 4, 4, 4)))
    for _ in range(2):
        vec = rng.standard_normal(eng.t_size)
        eng.set_t(vec)
        np.testing.assert_array_equal(eng.get_t(), vec)
    pinned = torch.empty(eng.t_size, dtype=torch.float64, pin_memory=True)
    assert eng.lib.ccq_hip_get_t(eng.h, ctypes.c_void_p(pinned.data_ptr()), eng.t_size) == 0
    np.testing.assert_array_equal(pinned.numpy(), vec)
    eng.close()
