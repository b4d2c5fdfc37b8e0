"""ccq_hip_set_ints that ran out of device memory can be called again once there
is some: the sweeps are those of a fresh context."""

import numpy as np
import pytest
import torch

from ccq_amd import engine as E
from gpu_helpers import Case, leave_free

pytestmark = pytest.mark.gpu


def test_set_ints_after_out_of_memory():
    print("case set_ints again after it ran out of memory, CCSD n=72", flush=True)
    c = Case(72, 9, 144, 23, occ_b=8)

    def engine():
        return E.Engine(0, c.oa, c.ob, c.n, "CCSD", shift=0.02)

    eng = engine()
    # set_ints needs about 1 GB here; a quarter of it is left
    block = leave_free(256 << 20)
    with pytest.raises(E.EngineError, match="memory"):
        eng.set_ints(c.fa, c.fb, c.vaa, c.vab, c.vbb)
    del block
    torch.cuda.empty_cache()
    out = []
    for e in (eng, engine()):
        e.set_ints(c.fa, c.fb, c.vaa, c.vab, c.vbb)
        e.guess("mp2")
        energies = []
        for _ in range(2):
            e.update()
            energies.append(e.energy())
        out.append((energies, e.debug_read("T2.oovv.abab", (c.oa, c.ob, c.va, c.vb))))
        e.close()
    assert out[0][0] == out[1][0]
    np.testing.assert_array_equal(out[0][1], out[1][1])
