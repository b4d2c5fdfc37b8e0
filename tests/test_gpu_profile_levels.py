"""Profile 2 times the launches that an untimed sweep makes: the sweep's result is
the untimed one bit for bit, every level launch has a class, and the products
counted are those of the per-operation profile."""

import numpy as np
import pytest

from ccq_amd import engine as E
from gpu_helpers import Case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("method,n,o,ob,prec", [("CCSD", 24, 5, 4, 0), ("CCSD", 24, 5, 4, 2), ("CCSDT", 26, 4, 4, 0)])
def test_profile_of_level_launches(method, n, o, ob, prec):
    print(f"case profile of levels {method} n={n} o={o} ob={ob} precision {prec}", flush=True)
    c = Case(n, o, 2 * n, 23, occ_b=ob)
    out, flops = [], []
    for mode in (0, 2, 1):
        eng = E.Engine(0, c.oa, c.ob, c.n, method, shift=0.02)
        eng.set_ints(c.fa, c.fb, c.vaa, c.vab, c.vbb)
        eng.guess("mp2")
        eng.set_precision(prec)
        eng.profile(mode)
        eng.update()
        rep, secs = eng.profile_report(), eng.profile_report(sections=True)
        eng.profile(0)
        out.append((eng.energy(), eng.get_t()))
        flops.append(sum(v["flops"] for v in rep.values()))
        levels = [k for k in rep if k.startswith("level:sweep:")]
        if mode == 2:
            assert len(levels) > 10 and all(rep[k]["calls"] == 1 and rep[k]["ms"] > 0 for k in levels)
            assert "section:levels:sweep" in secs
            # the triples' products with a short summed range have launches of their own
            assert any(k.startswith("gemm:") for k in rep) == (method == "CCSDT")
        else:
            assert not levels and bool(rep) == (mode == 1)
        eng.close()
    assert out[0][0] == out[1][0]
    np.testing.assert_array_equal(out[0][1], out[1][1])
    assert flops[1] == pytest.approx(flops[2], rel=1e-12)
