"""The correlation energy of given amplitudes at the edges of its kernel's tiles
(runs of 16 virtuals, one occupied orbital, more tiles than
blocks) against the same sums in numpy."""

import numpy as np
import pytest

from gpu_helpers import Case
from ccq_amd import engine as E

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,oa,ob", [(4, 1, 1), (19, 3, 2), (20, 4, 4), (36, 4, 3), (80, 2, 2)])
def test_energy_sums(n, oa, ob):
    print(f"case energy n={n} oa={oa} ob={ob}", flush=True)
    c = Case(n, oa, 2 * n, 5, occ_b=ob)
    rng = np.random.default_rng(n)
    eng = E.Engine(0, oa, ob, n, "CCSD")
    eng.set_ints(c.fa, c.fb, c.vaa, c.vab, c.vbb)
    va, vb = n - oa, n - ob
    shapes = [(oa, va), (ob, vb), (oa, oa, va, va), (oa, ob, va, vb), (ob, ob, vb, vb)]
    t = [rng.standard_normal(s) for s in shapes]
    vec = np.zeros(eng.t_size)
    flat = np.concatenate([x.ravel() for x in t])
    vec[:flat.size] = flat
    eng.set_t(vec)
    got = eng.energy()
    eng.close()
    a, b, aa, ab, bb = t
    terms = [c.fa[:oa, oa:] * a, c.fb[:ob, ob:] * b]
    for v, t2, x, y, o1, o2, w in ((c.vaa, aa, a, a, oa, oa, (0.25, 0.5)), (c.vab, ab, a, b, oa, ob, (1.0, 1.0)),
                                   (c.vbb, bb, b, b, ob, ob, (0.25, 0.5))):
        vv = v[o1:, o2:, :o1, :o2].transpose(2, 3, 0, 1)
        terms.append(vv * (w[0] * t2 + w[1] * np.einsum("ma,nf->mnaf", x, y)))
    want = sum(np.sum(x) for x in terms)
    # every term rounded a few times, their sum once per addition
    assert abs(got - want) <= 1e-13 * sum(np.abs(x).sum() for x in terms)
