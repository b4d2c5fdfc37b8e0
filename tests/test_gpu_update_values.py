"""The values of the amplitude step (lanes of a tuple as its sizes choose): after
one sweep, t - <R>/(D + shift) on every canonical tuple, with R read back from the
residual the sweep left and <R> its signed mean over the images, in numpy."""

import numpy as np
import pytest

from oracle import solver as osolver
from ccq_amd import engine as E
from gpu_helpers import Case, antisym_random, antisymmetrize_block, canonical_mask

pytestmark = pytest.mark.gpu

# 1, 4 and 16 lanes a tuple; blocks with a single tuple and with none
RESID = {"t1a": "R1.ov.aa", "t2aa": "R2.oovv.aaaa", "t2ab": "R2.oovv.abab", "t2bb": "R2.oovv.bbbb",
         "t3aaa": "R3.ooovvv.aaaaaa", "t3aab": "R3.ooovvv.aabaab", "t3abb": "R3.ooovvv.abbabb", "t3bbb": "R3.ooovvv.bbbbbb"}


@pytest.mark.parametrize("n,o,ob", [(6, 3, 3), (9, 3, 2), (12, 4, 3), (17, 4, 4)])
def test_step_values(n, o, ob):
    print(f"case step values CCSDT n={n} o={o} ob={ob}", flush=True)
    shift = 0.3
    c = Case(n, o, 2 * n, 7, occ_b=ob)
    rng = np.random.default_rng(3)
    t = osolver.zero_amplitudes("CCSDT", c.ca, c.cb, c.va, c.vb)
    for k in t:
        t[k] = antisym_random(rng, k, c.ca, c.cb, c.va, c.vb, 0.02)
    eng = E.Engine(0, c.oa, c.ob, c.n, "CCSDT", shift=shift)
    eng.set_ints(c.fa, c.fb, c.vaa, c.vab, c.vbb)
    eng.set_t(E.join_tvec(t, c.ca, c.cb, c.va, c.vb))
    eng.update()
    new = E.split_tvec(eng.get_t(), c.ca, c.cb, c.va, c.vb)
    fd = {"a": np.diag(c.fa), "b": np.diag(c.fb)}
    occ = {"a": c.oa, "b": c.ob}
    for name, tid in RESID.items():
        spins, shape = name[2:], t[name].shape
        h = len(spins)
        if 0 in shape:
            continue
        R = antisymmetrize_block(eng.debug_read(tid, shape), name)
        D = np.full(shape, shift)
        for d in range(2 * h):
            e = fd[spins[d % h]]
            x = -e[:occ[spins[d]]] if d < h else e[occ[spins[d - h]]:]
            D = D + x.reshape([-1 if i == d else 1 for i in range(2 * h)])
        mask = canonical_mask(name, shape)
        want = (t[name] - R / D)[mask]
        if want.size:
            scale = np.abs(t[name]).max() + np.abs(R / D).max()
            assert np.abs(new[name][mask] - want).max() <= 1e-13 * scale, name
    eng.close()
