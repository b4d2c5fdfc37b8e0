"""The level launches against the operations in program order, and the storage
orders chosen for products against the declared ones, also with irrep blocks, the
active-space tuples and the CC(t;3) tail."""

import numpy as np
import pytest

from oracle import active as A
from oracle import integrals as I
from oracle import solver as osolver
from ccq_amd import engine as E
from ccq_amd import solve, synth
from gpu_helpers import Case, antisym_random

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("method,n,o,ob", [("CCSD", 24, 5, 4), ("CCSDT", 12, 3, 2), ("CCSDTQ", 8, 3, 2), ("CCSDt", 10, 3, 2)])
def test_levels_match_program_order(method, n, o, ob, monkeypatch):
    """Three sweeps of level launches agree with one launch per operation in
    program order (CCQ_HIP_GROUP=0) to 1e-11, and graph replays with eager levels
    bit for bit."""
    print(f"case levels and program order {method} n={n} o={o} ob={ob}", flush=True)
    c = Case(n, o, 2 * n, 53, occ_b=ob)
    rng = np.random.default_rng(19)
    t = osolver.zero_amplitudes("CCSDT", c.ca, c.cb, c.va, c.vb)
    for k in t:
        if method != "CCSD" or osolver.BLOCKS[k][0] <= 2:
            t[k] = antisym_random(rng, k, c.ca, c.cb, c.va, c.vb, 0.03)
    kw = dict(shift=0.03)
    vec = E.join_tvec(t, c.ca, c.cb, c.va, c.vb)
    if method == "CCSDt":
        kw.update(act_occ=1, act_unocc=2)
        act = A.ActiveSpace(0, c.oa, c.ob, c.n, 1, 2)
        for k in ("t3aaa", "t3aab", "t3abb", "t3bbb"):
            t[k][~A.p_mask(k, t[k].shape, act)] = 0.0
        vec = A.tvec(t, act, c.ca, c.cb, c.va, c.vb)
    out = []
    for group, graph in (("0", "0"), ("1", "0"), ("1", "1")):
        monkeypatch.setenv("CCQ_HIP_GROUP", group)
        monkeypatch.setenv("CCQ_HIP_GRAPH", graph)
        eng = E.Engine(0, c.oa, c.ob, c.n, method, **kw)
        eng.set_ints(c.fa, c.fb, c.vaa, c.vab, c.vbb)
        eng.set_t(vec)
        es = []
        for _ in range(3):
            eng.update()
            es.append(eng.energy())
        out.append([np.array(es), eng.get_t()] + ([eng.get_t4()] if method == "CCSDTQ" else []))
        eng.close()
    for x, y in zip(out[0], out[1]):
        assert np.abs(y - x).max() <= 1e-11 * np.abs(x).max()
    for x, y in zip(out[1], out[2]):
        np.testing.assert_array_equal(x, y)


@pytest.mark.parametrize("method,n,o,irreps,act", [("CCSD", 48, 6, True, None), ("CCSDT", 30, 4, False, None),
                                                   ("CCSDt", 32, 5, False, (2, 4)), ("CC(t;3)", 36, 5, True, (2, 4))])
def test_storage_orders(method, n, o, irreps, act, monkeypatch, capfd):
    """Sizes at which orders change: energies and amplitudes after three sweeps
    within 1e-11 of those in the declared orders (CCQ_HIP_VIEWPERM=0), and so
    the left amplitudes and the correction of CC(t;3)."""
    print(f"case storage orders {method} n={n} o={o} irreps={irreps} active={act}", flush=True)
    s = synth.make_system(n, o, 2 * n, 11, sigma=min(0.05, synth.regime_sigma(n, o, 2 * n)), d2h_irreps=irreps)
    e2 = s.e2int()
    ints = (*I.gen_fock(s.h, e2, o, o), *I.antisymmetrize(e2, 0))
    kw = dict(act_occ=act[0], act_unocc=act[1]) if act else {}
    out = []
    monkeypatch.setenv("CCQ_HIP_SCHEDULE", "1")   # prints the orders that are not the declared ones
    for perm in ("0", "1"):
        monkeypatch.setenv("CCQ_HIP_VIEWPERM", perm)
        capfd.readouterr()
        eng = E.Engine(0, o, o, n, method, shift=0.05, **kw)
        if irreps:
            eng.set_irreps(s.irreps + 1)
        eng.set_ints(*ints)
        moved = [x for x in capfd.readouterr().err.splitlines() if x.startswith("[orders]")]
        assert (len(moved) >= 10) == (perm == "1"), moved
        eng.guess("mp2")
        es = []
        for _ in range(3):
            eng.update()
            es.append(eng.energy())
        res = [np.array(es)]
        v = n - o
        res += [eng.debug_read("T2.oovv.abab", (o, o, v, v))] if method == "CCSD" else [eng.get_t()]
        if method == "CC(t;3)":
            eng.hbar()
            left = solve.solve_lcc(eng, es[-1], 0.0, 3, 5, out=None)
            res += [np.array([h[1] for h in left.history]), eng.get_l(), np.array(eng.cct3())]
        out.append(res)
        eng.close()
    for x, y in zip(*out):
        assert np.abs(y - x).max() <= 1e-11 * np.abs(x).max()
