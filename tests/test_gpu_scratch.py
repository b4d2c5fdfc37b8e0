"""Level launches without partial accumulators and split-K partials (chosen where
device memory is short; CCQ_HIP_SCRATCH_MB=0 asks for it): less memory, the same
sweeps to 1e-11, in FP32 storage to FP32 rounding."""

import numpy as np
import pytest
import torch

from ccq_amd import engine as E
from gpu_helpers import Case, antisym_random, leave_free
from oracle import solver as osolver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("method,n,o,ob,prec", [("CCSD", 24, 5, 4, 0), ("CCSD", 64, 8, 8, 0), ("CCSDT", 16, 4, 3, 0),
                                                ("CCSDTQ", 8, 3, 2, 0), ("CCSDT", 16, 4, 3, 2)])
def test_sweeps_without_scratch(method, n, o, ob, prec, monkeypatch):
    print(f"case without scratch {method} n={n} o={o} ob={ob} precision {prec}", flush=True)
    c = Case(n, o, 2 * n, 61, occ_b=ob)
    rng = np.random.default_rng(3)
    t = osolver.zero_amplitudes("CCSDT", c.ca, c.cb, c.va, c.vb) if method != "CCSD" else c.random_t(3, 0.02)
    if method != "CCSD":
        for k in t:
            t[k] = antisym_random(rng, k, c.ca, c.cb, c.va, c.vb, 0.02)
    vec = E.join_tvec(t, c.ca, c.cb, c.va, c.vb)
    out = []
    for mb in ("0", "100000"):
        monkeypatch.setenv("CCQ_HIP_SCRATCH_MB", mb)
        eng = E.Engine(0, c.oa, c.ob, c.n, method, shift=0.05)
        eng.set_ints(c.fa, c.fb, c.vaa, c.vab, c.vbb)
        eng.set_t(vec)
        eng.set_precision(prec)
        for _ in range(3):
            eng.update()
        out.append(eng.get_t4() if method == "CCSDTQ" else eng.get_t())
        eng.close()
    assert not np.array_equal(out[0], out[1])
    assert np.abs(out[0] - out[1]).max() <= (1e-11 if prec == 0 else 1e-6) * np.abs(out[1]).max()


def test_scratch_gives_way_to_the_rest(monkeypatch):
    """A bound that the scratch does not fit leaves it out, and with memory for the
    system but hardly for the scratch beside it set_ints works (the runtime may free
    memory of its own meanwhile, so either schedule may be the one)."""
    print("case scratch with little memory left, CCSDTQ n=12", flush=True)
    c = Case(12, 3, 24, 7)
    out, used = [], []
    for mb, short in (("100000", False), ("8", False), (None, True)):
        if mb is None:
            monkeypatch.delenv("CCQ_HIP_SCRATCH_MB")
        else:
            monkeypatch.setenv("CCQ_HIP_SCRATCH_MB", mb)
        eng = E.Engine(0, c.oa, c.ob, c.n, "CCSDTQ", shift=0.05)
        free = torch.cuda.mem_get_info()[0]
        block = leave_free(300 << 20) if short else None
        eng.set_ints(c.fa, c.fb, c.vaa, c.vab, c.vbb)
        if not short:
            used.append(free - torch.cuda.mem_get_info()[0])
        eng.guess("mp2")
        for _ in range(2):
            eng.update()
        out.append(eng.get_t())
        eng.close()
        del block
        torch.cuda.empty_cache()
    assert used[1] + (16 << 20) < used[0]
    assert not np.array_equal(out[0], out[1])
    assert any(np.array_equal(out[2], x) for x in out[:2])
