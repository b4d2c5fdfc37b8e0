"""The measuring autotuner at a size where a sweep has products with a launch of
their own, the ones whose plan it chooses: FP64 sweeps agree with the model's
plans to 1e-11, FP32-storage sweeps with and without FP32-storage plans to FP32
rounding."""

import numpy as np
import pytest

from ccq_amd import engine as E
from gpu_helpers import Case

pytestmark = pytest.mark.gpu


def test_tuned_own_launches(monkeypatch):
    n, o = 26, 4
    print(f"case tuned own launches CCSDT n={n} o={o}", flush=True)
    c = Case(n, o, 2 * n, 67)
    out = {}
    for tune, tune32, prec in (("0", "0", 0), ("1", "0", 0), ("1", "0", 2), ("1", "1", 2)):
        monkeypatch.setenv("CCQ_HIP_TUNE", tune)
        monkeypatch.setenv("CCQ_HIP_TUNE32", tune32)
        eng = E.Engine(0, c.oa, c.ob, c.n, "CCSDT", shift=0.02)
        eng.set_ints(c.fa, c.fb, c.vaa, c.vab, c.vbb)
        eng.guess("mp2")
        eng.set_precision(prec)
        eng.profile(2)
        eng.update()
        own = [k for k in eng.profile_report() if k.startswith("gemm:")]
        eng.profile(0)
        eng.update()
        out[tune, tune32, prec] = eng.get_t()
        eng.close()
        print("  own launches: " + ", ".join(own), flush=True)
        assert own or tune == "1"   # (a tuned plan may join its level)
    ref = out["0", "0", 0]
    scale = np.abs(ref).max()
    assert np.abs(out["1", "0", 0] - ref).max() <= 1e-11 * scale
    assert np.abs(out["1", "1", 2] - out["1", "0", 2]).max() <= 1e-6 * scale
    assert 0 < np.abs(out["1", "1", 2] - ref).max() <= 1e-6 * scale
