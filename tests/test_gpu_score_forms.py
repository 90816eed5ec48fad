"""The stripe kernel's two score forms are kernels of their own, so a plan
that holds pairs of both launches each: codes below 4 (byte table) and the
code 4 as an ordinary symbol under KSW_EZ_GENERIC_SC (compare form) in one
batch, at swept lengths around the 64-column blocks and the first block that
runs without the start and end rules, against the oracle."""
import numpy as np
import pytest

import oracle_py as O
from anchorwave_amd import ksw2, workloads as W
from helpers import diff, same

pytestmark = pytest.mark.gpu

SWEPT = [1, 48, 63, 64, 65, 127, 128, 129, 191, 192, 193, 255, 256, 257, 320, 449]


@pytest.mark.parametrize("flag", [0, ksw2.KSW_EZ_RIGHT, ksw2.KSW_EZ_SCORE_ONLY, ksw2.KSW_EZ_SINGLETRACK])
@pytest.mark.parametrize("rows", ["4", "8"])
def test_both_score_forms_in_one_plan(flag, rows, monkeypatch):
    monkeypatch.setenv("KSW2_HIP_ROWS", rows)
    monkeypatch.setenv("KSW2_HIP_TRANSPOSE", "0")
    rng = np.random.default_rng(900 + flag)
    pairs = []
    for k, n in enumerate(SWEPT):
        t = W.random_seq(rng, int(rng.choice([n, 700, 1300])))
        q = W.mutate(rng, t, 0.08, 0.02)
        q = np.concatenate([q, W.random_seq(rng, n)])[:n]
        if k % 2:
            t = t.copy()
            t[rng.random(len(t)) < 0.03] = 4
            q[rng.random(len(q)) < 0.03] = 4
        pairs.append((q, t))
    flag |= ksw2.KSW_EZ_GENERIC_SC
    assert all(ksw2.route(q, t, flag=flag) == 0 for q, t in pairs)
    got = ksw2.extd2_batch(pairs, flag=flag)
    for k, ((q, t), g) in enumerate(zip(pairs, got)):
        r = O.run_oracle(q, t, flag=flag)
        assert same(g, r), f"pair {k} qlen={len(q)} tlen={len(t)}: {diff(g, r)}"
