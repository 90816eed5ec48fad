"""The band kernel's geometry: lengths around its 128-position stripes, every
phase of a width against its 16-anti-diagonal blocks, widths around the team
sizes (one workgroup whose last wave hands on to its first, several that hand
on through device memory), one to several workgroups forced, bit-exact against
the oracle (every ez field and the CIGAR)."""
import numpy as np
import pytest

import oracle_py as O
from anchorwave_amd import ksw2, workloads as W
from helpers import diff, same

pytestmark = pytest.mark.gpu

FLAGS = [0, ksw2.KSW_EZ_RIGHT, ksw2.KSW_EZ_SCORE_ONLY, 0x04]  # 0x04: KSW_EZ_GENERIC_SC


def _check(tuples):
    got = ksw2.extd2_batch(tuples)
    for (q, t, f, w), g in zip(tuples, got):
        r = O.run_oracle(q, t, flag=f, w=w)
        assert same(g, r), f"qlen={len(q)} tlen={len(t)} w={w} flag={f:#x}: {diff(g, r)}"


def _pair(rng, ql, tl):
    t = W.random_seq(rng, tl)
    q = W.mutate(rng, t, 0.1, 0.02)
    return np.resize(q, ql) if len(q) < ql else q[:ql], t


@pytest.mark.parametrize("w", [1, 2, 15, 16, 31, 46, 47, 64])
def test_lengths_around_stripes(w):
    rng = np.random.default_rng(300 + w)
    tuples = []
    for tl in (1, 2, 15, 16, 17, 63, 64, 65, 127, 128, 129, 255, 256, 257, 385, 513):
        for ql in (tl, max(1, tl - 9), tl + 13, tl + 2 * w + 5):
            q, t = _pair(rng, ql, tl)
            tuples.append((q, t, FLAGS[len(tuples) % 4], w))
    _check(tuples)


@pytest.mark.parametrize("flag", FLAGS)
def test_width_phases(flag):
    rng = np.random.default_rng(310)
    _check([(*_pair(rng, int(rng.integers(900, 1100)), 1000), flag, w) for w in range(96, 130)])


@pytest.mark.parametrize("team", [None, "1", "2", "3", "4", "8", "12"])
def test_widths_around_team_sizes(team, monkeypatch):
    if team:
        monkeypatch.setenv("KSW2_HIP_BAND_TEAM", team)
    rng = np.random.default_rng(320)
    tuples = []
    for w in (45, 46, 174, 175, 301, 302, 303, 430, 700):
        for ql, tl in ((1500, 1600), (1900, 1750)):
            tuples.append((*_pair(rng, ql, tl), FLAGS[len(tuples) % 4], w))
    _check(tuples)
    for tup in tuples[:4]:  # and alone
        _check([tup])
