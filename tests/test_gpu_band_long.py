"""Banded pairs of more than 1.03 M anti-diagonals on the band kernel: its H,
held with a bias that grows with the anti-diagonal, against the oracle, with
AnchorWave's gap scores and with the largest the kernel takes."""
import numpy as np
import pytest

import oracle_py as O
from anchorwave_amd import ksw2, workloads as W
from helpers import diff, same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sc", [dict(q=8, e=2, q2=75, e2=1), dict(q=60, e=4, q2=62, e2=2)])
@pytest.mark.parametrize("flag", [0, ksw2.KSW_EZ_SCORE_ONLY])
def test_long_pair(sc, flag):
    rng = np.random.default_rng(720)
    t = W.random_seq(rng, 520_000)
    q = W.mutate(rng, t, 0.12, 0.0)
    q[250_000:250_020] = (q[250_000:250_020] + 1) % 4
    q = np.delete(q, np.arange(100_000, 100_030))
    plan = ksw2.Plan([(q, t)], w=64, flag=flag, **sc)
    plan.run()
    got, facts = plan.fetch()[0], plan.facts()
    plan.close()
    assert (facts["band_pairs"], facts["redone"]) == (1, 0)
    r = O.run_oracle(q, t, w=64, flag=flag, **sc)
    assert same(got, r), diff(got, r)


def test_buffer_of_more_than_two_billion_dwords():
    """600 letters against 540 million, of which the band reaches some 1,700:
    the buffer's clearing counts past 2^31, on two workgroups."""
    rng = np.random.default_rng(721)
    t = W.random_seq(rng, 600)
    q = np.zeros(540_000_000, dtype=np.uint8)
    head = W.mutate(rng, t, 0.1, 0.02)
    q[: len(head)] = head
    plan = ksw2.Plan([(q, t)], w=500, flag=ksw2.KSW_EZ_SCORE_ONLY)
    plan.run()
    got, facts = plan.fetch()[0], plan.facts()
    plan.close()
    assert (facts["band_pairs"], facts["waiting"], facts["redone"]) == (1, 2, 0)
    r = O.run_oracle(q[:4000], t, w=500, flag=ksw2.KSW_EZ_SCORE_ONLY)
    assert same(got, r), diff(got, r)
