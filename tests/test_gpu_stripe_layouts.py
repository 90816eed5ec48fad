"""Plans that leave the device idle, on the stripe kernel (KSW2_HIP_THIN=0:
the thin kernel takes them otherwise): graph replay, direction bytes and
tracks in the planner's own layout, the compare form of the scores, pairs
spread over CUs and their one-workgroup form, and lone pairs whose layout
comes from the measured table."""
import numpy as np
import pytest

import oracle_py as O
import test_gpu_parity as parity
import test_gpu_singletrack as singletrack
import test_gpu_wide as wide
from anchorwave_amd import ksw2, workloads as W
from helpers import diff, random_pairs, same

pytestmark = pytest.mark.gpu


@pytest.fixture
def stripe(monkeypatch):
    monkeypatch.setenv("KSW2_HIP_THIN", "0")
    return monkeypatch


def test_graph_switch(stripe):
    """The same plan replays its graph, and with KSW2_HIP_GRAPH=0 does not."""
    pairs = random_pairs(910, 40, 200, 1500)
    exp = [O.run_oracle(q, t) for q, t in pairs]
    for switch, replays in ((None, 2), ("0", 0)):
        if switch:
            stripe.setenv("KSW2_HIP_GRAPH", switch)
        plan = ksw2.Plan(pairs)
        for _ in range(3):
            plan.run()
            bad = [diff(g, r) for g, r in zip(plan.fetch(), exp) if not same(g, r)]
            assert not bad, bad[0]
        assert plan.graph_stats() == (3, replays)
        assert plan.facts()["stripe_pairs"] == len(pairs)
        plan.close()


def test_bytes_and_tracks_of_every_cell(stripe):
    parity.test_direction_bytes_every_cell()
    singletrack.test_singletrack_tracks_every_cell()


@pytest.mark.parametrize("flag", [0, ksw2.KSW_EZ_RIGHT, ksw2.KSW_EZ_SCORE_ONLY, ksw2.KSW_EZ_SINGLETRACK])
def test_score_forms(flag, stripe):
    parity.test_generic_score_path(flag, stripe)


def test_spread_and_concurrent_calls(stripe):
    wide.test_spread_pairs_exact_wide_or_one_workgroup(stripe)
    stripe.delenv("KSW2_HIP_SPREAD_FALLBACK")
    wide.test_concurrent_single_calls_from_threads()


@pytest.mark.parametrize("fallback", [False, True])
@pytest.mark.parametrize("shape,thin", [((5000, 5000), "0"), ((900, 4000), "1"), ((1000, 9000), "1")])
def test_spread_layouts(shape, thin, fallback, stripe):
    """A pair of the planner's own spread layout, and two of the table's, as
    laid out and on one workgroup."""
    stripe.setenv("KSW2_HIP_THIN", thin)
    if fallback:
        stripe.setenv("KSW2_HIP_SPREAD_FALLBACK", "1")
    rng = np.random.default_rng(sum(shape))
    t = W.random_seq(rng, shape[1])
    q = np.resize(W.mutate(rng, t[: shape[0] + 300], 0.08, 0.02), shape[0])
    for flag in (0, ksw2.KSW_EZ_RIGHT, ksw2.KSW_EZ_SCORE_ONLY, ksw2.KSW_EZ_SINGLETRACK):
        plan = ksw2.Plan([(q, t)], flag=flag)
        plan.run()
        g, f = plan.fetch()[0], plan.facts()
        plan.close()
        assert (f["stripe_pairs"], f["waiting"], f["one_workgroup"]) == (1, 0 if fallback else 1, 1 if fallback else 0)
        r = O.run_oracle(q, t, flag=flag)
        assert same(g, r), diff(g, r)
