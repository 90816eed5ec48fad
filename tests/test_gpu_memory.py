"""Calls that find no memory to keep, and what threads keep between calls."""
import pytest

import oracle_py as O
from anchorwave_amd import ksw2
from helpers import diff, random_pairs, same

pytestmark = pytest.mark.gpu


def _tuples(seed, n, hi):
    """Pairs of the thin or stripe, band and general kernels."""
    return [(q, t, *[(0, -1), (0, 60), (ksw2.KSW_EZ_SINGLETRACK, 80)][k % 3])
            for k, (q, t) in enumerate(random_pairs(seed, n, 100, hi))]


def _check(tuples):
    for (q, t, f, w), g in zip(tuples, ksw2.extd2_batch(tuples)):
        r = O.run_oracle(q, t, flag=f, w=w)
        assert same(g, r), f"qlen={len(q)} tlen={len(t)} w={w} flag={f:#x}: {diff(g, r)}"


@pytest.mark.parametrize("n", [1, 30])
def test_no_pinned_memory_to_keep(n, monkeypatch):
    """A call whose pinned buffer cannot be allocated runs without it."""
    ksw2.release_cached_memory()
    monkeypatch.setenv("KSW2_HIP_FAIL_PINNED", "1")
    for dense in (False, True):
        if dense:
            monkeypatch.setenv("KSW2_HIP_DENSE_FETCH", "1")
        _check(_tuples(750 + n, n, 900))
