"""Batches through a thread's kept streams, device block and pinned memory:
larger and smaller ones in turn, several kernels in one, after a release, from
several threads at once and from inside another call's progress callback, each
bit-exact against the oracle."""
import threading

import numpy as np
import pytest

import oracle_py as O
from anchorwave_amd import ksw2, workloads as W
from helpers import diff, same

pytestmark = pytest.mark.gpu


def _tuples(seed, n, tlen):
    rng = np.random.default_rng(seed)
    out = []
    for k in range(n):
        t = W.random_seq(rng, int(rng.integers(tlen // 2, tlen + 1)))
        q = W.mutate(rng, t, 0.1, 0.02)
        # stripe kernel, band kernel, score only, general kernel (Singletrack under a band)
        out.append((q, t, *[(0, -1), (0, 60), (ksw2.KSW_EZ_SCORE_ONLY, -1), (ksw2.KSW_EZ_SINGLETRACK, 80)][k % 4]))
    return out


def _bad(tuples):
    got = ksw2.extd2_batch(tuples)
    for (q, t, f, w), g in zip(tuples, got):
        r = O.run_oracle(q, t, flag=f, w=w)
        if not same(g, r):
            return f"qlen={len(q)} tlen={len(t)} w={w} flag={f:#x}: {diff(g, r)}"
    return None


def test_growing_and_shrinking_batches():
    for k, (n, tlen) in enumerate([(2, 50), (40, 700), (3, 40), (1, 900), (300, 200), (2, 2500), (5, 60)]):
        assert _bad(_tuples(400 + k, n, tlen)) is None
        if k == 3:
            ksw2.lib().ksw2_hip_release_cached_memory()


def test_threads():
    errors = []

    def work(seed):
        for k in range(4):
            b = _bad(_tuples(500 + 10 * seed + k, 3 + 9 * (k % 2), 300))
            if b:
                errors.append(b)

    threads = [threading.Thread(target=work, args=(s,)) for s in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors[0]


def test_call_from_progress_callback():
    """A call made inside another call's callback has its own resources: the
    thread's are in use."""
    inner = _tuples(600, 6, 150)
    outer = _tuples(601, 12, 1500)
    seen = []

    def callback(_args, _r, _total):
        if not seen:
            seen.append(None)
            L.ksw2_hip_clear_progress_callback()  # (the inner call polls none)
            seen[0] = _bad(inner)
            L.ksw2_hip_set_progress_callback(cb, None, 256)
        return 1

    L = ksw2.lib()
    import ctypes as C
    cb = C.CFUNCTYPE(C.c_int, C.c_void_p, C.c_int, C.c_int)(callback)
    L.ksw2_hip_set_progress_callback(cb, None, 256)
    try:
        b = _bad(outer)
    finally:
        L.ksw2_hip_clear_progress_callback()
    assert seen == [None], seen
    assert b is None, b
