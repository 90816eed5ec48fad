"""Calls that find no memory to keep, and what threads keep between calls."""
import ctypes as C
import threading

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


@pytest.mark.parametrize("n", [12, 60])
def test_no_device_block_for_a_batch(n, monkeypatch):
    """A batch whose block cannot be allocated is streamed through the memory
    there is; a single call reports it, and the thread's next calls run."""
    tuples = _tuples(760 + n, n, 900)
    ksw2.release_cached_memory()
    monkeypatch.setenv("KSW2_HIP_MEM_BUDGET", str(96 << 20))
    monkeypatch.setenv("KSW2_HIP_FAIL_BLOCK", str(1 << 20))
    _check(tuples)
    q, t, f, w = tuples[0]
    big = ksw2.extd2(*random_pairs(761, 1, 3000, 3000, 1.0)[0], check=False)
    assert big.zdropped == 1 and big.n_cigar == 0
    assert ksw2.lib().ksw2_hip_last_error() == -3  # KSW2_HIP_ENOMEM
    assert same(ksw2.extd2(q[:50], t[:50], flag=f), O.run_oracle(q[:50], t[:50], flag=f))
    monkeypatch.delenv("KSW2_HIP_FAIL_BLOCK")
    _check(tuples)


def _free_bytes():
    hip = C.CDLL("libamdhip64.so")
    free, total = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def test_threads_keep_a_bounded_sum():
    """Fourteen threads that each run a batch of some 0.9 GiB and live on: at
    most 8 GiB stays with them."""
    pairs = random_pairs(762, 1, 2000, 2000, 1.0) * 190
    ref = O.run_oracle(*pairs[0])
    ksw2.extd2_batch(pairs)
    ksw2.release_cached_memory()
    before = _free_bytes()
    ran, done = threading.Barrier(15), threading.Event()
    bad = []

    def work():
        bad.extend(k for k, g in enumerate(ksw2.extd2_batch(pairs)) if not same(g, ref))
        ran.wait()
        done.wait()

    threads = [threading.Thread(target=work) for _ in range(14)]
    for t in threads:
        t.start()
    ran.wait()
    kept = before - _free_bytes()
    done.set()
    for t in threads:
        t.join()
    assert not bad
    assert 1 << 30 < kept < (8 << 30) + (1 << 28), kept / 2**30


def test_plan_after_one_that_found_no_memory():
    """A plan of some 420 GB of direction bytes is refused, and the next one's
    launches do not report its error."""
    t = random_pairs(763, 1, 400, 400, 1.0)[0][1]
    long = t.repeat(1000)
    with pytest.raises(ksw2.KswError):
        ksw2.Plan([(long, long)] * 3)
    pairs = random_pairs(764, 20, 100, 900)
    plan = ksw2.Plan(pairs)
    plan.run()
    got = plan.fetch()
    plan.close()
    for (q, t), g in zip(pairs, got):
        r = O.run_oracle(q, t)
        assert same(g, r), diff(g, r)


def test_server_without_pinned_memory(monkeypatch):
    """A server's flights that get no pinned staging and no mirror run without."""
    monkeypatch.setenv("KSW2_HIP_FAIL_PINNED", "1")
    server = ksw2.Server(device_bytes=2 << 30)
    tasks = {server.submit(q, t, flag=f, w=w): (q, t, f, w) for q, t, f, w in _tuples(765, 40, 900)}
    left = len(tasks)
    while left:
        for ticket, got, _ in server.poll(64, -1):
            q, t, f, w = tasks[ticket]
            r = O.run_oracle(q, t, flag=f, w=w)
            assert same(got, r), diff(got, r)
            left -= 1
    server.close()
