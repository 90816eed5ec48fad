"""The thin kernel (128-row passes, one wave each), which plans that leave
most of the device idle run on: every flag, both score forms, lengths around
its 128-row passes, 16-column hand-offs, 4-step chunks and 160-column tiles,
direction bytes and tracks of every cell, one-workgroup teams, pairs computed
again by their epilogue workgroup, and the limit of its rule."""
import numpy as np
import pytest

import oracle_py as O
from anchorwave_amd import ksw2, workloads as W
from helpers import diff, random_pairs, same

pytestmark = pytest.mark.gpu

FLAGS = [0, ksw2.KSW_EZ_RIGHT, ksw2.KSW_EZ_SCORE_ONLY, ksw2.KSW_EZ_REV_CIGAR, ksw2.KSW_EZ_SEMIGLOBAL_END,
         ksw2.KSW_EZ_EXTZ_ONLY, ksw2.KSW_EZ_SEMIGLOBAL_END | ksw2.KSW_EZ_RIGHT, ksw2.KSW_EZ_SINGLETRACK]


def _edge_pairs():
    rng = np.random.default_rng(31)
    out = []
    for ql, tl in [(1, 1), (1, 2), (2, 1), (3, 127), (4, 128), (5, 129), (15, 255), (16, 256), (17, 257), (126, 130),
                   (127, 384), (128, 385), (129, 641), (130, 513), (143, 700), (144, 150), (145, 200), (257, 260),
                   (500, 1025), (1000, 1100)]:
        t = W.random_seq(rng, tl)
        q = np.concatenate([W.mutate(rng, t, 0.1, 0.02), W.random_seq(rng, ql)])[:ql] if ql > 2 else W.random_seq(rng, ql)
        out += [(q, t), (t, q)]
    return out


def _check(pairs, flag, **kw):
    got = ksw2.extd2_batch(pairs, flag=flag, **kw)
    bad = []
    for k, ((q, t), g) in enumerate(zip(pairs, got)):
        r = O.run_oracle(q, t, flag=flag, **kw)
        if not same(g, r):
            bad.append(f"pair {k} qlen={len(q)} tlen={len(t)} flag={flag:#x}: {diff(g, r)}")
    assert not bad, "\n".join(bad[:5]) + f"\n({len(bad)} of {len(pairs)} differ)"


@pytest.mark.parametrize("lut", ["1", "0"])
@pytest.mark.parametrize("flag", FLAGS)
def test_thin_edge_lengths(flag, lut, monkeypatch):
    monkeypatch.setenv("KSW2_HIP_LUT", lut)
    _check(_edge_pairs(), flag)


@pytest.mark.parametrize("how", ["KSW2_HIP_SPREAD_FALLBACK", "KSW2_HIP_WIDE_REDO"])
@pytest.mark.parametrize("flag", [0, ksw2.KSW_EZ_RIGHT, ksw2.KSW_EZ_SCORE_ONLY, ksw2.KSW_EZ_SINGLETRACK])
def test_thin_one_workgroup_and_redo(flag, how, monkeypatch):
    monkeypatch.setenv(how, "1")
    _check(random_pairs(640 + flag, 12, 1, 2600), flag)


@pytest.mark.parametrize("transpose", ["0", "1"])
@pytest.mark.parametrize("flag", [0, ksw2.KSW_EZ_RIGHT, ksw2.KSW_EZ_SINGLETRACK])
def test_thin_bytes_of_every_cell(flag, transpose, monkeypatch):
    monkeypatch.setenv("KSW2_HIP_TRANSPOSE", transpose)
    pairs = [p for p in _edge_pairs() if min(len(p[0]), len(p[1])) > 2][::3] + random_pairs(650 + flag, 3, 200, 900)
    plan = ksw2.Plan(pairs, flag=flag)
    plan.run()
    plan.fetch()
    for k, (q, t) in enumerate(pairs):
        assert plan.stored_geometry(k) == (4, transpose == "1")  # as the layout it is reported in
        _, ref = O.run_oracle(q, t, flag=flag, want_dirs=True)
        got = (plan.tracks if flag & ksw2.KSW_EZ_SINGLETRACK else plan.dirs)(k, len(q), len(t))
        nbad = int((got != ref).sum())
        assert nbad == 0, f"pair {k} qlen={len(q)} tlen={len(t)}: {nbad} cells differ"
    plan.close()


def test_thin_rule_limit():
    """96 and 97 pairs of 16 passes: the last plan on the thin kernel and the
    first past it give the same results."""
    pairs = W.fixed(seed=8, n=97)
    assert all(len(t) == 2000 for _, t in pairs)
    _check(pairs[:96], 0)
    _check(pairs, 0)


def test_thin_more_passes_than_waves():
    """A pair of more than 1,024 passes: each wave computes several."""
    rng = np.random.default_rng(33)
    t = W.random_seq(rng, 1024 * 128 + 700)
    q = np.concatenate([t[5000:5300], W.random_seq(rng, 40)])
    for flag in (ksw2.KSW_EZ_SCORE_ONLY, 0):
        _check([(q, t)], flag)
        # (a call may take a layout of the measured table; a server's flight
        # of a lone long task does not)
        server = ksw2.Server()
        server.submit(q, t, flag=flag)
        (_, got, _), = server.poll(1, -1)
        server.close()
        ref = O.run_oracle(q, t, flag=flag)
        assert same(got, ref), diff(got, ref)


def test_thin_in_server_flights():
    """A burst of long and short tasks to a server: flights on the thin kernel
    beside flights of one-workgroup teams, all as the oracle has them."""
    rng = np.random.default_rng(95)
    tasks = []
    for k, tl in enumerate([9000, 8300, 8192, 8193, 12000] + [300, 1500, 2000, 4100] * 5):
        t = W.random_seq(rng, tl)
        q = W.mutate(rng, t, 0.08, 0.02)
        tasks.append((q, t) if k % 3 else (t, q))
    flags = [FLAGS[k % len(FLAGS)] for k in range(len(tasks))]
    for count in (1, len(tasks)):  # alone, and all at once
        server = ksw2.Server()
        tickets = {server.submit(q, t, flag=f): k for k, ((q, t), f) in enumerate(zip(tasks[:count], flags))}
        seen = 0
        while seen < count:
            for ticket, got, _ in server.poll(count, -1):
                q, t = tasks[tickets[ticket]]
                ref = O.run_oracle(q, t, flag=flags[tickets[ticket]])
                assert same(got, ref), diff(got, ref)
                seen += 1
        server.close()
