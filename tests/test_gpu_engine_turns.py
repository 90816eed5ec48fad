"""Tasks of a server that arrive while two long flights hold the thin kernel's
turns: they run beside them instead of waiting for one to end."""
import time

import numpy as np
import pytest

import oracle_py as O
from anchorwave_amd import ksw2, workloads as W
from helpers import diff, same

pytestmark = pytest.mark.gpu


def test_short_tasks_pass_two_long_flights():
    rng = np.random.default_rng(740)
    t = W.random_seq(rng, 65_000)
    q = W.mutate(rng, t, 0.05, 0.001)
    # a class of sizes each, so that both find a stream: 18 and 12 ms of steps
    long = [(q, t), (q[:7600], t)]
    tasks = [(W.random_seq(rng, 300), 0, -1), (W.random_seq(rng, 400), ksw2.KSW_EZ_SINGLETRACK, 60),
             (W.random_seq(rng, 500), ksw2.KSW_EZ_RIGHT, -1)]
    tasks = [(W.mutate(rng, t, 0.1, 0.02), t, f, w) for t, f, w in tasks]
    server = ksw2.Server(device_bytes=8 << 30)

    def drain(n):
        out = []
        while len(out) < n:
            out += [(ticket, got) for ticket, got, _ in server.poll(8, -1)]
        return out

    for task in tasks:  # the kernels' first launches
        server.submit(*task[:2], flag=task[2], w=task[3])
        drain(1)
    for pair in long:
        server.submit(*pair, flag=ksw2.KSW_EZ_SCORE_ONLY)
        drain(1)
    # (three tries: a host that is held up for the flights' milliseconds
    # submits the tasks too late)
    for _ in range(3):
        for pair in long:
            server.submit(*pair, flag=ksw2.KSW_EZ_SCORE_ONLY)
            time.sleep(0.002)
        tickets = {server.submit(*task[:2], flag=task[2], w=task[3]): task for task in tasks}
        done = drain(len(long) + len(tasks))
        for ticket, got in done:
            if ticket in tickets:
                q, t, f, w = tickets[ticket]
                r = O.run_oracle(q, t, flag=f, w=w)
                assert same(got, r), diff(got, r)
        first = {ticket for ticket, _ in done[: len(tasks)]}
        if first == set(tickets):
            break
    server.close()
    assert first == set(tickets), [ticket for ticket, _ in done]
