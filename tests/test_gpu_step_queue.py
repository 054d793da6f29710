"""How much a Lanczos run leaves enqueued. A release waits for all that any engine stream holds, so a run
on one thread may hold up a release on another by a few of its steps, not by a batch of them; and a run
that breaks down at once does not first do a batch of steps. Times of one run against each other, the
lines well apart: with 16 steps enqueued at a time the release waits for eight or more of them, with 64 the
run that breaks down takes as long as one that does not. Every case prints its name before it touches the
device."""

import threading
import time

import numpy as np
import pytest

import qed_spin_amd as qs
from qed_spin_amd import _lib
from qed_spin_amd import symmetry as sym

pytestmark = pytest.mark.gpu


def ring(N, k, up):
    H = qs.HamiltonianBuilder(N).heisenberg([(i, (i + 1) % N) for i in range(N)], 1.0).to_operator()
    return qs.SectorMatvec(H, qs.Sector(sym.chain_group(N, k), up), lane=qs.LANE_CSR, tune=False)


def test_a_release_waits_for_a_few_steps():
    print("[case] release beside a run", flush=True)
    m = ring(30, 3, 15)
    v0 = np.random.default_rng(1).normal(size=m.dim) + 0j
    m.lanczos(v0, 8, reorth=0)
    step = m.lanczos(v0, 48, reorth=0)[2]["total_s"] / 48
    word = qs.DeviceArray.from_host(np.zeros(2))

    def release():
        s = qs.Sector(sym.chain_group(10, 0), 5)
        word.to_host()
        t = time.perf_counter()
        del s
        word.to_host()   # the releasing stream has passed the wait
        return time.perf_counter() - t

    alone = np.median([release() for _ in range(20)])   # an event for every stream that the process has made
    waits = []

    def go():
        _lib.call("qedh_thread_stream", 1)
        m.lanczos(v0, 200, reorth=0)

    run = threading.Thread(target=go)
    run.start()
    while run.is_alive() and len(waits) < 200:
        waits.append(release())
        time.sleep(0.37 * step)
    run.join()
    assert len(waits) >= 10
    assert np.median(waits) < alone + 4 * step, (np.median(waits), alone, step)


def test_a_run_that_breaks_down_at_once_is_short():
    print("[case] early breakdown", flush=True)
    b = qs.HamiltonianBuilder(24)
    for i in range(23):
        b.heisenberg([(i, i + 1)], 1.0)
    m = qs.SectorMatvec(b.to_operator(), qs.Sector(sym.trivial_group(24), 2), lane=qs.LANE_CSR, tune=False)
    ferromagnet = np.ones(m.dim)   # an eigenvector
    times = []
    for v0, tol in ((ferromagnet, 1e-9), (np.random.default_rng(2).normal(size=m.dim), 0.0)):
        best = 1.0
        for _ in range(6):
            a, _, t = m.lanczos(v0, 60, reorth=0, breakdown_tol=tol)
            best = min(best, t["total_s"])
        times.append(best)
        assert len(a) == (1 if tol else 60)
    assert times[0] < 0.5 * times[1], times


@pytest.mark.parametrize("reorth", [0, 1, 2])
def test_the_steps_between_looks_do_not_show(reorth):
    print("[case] looks", reorth, flush=True)
    m = ring(14, 3, 7)
    v0 = np.random.default_rng(3).normal(size=m.dim) + 0j
    a, b, _ = m.lanczos(v0, 160, reorth=reorth)
    for steps in (1, 15, 16, 17, 79, 80, 81, 144, 145):   # the host looks after 16, 80 and 144
        a1, b1, _ = m.lanczos(v0, steps, reorth=reorth)
        assert np.array_equal(a1, a[:steps]) and np.array_equal(b1, b[:steps + 1])
