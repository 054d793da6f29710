"""The batched engine's tile schedule (which workgroup runs which tile: in order, or a run of neighbouring
tiles per XCD, the default) must never show in a result: both give the same bits. Pinned here through QED_SPIN_AMD_BATCH_SCHEDULE."""

import sys

import numpy as np
import pytest

import qed_spin_amd as qs
from qed_spin_amd import dynamics as dy
from qed_spin_amd import thermal as th

pytestmark = pytest.mark.gpu


def say(*a):
    print("[case]", *a, flush=True)
    sys.stdout.flush()


def bits(a):
    return np.ascontiguousarray(a, np.float64).view(np.uint64)


def xxz(N):
    return qs.HamiltonianBuilder(N).xxz([(i, (i + 1) % N) for i in range(N)], 1.0, 0.5).to_operator()


def test_ftlm_same_under_every_schedule(monkeypatch):
    say("ftlm schedules")
    H = xxz(14)
    T = np.linspace(0.2, 3.0, 12)
    out = []
    for kind in ("0", "1"):
        monkeypatch.setenv("QED_SPIN_AMD_BATCH_SCHEDULE", kind)
        r = th.thermal(H, T, sym=qs.Symmetry(), samples=12, krylov=40, seed=5, dense_max_dim=0)
        assert int(r.engine["schedule"]) == int(kind)
        out.append(r)
    for name in ("lnZ", "E", "C"):
        assert np.array_equal(bits(getattr(out[0], name)), bits(getattr(out[1], name))), name


def test_continued_fractions_same_under_every_schedule(monkeypatch):
    say("cf schedules")
    N = 14
    b = qs.HamiltonianBuilder(N)
    b.heisenberg([(i, (i + 1) % N) for i in range(N)], 1.0)
    H = b.to_operator()
    omega = np.linspace(0.0, 3.0, 64)
    probes = [dy.sz_q(N, 2 * np.pi * m / N) for m in range(N)]
    out = []
    for kind in ("0", "1"):
        monkeypatch.setenv("QED_SPIN_AMD_BATCH_SCHEDULE", kind)
        r = dy.dynamics(H, probes, omega, eta=0.1, sym=qs.Symmetry(sz=[N // 2]), krylov=60)
        assert int(r.engine["schedule"]) == int(kind)
        out.append(r)
    assert np.array_equal(bits(np.asarray(out[0].S)), bits(np.asarray(out[1].S)))
