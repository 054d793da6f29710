"""Where a Lanczos run ends, whatever the number of steps the device is given at a time. Two open chains of
ka and kb spins, not coupled, one spin up in each at its end: the states reached are the ka kb placings
of the two, and no rounding leads out of them (the other entries of every vector stay exactly zero), so
the run breaks down at step ka kb: at one step, in the first and the later batches of steps that are
enqueued at a time, and where max_iter ends it first. What is returned of a longer run is what a run of
that length returns. Every case prints its name before it touches the device.

The last norm is rounding, below 1e-10 ||H|| while the betas before it stay above 1e-4 ||H|| (asserted);
the Ritz values are the ka kb levels of that subspace within k ||H|| eps times the orthogonality that the
Gram-Schmidt passes keep (a few eps sqrt(n)): 1e-12 ||H||. Without reorthogonalisation the chains are
short enough (k <= 4) for the same bounds."""

import numpy as np
import pytest

import qed_spin_amd as qs
from qed_spin_amd import symmetry as sym

pytestmark = pytest.mark.gpu


def matvec(ka, kb, N=24):
    """(the block of two spins up, ||H|| bound, index of the start, the subspace's Hamiltonian)"""
    rng = np.random.default_rng(ka * 100 + kb)
    b = qs.HamiltonianBuilder(N)
    hop = {}
    for i0, k, s in ((0, ka, 1.0), (ka, kb, 1.37)):
        for i in range(i0, i0 + k - 1):
            hop[i] = s * (1.0 + 0.2 * rng.random())
            b.heisenberg([(i, i + 1)], float(hop[i]))
    H = b.to_operator()
    m = qs.SectorMatvec(H, qs.Sector(sym.trivial_group(N), 2), lane=qs.LANE_CSR, tune=False)
    places = [(i, ka + j) for i in range(ka) for j in range(kb)]
    h = np.zeros((len(places), len(places)))
    for p, (i, j) in enumerate(places):
        up = {i, j}
        for q, J in hop.items():
            h[p, p] += 0.25 * J * (1 if (q in up) == (q + 1 in up) else -1)
            if (q in up) != (q + 1 in up):
                to = tuple(sorted(up ^ {q, q + 1}))
                h[places.index(to), p] += 0.5 * J
    return m, H.norm_bound() or 1.0, h   # (no bond at all: the zero operator)


def start_of(m, N, up):
    """The unit vector of the basis state with the spins `up` up."""
    states = [sum(1 << q for q in (i, j)) for j in range(N) for i in range(j)]
    v = np.zeros(m.dim)
    v[sorted(states).index(sum(1 << q for q in up))] = 1.0
    return v


@pytest.mark.parametrize("reorth,ka,kb,extra", [(1, 1, 1, 30), (1, 2, 1, 5), (1, 7, 9, 0), (1, 7, 9, 1), (1, 8, 8, 9),
                                                (1, 5, 13, 40), (0, 1, 1, 30), (0, 2, 2, 30), (2, 2, 2, 30)])
@pytest.mark.parametrize("cv", [False, True])
def test_run_ends_at_the_invariant_subspace(cv, reorth, ka, kb, extra):
    print("[case] lanczos", cv, reorth, ka, kb, extra, flush=True)
    m, scale, h = matvec(ka, kb)
    k = ka * kb
    v0 = start_of(m, 24, (0, ka))
    a, b, t = m.lanczos(v0, k + extra, reorth=reorth, breakdown_tol=1e-10 * scale, complex_vectors=cv)
    assert len(a) == k and len(b) == k + 1 and b[0] == 0.0 and b[k] < 1e-10 * scale
    assert np.all(b[1:k] > 1e-4 * scale)
    ritz = np.linalg.eigvalsh(np.diag(a) + np.diag(b[1:k], 1) + np.diag(b[1:k], -1))
    assert np.max(np.abs(ritz - np.linalg.eigvalsh(h))) < 1e-12 * scale
    assert t["apply_s"] > 0.0 and t["total_s"] > 0.0


@pytest.mark.parametrize("reorth", [0, 1, 2])
def test_a_shorter_run_is_a_longer_ones_head(reorth):
    print("[case] lanczos head", reorth, flush=True)
    m, _, _ = matvec(12, 12)
    v0 = np.random.default_rng(2).normal(size=m.dim)
    a, b, _ = m.lanczos(v0, 150, reorth=reorth)
    assert len(a) == 150
    for steps in (1, 2, 63, 64, 65, 128):
        a1, b1, _ = m.lanczos(v0, steps, reorth=reorth)
        assert np.array_equal(a1, a[:steps]) and np.array_equal(b1, b[:steps + 1])
