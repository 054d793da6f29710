"""The batched engine's row order: blocks whose vectors take more than 2 MB (eight vectors at most) are
stored by breadth-first level of their matrix's graph, the others as they are. Every way a vector comes
in (from the host, placed from the device, drawn on the device, through a probe) and every result must
be what the states' order gives. Rounding alone differs (the order of a block's sums), hence the
tolerances: 1e-10 for ten unconverged Lanczos steps, 1e-9 for curves. Every case prints its name before
it touches the device."""

import sys

import numpy as np
import pytest

from oracle import pyoracle as po

import qed_spin_amd as qs
from qed_spin_amd import _lib
from qed_spin_amd import dynamics as dy
from qed_spin_amd import symmetry as sym
from qed_spin_amd import thermal as th

pytestmark = pytest.mark.gpu

STEPS = 10


def say(*a):
    print("[case]", *a, flush=True)
    sys.stdout.flush()


def chain(N, closed=True, cut=()):
    """A Heisenberg chain; cut: bonds left out (the sector falls into parts no level sweep crosses)."""
    b = qs.HamiltonianBuilder(N)
    b.heisenberg([(i, (i + 1) % N) for i in range(N if closed else N - 1) if i not in cut], 1.0)
    return b.to_operator()


def recurrence(H, N, n_up, v):
    g = sym.trivial_group(N)
    o = po.OracleSector(N, n_up, g.perms, g.chars)
    row_ptr, col, val = po.sector_csr(qs.Program(H).export(), o)
    alpha, beta = [], []
    v, p, b = v / np.linalg.norm(v), np.zeros_like(v), 0.0
    for _ in range(STEPS):
        w = po.csr_matvec(row_ptr, col, val, v) - b * p
        alpha.append(np.vdot(v, w).real)
        w = w - alpha[-1] * v
        b = np.linalg.norm(w)
        beta.append(b)
        p, v = v, w / b
    return np.array(alpha), np.array(beta)


# (R, sites and up spins of the blocks): a reordered block alone, between small ones, and at R = 1
@pytest.mark.parametrize("R,dims,closed,cut", [
    (4, [(18, 9)], True, ()),
    (8, [(10, 5), (17, 8), (9, 4), (17, 7)], False, ()),
    (11, [(17, 8), (8, 4)], False, (3, 9)),
    (1, [(20, 10), (8, 3)], True, ()),
])
def test_steps_from_host_vectors(R, dims, closed, cut):
    say("row order", R, dims)
    Hs = [chain(N, closed, cut if N > 12 else ()) for N, _ in dims]
    secs = [qs.Sector(sym.trivial_group(N), up) for N, up in dims]
    mats = [qs.SectorMatvec(H, s, lane=qs.LANE_CSR, tune=False) for H, s in zip(Hs, secs)]
    assert max(s.dim for s in secs) * min(R, 8) * 16 > 2 << 20
    rows = sum(s.dim for s in secs)
    rng = np.random.default_rng(R)
    start = rng.normal(size=(rows, R)) + 1j * rng.normal(size=(rows, R))
    a, b, _, _ = th.batch_lanczos(mats, R, STEPS, start, reorth=0)
    r0 = 0
    for q, (H, (N, up), s) in enumerate(zip(Hs, dims, secs)):
        for t in sorted({0, R - 1}):
            al, be = recurrence(H, N, up, start[r0:r0 + s.dim, t])
            assert np.max(np.abs(a[:, q, t] - al)) <= 1e-10 * np.max(np.abs(al)), (q, t)
            assert np.max(np.abs(b[:, q, t] - be)) <= 1e-10 * np.max(np.abs(be)), (q, t)
        r0 += s.dim


@pytest.mark.parametrize("samples", [3, 9])
def test_vectors_drawn_on_the_device(samples):
    say("row order: ftlm", samples)
    H = chain(18)
    m = qs.SectorMatvec(H, qs.Sector(sym.trivial_group(18), 9), lane=qs.LANE_CSR, tune=False)
    betas = 1.0 / np.linspace(0.3, 3.0, 7)
    lnZ, E, V, _, _ = th.ftlm_batched([m], samples, 60, [77], betas)
    ref = m.ftlm(samples, 60, 77, betas)   # one vector at a time, the states' order
    for got, want in zip((lnZ, E, V), ref[:3]):
        assert np.max(np.abs(got[0] - want)) <= 1e-9 * np.max(np.abs(want))


def test_vectors_placed_from_the_device():
    say("row order: continued fraction")
    N = 20
    H = chain(N)
    omega = np.linspace(0.0, 4.0, 50)
    no_space = qs.Symmetry(sz=[N // 2], translations=False)
    r = dy.dynamics(H, [dy.sz_q(N, np.pi)], omega, eta=0.2, sym=no_space, krylov=60)
    k = dy.dynamics(H, [dy.sz_q(N, np.pi)], omega, eta=0.2, sym=qs.Symmetry(sz=[N // 2]), krylov=60)
    assert np.max(np.abs(r.S[0] - k.S[0])) <= 1e-7 * np.max(k.S[0])


def test_kept_bases_and_probes(monkeypatch):
    """Five samples in one round (the source and target reordered, the probe between them) against
    one sample a round (small enough to stay as they are)."""
    say("row order: T > 0")
    N = 18
    H = chain(N)
    omega = np.linspace(0.0, 4.0, 40)
    kw = dict(eta=0.2, T=[0.7], samples=5, seed=3, krylov=30, sym=qs.Symmetry(sz=[9], translations=False))
    wide = dy.dynamics(H, [dy.sz_q(N, np.pi)], omega, **kw)
    call = _lib.call

    def small_budget(name, *args):
        if name == "qedh_ftlm_dynamics_walk":
            args = list(args)
            at = [i for i, x in enumerate(args) if type(x).__name__ == "c_ulong" and x.value == 0]
            args[at[0]] = type(args[at[0]])(16 * 31 * 48620 * 4)   # one sample's kept vectors and a little
        return call(name, *args)

    monkeypatch.setattr(_lib, "call", small_budget)
    one = dy.dynamics(H, [dy.sz_q(N, np.pi)], omega, **kw)
    assert wide.engine["waves"] == 1 and one.engine["waves"] == 5
    assert np.max(np.abs(wide.S[0] - one.S[0])) <= 1e-9 * np.max(np.abs(one.S[0]))
