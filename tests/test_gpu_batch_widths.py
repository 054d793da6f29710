"""The batched engine's SpMV and recurrence for every number of vectors per block that has a kernel or
a branch of its own (R = 1, 2, 3-4, 5-7, 8 and more), on blocks whose rows end below, at and past a
tile of 256 rows and whose values sit in a dictionary in LDS, in a dictionary too large for it, or in
full: alpha and beta of the first Lanczos steps against the recurrence on the oracle's matrix. Ten
steps without reorthogonalisation amplify the rounding of a row's sum (1e-15) by less than 1e3 on these
spectra, hence 1e-11. Every case prints its name before it touches the device."""

import sys

import numpy as np
import pytest

from oracle import pyoracle as po

import qed_spin_amd as qs
from qed_spin_amd import symmetry as sym
from qed_spin_amd import thermal as th

pytestmark = pytest.mark.gpu

STEPS = 10


def ring(N, fields=(), bonds=None):
    b = qs.HamiltonianBuilder(N)
    b.heisenberg([(i, (i + 1) % N) for i in range(N)] if bonds is None else bonds, 1.0)
    H = b.to_operator()
    for i, f in enumerate(fields):
        H.add_product("z", (i,), float(f))
    return H


def blocks(values):
    """[(operator, sector, oracle sector)] with the dictionary sizes `values` asks for."""
    rng = np.random.default_rng(2)
    if values == "dictionary":   # 1, 92, 252, 462 and 792 rows: below a tile, just below, across one, three
        what = [(ring(8), sym.chain_group(8, 0), 0), (ring(12), sym.chain_group(12, 3), 5),
                (ring(10), sym.trivial_group(10), 5), (ring(11), sym.trivial_group(11), 5),
                (ring(12), sym.trivial_group(12), 5)]
    elif values == "large dictionary":   # a random field: a value per diagonal entry
        what = [(ring(11, rng.random(11)), sym.trivial_group(11), -1)]
    else:   # "full": as many values as entries
        what = [(ring(10, rng.random(10), []), sym.trivial_group(10), -1)]
    return [(H, qs.Sector(g, up), po.OracleSector(g.N, up, g.perms, g.chars)) for H, g, up in what]


@pytest.mark.parametrize("R", [1, 2, 3, 4, 5, 7, 8, 11, 16, 40])
@pytest.mark.parametrize("values", ["dictionary", "large dictionary", "full"])
def test_batched_steps_match_the_recurrence(values, R):
    print("[case] batch width", values, R, flush=True)
    sys.stdout.flush()
    bl = blocks(values)
    mats = [qs.SectorMatvec(H, s, lane=qs.LANE_CSR, tune=False) for H, s, _ in bl]
    if values == "large dictionary":
        assert mats[0].info["dict_size"] > 1024 and mats[0].info["value_bytes"] == 2
    if values == "full":
        assert mats[0].info["value_bytes"] in (8, 16)
    rows = sum(m.dim for m in mats)
    rng = np.random.default_rng(R)
    start = rng.normal(size=(rows, R)) + 1j * rng.normal(size=(rows, R))
    for reorth in (0, 2):
        a, b, steps, _ = th.batch_lanczos(mats, R, STEPS, start, reorth=reorth)
        r0 = 0
        for q, (H, s, o) in enumerate(bl):
            row_ptr, col, val = po.sector_csr(qs.Program(H).export(), o)
            M = min(STEPS, s.dim)
            for t in range(R):
                v = start[r0:r0 + s.dim, t] / np.linalg.norm(start[r0:r0 + s.dim, t])
                p = np.zeros_like(v)
                beta = 0.0
                for j in range(M):
                    w = po.csr_matvec(row_ptr, col, val, v) - beta * p
                    alpha = np.vdot(v, w).real
                    w = w - alpha * v
                    beta = np.linalg.norm(w)
                    assert abs(a[j, q, t] - alpha) <= 1e-11 * (1 + abs(alpha)), (q, t, j)
                    if beta < 1e-9:   # the block's Krylov space is full
                        break
                    assert abs(b[j, q, t] - beta) <= 1e-11 * beta, (q, t, j)
                    p, v = v, w / beta
            r0 += s.dim
