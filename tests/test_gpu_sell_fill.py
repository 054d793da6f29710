"""The SELL copy of a CSR matrix, rows of every length modulo the groups of four, every value format (u8
ids in the column words, u16 ids, full real and complex values), with and without the diagonal
entry first: applies equal the exported CSR's rows summed in numpy, n products of one row rounding by
less than 2 n eps of their moduli's sum (n <= 20). Every case prints its name before it touches the device."""

import numpy as np
import pytest

import qed_spin_amd as qs
from qed_spin_amd import _lib
from qed_spin_amd import symmetry as sym

pytestmark = pytest.mark.gpu

XCD, UNROLL, SELL, DIAG = 2, 4, 1024, 4096


def model(name):
    rng = np.random.default_rng(7)
    N = 17 if name.startswith("full") else 12
    b = qs.HamiltonianBuilder(N)
    b.heisenberg([(i, i + 1) for i in range(0, N - 1, 5 if name.startswith("full") else 1)], 1.0)
    H = b.to_operator()
    if name in ("u16", "full real", "full complex"):
        for i in range(N):
            H.add_product("z", (i,), float(rng.random()))
    if name == "full complex":
        H.add_product("+-", (3, 9), 0.3 + 0.7j)
        H.add_product("+-", (9, 3), 0.3 - 0.7j)
    return H, sym.trivial_group(N), 6 if name.startswith("u") else -1


@pytest.mark.parametrize("diag", [0, DIAG])
@pytest.mark.parametrize("name", ["u8", "u16", "full real", "full complex"])
def test_fill(name, diag):
    print("[case] sell fill", name, diag, flush=True)
    H, g, n_up = model(name)
    s = qs.Sector(g, n_up)
    m = qs.SectorMatvec(H, s, lane=qs.LANE_CSR, tune=False)
    assert (m.info["dict_size"] == 0) == name.startswith("full")
    rp, col, val = m.export_csr()
    rows = np.repeat(np.arange(s.dim), np.diff(rp.astype(np.int64)))
    _lib.call("qedh_matvec_set_tuning", m.h, 0, XCD | UNROLL | SELL | diag)
    x = np.random.default_rng(1).normal(size=s.dim)
    if not m.is_real:
        x = x + 1j * x[::-1]
    y = m.apply_host(x)
    part = val * x[col]
    ref = np.zeros(s.dim, complex)
    size = np.zeros(s.dim)
    np.add.at(ref, rows, part)
    np.add.at(size, rows, np.abs(part))
    assert np.all(np.abs(y - ref) <= 40 * np.finfo(float).eps * size)
