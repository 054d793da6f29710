"""Where the SpMV reads an operator's value dictionary: u8 ids from a copy in LDS, u16 ids too where a
workgroup's lookups pay for the copy, larger dictionaries (above 63.5 KB) from global memory. Both give the
same bits, in the CSR and the SELL layout, for one vector, several, and row-interleaved ones, and match the
oracle within 1e-13. Every case prints its name before it touches the device."""

import sys

import numpy as np
import pytest

from oracle import pyoracle as po

import qed_spin_amd as qs
from qed_spin_amd import _lib
from qed_spin_amd import symmetry as sym

pytestmark = pytest.mark.gpu

XCD, UNROLL, GLOBAL_DICT, SELL = 2, 4, 16, 1024


def model(name):
    """(operator, group, n_up, dictionary sizes allowed)."""
    rng = np.random.default_rng(3)
    if name == "u8":
        N = 14
        H = qs.HamiltonianBuilder(N).heisenberg([(i, (i + 1) % N) for i in range(N)], 1.0).to_operator()
        return H, sym.chain_group(N, 3), 7, (2, 256)
    if name == "u16 real":
        N = 12
        b = qs.HamiltonianBuilder(N)
        for i in range(N):
            b.heisenberg([(i, (i + 1) % N)], float(rng.random()))
        return b.to_operator(), sym.trivial_group(N), 6, (257, 8192)
    if name == "u16 complex":
        N = 16
        b = qs.HamiltonianBuilder(N)
        for d in (1, 2, 3, 4):
            b.heisenberg([(i, (i + d) % N) for i in range(N)], float(rng.random()))
        return b.to_operator(), sym.chain_group(N, 3), 8, (257, 4096)
    N = 14   # a random field: nearly every diagonal entry is its own value
    b = qs.HamiltonianBuilder(N)
    for i in range(N):
        b.heisenberg([(i, (i + 1) % N)], float(rng.random()))
    H = b.to_operator()
    for i in range(N):
        H.add_product("z", (i,), float(rng.random()))
    return H, sym.trivial_group(N), -1, (8193, 65536)


def bits(a):
    return np.ascontiguousarray(a).view(np.uint64)


@pytest.mark.parametrize("layout", [0, SELL])
@pytest.mark.parametrize("name", ["u8", "u16 real", "u16 complex", "above 64 KB"])
def test_dictionary_in_lds_and_in_global_memory_agree(name, layout):
    print("[case] dictionary", name, layout, flush=True)
    sys.stdout.flush()
    H, g, n_up, (lo, hi) = model(name)
    s = qs.Sector(g, n_up)
    m = qs.SectorMatvec(H, s, lane=qs.LANE_CSR, tune=False)
    assert lo <= m.info["dict_size"] <= hi
    o = po.OracleSector(g.N, n_up, g.perms, g.chars)
    row_ptr, col, val = po.sector_csr(qs.Program(H).export(), o)
    rng = np.random.default_rng(5)
    for cv in ([False, True] if m.is_real else [True]):
        xs = [rng.normal(size=s.dim) + (1j * rng.normal(size=s.dim) if cv else 0.0) for _ in range(7)]
        got = {}
        for where in (0, GLOBAL_DICT):
            _lib.call("qedh_matvec_set_tuning", m.h, 0, XCD | UNROLL | layout | where)
            X = [qs.DeviceArray.from_host(x.astype(m.dtype(cv))) for x in xs]
            Y = [qs.DeviceArray(s.dim, m.dtype(cv)) for _ in xs]
            m.apply_multi(X, Y, complex_vectors=cv)
            single = m.apply_host(xs[0], complex_vectors=cv)
            B = qs.DeviceArray.from_host(np.stack(xs[:4], axis=1).astype(m.dtype(cv)).ravel())
            Z = qs.DeviceArray(4 * s.dim, m.dtype(cv))
            m.apply_block(4, B, Z, complex_vectors=cv)
            multi = np.stack([y.to_host() for y in Y], axis=1)
            block = Z.to_host().reshape(s.dim, 4)
            assert np.array_equal(bits(multi[:, 0]), bits(single))
            assert np.array_equal(bits(multi[:, :4]), bits(block))
            got[where] = multi
        assert np.array_equal(bits(got[0]), bits(got[GLOBAL_DICT]))
        for i, x in enumerate(xs):
            ref = po.csr_matvec(row_ptr, col, val, x.astype(complex))
            assert np.linalg.norm(got[0][:, i] - ref) <= 1e-13 * np.linalg.norm(ref)
