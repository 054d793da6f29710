"""Row-interleaved vectors on the SELL layout, 16 bytes of a row per lane: 1, 2, 4 and 8 vectors, real and
complex, with one and with four partial sums, rows below, at and past a slice, in memory aligned to 8
bytes only. Bit for bit the single applies; the oracle within 1e-13. Every case prints its name before it
touches the device."""

import ctypes as C

import numpy as np
import pytest

from oracle import pyoracle as po

import qed_spin_amd as qs
from qed_spin_amd import _lib
from qed_spin_amd import symmetry as sym

pytestmark = pytest.mark.gpu

XCD, UNROLL, SELL, ONE_SUM = 2, 4, 1024, 2048


def bits(a):
    return np.ascontiguousarray(a).view(np.uint64)


@pytest.mark.parametrize("nv", [1, 2, 4, 8])
@pytest.mark.parametrize("N,n_up,momentum", [(8, 0, None), (8, 4, None), (11, 1, None), (12, 6, 0), (14, 7, 3), (12, -1, None)])
def test_interleaved_vectors(N, n_up, momentum, nv):
    print("[case] block vectors", N, n_up, momentum, nv, flush=True)
    b = qs.HamiltonianBuilder(N)
    b.heisenberg([(i, (i + 1) % N) for i in range(N)], 1.0)
    H = b.to_operator()
    g = sym.trivial_group(N) if momentum is None else sym.chain_group(N, momentum)
    s = qs.Sector(g, n_up)
    m = qs.SectorMatvec(H, s, lane=qs.LANE_CSR, tune=False)
    o = po.OracleSector(g.N, n_up, g.perms, g.chars)
    csr = po.sector_csr(qs.Program(H).export(), o)
    rng = np.random.default_rng(nv)
    for sums, cv in [(f, c) for f in (0, ONE_SUM) for c in ([False, True] if m.is_real else [True])]:
        _lib.call("qedh_matvec_set_tuning", m.h, 0, XCD | UNROLL | SELL | sums)
        dt = m.dtype(cv)
        x = rng.normal(size=(s.dim, nv)) + (1j * rng.normal(size=(s.dim, nv)) if cv else 0.0)
        x = x.astype(dt)
        words = x.ravel().view(np.float64).size
        X = qs.DeviceArray.from_host(np.concatenate([[0.0], x.ravel().view(np.float64)]))
        Y = qs.DeviceArray(words + 2, np.float64)
        Y.zero()
        at = lambda a: C.c_void_p(a.ptr.value + 8)
        _lib.call("qedh_matvec_apply_block", m.h, nv, at(X), at(Y), int(cv))
        out = Y.to_host()
        assert out[0] == 0.0 and out[-1] == 0.0
        y = np.ascontiguousarray(out[1:-1]).view(dt).reshape(s.dim, nv)
        for q in range(nv):
            assert np.array_equal(bits(y[:, q]), bits(m.apply_host(np.ascontiguousarray(x[:, q]), complex_vectors=cv)))
            ref = po.csr_matvec(*csr, x[:, q].astype(complex))
            assert np.linalg.norm(y[:, q] - ref) <= 1e-13 * np.linalg.norm(ref)
