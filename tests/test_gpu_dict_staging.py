"""When the SpMV copies an operator's u16 dictionary into LDS: a launch whose workgroups look up too little
for their copy must not be slower for it (the two placements give the same bits, so only time shows which
one ran). 5.17 million rows of 32 entries and 996 values, one vector: staged 6 to 9% slower. And each placement on either side of the rule's lines gives the other's bits.
Every case prints its name before it touches the device."""

import ctypes as C

import numpy as np
import pytest

import qed_spin_amd as qs
from qed_spin_amd import _lib
from qed_spin_amd import symmetry as sym

pytestmark = pytest.mark.gpu

XCD, UNROLL, GLOBAL_DICT = 2, 4, 16


def ring(N, k, couplings):
    b = qs.HamiltonianBuilder(N)
    for d, J in enumerate(couplings, 1):
        b.heisenberg([(i, (i + d) % N) for i in range(N)], float(J))
    return qs.SectorMatvec(b.to_operator(), qs.Sector(sym.chain_group(N, k), N // 2), lane=qs.LANE_CSR, tune=False)


def microseconds(m, vectors):
    """Device time of an apply: by the rule, and with the dictionary in global memory."""
    best = [1e9, 1e9]
    for _ in range(4):
        for i, where in enumerate((0, GLOBAL_DICT)):
            _lib.call("qedh_matvec_set_tuning", m.h, 0, XCD | UNROLL | where)
            s = C.c_double()
            _lib.call("qedh_matvec_benchmark", m.h, vectors, 0, 0, 5, 40, C.byref(s))
            best[i] = min(best[i], s.value * 1e6)
    return best


@pytest.mark.parametrize("N,couplings,vectors", [(30, (0.801, 0.236), 1), (24, (0.801, 0.236, 0.517, 0.623), 4)])
def test_no_copy_that_does_not_pay(N, couplings, vectors):
    print("[case] staging", N, vectors, flush=True)
    m = ring(N, 0, couplings)
    assert m.info["dict_size"] > 900
    here, elsewhere = microseconds(m, vectors)
    assert here < 1.04 * elsewhere, (here, elsewhere)


@pytest.mark.parametrize("N,k", [(14, 3), (16, 0), (16, 3), (20, 0), (22, 0), (22, 3)])
def test_either_placement_gives_the_same_bits(N, k):
    print("[case] staging bits", N, k, flush=True)
    m = ring(N, k, (0.801, 0.236, 0.517, 0.623))
    assert m.info["dict_size"] > 256
    for vectors in (1, 3):
        got = []
        for where in (0, GLOBAL_DICT):
            _lib.call("qedh_matvec_set_tuning", m.h, 0, XCD | UNROLL | where)
            rng = np.random.default_rng(4)
            X = [qs.DeviceArray.from_host(rng.normal(size=m.dim).astype(m.dtype(False))) for _ in range(vectors)]
            Y = [qs.DeviceArray(m.dim, m.dtype(False)) for _ in range(vectors)]
            m.apply_multi(X, Y)
            got.append([np.ascontiguousarray(y.to_host()).view(np.uint64) for y in Y])
        assert all(np.array_equal(a, b) for a, b in zip(*got))
