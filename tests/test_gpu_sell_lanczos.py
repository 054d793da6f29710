"""The Lanczos first pass fused into the SELL apply: alpha and beta have the same bits whatever the workgroup
size, whether the value dictionary lies in LDS or in global memory, and just below, at and past the sizes
where it changes place: 16 KB (workgroups of 1024 from there) and 63.5 KB (global memory above). The diagonal
of a field that doubles from site to site takes every value from -w/2 to w/2, so the number of values is
chosen exactly; its last weight fills up to it. Rows below, at and past a partial sum's 256. Against the CSR
layout within rounding. Every case prints its name before it touches the device."""

import numpy as np
import pytest

import qed_spin_amd as qs
from qed_spin_amd import _lib
from qed_spin_amd import symmetry as sym

pytestmark = pytest.mark.gpu

XCD, UNROLL, GLOBAL_DICT, WG256, WG1024, CSR, SELL = 2, 4, 16, 32, 64, 512, 1024


def matvec(values, cplx, N=14):
    """An operator of exactly `values` distinct entries: an even number on the diagonal, one hopping amplitude
    (real) or a conjugate pair (complex)."""
    diagonal = values - (2 if cplx else 1)
    assert diagonal % 2 == 0
    weights, left = [], diagonal - 1
    while left > 0:
        w = min(2 ** len(weights), left)
        weights.append(w)
        left -= w
    H = qs.Operator(N)
    for i, w in enumerate(weights):
        H.add_product("z", (i,), float(w))
    for i in range(N):
        j = (i + 1) % N
        H.add_product("+-", (i, j), 0.3 + 0.11j if cplx else 0.3)
        H.add_product("-+", (i, j), 0.3 - 0.11j if cplx else 0.3)
    return qs.SectorMatvec(H, qs.Sector(sym.trivial_group(N), -1), lane=qs.LANE_CSR, tune=False)


def run(m, v0, flags, steps=8):
    _lib.call("qedh_matvec_set_tuning", m.h, 0, XCD | UNROLL | flags)
    a, b, _ = m.lanczos(v0, steps, reorth=0)
    return np.concatenate([a, b])


@pytest.mark.parametrize("values,cplx", [(300, True), (1022, True), (1024, True), (1026, True), (4062, True), (4064, True),
                                         (4066, True), (301, False), (2047, False), (2049, False), (8127, False),
                                         (8129, False), (8191, False)])
def test_same_bits_wherever_the_dictionary_lies(values, cplx):
    print("[case] sell lanczos", values, cplx, flush=True)
    m = matvec(values, cplx)
    assert m.info["dict_size"] == values and m.is_real != cplx
    v0 = np.random.default_rng(values).normal(size=m.dim).astype(m.dtype(False))
    got = [run(m, v0, SELL | wg | where) for wg in (WG256, 0, WG1024) for where in (0, GLOBAL_DICT)]
    assert all(np.array_equal(got[0].view(np.uint64), g.view(np.uint64)) for g in got)
    ref = run(m, v0, CSR)
    assert np.max(np.abs(got[0] - ref)) <= 1e-11 * np.max(np.abs(ref))   # eight steps from a generic start


@pytest.mark.parametrize("N,up", [(6, 3), (9, 1), (8, -1), (10, 4), (11, 4), (12, 5), (13, 6)])   # 9 to 1716 rows, 256 among them
def test_same_bits_at_every_workgroup_size(N, up):
    print("[case] sell lanczos rows", N, up, flush=True)
    H = qs.HamiltonianBuilder(N).heisenberg([(i, (i + 1) % N) for i in range(N)], 1.0).to_operator()
    m = qs.SectorMatvec(H, qs.Sector(sym.trivial_group(N), up), lane=qs.LANE_CSR, tune=False)
    v0 = np.random.default_rng(N).normal(size=m.dim)
    got = [run(m, v0, SELL | wg, 6) for wg in (WG256, 0, WG1024)]
    assert all(np.array_equal(got[0].view(np.uint64), g.view(np.uint64)) for g in got)
    ref = run(m, v0, CSR, 6)
    assert np.max(np.abs(got[0] - ref)) <= 1e-11 * np.max(np.abs(ref))
