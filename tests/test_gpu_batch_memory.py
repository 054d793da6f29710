"""What a batched engine takes beside its vectors, and what it does when there is no more. Its matrix is
written once, straight from the blocks' own into the row order and layout that it keeps: at one vector a
block the peak stays below 6 bytes an entry (column and 16-bit id) filled up by a quarter, and 100 bytes a
row (three vectors, a row's length, place and sort words), also where one block has more values than LDS
holds. Without room for the order or the slices (a limit set here) it keeps the states' order and the
packed matrix: Lanczos coefficients within rounding of the ordered engine's and the dense block's levels.
Every case prints its name before it touches the device."""

import ctypes as C

import numpy as np
import pytest

import qed_spin_amd as qs
from qed_spin_amd import _lib
from qed_spin_amd import symmetry as sym
from qed_spin_amd import thermal as th

pytestmark = pytest.mark.gpu

USED_HIGH = 8   # hipMemPoolAttrUsedMemHigh
USED = 7        # hipMemPoolAttrUsedMemCurrent


class Pool:
    """The device's default memory pool."""

    def __init__(self):
        self.hip = C.CDLL("libamdhip64.so")
        self.pool = C.c_void_p()
        assert self.hip.hipDeviceGetDefaultMemPool(C.byref(self.pool), 0) == 0

    def get(self, what):
        v = C.c_uint64()
        assert self.hip.hipMemPoolGetAttribute(self.pool, what, C.byref(v)) == 0
        return v.value

    def reset_high(self):
        v = C.c_uint64(0)
        assert self.hip.hipMemPoolSetAttribute(self.pool, USED_HIGH, C.byref(v)) == 0


def ring_blocks(N):
    b = qs.HamiltonianBuilder(N)
    b.heisenberg([(i, (i + 1) % N) for i in range(N)], 1.0)
    b.heisenberg([(i, (i + 2) % N) for i in range(N)], 0.37)
    return b.to_operator(), [sym.chain_group(N, k) for k in (0, 1, 2)], N // 2


def uneven_blocks(N=14):
    """One block of thousands of values (a random field), beside blocks of a few."""
    rng = np.random.default_rng(1)
    out = []
    for field in (0.0, 1.0, 0.0):
        b = qs.HamiltonianBuilder(N)
        b.heisenberg([(i, (i + 1) % N) for i in range(N)], 1.0)
        H = b.to_operator()
        if field:
            for i in range(N):
                H.add_product("z", (i,), float(rng.random()))
        out.append(qs.SectorMatvec(H, qs.Sector(sym.trivial_group(N), N // 2), lane=qs.LANE_CSR, tune=False))
    return out


def mats(N):
    H, groups, up = ring_blocks(N)
    return [qs.SectorMatvec(H, qs.Sector(g, up), lane=qs.LANE_CSR, tune=False) for g in groups]


def starts(ms, R, seed=2):
    rng = np.random.default_rng(seed)
    n = sum(m.dim for m in ms)
    return rng.normal(size=(n, R)) + 1j * rng.normal(size=(n, R))


@pytest.mark.parametrize("which", ["ring", "uneven"])
def test_peak_of_one_vector_a_block(which):
    print("[case] peak", which, flush=True)
    ms = mats(26) if which == "ring" else uneven_blocks(18)
    rows, nnz = sum(m.dim for m in ms), sum(m.info["nnz"] for m in ms)
    start = starts(ms, 1)
    pool = Pool()
    th.batch_lanczos(ms, 1, 2, start)
    _lib.call("qedh_synchronize")
    before = pool.get(USED)
    pool.reset_high()
    th.batch_lanczos(ms, 1, 2, start)
    took = pool.get(USED_HIGH) - before
    assert took <= 6 * 1.25 * nnz + 100 * rows + (16 << 20), (took / rows, nnz / rows)


@pytest.mark.parametrize("R", [1, 2, 8, 12])
def test_without_room_for_the_order(R, monkeypatch):
    print("[case] no room", R, flush=True)
    ms = mats(22) + uneven_blocks(14)   # 32,066 rows: ordered from R = 8 on, sliced at 1
    scale = max(m.op.norm_bound() for m in ms)
    start = starts(ms, R)
    a, b, steps, _ = th.batch_lanczos(ms, R, 10, start)
    monkeypatch.setenv("QED_SPIN_AMD_BATCH_EXTRA_BYTES", "1")
    a1, b1, steps1, _ = th.batch_lanczos(ms, R, 10, start)
    assert np.array_equal(steps, steps1)
    # ten steps from generic starts: rounding grows by no more than a factor of some hundred
    assert np.max(np.abs(a - a1)) <= 1e-12 * scale and np.max(np.abs(b - b1)) <= 1e-12 * scale


@pytest.mark.parametrize("R", [1, 2, 9])
def test_a_block_of_many_values_among_others(R):
    print("[case] many values", R, flush=True)
    ms = uneven_blocks(14)
    assert max(m.info["dict_size"] for m in ms) > 1024 and ms[0].info["dict_size"] < 1024
    start = starts(ms, R)
    a, b, steps, _ = th.batch_lanczos(ms, R, 6, start)
    row = 0
    for i, m in enumerate(ms):
        for s in range(R):
            v = start[row:row + m.dim, s]
            a1, b1, _ = m.lanczos(v, 6, reorth=2, complex_vectors=True)
            tol = 1e-12 * m.op.norm_bound()
            assert np.max(np.abs(a[:, i, s] - a1)) <= tol and np.max(np.abs(b[:6, i, s] - b1[1:7])) <= tol
        row += m.dim


def test_times_go_by_their_names():
    print("[case] names", flush=True)
    ms = mats(14)
    engine = th.ftlm_batched(ms, 2, 10, [1, 2, 3], np.array([1.0]))[4]
    assert engine["tune_s"] == 0.0 and 0.0 <= engine["order_s"] <= engine["pack_s"]
