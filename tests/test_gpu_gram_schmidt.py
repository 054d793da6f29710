"""The Gram-Schmidt kernels at the sizes where their split of the work changes: rows below, at and past a
block's rows and tile, 65536 (workgroups of one or four wavefronts), 2^19 (a row a thread below, rows in
strides above) and 2^20 (more rows than threads); columns below, at and past four, a launch's 256, and more. Against numpy in
double: a sum of n products of order one rounds by less than n eps, and the results are divided by
sqrt(n), hence 4 eps sqrt(n). dot_many_noalloc gives dot_many's bits. Every case prints its name before
it touches the device."""

import ctypes as C

import numpy as np
import pytest

import qed_spin_amd as qs
from qed_spin_amd import _lib

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps


def handles(vs):
    return (C.c_void_p * len(vs))(*[v.ptr.value for v in vs])


@pytest.mark.parametrize("cv", [0, 1])
@pytest.mark.parametrize("n,m", [(1, 1), (63, 3), (64, 4), (65, 5), (1023, 9), (1025, 300), (9252, 100), (65536, 8),
                                 (65537, 7), (140000, 13), ((1 << 19) - 1, 6), (1 << 19, 6), ((1 << 20) + 3, 5)])
def test_gram_schmidt_kernels(n, m, cv):
    print("[case] gram schmidt", n, m, cv, flush=True)
    rng = np.random.default_rng(n + m)
    dt = np.complex128 if cv else np.float64

    def draw(*shape):
        x = rng.normal(size=shape)
        return (x + 1j * rng.normal(size=shape) if cv else x).astype(dt) / np.sqrt(n)

    V, w, a = draw(m, n), draw(n), draw(m) * np.sqrt(n)
    dV, dw = [qs.DeviceArray.from_host(v) for v in V], qs.DeviceArray.from_host(w)
    out, again = np.zeros(m, dt), np.zeros(m, dt)
    for name, o in (("qedh_dot_many", out), ("qedh_dot_many_noalloc", again)):
        _lib.call(name, cv, handles(dV), C.c_size_t(m), dw.ptr, C.c_size_t(n), _lib.ptr(o.view(np.float64), C.c_double))
    assert np.array_equal(out.view(np.uint64), again.view(np.uint64))
    assert np.max(np.abs(out - V.conj() @ w)) <= 4 * EPS * np.sqrt(n) * 4
    _lib.call("qedh_axpy_many", cv, _lib.ptr(a.view(np.float64), C.c_double), handles(dV), C.c_size_t(m), dw.ptr,
              C.c_size_t(n))
    ref = w + a @ V
    assert np.max(np.abs(dw.to_host() - ref)) <= 8 * EPS * (m + 1) * np.max(np.abs(V)) * np.max(np.abs(a)) + 4 * EPS * np.max(np.abs(ref))
