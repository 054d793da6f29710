"""axpy_many adds a row's columns one after the other, whichever kernel runs it: below 2^16 rows, from there
to 2^19 and above, and with every remainder of the columns it loads together (16, then 4, then one). No
multiply-add is fused, so numpy doing the same additions in the same order gives the same bits. Every case
prints its name before it touches the device."""

import ctypes as C

import numpy as np
import pytest

import qed_spin_amd as qs
from qed_spin_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cv", [0, 1])
@pytest.mark.parametrize("n,m", [(1, 3), (64, 21), (65, 16), (65536, 7), (65537, 23), (262145, 5), ((1 << 19) - 1, 20),
                                 (1 << 19, 6)])
def test_columns_in_order(n, m, cv):
    print("[case] axpy columns", n, m, cv, flush=True)
    rng = np.random.default_rng(n + m)
    dt = np.complex128 if cv else np.float64

    def draw(*shape):
        return (rng.normal(size=shape) + (1j * rng.normal(size=shape) if cv else 0.0)).astype(dt)

    V, w, a = draw(m, n), draw(n), draw(m)
    dV, dw = [qs.DeviceArray.from_host(v) for v in V], qs.DeviceArray.from_host(w)
    _lib.call("qedh_axpy_many", cv, _lib.ptr(a.view(np.float64), C.c_double), (C.c_void_p * m)(*[v.ptr.value for v in dV]),
              C.c_size_t(m), dw.ptr, C.c_size_t(n))
    re, im = w.real.copy(), w.imag.copy()
    for c, v in zip(a, V):
        re, im = re + ((c.real * v.real - c.imag * v.imag) if cv else c * v), im + (c.real * v.imag + c.imag * v.real)
    got = dw.to_host()
    assert np.array_equal(got.real, re) and (not cv or np.array_equal(got.imag, im))
