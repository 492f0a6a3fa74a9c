"""Blocked QR of one matrix at the edges of its panels, row blocks and row
classes (16, 64, 128, 256, 512 rows and beyond), wide and tall, both types and
every operand option, against LAPACK's factors (the same Householder signs).

Tolerance: the factors' errors grow like a small multiple of sqrt(k) units of
FP64 times the condition of a Gaussian matrix (below 1e3 for every shape):
1e-12 in complex128; in complex64 the result is rounded to 24 bits: 1e-6."""
import ctypes as C

import numpy as np
import pytest

import tenet_hip as T
from tenet_hip import _lib as L

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt,tol", [(np.complex128, 1e-12), (np.complex64, 1e-6)])
@pytest.mark.parametrize("m,n", [(65, 1), (1, 65), (66, 16), (80, 17), (65, 65), (129, 31), (130, 100), (257, 48),
                                 (100, 300), (272, 33), (273, 250), (511, 70), (513, 40), (528, 33), (1000, 20),
                                 (1024, 129), (300, 530)])
def test_factors(ctx, m, n, dt, tol):
    rng = np.random.default_rng(m * 1000 + n)
    a = ((rng.standard_normal((m, n)) + 1j * rng.standard_normal((m, n))) / np.sqrt(2)).astype(dt)
    k = min(m, n)
    q0, r0 = np.linalg.qr(a.astype(np.complex128))
    A, Ah = T.DeviceArray.from_host(ctx, a, dt), T.DeviceArray.from_host(ctx, a.conj().T, dt)
    for flags in (0, 1, 2 | 4, 1 | 2 | 4):
        Q = T.DeviceArray(ctx, (k, m) if flags & 2 else (m, k), dt)
        R = T.DeviceArray(ctx, (n, k) if flags & 4 else (k, n), dt)
        src = Ah if flags & 1 else A
        L.check(L.lib.tenet_qr_thin_ex(ctx.h, None, A.code, flags, m, n, C.c_void_p(src.ptr), src.shape[0],
                                       C.c_void_p(Q.ptr), Q.shape[0], C.c_void_p(R.ptr), R.shape[0]), "qr")
        q, r = Q.to_host().astype(np.complex128), R.to_host().astype(np.complex128)
        q, r = (q.conj().T if flags & 2 else q), (r.conj().T if flags & 4 else r)
        assert np.linalg.norm(q.conj().T @ q - np.eye(k)) <= tol * np.sqrt(k)
        assert np.linalg.norm(q @ r - a) <= tol * np.linalg.norm(a)
        assert np.linalg.norm(r - r0) <= tol * np.linalg.norm(r0)
        assert np.linalg.norm(np.tril(r, -1)) == 0
    if m == 80:  # rank deficient: exact zero columns and a repeated one
        a[:, 3] = 0
        a[:, 9] = a[:, 8]
        q, r = T.tensor_qr_thin(T.Tensor.from_host(ctx, a, "mn", dt), ["m"], ["n"], "v")
        q, r = q.to_host().astype(np.complex128), r.to_host().astype(np.complex128)
        assert np.linalg.norm(q.conj().T @ q - np.eye(k)) <= tol * np.sqrt(k)
        assert np.linalg.norm(q @ r - a) <= tol * np.linalg.norm(a)


@pytest.mark.parametrize("dt,tol", [(np.complex128, 1e-12), (np.complex64, 1e-6)])
@pytest.mark.parametrize("m,n", [(768, 256), (769, 5), (769, 256), (769, 257), (1024, 240), (600, 527), (600, 529),
                                 (640, 1000), (1024, 1)])
def test_above_512_rows(ctx, m, n, dt, tol):
    """Either side of the lines between the row chunks and the 16-wave
    workgroups: 768 rows and 256 columns for Q, 32 column blocks right of a
    panel for its update."""
    test_factors(ctx, m, n, dt, tol)
