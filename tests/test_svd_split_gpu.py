"""Jacobi rounds that share a pair's rows among workgroups, against LAPACK's
singular values, the product and the factors' orthonormality.

Shapes sit at the edges of the rule and of the strips: one column over a single
pair (33), ragged last strips and blocks (100 x 70, 257 x 130), three and two pairs on
an XCD (530 x 530, 768 x 300), the last row count of the one-launch rounds (768)
and the next, and a batch whose rounds are cut for some problems and not for
others.

Tolerance: each of the n = min(shape) columns takes part in at most n rotations a
sweep and about 16 sweeps, each adding a few eps of its norm: 100 n eps of FP64;
norms and products over m = max(shape) rows add at most m eps; complex64 factors
are rounded to 24 bits at the end: 8 eps of FP32 more."""
import ctypes as C

import numpy as np
import pytest

import tenet_hip as T
from tenet_hip import _lib as L
from tenet_hip.grouped import grouped_svd

pytestmark = pytest.mark.gpu


def _matrix(rng, m, n, dt):
    return (rng.standard_normal((m, n)) + 1j * rng.standard_normal((m, n))).astype(dt)


def _check(a, u, s, vh):
    n, tol = min(a.shape), (100 * min(a.shape) + max(a.shape)) * 2.0 ** -52
    if a.dtype == np.complex64:
        tol += 8 * 2.0 ** -23
    a, vh = a.astype(np.complex128), vh.astype(np.complex128)
    s0 = np.linalg.svd(a, compute_uv=False)
    assert np.abs(s - s0).max() <= tol * s0[0]
    assert np.abs(vh @ vh.conj().T - np.eye(n)).max() <= tol
    if u is not None:
        u = u.astype(np.complex128)
        assert np.abs(u.conj().T @ u - np.eye(n)).max() <= tol
        assert np.linalg.norm((u * s) @ vh - a) <= tol * np.linalg.norm(a)


@pytest.mark.parametrize("precondition", [False, True])
@pytest.mark.parametrize("m,n", [(33, 33), (100, 70), (70, 100), (257, 130), (256, 256), (768, 48), (769, 48), (530, 530), (768, 300)])
def test_one_matrix(ctx, m, n, precondition):
    a, k = _matrix(np.random.default_rng(m + n), m, n, np.complex128), min(m, n)
    A = T.DeviceArray.from_host(ctx, a)
    U, S, V = T.DeviceArray(ctx, (m, k)), T.DeviceArray(ctx, (k,)), T.DeviceArray(ctx, (k, n))
    ctx.svd_precondition(precondition)
    try:
        for _ in range(2):
            L.check(L.lib.tenet_svd_thin(ctx.h, None, 0, m, n, C.c_void_p(A.ptr), m, C.c_void_p(U.ptr), m,
                                         C.c_void_p(S.ptr), C.c_void_p(V.ptr), k, 0, 0.0, None, None))
            _check(a, U.to_host(), S.to_host().view(np.float64)[:k], V.to_host())
    finally:
        ctx.svd_precondition(True)


@pytest.mark.parametrize("dt", [np.complex128, np.complex64])
@pytest.mark.parametrize("want_u", [True, False])
def test_batch(ctx, dt, want_u):
    rng = np.random.default_rng(7)
    shapes = [(256, 250), (130, 129), (70, 300), (48, 33), (31, 31), (300, 5), (64, 64)] + [(40, 40)] * 9
    mats = [_matrix(rng, m, n, dt) for m, n in shapes]
    dev = [T.DeviceArray.from_host(ctx, a, dt) for a in mats]
    for a, (u, s, vh, k, _) in zip(mats, grouped_svd(ctx, dev, want_u=want_u)):
        assert k == min(a.shape)
        _check(a, u.to_host() if want_u else None, np.asarray(s), vh.to_host())
