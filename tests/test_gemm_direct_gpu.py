"""The direct contraction kernel at the edges of its tiles and K groups, for
every operand order, both types, conjugations, batch labels and alpha / beta,
against numpy in complex128.

Tolerance: the products are exact to one rounding and summed in the dtype's
own precision in chains of at most 2 K terms, so the relative error of the
result's norm stays below about sqrt(2 K) units of that precision for
Gaussian entries; four times that is allowed."""
import ctypes as C

import numpy as np
import pytest

import tenet_hip as T
from tenet_hip import _lib as L
from tenet_hip.device import tdesc

pytestmark = pytest.mark.gpu


def _gauss(rng, shape, dt):
    return ((rng.standard_normal(shape) + 1j * rng.standard_normal(shape)) / np.sqrt(2)).astype(dt)


def _tol(K, dt):
    return 4.0 * np.sqrt(2.0 * K + 2.0) * np.finfo(dt).eps


def _check(got, ref, K, dt):
    assert np.linalg.norm(got - ref) <= _tol(K, dt) * np.linalg.norm(ref)


# (M, N, K): one element, edges of the 16 / 32 / 64 / 128 wide tiles, K remainders
# of the 4-, 8- and 32-wide groups, few and many tiles, a short K over many rows
SIZES = [(1, 1, 1), (1, 3, 9), (15, 17, 3), (16, 16, 4), (17, 33, 5), (31, 64, 16), (33, 129, 17), (65, 63, 31),
         (128, 20, 20), (40000, 20, 20), (40000, 11, 9), (300, 260, 127), (257, 500, 128), (513, 511, 130),
         (1000, 700, 33), (2049, 300, 131)]


@pytest.mark.parametrize("dt", [np.complex128, np.complex64])
@pytest.mark.parametrize("order", ["mk,kn->mn", "km,kn->mn", "mk,nk->mn", "mk,kn->nm", "km,nk->nm"])
@pytest.mark.parametrize("size", SIZES)
def test_plain_orders(ctx, size, order, dt):
    M, N, K = size
    ext = {"m": M, "n": N, "k": K}
    la, rest = order.split(",")
    lb, lc = rest.split("->")
    rng = np.random.default_rng(M * 7 + N * 3 + K)
    a, b = _gauss(rng, [ext[x] for x in la], dt), _gauss(rng, [ext[x] for x in lb], dt)
    for ca, cb in ((0, 0), (1, 0), (0, 1), (1, 1)):
        got = T.binary_einsum(T.Tensor.from_host(ctx, a, la), T.Tensor.from_host(ctx, b, lb), conj_a=ca, conj_b=cb,
                              out_labels=list(lc)).to_host()
        A, B = (a.conj() if ca else a).astype(np.complex128), (b.conj() if cb else b).astype(np.complex128)
        A, B = (A if la == "mk" else A.T), (B if lb == "kn" else B.T)
        ref = A @ B
        _check(got, ref if lc == "mn" else ref.T, K, dt)


@pytest.mark.parametrize("dt", [np.complex128, np.complex64])
@pytest.mark.parametrize("spec,ext", [
    ("bqov,boB->Bvq", dict(b=37, q=29, o=3, v=5, B=41)),     # split K and row classes, output permuted
    ("wlxk,wxpr->krlp", dict(w=5, l=33, x=2, k=70, p=7, r=3)),
    ("axbyc,dyxe->cdaeb", dict(a=4, x=9, b=3, y=6, c=11, d=5, e=2)),
    ("zab,zbc->zac", dict(z=9, a=18, b=21, c=35)),           # batch label, fastest
    ("abz,bcz->acz", dict(z=5, a=33, b=13, c=17)),           # batch label, slowest
    ("z,zab->zab", dict(z=70, a=3, b=31)),                   # Hadamard scaling
    ("abc,->cba", dict(a=19, b=2, c=23)),                    # permutation
    ("ab,ab->", dict(a=33, b=65)),                           # full contraction
    ("a,b->ba", dict(a=31, b=77)),                           # outer product
])
def test_gathered_orders(ctx, spec, ext, dt):
    la, rest = spec.split(",")
    lb, lc = rest.split("->")
    rng = np.random.default_rng(len(spec))
    a, b = _gauss(rng, [ext[x] for x in la], dt), _gauss(rng, [ext[x] for x in lb], dt)
    shared = [x for x in la if x in lb]
    dims = [x for x in shared if x not in lc]
    for cb in (0, 1):
        got = T.binary_einsum(T.Tensor.from_host(ctx, a, la), T.Tensor.from_host(ctx, b, lb), dims=dims, conj_b=cb,
                              out_labels=list(lc)).to_host()
        B = (b.conj() if cb else b).astype(np.complex128)
        ref = np.einsum(spec, a.astype(np.complex128), B, optimize=True)
        _check(got, ref, int(np.prod([ext[x] for x in dims], dtype=np.int64)), dt)


@pytest.mark.parametrize("dt", [np.complex128, np.complex64])
@pytest.mark.parametrize("size", [(5, 1, 3), (20, 70, 40), (200, 90, 150), (3, 2, 0)])
def test_alpha_beta_strided(ctx, size, dt):
    """alpha A B + beta C with padded column strides on all three operands."""
    M, N, K = size
    rng = np.random.default_rng(M)
    a, b, c = _gauss(rng, (M + 3, max(K, 1)), dt), _gauss(rng, (K + 2, N), dt), _gauss(rng, (M + 1, N), dt)
    A, B, Cd = (T.DeviceArray.from_host(ctx, x, dt) for x in (a, b, c))
    da, db, dc = tdesc((M, K), [1, 2], [1, M + 3]), tdesc((K, N), [2, 3], [1, K + 2]), tdesc((M, N), [1, 3], [1, M + 1])
    h = C.c_void_p()
    L.check(L.lib.tenet_einsum_plan(ctx.h, A.code, 0, C.byref(da), C.byref(db), C.byref(dc), C.byref(h)), "plan")
    al, be = 0.75 - 0.5j, -0.25 + 1.5j
    L.check(L.lib.tenet_einsum_exec(h, None, C.c_void_p(A.ptr), C.c_void_p(B.ptr), C.c_void_p(Cd.ptr), 0, 0,
                                    (C.c_double * 2)(al.real, al.imag), (C.c_double * 2)(be.real, be.imag)), "exec")
    got = Cd.to_host()
    L.lib.tenet_plan_destroy(h)
    a, b, c = (x.astype(np.complex128) for x in (a, b, c))
    ref = c.copy()
    ref[:M] = al * (a[:M, :K] @ b[:K]) + be * c[:M]
    _check(got, ref, K, dt)
    assert np.array_equal(got[M:], c[M:].astype(dt))
