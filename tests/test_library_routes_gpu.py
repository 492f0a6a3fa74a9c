"""Which plain matrix products of at least 1e8 flops run in the vendor library
and which in the direct kernel, either side of each line of the rule, and the
results of both against numpy.  A library GEMM is none of the contraction
kernels' launches.

Tolerance as for the direct kernel: sums of at most 2 K terms in the dtype's
precision, four times sqrt(2 K) units of it on the result's norm."""
import ctypes as C

import numpy as np
import pytest

import tenet_hip as T
from tenet_hip import _lib as L
from tenet_hip.device import tdesc

pytestmark = pytest.mark.gpu

Z, F = np.complex128, np.complex64


def _gauss(rng, shape, dt):
    return ((rng.standard_normal(shape) + 1j * rng.standard_normal(shape)) / np.sqrt(2)).astype(dt)


# (M, N, K, batch), A and B as stored (n) or transposed (t), library?
@pytest.mark.parametrize("dt,size,ops,library", [
    # many tiles, either type and any order, but not along a narrow edge or for a tiny K
    (Z, (1536, 2048, 33, 1), "nt", True), (Z, (1536, 2048, 31, 1), "nt", False), (F, (1536, 2048, 16, 1), "nn", True),
    (F, (1536, 1984, 50, 1), "nn", False), (F, (63, 50000, 20, 1), "nt", False), (Z, (250, 255, 40, 48), "tn", True),
    # complex128, full rounds of 5 GFLOP
    (Z, (1024, 1024, 600, 1), "tt", True), (Z, (1024, 1024, 590, 1), "tt", False),
    (Z, (1024, 1152, 600, 1), "tn", False),
    # few tiles: complex128 as stored, complex64 with A along K
    (Z, (500, 500, 500, 1), "nn", True), (Z, (500, 500, 500, 1), "tn", False), (Z, (179, 1030, 100, 1), "nn", False),
    (Z, (384, 440, 100, 1), "nn", False), (F, (640, 640, 640, 1), "tn", True), (F, (640, 640, 640, 1), "nn", False),
    (F, (448, 570, 60, 1), "tn", False), (F, (512, 512, 60, 1), "tn", True), (Z, (300, 700, 4001, 1), "nn", False),
    # batches of narrow products
    (Z, (8, 8, 8, 30000), "nn", True), (Z, (8, 9, 12, 30000), "tn", False), (Z, (30, 40, 64, 1000), "nt", True),
    (Z, (30, 40, 65, 1000), "nt", False), (Z, (40, 40, 10, 999), "nn", False), (Z, (2, 9, 20, 50000), "nn", False),
    (F, (20, 20, 24, 2000), "tn", True), (F, (20, 20, 25, 2000), "tn", False), (F, (20, 20, 24, 2000), "nn", False),
    # few tiles and a long K: never
    (Z, (128, 128, 65536, 1), "nt", False), (F, (64, 64, 20000, 1), "tn", False),
])
def test_route_and_result(ctx, dt, size, ops, library):
    M, N, K, Bt = size
    rng = np.random.default_rng(M + N + K)
    a = _gauss(rng, (M, K, Bt) if ops[0] == "n" else (K, M, Bt), dt)
    b = _gauss(rng, (K, N, Bt) if ops[1] == "n" else (N, K, Bt), dt)
    A, B, Cd = T.DeviceArray.from_host(ctx, a, dt), T.DeviceArray.from_host(ctx, b, dt), T.DeviceArray(ctx, (M, N, Bt), dt)
    da = tdesc(a.shape, [1, 2, 4] if ops[0] == "n" else [2, 1, 4])
    db = tdesc(b.shape, [2, 3, 4] if ops[1] == "n" else [3, 2, 4])
    dc = tdesc((M, N, Bt), [1, 3, 4])
    ctx.stats_enable(L.KSTAT_GEMM)
    L.check(L.lib.tenet_einsum(ctx.h, None, A.code, 0, C.byref(da), C.c_void_p(A.ptr), C.byref(db),
                               C.c_void_p(B.ptr), C.byref(dc), C.c_void_p(Cd.ptr), 0, 0), "einsum")
    launches = ctx.stats_read()["launches"]
    ctx.stats_enable(L.KSTAT_OFF)
    assert launches == (0 if library else 1)
    got = Cd.to_host()
    for z in range(Bt):
        x = (a if ops[0] == "n" else a.transpose(1, 0, 2))[..., z].astype(np.complex128)
        y = (b if ops[1] == "n" else b.transpose(1, 0, 2))[..., z].astype(np.complex128)
        ref = x @ y
        assert np.linalg.norm(got[..., z] - ref) <= 4 * np.sqrt(2 * K + 2) * np.finfo(dt).eps * np.linalg.norm(ref)


# (M, N, K), A and B as stored (n) or transposed (t), copies, a small product beside them, library?
@pytest.mark.parametrize("dt,size,ops,copies,beside,library", [
    # the only problem of its plan: as the single product
    (Z, (500, 500, 500), "nn", 1, False, True), (Z, (500, 500, 500), "tn", 1, False, False),
    (F, (512, 512, 60), "tn", 1, False, True), (F, (2000, 2000, 1000), "nn", 1, False, True),
    # a few: in the kernel, but for full rounds of 5 GFLOP in complex128 and a band of complex64
    (Z, (500, 500, 500), "nn", 1, True, False), (Z, (500, 500, 500), "nn", 7, False, False),
    (Z, (1024, 1024, 600), "tt", 1, True, True), (Z, (512, 512, 640), "nn", 4, False, True),
    (Z, (512, 576, 640), "nn", 4, False, False),
    (F, (512, 512, 60), "tn", 2, True, False), (F, (640, 640, 640), "tn", 1, True, True),
    (F, (640, 640, 640), "nn", 2, True, False), (F, (640, 640, 640), "tn", 3, False, False),
    (F, (2000, 2000, 1000), "nn", 1, True, True),
])
def test_route_of_grouped_products(ctx, dt, size, ops, copies, beside, library):
    from tenet_hip.grouped import GroupedPlan
    M, N, K = size
    rng = np.random.default_rng(M + N + K + copies)
    probs, hosts, outs, ptrs, small = [], [], [], [], 8.0 * 9 * 11 * 7
    for m, n, k, o in [(M, N, K, ops)] * copies + [(9, 11, 7, "nn")] * beside:
        a = _gauss(rng, (m, k) if o[0] == "n" else (k, m), dt)
        b = _gauss(rng, (k, n) if o[1] == "n" else (n, k), dt)
        A, B, Cd = T.DeviceArray.from_host(ctx, a, dt), T.DeviceArray.from_host(ctx, b, dt), T.DeviceArray(ctx, (m, n), dt)
        probs.append((a.shape, "mk" if o[0] == "n" else "km", b.shape, "kn" if o[1] == "n" else "nk", (m, n), "mn"))
        hosts.append((a if o[0] == "n" else a.T, b if o[1] == "n" else b.T))
        outs.append((A, B, Cd))
        ptrs += [A.ptr, B.ptr, Cd.ptr]
    plan = GroupedPlan(ctx, probs, dt)
    ctx.stats_enable(L.KSTAT_GEMM)
    plan.exec(ptrs)
    flops = ctx.stats_read()["flops"]
    ctx.stats_enable(L.KSTAT_OFF)
    got = [o[2].to_host() for o in outs]
    plan.close()
    assert flops == (0 if library else 8.0 * M * N * K * copies) + small * beside
    for (a, b), x in zip(hosts, got):
        ref = a.astype(np.complex128) @ b.astype(np.complex128)
        assert np.linalg.norm(x - ref) <= 4 * np.sqrt(2 * a.shape[1] + 2) * np.finfo(dt).eps * np.linalg.norm(ref)
