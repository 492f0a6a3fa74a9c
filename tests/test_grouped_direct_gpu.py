"""Grouped contractions at the edges of the work units: tile edges, K chunks
with odd lengths and one-step remainders, paired and unpaired contracted
entries, output orders, against numpy in complex128.

Tolerance as for the single contraction: sums of at most 2 K terms in the
dtype's precision, four times sqrt(2 K) units of it on the result's norm."""
import numpy as np
import pytest

import tenet_hip as T
from tenet_hip.grouped import GroupedPlan

pytestmark = pytest.mark.gpu


def _run(ctx, specs, dt, conj=None, reps=2):
    rng = np.random.default_rng(len(specs))
    probs, hosts, dev, ptrs = [], [], [], []
    for la, lb, lc, ext in specs:
        sh = [tuple(ext[x] for x in ls) for ls in (la, lb, lc)]
        a, b = (((rng.standard_normal(s) + 1j * rng.standard_normal(s)) / np.sqrt(2)).astype(dt) for s in sh[:2])
        probs.append((sh[0], la, sh[1], lb, sh[2], lc))
        hosts.append((a, b))
        d = [T.DeviceArray.from_host(ctx, a, dt), T.DeviceArray.from_host(ctx, b, dt), T.DeviceArray(ctx, sh[2], dt)]
        dev.append(d)
        ptrs += [x.ptr for x in d]
    plan = GroupedPlan(ctx, probs, dt, conj=conj)
    first = None
    for _ in range(reps):  # the queue is ready again after every launch
        for d in dev:
            d[2].zero_()
        plan.exec(ptrs)
        got = [d[2].to_host() for d in dev]
        if first is not None:
            assert all(np.array_equal(x, y) for x, y in zip(first, got))
        first = got
    info = plan.info()
    plan.close()
    for i, ((la, lb, lc, ext), (a, b), g) in enumerate(zip(specs, hosts, first)):
        a, b = a.astype(np.complex128), b.astype(np.complex128)
        if conj:
            a, b = (x.conj() if c else x for x, c in zip((a, b), conj[i]))
        ref = np.einsum(f"{la},{lb}->{lc}", a, b, optimize=True)
        K = np.prod([ext[x] for x in la if x in lb and x not in lc], dtype=float)
        assert np.linalg.norm(g - ref) <= 4 * np.sqrt(2 * K + 2) * np.finfo(dt).eps * np.linalg.norm(ref), (la, lb, lc, ext)
    return info


@pytest.mark.parametrize("dt", [np.complex128, np.complex64])
def test_edges_and_orders(ctx, dt):
    specs = []
    orders = ["mk,kn->mn", "km,kn->mn", "mk,nk->nm", "km,nk->mn", "kml,lnk->mn", "mlk,kln->nm"]
    for i, (m, n, k) in enumerate([(1, 1, 9), (15, 17, 16), (16, 16, 17), (33, 31, 31), (64, 65, 64), (129, 63, 5),
                                   (200, 190, 33), (70, 300, 130)]):
        for o in orders:
            la, r = o.split(",")
            lb, lc = r.split("->")
            specs.append((la, lb, lc, dict(m=m, n=n, k=k, l=3)))
    conj = [(i % 2, (i // 2) % 2) for i in range(len(specs))]
    _run(ctx, specs, dt, conj)


@pytest.mark.parametrize("dt", [np.complex128, np.complex64])
@pytest.mark.parametrize("K", [4097, 5000, 8191, 30003])
def test_k_chunks(ctx, dt, K):
    """Long contracted ranges among short ones are cut into chunks (odd
    remainders included); the sums are the same on every launch."""
    specs = [("mk", "kn", "mn", dict(m=9, n=5, k=K)), ("km", "kn", "nm", dict(m=40, n=33, k=K)),
             ("mk", "nk", "mn", dict(m=70, n=66, k=K)), ("k", "k", "", dict(k=K))]
    specs += [("mk", "kn", "mn", dict(m=20, n=21, k=11))] * 20
    assert _run(ctx, specs, dt)["split_tiles"] > 0
