"""Transfer-matrix sweeps (overlap, Pauli strings) whose environments lie below,
at and above the 4096 entries where their rescaling changes from one workgroup
to two launches over many, mixed in one chain, with sites scaled so far apart
that only the running log-scale holds the result, against numpy in complex128.

Tolerance: a site is two contractions, each a sum of at most 2 K products in the
dtype's precision (relative sqrt(2 K) units), independent from site to site:
four times sqrt(2 K) sqrt(2 n) units.  The log-scale is a sum of n logarithms in
double that grows to 1400 here, so its own rounding, n + 1 spacings of doubles of
its size, adds to that where a value is put together from it."""
import numpy as np
import pytest

import tenet_hip as T
from oracle import tenet_oracle as O

pytestmark = pytest.mark.gpu

PAULI = {"I": np.eye(2), "X": np.array([[0, 1], [1, 0]]), "Y": np.array([[0, -1j], [1j, 0]]), "Z": np.diag([1, -1])}


def _sites(rng, bonds, dt, scales):
    return [(O.complex_gaussian(rng, (l, 2, r)) / np.sqrt(2 * r) * s).astype(dt)
            for l, r, s in zip(bonds, bonds[1:], scales)]


def _tol(bonds, dt):
    return 4 * np.sqrt(2 * 2 * max(bonds)) * np.sqrt(2 * len(bonds)) * np.finfo(dt).eps


@pytest.mark.parametrize("dt", [np.complex128, np.complex64])
def test_overlap(ctx, dt):
    # environments of 15, 4095, 4096, 4160, 12610, 6000, 64 and 1 entries
    ba, bb = [1, 3, 63, 64, 64, 130, 20, 64, 1], [1, 5, 65, 64, 65, 97, 300, 1, 1]
    rng = np.random.default_rng(1)
    big = 1e150 if dt == np.complex128 else 1e14
    sa = [big, 1, 1 / big, big, big, 1, big, big]
    a, b = _sites(rng, ba, dt, sa), _sites(rng, bb, dt, [1] * 8)
    A, B = T.MPS.from_host(ctx, a, dt), T.MPS.from_host(ctx, b, dt)
    ref, lg = O.overlap_mps_logscaled(O.OMPS([x.astype(np.complex128) for x in a]),
                                      O.OMPS([x.astype(np.complex128) for x in b]))
    assert lg > np.log(np.finfo(dt).max) / 2  # (a plain product would have left the type's range on its way)
    for _ in range(2):
        m, got = A.overlap(B, log=True)
        assert abs(m * np.exp(got - lg) - ref) <= (_tol(ba + bb, dt) + 9 * np.spacing(lg)) * abs(ref)
    # a state that is zero from a large environment on
    a[4] = np.zeros_like(a[4])
    m, got = T.MPS.from_host(ctx, a, dt).overlap(B, log=True)
    assert m == 0 and np.isfinite(got)


@pytest.mark.parametrize("dt", [np.complex128, np.complex64])
def test_pauli_string(ctx, dt):
    bonds = [7, 64, 65, 63, 130, 64, 66]
    rng = np.random.default_rng(2)
    inner = _sites(rng, bonds, dt, [1e3, 1e-4, 1e5, 1, 1e-3, 1e2])
    psi = T.MPS.from_host(ctx, _sites(rng, [1, 7], dt, [1]) + inner + _sites(rng, [66, 1], dt, [1]), dt,
                          form=("mixed", 1, 6))  # only the sites 1 .. 6 and the string enter
    ps = "XIZYZX"
    env = np.eye(7, dtype=np.complex128)
    for p, x in zip(ps, inner):
        x = x.astype(np.complex128)
        px = np.einsum("xi,lir->lxr", PAULI[p], x)
        env = np.tensordot(np.tensordot(env, px, axes=([0], [0])), x.conj(), axes=([0, 1], [0, 1]))
    ref, scale = np.trace(env), np.linalg.norm(env) * np.sqrt(66)
    for _ in range(2):
        assert abs(psi.expect_pauli(1, ps) - ref) <= _tol(bonds, dt) * scale
