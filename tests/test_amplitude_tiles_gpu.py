"""Site-parallel amplitudes with requests of several states in one batch:
tiles of 1..16 rows, odd and even bonds around the tile and step edges, sites
of different length, against numpy; a request's value is the same to the bit
alone and in the batch.

Tolerance: the vectors are FP64 and each of the n steps sums at most 2 chi
products; 1e-12 is above n * sqrt(2 chi) * 1.1e-16 for every case here."""
import ctypes as C

import numpy as np
import pytest

import tenet_hip as T
from tenet_hip import _lib as L
from tenet_hip.serving import ServedState

pytestmark = pytest.mark.gpu


def _state(ctx, rng, bonds, d, dt):
    dims = [1] + list(bonds) + [1]
    host = [((rng.standard_normal((a, d, b)) + 1j * rng.standard_normal((a, d, b))) / np.sqrt(2 * d * b)).astype(dt)
            for a, b in zip(dims, dims[1:])]
    return host, ServedState(ctx, T.MPS.from_host(ctx, host, dt))


def _amplitudes(ctx, states, reqs, d, dt):
    bits = [np.asarray(b, dtype=np.uint8) for _, b in reqs]
    off = np.concatenate([[0], np.cumsum([len(b) for b in bits])]).astype(np.uint64)
    k = len(reqs)
    flat = np.concatenate(bits)
    buf = ctx.malloc(flat.nbytes + 64 + k * 56)
    p_tab = (buf + flat.nbytes + 63) // 64 * 64
    tab = np.empty((4, k), dtype=np.uint64)
    tab[0] = [states[s].n for s, _ in reqs]
    tab[1] = [states[s].site_tab for s, _ in reqs]
    tab[2] = [states[s].chi_tab for s, _ in reqs]
    tab[3] = buf + off[:-1]
    for src, dst in ((flat, buf), (tab, p_tab)):
        L.check(L.lib.tenet_memcpy_h2d(ctx.h, C.c_void_p(dst), src.ctypes.data_as(C.c_void_p), src.nbytes, None))
    n_max = max(states[s].n for s, _ in reqs)
    chi_max = max(int(states[s].chis.max()) for s, _ in reqs)
    L.check(L.lib.tenet_amplitudes_sites(ctx.h, None, L.C128 if dt == np.complex128 else L.C64, k, n_max, chi_max,
                                         C.c_void_p(p_tab), C.c_void_p(p_tab + 8 * k), C.c_void_p(p_tab + 16 * k),
                                         C.c_void_p(p_tab + 24 * k), d, C.c_void_p(p_tab + 32 * k)), "amplitudes_sites")
    h = np.zeros((k, 3))
    L.check(L.lib.tenet_memcpy_d2h(ctx.h, h.ctypes.data_as(C.c_void_p), C.c_void_p(p_tab + 32 * k), h.nbytes, None))
    ctx.free(buf)
    return h


@pytest.mark.parametrize("dt", [np.complex128, np.complex64])
@pytest.mark.parametrize("d", [2, 3])
def test_mixed_states(ctx, d, dt):
    rng = np.random.default_rng(d)
    shapes = [[2, 3, 1, 7, 8, 9], [15, 16, 17, 33], [65, 130, 64, 63, 127], [1], []]
    built = [_state(ctx, rng, s, d, dt) for s in shapes]
    hosts, states = [b[0] for b in built], [b[1] for b in built]
    reqs = []
    for s, count in enumerate([37, 9, 70, 5, 3]):
        reqs += [(s, rng.integers(0, d, states[s].n)) for _ in range(count)]
    reqs = [reqs[i] for i in rng.permutation(len(reqs))]
    h = _amplitudes(ctx, states, reqs, d, dt)
    got = (h[:, 0] + 1j * h[:, 1]) * np.exp(h[:, 2])
    for (s, b), g in zip(reqs, got):
        v = np.ones(1, dtype=np.complex128)
        for A, x in zip(hosts[s], b):
            v = v @ A[:, x, :].astype(np.complex128)
        assert abs(g - v[0]) <= 1e-12 * max(abs(v[0]), np.prod([np.linalg.norm(A) for A in hosts[s]]) * 1e-3)
    for i in (0, 1, 17, len(reqs) - 1):
        assert np.array_equal(_amplitudes(ctx, states, [reqs[i]], d, dt)[0], h[i])
    for st in states:
        st.close()
