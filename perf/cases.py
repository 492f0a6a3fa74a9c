"""Performance cases: the calls that programs built on tenet_hip spend their
time in, at sizes taken from the benchmark, the tests and the ranges those
draw from.

A case is a dict of plain values; ``kind`` names the path:

  site    one small contraction of a bond matrix (or of singular values) with
          an MPS site: what every canonize / evolve step is made of
  env     one left-environment update of DMRG (three contractions, the last
          one conjugated and with permuted labels)
  heff    the two-site effective Hamiltonian on a state (DMRG's inner loop),
          in the native precision or with split operands
  norm    canonize_ to the first site, overlap with itself and norm
  gate    one gate of a gate-by-gate TEBD sweep: the centre moves one site
          (QR), then the fused update with its truncated SVD
  vidal   a whole Vidal-gauge TEBD sweep from |0...0> and the amplitudes of
          the final state
  svds    a batch of unlike truncated SVDs, singular values absorbed into
          V^H and the factors multiplied (the truncated matrices)
  batch   a planned batch of unlike pairwise contractions
  amps    amplitudes of a batch of bitstrings
  pauli   expectation values of Pauli strings near the orthogonality centre

Outputs are free of the arbitrary phases of singular vectors: factors that
carry them come back multiplied together.
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tenet.jl_amd"))

import tenet_hip as T  # noqa: E402
from tenet_hip.dmrg import heff_apply  # noqa: E402
from tenet_hip.grouped import GroupedPlan, grouped_svd  # noqa: E402
from tenet_hip.tebd import upload_gates  # noqa: E402
from tenet_hip.vidal import brickwork_layers, tebd_vidal_sweep  # noqa: E402

NP = {"c128": np.complex128, "c64": np.complex64}
TORCH = {"c128": torch.complex128, "c64": torch.complex64}
PREC = {"native": 0, "fp32": 1, "split_bf16": 2, "split_fp16": 3, "split_i8": 4, "split_i8_fast": 5}
THRESHOLD = 1e-10


def listed():
    return [
        # the smallest call: a bond matrix into a site, launch and host cost only
        {"name": "site_chi24", "kind": "site", "dtype": "c128", "chi": 24, "chir": 19, "d": 2, "absorb": False},
        # environment of a ragged bond in single precision (gathered operands)
        {"name": "env_chi250_c64", "kind": "env", "dtype": "c64", "chi": 250, "chir": 231, "w": 5},
        # the DMRG inner loop at an ordinary large bond, double precision
        {"name": "heff_chi768", "kind": "heff", "dtype": "c128", "chi": 768, "prec": "native"},
        # the same with operands split into int8 slices (FP64-grade results)
        {"name": "heff_chi512_i8", "kind": "heff", "dtype": "c128", "chi": 512, "prec": "split_i8"},
        # the benchmark's plain workload: a 20-site chain of bond 32, latency
        {"name": "norm_n20_chi32", "kind": "norm", "dtype": "c128", "n": 20, "chi": 32},
        # canonical form, overlap and norm of a longer chain of ordinary bond
        {"name": "norm_n40_chi160", "kind": "norm", "dtype": "c128", "n": 40, "chi": 160},
        # one gate-by-gate TEBD step at an ordinary bond
        {"name": "gate_chi128", "kind": "gate", "dtype": "c128", "chi": 128, "prec": "native"},
        # the benchmark's headline: the 630-gate Vidal sweep, the largest case
        {"name": "vidal_n64_chi256", "kind": "vidal", "dtype": "c128", "n": 64, "chi": 256, "depth": 20},
        # part of the benchmark's batch of truncated SVDs, sides 16..512
        {"name": "svds_256_c64", "kind": "svds", "dtype": "c64", "count": 256, "shapes": 5, "hi": 512},
        # part of the benchmark's batch of contractions, rank 3..5
        {"name": "batch_1024_c64", "kind": "batch", "dtype": "c64", "count": 1024, "shapes": 3},
        # a served state asked for a batch of amplitudes
        {"name": "amps_n96_chi400_c64", "kind": "amps", "dtype": "c64", "n": 96, "chi": 400, "count": 128},
        # energy terms of a served state
        {"name": "pauli_chi300_c64", "kind": "pauli", "dtype": "c64", "chi": 300, "count": 12, "weight": 2},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["site", "env", "heff", "norm", "gate", "vidal", "svds", "batch", "amps", "pauli"])
    c = {"kind": kind, "dtype": rng.choice(["c128", "c64"])}
    if kind == "site":
        c |= {"chi": _log_int(rng, 4, 96), "chir": _log_int(rng, 4, 96), "d": rng.randint(2, 4),
              "absorb": rng.random() < 0.3}
    elif kind == "env":
        c |= {"chi": _log_int(rng, 16, 512), "w": rng.randint(3, 8)}
        c["chir"] = max(16, min(512, int(c["chi"] * rng.uniform(0.6, 1.6))))
    elif kind == "heff":
        c |= {"chi": _log_int(rng, 32, 1024), "prec": "native"}
        if c["dtype"] == "c128":
            c["prec"] = rng.choice(["native", "split_i8", "split_i8_fast", "split_bf16", "split_fp16"])
    elif kind == "norm":
        c |= {"n": _log_int(rng, 8, 60), "chi": _log_int(rng, 4, 200), "dtype": "c128"}
    elif kind == "gate":
        c |= {"chi": _log_int(rng, 8, 256), "prec": "native"}
        if c["dtype"] == "c128":
            c["prec"] = rng.choice(["native", "native", "split_bf16"])
    elif kind == "vidal":
        c |= {"n": rng.randint(12, 64), "chi": _log_int(rng, 16, 256), "depth": rng.randint(6, 20), "dtype": "c128"}
    elif kind == "svds":
        c |= {"count": _log_int(rng, 16, 256), "shapes": rng.randrange(1 << 20), "hi": _log_int(rng, 48, 512)}
    elif kind == "batch":
        c |= {"count": _log_int(rng, 32, 1024), "shapes": rng.randrange(1 << 20)}
    elif kind == "amps":
        c |= {"n": _log_int(rng, 16, 128), "chi": _log_int(rng, 16, 512), "count": _log_int(rng, 1, 512)}
    else:
        c |= {"chi": _log_int(rng, 16, 512), "count": rng.randint(4, 16), "weight": rng.randint(1, 4)}
    return c


# ---- inputs ------------------------------------------------------------------
_CTX = []


def _ctx():
    """A program keeps one context for its device."""
    if not _CTX:
        _CTX.append(T.Context(0))
    return _CTX[0]


class _Span:
    """A DeviceArray as torch sees it (column-major, no copy)."""

    def __init__(self, d):
        self.d = d
        st, acc = [], d.dtype.itemsize
        for s in d.shape:
            st.append(acc)
            acc *= s
        self.__cuda_array_interface__ = {"shape": d.shape, "typestr": d.dtype.str, "data": (d.ptr, False),
                                         "strides": tuple(st), "version": 2}


def _out(d):
    return torch.as_tensor(_Span(d), device="cuda")


def _dev(t):
    """A DeviceArray holding the values of a CUDA tensor."""
    a = T.DeviceArray(_ctx(), tuple(t.shape), np.complex128 if t.dtype == torch.complex128 else np.complex64)
    _out(a).copy_(t)
    return a


class _Gauss:
    def __init__(self, case, seed):
        self.dt = TORCH[case["dtype"]]
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(int(seed))

    def __call__(self, *shape):
        """Standard complex Gaussian entries."""
        return torch.randn(shape, dtype=torch.complex128, device="cuda", generator=self.g).to(self.dt)

    def iso(self, m, n):
        """A random m x n isometry (m >= n)."""
        z = torch.randn((m, n), dtype=torch.complex128, device="cuda", generator=self.g)
        return torch.linalg.qr(z)[0].to(self.dt)


def _xxz(dt):
    """Bulk tensor W[l, r, o, i] of the XXZ chain (J = 1, Delta = 0.5)."""
    sp = np.array([[0.0, 1.0], [0.0, 0.0]])
    sz = 0.5 * np.array([[1.0, 0.0], [0.0, -1.0]])
    W = np.zeros((5, 5, 2, 2))
    W[0, 0], W[4, 4] = np.eye(2), np.eye(2)
    W[1, 0], W[2, 0], W[3, 0] = sp, sp.T, sz
    W[4, 1], W[4, 2], W[4, 3] = 0.5 * sp.T, 0.5 * sp, 0.5 * sz
    return torch.from_numpy(W).to(dt).cuda()


def _haar(rng):
    z = (rng.standard_normal((4, 4)) + 1j * rng.standard_normal((4, 4))) / math.sqrt(2)
    q, r = np.linalg.qr(z)
    return q * (np.diag(r) / np.abs(np.diag(r)))


def _contractions(case):
    """Shapes of the batch: ranks 3..5, 1..3 shared labels, extents
    log-uniform in 2..128, every tensor at most 2^20 elements."""
    rng = np.random.default_rng(case["shapes"])
    got = []
    while len(got) < case["count"]:
        ra, rb = int(rng.integers(3, 6)), int(rng.integers(3, 6))
        s = min(int(rng.integers(1, 4)), ra, rb)
        sh = "xyz"[:s]
        la, lb = "abcde"[:ra - s] + sh, sh + "fghij"[:rb - s]
        la = "".join(la[i] for i in rng.permutation(ra))
        lb = "".join(lb[i] for i in rng.permutation(rb))
        ext = {x: int(round(math.exp(rng.uniform(math.log(2), math.log(128))))) for x in sorted(set(la + lb))}
        lc = "".join(x for x in la if x not in sh) + "".join(x for x in lb if x not in sh)
        shp = [tuple(ext[x] for x in ls) for ls in (la, lb, lc)]
        if max(math.prod(x) for x in shp) <= 1 << 20:
            got.append((la, lb, lc, shp))
    return got


def _sides(case):
    rng = np.random.default_rng(case["shapes"])
    lim = (math.log(16), math.log(case["hi"]))
    return [tuple(int(round(math.exp(rng.uniform(*lim)))) for _ in "mn") for _ in range(case["count"])]


def _bonds(n, chi):
    return [1] + [min(chi, 2 ** min(b, n - b, 30)) for b in range(1, n)] + [1]


def _inputs(case, seed):
    """The case's numbers as CUDA tensors and host arrays, from the seed alone."""
    g, kind = _Gauss(case, seed), case["kind"]
    rng = np.random.default_rng(seed)
    if kind == "site":
        x, r, d = case["chi"], case["chir"], case["d"]
        first = torch.exp(-torch.arange(x, device="cuda") / x).to(g.dt) * (1 + rng.random()) if case["absorb"] else g(x, x)
        return {"E": first, "A": g(x, d, r)}
    if kind == "env":
        x, r, w = case["chi"], case["chir"], case["w"]
        return {"L": g(x, w, x) / x, "A": g(x, 2, r) / math.sqrt(x), "W": g(w, 2, 2, w)}
    if kind == "heff":
        x = case["chi"]
        return {"L": g(x, 5, x) / x, "R": g(x, 5, x) / x, "W": _xxz(g.dt), "theta": g(x, 2, 2, x) / (2 * x)}
    if kind == "norm":
        n, x = case["n"], case["chi"]
        dims = [1] + [x] * (n - 1) + [1]
        return {"sites": [g(dims[i], 2, dims[i + 1]) / math.sqrt(2 * dims[i + 1]) for i in range(n)]}
    if kind == "gate":
        # three sites of a chain: the centre (a decaying Schmidt spectrum), then two right isometries
        x = case["chi"]
        lam = torch.exp(-torch.arange(x, device="cuda", dtype=torch.float64) * (9.0 / x)).to(g.dt)
        lam = lam / torch.linalg.norm(lam)
        right = [g.iso(2 * x, x).T.reshape(x, 2, x).contiguous() for _ in range(2)]
        return {"sites": [(g.iso(2 * x, x) * lam).reshape(x, 2, x)] + right, "gate": _haar(rng)}
    if kind == "vidal":
        layers = brickwork_layers(case["n"], case["depth"])
        gates = np.stack([_haar(rng) for la in layers for _ in la])
        return {"gates": gates, "bits": rng.integers(0, 2, (256, case["n"])).astype(np.uint8)}
    if kind == "svds":
        return {"flat": g(sum(m * n for m, n in _sides(case)))}
    if kind == "batch":
        sp = _contractions(case)
        return {"A": g(sum(math.prod(s[3][0]) for s in sp)), "B": g(sum(math.prod(s[3][1]) for s in sp))}
    if kind == "amps":
        dims = _bonds(case["n"], case["chi"])
        sites = [g(dims[i], 2, dims[i + 1]) / math.sqrt(2 * dims[i + 1]) for i in range(case["n"])]
        return {"sites": sites, "bits": rng.integers(0, 2, (case["count"], case["n"])).astype(np.uint8)}
    # pauli: left isometries, the centre, right isometries
    n, c, w = _pauli_chain(case)
    dims = _bonds(n, case["chi"])
    sites = []
    for i in range(n):
        a, b = dims[i], dims[i + 1]
        if i < c:
            sites.append(g.iso(2 * a, b).reshape(a, 2, b))
        elif i == c:
            z = g(a, 2, b)
            sites.append(z / torch.linalg.norm(z))
        else:
            sites.append(g.iso(2 * b, a).T.reshape(a, 2, b))
    terms = [(c + int(rng.integers(0, 4)), "".join(rng.choice(list("XYZ"), w))) for _ in range(case["count"])]
    return {"sites": sites, "terms": terms}


def _pauli_chain(case):
    half = max(4, math.ceil(math.log2(case["chi"])))
    return 2 * half + 8, half, case["weight"]


def prepare(case, seed):
    ctx, kind, dt = _ctx(), case["kind"], NP[case["dtype"]]
    x = _inputs(case, seed)
    st = {"case": case}
    if kind == "site":
        st["E"] = T.Tensor(_dev(x["E"]), ["l"] if case["absorb"] else ["x", "l"])
        st["A"] = T.Tensor(_dev(x["A"]), ["l", "s", "r"])
    elif kind == "env":
        st["L"] = T.Tensor(_dev(x["L"]), ["b", "w", "k"])
        A = _dev(x["A"])
        st["A"], st["Ac"] = T.Tensor(A, ["k", "p", "k2"]), T.Tensor(A, ["b", "o", "b2"])
        st["W"] = T.Tensor(_dev(x["W"]), ["w", "o", "p", "w2"])
    elif kind == "heff":
        W = _dev(x["W"])
        st["L"], st["R"] = T.Tensor(_dev(x["L"]), ["l", "w", "lk"]), T.Tensor(_dev(x["R"]), ["r", "wr", "rk"])
        st["W1"], st["W2"] = T.Tensor(W, ["w", "m", "o1", "i1"]), T.Tensor(W, ["m", "wr", "o2", "i2"])
        st["theta"] = T.Tensor(_dev(x["theta"]), ["lk", "i1", "i2", "rk"])
    elif kind in ("norm", "gate", "pauli"):
        st["sites"] = [_dev(s) for s in x["sites"]]
        if kind == "gate":
            G = np.asfortranarray(x["gate"].reshape(2, 2, 2, 2))
            st["gate"] = T.DeviceArray.from_host(ctx, G, dt)
        st["terms"] = x.get("terms")
    elif kind == "vidal":
        st["layers"] = brickwork_layers(case["n"], case["depth"])
        st["gates"], st["bits"] = upload_gates(ctx, x["gates"]), x["bits"]
    elif kind == "svds":
        sides = _sides(case)
        arena, lows, es = _dev(x["flat"]), [], np.dtype(dt).itemsize
        st["mats"], off = [], 0
        for m, n in sides:
            st["mats"].append(T.DeviceArray(ctx, (m, n), dt, ptr=arena.ptr + off * es, owner=False))
            off += m * n
        st["low"] = T.DeviceArray(ctx, (off,), dt)
        ks = [(min(m, n) + 1) // 2 for m, n in sides]
        st["scaled"] = T.DeviceArray(ctx, (sum(k * n for k, (_, n) in zip(ks, sides)),), dt)
        # the kept counts of generic matrices are known: the plans are made once
        st["absorb"] = GroupedPlan(ctx, [((k,), "k", (k, n), "kn", (k, n), "kn", None, (1, min(m, n)))
                                         for k, (m, n) in zip(ks, sides)], dt)
        st["join"] = GroupedPlan(ctx, [((m, k), "mk", (k, n), "kn", (m, n), "mn") for k, (m, n) in zip(ks, sides)], dt)
        st["arena"], st["sides"], st["ks"] = arena, sides, ks
    elif kind == "batch":
        sp, es = _contractions(case), np.dtype(dt).itemsize
        st["A"], st["B"] = _dev(x["A"]), _dev(x["B"])
        st["C"] = T.DeviceArray(ctx, (sum(math.prod(s[3][2]) for s in sp),), dt)
        st["plan"] = GroupedPlan(ctx, [(s[3][0], s[0], s[3][1], s[1], s[3][2], s[2]) for s in sp], dt)
        at, st["ptrs"] = [st["A"].ptr, st["B"].ptr, st["C"].ptr], []
        for s in sp:
            st["ptrs"] += at
            at = [p + math.prod(e) * es for p, e in zip(at, s[3])]
    else:
        st["psi"] = T.MPS(ctx, [_dev(s) for s in x["sites"]], dtype=dt)
        st["bits"] = x["bits"]
    torch.cuda.synchronize()
    return st


# ---- one pass ------------------------------------------------------------------
def run(st):
    ctx, case = _ctx(), st["case"]
    kind, dt = case["kind"], NP[case["dtype"]]
    if kind == "site":
        return _out(T.binary_einsum(st["E"], st["A"], dims=[] if case["absorb"] else None).data)
    if kind == "env":
        t1 = T.binary_einsum(st["L"], st["A"], out_labels=["b", "w", "p", "k2"])
        t2 = T.binary_einsum(t1, st["W"], out_labels=["b", "k2", "o", "w2"])
        return _out(T.binary_einsum(t2, st["Ac"], conj_b=True, out_labels=["b2", "w2", "k2"]).data)
    if kind == "heff":
        return _out(heff_apply(st["L"], st["W1"], st["W2"], st["R"], st["theta"], prec=PREC[case["prec"]]).data)
    if kind == "norm":
        p = T.MPS(ctx, list(st["sites"]), dtype=dt)
        p.canonize_(0)
        return {"sites": [_out(s) for s in p.sites], "overlap": np.complex128(p.overlap(p)), "norm": p.norm()}
    if kind == "gate":
        p = T.MPS(ctx, list(st["sites"]), form=("mixed", 0, 0), dtype=dt)
        k = p.simple_update_(st["gate"], 1, maxdim=case["chi"], threshold=THRESHOLD, prec=PREC[case["prec"]])
        left = T.binary_einsum(T.Tensor(p.sites[0], "lpa"), T.Tensor(p.sites[1], "aqb"))
        return {"k": k, "block": _out(T.binary_einsum(left, T.Tensor(p.sites[2], "bsr")).data)}
    if kind == "vidal":
        v = tebd_vidal_sweep(ctx, case["n"], st["layers"], st["gates"], case["chi"], THRESHOLD)
        return {"amps": v.to_mps().amplitudes(st["bits"]), "bonds": np.array(v.bondsizes()),
                "lambdas": np.concatenate(v.lam_host)}
    if kind == "svds":
        sides, ks, es = st["sides"], st["ks"], np.dtype(dt).itemsize
        got = grouped_svd(ctx, st["mats"], maxdims=ks, threshold=THRESHOLD)
        s = T.DeviceArray.from_host(ctx, np.concatenate([g[1][:k] for g, k in zip(got, ks)]), dt)
        first, second, a, b, c = [], [], s.ptr, st["scaled"].ptr, st["low"].ptr
        for (U, _, Vh, _, _), k, (m, n) in zip(got, ks, sides):
            first += [a, Vh.ptr, b]
            second += [U.ptr, b, c]
            a, b, c = a + k * es, b + k * n * es, c + m * n * es
        st["absorb"].exec(first)
        st["join"].exec(second)
        return {"low": _out(st["low"]), "s": np.concatenate([g[1] for g in got]),
                "k": np.array([g[3] for g in got]), "discarded": np.array([g[4] for g in got])}
    if kind == "batch":
        st["plan"].exec(st["ptrs"])
        return _out(st["C"])
    if kind == "amps":
        return st["psi"].amplitudes(st["bits"])
    c = _pauli_chain(case)[1]
    p = T.MPS(ctx, list(st["sites"]), form=("mixed", c, c), dtype=dt)
    return np.array([p.expect_pauli(a, s) for a, s in st["terms"]], dtype=dt)


# ---- work ------------------------------------------------------------------------
def _qr(m, n):
    p, q = max(m, n), min(m, n)
    return 4.0 * (4.0 * p * q * q - 4.0 * q ** 3 / 3.0)


def _svd(m, n):
    p, q = max(m, n), min(m, n)
    return 4.0 * (4.0 * p * p * q + 8.0 * p * q * q + 9.0 * q ** 3)


def work(case):
    """Complex multiply-add = 8 flops; thin QR and SVD by the usual counts."""
    kind, es = case["kind"], 16 if case["dtype"] == "c128" else 8
    x = case.get("chi", 0)
    if kind == "site":
        r, d = case["chir"], case["d"]
        el = x * d * r * 2 + (x if case["absorb"] else x * x)
        return {"bytes": el * es, "flops": 8.0 * x * d * r * (1 if case["absorb"] else x)}
    if kind == "env":
        r, w = case["chir"], case["w"]
        el = x * w * x + x * 2 * r + 4 * w * w + r * w * r
        return {"bytes": el * es, "flops": 8.0 * (x * w * x * 2 * r + x * r * 4 * w * w + r * w * r * x * 2)}
    if kind == "heff":
        el = 2 * 5 * x * x + 2 * 4 * x * x
        return {"bytes": el * es, "flops": 8.0 * (2 * 20 * x ** 3 + 400 * x * x)}
    if kind == "norm":
        n = case["n"]
        dims = [1] + [x] * (n - 1) + [1]
        fl, el = 0.0, 0
        for i in range(n):
            a, b = dims[i], dims[i + 1]
            el += 2 * a * 2 * b
            fl += _qr(2 * b, a) + 8.0 * (a * a * 2 * b + a * 2 * b * b) + (8.0 * dims[i - 1] * 2 * a * a if i else 0)
        return {"bytes": el * es, "flops": fl}
    if kind == "gate":
        fl = _qr(2 * x, x) + 8.0 * (2 * x ** 3 + 4 * x ** 3 + 16 * x * x + 12 * x ** 3) + _svd(2 * x, 2 * x)
        return {"bytes": (3 * 2 * x * x + 16 + 8 * x * x) * es, "flops": fl}
    if kind == "vidal":
        n, dims, fl, el = case["n"], [1] * (case["n"] + 1), 0.0, 0
        for bonds in brickwork_layers(n, case["depth"]):
            for a in bonds:
                li, b, r = dims[a], dims[a + 1], dims[a + 2]
                dims[a + 1] = k = min(x, 2 * li, 2 * r)
                fl += 8.0 * (4 * li * b * r + 16 * li * r + 4 * li * r * k) + _svd(2 * li, 2 * r)
                el += 16 + k
        el += sum(2 * dims[i] * dims[i + 1] for i in range(n))
        return {"bytes": el * es, "flops": fl}
    if kind == "svds":
        sides = _sides(case)
        fl = sum(_svd(m, n) + 8.0 * m * n * ((min(m, n) + 1) // 2) for m, n in sides)
        return {"bytes": 2.0 * es * sum(m * n for m, n in sides), "flops": fl}
    if kind == "batch":
        fl, el = 0.0, 0
        for la, lb, lc, shp in _contractions(case):
            ext = dict(zip(la, shp[0])) | dict(zip(lb, shp[1]))
            fl += 8.0 * math.prod(ext.values())
            el += sum(math.prod(s) for s in shp)
        return {"bytes": float(el * es), "flops": fl}
    if kind == "amps":
        dims = _bonds(case["n"], x)
        el = sum(a * b for a, b in zip(dims, dims[1:]))
        # each physical value's slice is needed at most once, and once per request
        return {"bytes": float(min(2, case["count"]) * el * es), "flops": 8.0 * el * case["count"]}
    # the strings start at most 3 sites right of the centre: the mean sweep length
    span = case["weight"] + 1.5
    return {"bytes": (3 + case["weight"]) * 2.0 * x * x * es, "flops": 8.0 * case["count"] * span * 4 * x ** 3}


# ---- the same in 64 bits, plain torch and numpy ------------------------------------
def _up(v):
    return v.to(torch.complex128) if torch.is_tensor(v) else v


def _mul(A, B, k):
    """Contract A's last k axes with B's first k."""
    sa, sb = A.shape, B.shape
    m = math.prod(sb[:k])
    return (A.reshape(-1, m) @ B.reshape(m, -1)).reshape(tuple(sa[:len(sa) - k]) + tuple(sb[k:]))


def exact(case, seed):
    kind = case["kind"]
    if kind == "vidal" and case["n"] * case["depth"] * case["chi"] ** 3 > 3e8:
        return None
    x = _inputs(case, seed)
    if kind == "site":
        E, A = _up(x["E"]), _up(x["A"])
        return E[:, None, None] * A if case["absorb"] else _mul(E, A, 1)
    if kind == "env":
        L, A, W = _up(x["L"]), _up(x["A"]), _up(x["W"])
        t = _mul(L, A, 1)  # b w p k2
        t = _mul(t.permute(0, 3, 1, 2), W.permute(0, 2, 1, 3), 2)  # b k2 o w2
        return _mul(A.conj().permute(2, 0, 1), t.permute(0, 2, 3, 1), 2)  # b2 w2 k2
    if kind == "heff":
        L, R, W, th = (_up(x[k]) for k in ("L", "R", "W", "theta"))
        op = _mul(W.permute(0, 2, 3, 1), W, 1)  # w o1 i1 wr o2 i2
        t = _mul(L, th, 1)  # l w i1 i2 rk
        t = _mul(t.permute(0, 4, 1, 2, 3), op.permute(0, 2, 5, 1, 4, 3), 3)  # l rk o1 o2 wr
        return _mul(t.permute(0, 2, 3, 1, 4), R.permute(2, 1, 0), 2)  # l o1 o2 r
    if kind == "norm":
        s = [_up(v).cpu().numpy() for v in x["sites"]]
        for i in range(len(s) - 1, 0, -1):
            a, d, b = s[i].shape
            if a == 1:
                continue
            q, r = np.linalg.qr(s[i].reshape(a, d * b, order="F").conj().T)
            s[i] = q.conj().T.reshape(-1, d, b, order="F")
            s[i - 1] = np.tensordot(s[i - 1], r.conj().T, 1)
        nrm = float(np.linalg.norm(s[0]))
        return {"sites": [torch.from_numpy(np.ascontiguousarray(v)) for v in s], "overlap": np.complex128(nrm ** 2),
                "norm": nrm}
    if kind == "gate":
        A, B, C = (_up(v).cpu().numpy() for v in x["sites"])
        G, X = x["gate"].astype(NP[case["dtype"]]).astype(np.complex128).reshape(2, 2, 2, 2), case["chi"]
        q, r = np.linalg.qr(A.reshape(2 * X, X))
        th = np.tensordot(np.tensordot(np.tensordot(r, B, 1), C, 1), G, [[1, 2], [2, 3]])  # l r oa ob
        u, s, v = np.linalg.svd(th.transpose(0, 2, 3, 1).reshape(2 * X, 2 * X))
        k = min(X, int(np.count_nonzero(s > THRESHOLD)))
        th = ((u[:, :k] * s[:k]) @ v[:k]).reshape(X, -1)
        return {"k": k, "block": torch.from_numpy((q @ th).reshape(X, 2, 2, 2, X))}
    if kind == "vidal":
        return _vidal(case, x)
    if kind == "svds":
        flat, low, sv, ks, disc, off = x["flat"].cpu().numpy().astype(np.complex128), [], [], [], [], 0
        for m, n in _sides(case):
            u, s, v = np.linalg.svd(flat[off:off + m * n].reshape(m, n, order="F"), full_matrices=False)
            k = min((min(m, n) + 1) // 2, int(np.count_nonzero(s > THRESHOLD)))
            low.append(((u[:, :k] * s[:k]) @ v[:k]).reshape(-1, order="F"))
            sv.append(s)
            ks.append(k)
            disc.append(float(np.sum(s[k:] ** 2)))
            off += m * n
        return {"low": torch.from_numpy(np.concatenate(low)), "s": np.concatenate(sv), "k": np.array(ks),
                "discarded": np.array(disc)}
    if kind == "batch":
        A, B, oa, ob, got = x["A"], x["B"], 0, 0, []
        for la, lb, lc, (sa, sb, _) in _contractions(case):
            a = _up(A[oa:oa + math.prod(sa)]).reshape(sa[::-1])  # reversed axes: column-major
            b = _up(B[ob:ob + math.prod(sb)]).reshape(sb[::-1])
            got.append(torch.einsum(f"{la[::-1]},{lb[::-1]}->{lc[::-1]}", a, b).reshape(-1))
            oa, ob = oa + a.numel(), ob + b.numel()
        return torch.cat(got)
    if kind == "amps":
        return _amplitudes([_up(v) for v in x["sites"]], x["bits"]).cpu().numpy()
    c = _pauli_chain(case)[1]
    P = {"I": [[1, 0], [0, 1]], "X": [[0, 1], [1, 0]], "Y": [[0, -1j], [1j, 0]], "Z": [[1, 0], [0, -1]]}
    P = {k: torch.tensor(v, dtype=torch.complex128, device="cuda") for k, v in P.items()}
    got = []
    for a, letters in x["terms"]:
        E = torch.eye(x["sites"][c].shape[0], dtype=torch.complex128, device="cuda")
        for i in range(c, a + len(letters)):
            A = _up(x["sites"][i])
            PA = _mul(P[letters[i - a] if i >= a else "I"], A.permute(1, 0, 2), 1).permute(1, 0, 2)
            E = _mul(A.conj().permute(2, 0, 1), _mul(E, PA, 1), 2)
        got.append(complex(torch.trace(E)))
    return np.array(got)


def _amplitudes(sites, bits):
    b = torch.from_numpy(bits.astype(np.int64)).to(sites[0].device)
    v = torch.ones((len(bits), 1), dtype=torch.complex128, device=sites[0].device)
    for i, A in enumerate(sites):
        v = torch.where((b[:, i] == 0)[:, None], v @ A[:, 0, :], v @ A[:, 1, :])
    return v[:, 0]


def _vidal(case, x):
    n = case["n"]
    B = [np.array([1.0, 0.0], dtype=np.complex128).reshape(1, 2, 1) for _ in range(n)]
    lam = [np.ones(1) for _ in range(n - 1)]
    g = 0
    for bonds in brickwork_layers(n, case["depth"]):
        for a in bonds:
            U = x["gates"][g].reshape(2, 2, 2, 2)
            g += 1
            th = np.tensordot(np.tensordot(B[a], B[a + 1], 1), U, [[1, 2], [2, 3]]).transpose(0, 2, 3, 1)
            li, _, _, r = th.shape
            X = (th if a == 0 else lam[a - 1][:, None, None, None] * th).reshape(2 * li, 2 * r)
            s, v = np.linalg.svd(X, full_matrices=False)[1:]
            k = min(case["chi"], int(np.count_nonzero(s > THRESHOLD)))
            v = v[:k].reshape(k, 2, r)
            B[a], B[a + 1], lam[a] = np.tensordot(th, v.conj(), [[2, 3], [1, 2]]), v, s[:k]
    amps = _amplitudes([torch.from_numpy(np.ascontiguousarray(b)) for b in B], x["bits"])
    return {"amps": amps.numpy(), "bonds": np.array([b.shape[2] for b in B[:-1]]), "lambdas": np.concatenate(lam)}
