"""The work that is timed: batched symmetric eigendecompositions as programs run them.

A pass takes matrices to eigenpairs through the binding's entry points and then forms
what a program forms of eigenpairs: Z diag(w) Z^T, or (for the ensemble filter) the
transform sqrt(k-1) A^{-1/2} from a scaled power of the eigenvalues.  An eigenvector's
sign, and the basis of a close pair of eigenvalues, are arbitrary, so the eigenvalues and
that product, which uses every eigenvector whole, are what a pass returns.

Three kinds of case:
  letkf   analysis step: A = (k-1)/rho I + Y^T Y from the observations (gram), the solve,
          and the transform (matpow).  FP32, Y ~ N(0, 0.1^2).
  eig     one uniform batch: A copied into the buffer that is solved in place, the solve,
          the product (symdmt).  Spectra: "random" A = (B + B^T)/2 with B ~ U[-1, 1];
          "pairs" A = Q diag(lam) Q^T, lam ~ U[-1, 1] with 5 % of them in pairs split by
          1e-8.  solver: "plain" or "mixed" (FP32 solve and FP64 refinement).
  uneven  one batch of many orders, lam log-spaced over 1..1e-6 in random order, packed
          matrix after matrix; the products are formed per order.
"""
from __future__ import annotations

import math
import os
import sys
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "eigeng-batched_amd"))
import eigeng_batched as eg  # noqa: E402

DT = {"f32": torch.float32, "f64": torch.float64}
SOLVER = {"plain": eg.IMTQL2, "mixed": eg.MIXED}
RHO = 1.1


def listed():
    return [
        # a few grid points with a small ensemble: launches and latency are all there is
        {"name": "letkf n20 L16", "kind": "letkf", "dtype": "f32", "n": 20, "p": 60, "L": 16},
        # the small FP64 batch of the configurations: 1024 matrices of order 32
        {"name": "eig f64 n32 L1024", "kind": "eig", "dtype": "f64", "n": 32, "nm": 32, "L": 1024,
         "spectrum": "random", "solver": "plain"},
        # the headline: an analysis step of 64 members and 400 observations at 16384 points
        {"name": "letkf n64 L16384", "kind": "letkf", "dtype": "f32", "n": 64, "p": 400, "L": 16384},
        # one step of the drifting stream of 48 members and 300 observations at 65536 points
        {"name": "letkf n48 L65536", "kind": "letkf", "dtype": "f32", "n": 48, "p": 300, "L": 65536},
        # FP64, an order that fills no tile, padded columns, a batch between small and large
        {"name": "eig f64 n60 L3000", "kind": "eig", "dtype": "f64", "n": 60, "nm": 64, "L": 3000,
         "spectrum": "random", "solver": "plain"},
        # a small batch of an order past one wave's 64 rows, ragged
        {"name": "eig f32 n100 L500", "kind": "eig", "dtype": "f32", "n": 100, "nm": 104, "L": 500,
         "spectrum": "random", "solver": "plain"},
        # the FP32 batch of order 128
        {"name": "eig f32 n128 L8192", "kind": "eig", "dtype": "f32", "n": 128, "nm": 128, "L": 8192,
         "spectrum": "pairs", "solver": "plain"},
        # the large FP64 batch: 8192 matrices of order 256
        {"name": "eig f64 n256 L8192", "kind": "eig", "dtype": "f64", "n": 256, "nm": 256, "L": 8192,
         "spectrum": "random", "solver": "plain"},
        # a handful of large FP64 matrices: one call of a program that has few of them
        {"name": "eig f64 n200 L64", "kind": "eig", "dtype": "f64", "n": 200, "nm": 200, "L": 64,
         "spectrum": "random", "solver": "plain"},
        # the largest order
        {"name": "eig f64 n512 L64", "kind": "eig", "dtype": "f64", "n": 512, "nm": 512, "L": 64,
         "spectrum": "random", "solver": "plain"},
        # every order from 8 to 128 in one call
        {"name": "uneven f32 n8-128 L20000", "kind": "uneven", "dtype": "f32", "n": 128, "nlo": 8, "L": 20000},
        # mixed precision: FP64 results by refinement of an FP32 solve, clustered spectrum
        {"name": "mixed f64 n256 L2048", "kind": "eig", "dtype": "f64", "n": 256, "nm": 256, "L": 2048,
         "spectrum": "pairs", "solver": "mixed"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["letkf", "letkf", "eig", "eig", "eig", "eig", "uneven", "mixed"])
    if kind == "letkf":
        n = rng.randint(8, 64)
        top = min(65536, int(1.2e9 / n ** 2))
        return {"kind": "letkf", "dtype": "f32", "n": n, "p": rng.randint(n, 400), "L": _log(rng, 16, top)}
    if kind == "uneven":
        nlo = rng.randint(8, 24)
        return {"kind": "uneven", "dtype": rng.choice(["f32", "f32", "f64"]), "n": rng.randint(48, 128), "nlo": nlo,
                "L": _log(rng, 1000, 20000)}
    if kind == "mixed":
        n = _log(rng, 64, 256)
        return {"kind": "eig", "dtype": "f64", "n": n, "nm": n, "L": _log(rng, 64, min(4096, int(1.3e8 / n ** 2))),
                "spectrum": "pairs", "solver": "mixed"}
    n = _log(rng, 8, 512)
    top = 16384 if n <= 64 else 8192 if n <= 128 else 2048 if n <= 256 else 128
    return {"kind": "eig", "dtype": rng.choice(["f32", "f64"]), "n": n, "nm": n + rng.choice([0, 0, 1, 4]),
            "L": _log(rng, 16, top), "spectrum": "random", "solver": "plain"}


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _orthogonal(L, n, g):
    """Q of a Gaussian matrix, FP64, as its n-1 Householder reflections applied to I."""
    G = torch.randn((L, n, n), generator=g, device="cuda", dtype=torch.float64)
    V = []
    for k in range(n - 1):
        v = G[:, k:, k].clone()
        v[:, 0] += torch.where(v[:, 0] >= 0, 1.0, -1.0) * torch.linalg.vector_norm(v, dim=1)
        v /= torch.linalg.vector_norm(v, dim=1, keepdim=True)
        S = G[:, k:, k:]
        S -= 2.0 * v.unsqueeze(2) * torch.bmm(v.unsqueeze(1), S)
        V.append(v)
    Q = torch.eye(n, dtype=torch.float64, device="cuda").expand(L, n, n).contiguous()
    for k in reversed(range(n - 1)):
        S = Q[:, k:, :]
        S -= 2.0 * V[k].unsqueeze(2) * torch.bmm(V[k].unsqueeze(1), S)
    return Q


def _from_spectrum(lam, g):
    Q = _orthogonal(lam.shape[0], lam.shape[1], g)
    A = torch.bmm(Q * lam[:, None, :], Q.transpose(1, 2).contiguous())
    return 0.5 * (A + A.transpose(1, 2))


def _matrices(case, seed):
    """The batch (L, n, nm) of an "eig" case; the padding rows are not read."""
    L, n, nm, dt = case["L"], case["n"], case["nm"], DT[case["dtype"]]
    g = _generator(seed)
    a = torch.zeros((L, n, nm), dtype=dt, device="cuda")
    if case["spectrum"] == "random":
        b = torch.rand((L, n, n), generator=g, dtype=dt, device="cuda") * 2 - 1
        a[:, :, :n] = 0.5 * (b + b.transpose(1, 2))
    else:
        pairs = max(1, int(round(0.025 * n)))
        lam = torch.rand((L, n), generator=g, dtype=torch.float64, device="cuda") * 2 - 1
        idx = torch.argsort(torch.rand((L, n), generator=g, device="cuda"), dim=1)[:, : 2 * pairs]
        lam.scatter_(1, idx[:, 1::2], torch.gather(lam, 1, idx[:, 0::2]) + 1e-8)
        a[:, :, :n] = _from_spectrum(lam, g)
    return a


def _observations(case, seed):
    g = _generator(seed)
    return torch.randn((case["L"], case["n"], case["p"]), generator=g, device="cuda", dtype=torch.float32) * 0.1


def _orders(case):
    """The orders of an uneven batch: nlo..n in equal numbers, ascending."""
    return case["nlo"] + np.arange(case["L"], dtype=np.int64) * (case["n"] - case["nlo"] + 1) // case["L"]


def _uneven(case, seed):
    """(packed batch, orders, [(order, how many)])."""
    ns = _orders(case)
    g = _generator(seed)
    parts, runs = [], []
    for n, count in zip(*np.unique(ns, return_counts=True)):
        n, count = int(n), int(count)
        lam = torch.logspace(0, -6, n, dtype=torch.float64, device="cuda")
        lam = lam[torch.argsort(torch.rand((count, n), generator=g, device="cuda"), dim=1)]
        parts.append(_from_spectrum(lam, g).to(DT[case["dtype"]]).reshape(-1))
        runs.append((n, count))
    return torch.cat(parts), ns, runs


def prepare(case, seed):
    L, n, dt = case["L"], case["n"], DT[case["dtype"]]
    s = {"kind": case["kind"], "info": torch.empty(L, dtype=torch.int32, device="cuda")}
    if case["kind"] == "letkf":
        s["y"], s["p"], s["k"] = _observations(case, seed), case["p"], n
        s["a"] = torch.empty((L, n, n), dtype=dt, device="cuda")
        s["w"] = torch.empty((L, n), dtype=dt, device="cuda")
        s["c"] = torch.empty_like(s["a"])
        size = eg.bufsize(L, n, n, n, 4)
        s["solver"] = eg.IMTQL2
    elif case["kind"] == "eig":
        s["a0"] = _matrices(case, seed)
        s["a"] = torch.empty_like(s["a0"])
        s["w"] = torch.empty((L, n), dtype=dt, device="cuda")
        s["c"] = torch.zeros_like(s["a0"])
        s["solver"] = SOLVER[case["solver"]]
        size = eg.bufsize(L, case["nm"], n, n, s["a"].element_size(), s["solver"])
    else:
        s["a0"], ns, s["runs"] = _uneven(case, seed)
        s["a"], s["c"] = torch.empty_like(s["a0"]), torch.empty_like(s["a0"])
        s["w"] = torch.empty(int(ns.sum()), dtype=dt, device="cuda")
        s["nv"] = torch.from_numpy(ns.astype(np.int32)).to("cuda")
        s["n"] = n
        size = eg.uneven_bufsize(L, n, s["a"].element_size())
    s["ws"] = torch.empty(max(size, 1), dtype=torch.uint8, device="cuda")
    return s


def run(s):
    a, w, c = s["a"], s["w"], s["c"]
    if s["kind"] == "letkf":
        eg.gram(s["y"], s["p"], alpha=(s["k"] - 1) / RHO, a=a)
        eg.eigen_batch(a, w=w, info=s["info"], workspace=s["ws"])
        eg.matpow(a, w, -0.5, scale=math.sqrt(s["k"] - 1), c=c)
    elif s["kind"] == "eig":
        a.copy_(s["a0"])
        eg.eigen_batch(a, w=w, solver=s["solver"], info=s["info"], workspace=s["ws"])
        eg.symdmt(a, w, c=c)
    else:
        a.copy_(s["a0"])
        eg.eigen_batch_uneven(a, s["nv"], s["n"], w=w, info=s["info"], workspace=s["ws"])
        oa = ow = 0
        for n, count in s["runs"]:
            ea, ew = oa + count * n * n, ow + count * n
            eg.symdmt(a[oa:ea].view(count, n, n), w[ow:ew].view(count, n), c=c[oa:ea].view(count, n, n))
            oa, ow = ea, ew
    return {"w": w, "product": c, "info": s["info"]}


def work(case):
    """The input read once (the upper triangle, or the observations), eigenvectors, eigenvalues
    and product written once; (10/3) n^3 operations a solve and n^2 (n+1) a product."""
    size = 4 if case["dtype"] == "f32" else 8
    L = case["L"]
    if case["kind"] == "uneven":
        ns = np.arange(case["nlo"], case["n"] + 1, dtype=np.float64)
    else:
        ns = np.array([case["n"]], dtype=np.float64)
    source = case["p"] * ns if case["kind"] == "letkf" else ns * (ns + 1) / 2
    extra = case["p"] * ns * (ns + 1) if case["kind"] == "letkf" else 0
    return {"bytes": float(L * size * np.mean(source + 2 * ns * ns + ns)),
            "flops": float(L * np.mean(10.0 / 3.0 * ns ** 3 + ns * ns * (ns + 1) + extra))}


def _threads(fn, parts):
    with ThreadPoolExecutor(max_workers=min(16, os.cpu_count() or 1)) as ex:
        return list(ex.map(fn, parts))


def _eigenvalues(A):
    """Ascending eigenvalues of a batch, FP64, on the host."""
    A = A.cpu().numpy()
    step = max(1, min(256, A.shape[0] // 32))
    got = _threads(np.linalg.eigvalsh, [A[i:i + step] for i in range(0, A.shape[0], step)])
    return torch.from_numpy(np.concatenate(got))


def _transform(A, k):
    """sqrt(k-1) A^{-1/2} in FP64 (A well conditioned): the coupled Newton-Schulz iteration."""
    size = A.diagonal(dim1=1, dim2=2).abs().amax(1)[:, None, None] * 2
    eye = torch.eye(A.shape[1], dtype=A.dtype, device=A.device).expand_as(A)
    Y, Z = A / size, eye.clone()
    for _ in range(24):
        T = 0.5 * (3.0 * eye - torch.bmm(Z, Y))
        Y, Z = torch.bmm(Y, T), torch.bmm(T, Z)
    return math.sqrt(k - 1) * Z / torch.sqrt(size)


def exact(case, seed):
    L, n = case["L"], case["n"]
    info = torch.zeros(L, dtype=torch.int32)
    if case["kind"] == "letkf":
        y = _observations(case, seed)
        A = torch.empty((L, n, n), dtype=torch.float64, device="cuda")
        c = torch.empty_like(A)
        for i in range(0, L, 4096):
            z = y[i:i + 4096].double()
            A[i:i + 4096] = torch.bmm(z, z.transpose(1, 2).contiguous())
            A[i:i + 4096] += torch.eye(n, dtype=torch.float64, device="cuda") * ((n - 1) / RHO)
            c[i:i + 4096] = _transform(A[i:i + 4096], n)
        return {"w": _eigenvalues(A), "product": c, "info": info}
    if case["kind"] == "eig":
        A = _matrices(case, seed).double()
        return {"w": _eigenvalues(A[:, :, :n].contiguous()), "product": A, "info": info}
    packed, _, runs = _uneven(case, seed)
    packed, at, w = packed.double(), 0, []
    for n, count in runs:
        w.append(_eigenvalues(packed[at:at + count * n * n].view(count, n, n)).reshape(-1))
        at += count * n * n
    return {"w": torch.cat(w), "product": packed, "info": info}
