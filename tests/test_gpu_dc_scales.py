"""Divide and conquer on matrices whose parts differ much in scale.

Bounds as in test_gpu_dc.py, against the norm of the whole matrix: the small part adds
nothing to the backward error, but its vectors have to be orthogonal like the others.
The tridiagonalisation squares the entries it meets, so below about 1e-19 (FP32) and
1e-154 (FP64) of the largest they underflow; a matrix it cannot reduce is reported in
info (batches of fewer than 2048 matrices) and is not checked."""
import numpy as np
import pytest
import torch

import eigeng_batched as eg
from test_gpu_dc import check

pytestmark = pytest.mark.gpu
DEV = "cuda"
KINDS = ["last", "first", "middle", "weak", "dbd", "dbd reversed", "tridiagonal", "tridiagonal reversed"]


def parts(kind, n, s, count, rng):
    """Symmetric matrices with a part s times the rest: a decoupled block in each place,
    a block coupled at its own scale, D B D with D graded either way, and a graded
    tridiagonal."""
    b = rng.uniform(-1, 1, (count, n, n))
    b = (b + b.transpose(0, 2, 1)) / 2
    a = np.zeros_like(b)
    h, q, r = n // 2, n // 3, 2 * n // 3
    d = np.logspace(0, np.log10(s), n)
    if kind == "last":
        a[:, :h, :h], a[:, h:, h:] = b[:, :h, :h], s * b[:, h:, h:]
    elif kind == "first":
        a[:, :h, :h], a[:, h:, h:] = s * b[:, :h, :h], b[:, h:, h:]
    elif kind == "middle":
        a[:, :q, :q], a[:, q:r, q:r], a[:, r:, r:] = b[:, :q, :q], s * b[:, q:r, q:r], b[:, r:, r:]
    elif kind == "weak":
        a = s * b
        a[:, :h, :h] = b[:, :h, :h]
    elif kind.startswith("dbd"):
        a = np.sqrt(d)[:, None] * b * np.sqrt(d)
    else:
        i = np.arange(n)
        a[:, i, i] = d * b[:, i, i]
        a[:, i[1:], i[:-1]] = a[:, i[:-1], i[1:]] = d[1:] * b[:, i[1:], i[:-1]]
    return a[:, ::-1, ::-1].copy() if kind.endswith("reversed") else a


@pytest.mark.parametrize("dtype,scales", [(np.float32, (1e-12, 1e-16, 1e-17, 4e-18)), (np.float64, (1e-100, 1e-150))])
@pytest.mark.parametrize("n,reps", [(8, 1), (16, 1), (20, 1), (20, 3), (33, 1), (48, 1), (64, 1), (100, 1), (130, 1),
                                    (300, 1)])
def test_parts_of_different_scale(n, reps, dtype, scales):
    """Every order class (reps: batches of 512 and more take other shapes for n <= 32)."""
    rng = np.random.default_rng(n)
    for s in scales:
        a = np.concatenate([parts(k, n, s, 24 if n <= 130 else 4, rng) for k in KINDS]).astype(dtype)
        print(f"[dc scales] n={n} {np.dtype(dtype).name} s={s:g} L={reps * len(a)}", flush=True)
        z, w, info = eg.eigen_batch(torch.from_numpy(a).repeat(reps, 1, 1).to(DEV), path="dc")
        torch.cuda.synchronize()
        z, w, info = z.cpu().numpy(), w.cpu().numpy(), info.cpu().numpy()
        ok = info == 0
        assert ok.all() if s >= (1e-12 if dtype == np.float32 else 1e-100) else ok.mean() > 0.5
        check(np.tile(a, (reps, 1, 1))[ok], z[ok], w[ok], dtype)
