"""Tridiagonalisation of matrices that are exhausted early: every column leaves a rest eps
times smaller than the one before, down to where its squares underflow."""
import numpy as np
import pytest
import torch

import eigeng_batched as eg
from test_gpu_dc import check
from test_gpu_dc_scales import parts

pytestmark = pytest.mark.gpu
# groups of lanes (2..16), wave kernel (17..64), register kernel in its three forms (65..128,
# ..192, ..256), streamed
ORDERS = [2, 3, 5, 7, 8, 9, 10, 11, 12, 13, 14, 15, 16, 17, 20, 22, 31, 32, 33, 47, 63, 64, 65, 66, 79, 81, 96, 127, 128, 129, 160, 192, 193, 255, 256, 257, 283, 321,
          334, 384, 385, 449, 453, 512]


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n", ORDERS)
def test_all_ones(n, dtype):
    """The all-ones matrix, its negative, and one with random signs, at several scales:
    solved, bounds as in test_gpu_dc.py."""
    s = np.random.default_rng(n).choice([-1.0, 1.0], n)
    one = np.stack([np.ones((n, n)), -np.ones((n, n)), np.outer(s, s)])
    a = np.concatenate([c * one for c in (1, 3, 1e6, 1e-3)]).astype(dtype)
    # (second forms: 17..32 above 2048 matrices, 129..192 above 256)
    reps = 200 if n <= 32 else 30 if 128 < n <= 192 else 1
    for r in {1, reps}:
        print(f"[all ones] n={n} {np.dtype(dtype).name} L={r * len(a)}", flush=True)
        z, w, info = eg.eigen_batch(torch.from_numpy(a).repeat(r, 1, 1).cuda(), path="dc")
        torch.cuda.synchronize()
        assert int(info.abs().max()) == 0
        check(np.tile(a, (r, 1, 1)), z.cpu().numpy(), w.cpu().numpy(), dtype)


@pytest.mark.parametrize("dtype,scales", [(np.float32, (1e-18, 1e-20, 1e-22, 1e-26)), (np.float64, (1e-154, 1e-160, 1e-200))])
@pytest.mark.parametrize("n,reps", [(8, 1), (9, 60), (16, 1), (16, 60), (17, 1), (20, 50), (20, 60), (32, 1), (33, 1), (48, 60), (64, 1), (100, 1), (130, 1), (200, 1), (300, 1)])
def test_blocks_whose_squares_underflow(n, reps, dtype, scales):
    """A decoupled block that small, last, first or in the middle: solved, from 2048 matrices
    on too, bounds against the norm of the whole matrix."""
    rng = np.random.default_rng(n)
    for s in scales:
        a = np.concatenate([parts(k, n, s, 12 if n <= 130 else 2, rng) for k in ("last", "first", "middle")]).astype(dtype)
        print(f"[small blocks] n={n} {np.dtype(dtype).name} s={s:g} L={reps * len(a)}", flush=True)
        z, w, info = eg.eigen_batch(torch.from_numpy(a).repeat(reps, 1, 1).cuda(), path="dc")
        torch.cuda.synchronize()
        assert int(info.abs().max()) == 0
        check(np.tile(a, (reps, 1, 1)), z.cpu().numpy(), w.cpu().numpy(), dtype)
