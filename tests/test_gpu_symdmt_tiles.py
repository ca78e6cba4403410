"""C = Z diag(d) Z^T by 64 x 64 tiles (n > 64) at the edges of the tiles.

Bound: a sum of n products accumulated one after the other in the working
precision, each with its own rounding of z d: |error| <= (n + 2) eps |Z| |d| |Z|^T.
"""
import numpy as np
import pytest
import torch

import eigeng_batched as eg

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("n", [65, 79, 80, 81, 127, 128, 129, 192, 193, 511, 512])
@pytest.mark.parametrize("L", [1, 8])
def test_edges_of_the_tiles(n, dtype, L):
    print(f"[symdmt] n={n} {dtype} L={L}", flush=True)
    rng = np.random.default_rng(n)
    nm = n + 3
    z = rng.normal(size=(L, n, n)).astype(np.float32 if dtype == torch.float32 else np.float64)
    d = rng.normal(size=(L, n))
    zt = torch.full((L, n, nm), float("nan"), dtype=dtype)
    zt[:, :, :n] = torch.from_numpy(z)
    dt = torch.from_numpy(d).to(dtype)
    c = torch.full((L, n, nm), -7.0, dtype=dtype, device=DEV)
    eg.symdmt(zt.to(DEV), dt.to(DEV), c)
    torch.cuda.synchronize()
    c = c.cpu()
    assert bool((c[:, :, n:] == -7.0).all())
    c = c[:, :, :n]
    assert torch.equal(c, c.transpose(1, 2))
    z, d = z.astype(np.longdouble), dt.numpy().astype(np.longdouble)
    for k in {0, L - 1}:
        ref = z[k].T @ (d[k][:, None] * z[k])
        mag = np.abs(z[k]).T @ (np.abs(d[k])[:, None] * np.abs(z[k]))
        assert (np.abs(c[k].numpy() - ref) <= (n + 2) * float(torch.finfo(dtype).eps) * mag).all()
