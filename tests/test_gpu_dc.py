"""The divide and conquer path (csrc/eig_dc.hpp) at the edges of its tiles.

Bounds, derived from backward stability with every step's error a small multiple
of eps ||A||: eigenvalues within 8 n eps ||A|| of LAPACK's in float64, residual
||A Z - Z D||_F <= 8 n eps ||A||, ||Z^T Z - I||_max <= 8 n eps.
"""
import numpy as np
import pytest
import torch

import eigeng_batched as eg

pytestmark = pytest.mark.gpu
DEV = "cuda"


def families(n, rng):
    """Symmetric matrices on which merges meet every kind of node: generic,
    symmetric halves (equal poles), graded, clustered, low rank, decoupled."""
    def spec(lam):
        q = np.linalg.qr(rng.normal(size=(n, n)))[0]
        return (q * lam) @ q.T
    b = [rng.uniform(-1, 1, (n, n)) for _ in range(5)]
    y = rng.normal(0, 0.1, (n // 2, n))
    lam = rng.uniform(-1, 1, n)
    pairs = lam.copy()
    pairs[1::2] = pairs[0::2][: len(pairs[1::2])] + 1e-8
    block = np.zeros((n, n))
    h = n // 3
    block[:h, :h], block[h:, h:] = b[0][:h, :h], b[1][h:, h:]
    low = np.ones(n)
    low[:2] = [3.0, 2.0][:n]
    out = b[:3] + [
        2 * np.eye(n) - np.eye(n, k=1) - np.eye(n, k=-1), np.eye(n, k=1) + np.eye(n, k=-1),
        np.minimum.outer(np.arange(1.0, n + 1), np.arange(1.0, n + 1)),
        np.eye(n) * (n - 1) / 1.1 + y.T @ y, spec(np.logspace(0, -6, n)), spec(pairs), spec(low), block,
        np.eye(n), np.zeros((n, n)), np.diag(lam), 1e10 * b[3], 1e-10 * b[4]]
    return np.array([(a + a.T) / 2 for a in out])


def check(a, z, w, dtype):
    n, eps = a.shape[1], float(np.finfo(dtype).eps)
    a, z, w = a.astype(np.float64), z.astype(np.float64), w.astype(np.float64)
    we = np.linalg.eigvalsh(a)
    nrm = np.maximum(np.abs(we).max(axis=1), 1e-300)
    assert (np.diff(w, axis=1) >= 0).all()
    assert (np.abs(w - we).max(axis=1) <= 8 * n * eps * nrm).all()
    v = z.transpose(0, 2, 1)
    assert (np.linalg.norm(a @ v - v * w[:, None, :], axis=(1, 2)) <= 8 * n * eps * nrm).all()
    assert (np.abs(z @ v - np.eye(n)).max(axis=(1, 2)) <= 8 * n * eps).all()


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n", [1, 2, 3, 7, 8, 9, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64])
@pytest.mark.parametrize("reps", [1, 40])
def test_families(n, dtype, reps):
    """Every order class, in the small-batch (two-wave) and the large-batch shape."""
    print(f"[dc] n={n} {np.dtype(dtype).name} x{reps}", flush=True)
    a = np.tile(families(n, np.random.default_rng(n)).astype(dtype), (reps, 1, 1))
    nm = n + 1
    t = torch.full((a.shape[0], n, nm), float("nan"), dtype=torch.float32 if dtype == np.float32 else torch.float64)
    t[:, :, :n] = torch.from_numpy(np.tril(a))           # t[k, c, r]: the upper triangle r <= c
    z, w, info = eg.eigen_batch(t.to(DEV), path="dc")
    torch.cuda.synchronize()
    assert int(info.abs().max()) == 0
    z = z.cpu().numpy()
    assert np.isnan(z[:, :, n:]).all()
    check(a, z[:, :, :n], w.cpu().numpy(), dtype)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n", [65, 66, 128, 129, 192, 193, 256, 257, 320, 321, 384, 385, 449, 512])
def test_families_of_several_blocks(n, dtype):
    """Every shape of the merge tree over blocks of 64 columns (one column in the
    last block, full blocks, uneven halves) and every back-transformation size."""
    print(f"[dc] n={n} {np.dtype(dtype).name}", flush=True)
    a = families(n, np.random.default_rng(n)).astype(dtype)
    t = torch.full((a.shape[0], n, n + 1), float("nan"), dtype=torch.float32 if dtype == np.float32 else torch.float64)
    t[:, :, :n] = torch.from_numpy(np.tril(a))
    z, w, info = eg.eigen_batch(t.to(DEV), path="dc")
    torch.cuda.synchronize()
    assert int(info.abs().max()) == 0
    z = z.cpu().numpy()
    assert np.isnan(z[:, :, n:]).all()
    check(a, z[:, :, :n], w.cpu().numpy(), dtype)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n", [65, 128, 129, 160, 191, 192, 193])
def test_families_in_large_batches(n, dtype):
    """More than 256 matrices (128 < n <= 192: the three-block tridiagonalisation)."""
    print(f"[dc] n={n} {np.dtype(dtype).name}", flush=True)
    f = families(n, np.random.default_rng(n)).astype(dtype)
    t = torch.from_numpy(np.tril(f)).repeat(17, 1, 1).to(DEV)
    z, w, info = eg.eigen_batch(t, path="dc")
    torch.cuda.synchronize()
    assert int(info.abs().max()) == 0
    z, w = z.view(17, *f.shape), w.view(17, *f.shape[:2])
    assert torch.equal(z, z[:1].expand_as(z)) and torch.equal(w, w[:1].expand_as(w))
    check(f, z[0].cpu().numpy(), w[0].cpu().numpy(), dtype)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n", [257, 264, 272])
def test_more_matrices_than_workgroups(n, dtype):
    """Above 1024 matrices a workgroup of the tridiagonalisation takes a second one:
    copies of one matrix give the same bits wherever they stand in the batch."""
    a = families(n, np.random.default_rng(n))[:5].astype(dtype)
    z0, w0, _ = eg.eigen_batch(torch.from_numpy(np.tril(a)).to(DEV), path="dc")
    check(a, z0.cpu().numpy(), w0.cpu().numpy(), dtype)
    z, w, info = eg.eigen_batch(torch.from_numpy(np.tril(a)).to(DEV).repeat(206, 1, 1), path="dc")
    torch.cuda.synchronize()
    assert int(info.abs().max()) == 0
    assert torch.equal(z.view(206, *z0.shape), z0.expand(206, *z0.shape))
    assert torch.equal(w.view(206, *w0.shape), w0.expand(206, *w0.shape))


# Q is formed explicitly nowhere for n > 64 any more: these batches take the reflectors and
# the blocked back-transformation as smaller ones do, and no small batch is compared with.
@pytest.mark.parametrize("n", [65, 100, 128])
def test_families_with_explicit_q(n):
    """FP32 batches of 2048 and more, n <= 128: Q formed by the tridiagonalisation
    and multiplied; the same bound, and the small batch's eigenvalues."""
    a = np.tile(families(n, np.random.default_rng(n)).astype(np.float32), (130, 1, 1))
    t = torch.from_numpy(np.tril(a)).to(DEV)
    z, w, info = eg.eigen_batch(t.clone())
    torch.cuda.synchronize()
    assert int(info.abs().max()) == 0
    check(a, z.cpu().numpy(), w.cpu().numpy(), np.float32)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("n", [8, 33, 64, 100, 130, 300])
def test_first_columns_and_smaller_chunks(n, dtype):
    """m < n stores the same first columns and eigenvalues; a divided chunk and a
    call phase by phase give the same bits."""
    g = torch.Generator(device=DEV)
    g.manual_seed(n)
    L = 900 if n <= 130 else 20
    b = torch.rand((L, n, n), generator=g, device=DEV, dtype=dtype) - 0.5
    a = (b + b.transpose(1, 2)).contiguous()
    z, w, _ = eg.eigen_batch(a.clone(), path="dc")
    m = n // 2
    zm, wm, _ = eg.eigen_batch(a.clone(), m=m, path="dc")
    assert torch.equal(w, wm) and torch.equal(z[:, :m], zm[:, :m]) and torch.equal(zm[:, m:], a[:, m:])
    zc, wc, _ = eg.eigen_batch(a.clone(), solver=eg.IMTQL2 | (3 << eg.CHUNK_SHIFT), path="dc")
    assert torch.equal(w, wc) and torch.equal(z, zc)
    ws = torch.empty(eg.bufsize(L, n, n, n, a.element_size(), eg.FLAG_DC), dtype=torch.uint8, device=DEV)
    zp, wp, info = a.clone(), torch.empty_like(w), torch.empty(L, dtype=torch.int32, device=DEV)
    for ph in ("tri", "ql", "apply"):
        eg.eigen_batch(zp, w=wp, info=info, workspace=ws, path="dc", phases=[ph])
    assert torch.equal(w, wp) and torch.equal(z, zp)


# From 2048 matrices on, "split" is divide and conquer itself for n <= 64:
# test_gpu_dc_status.py compares with routes that are QL at every size.
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("n,L", [(20, 40), (20, 3000), (48, 100), (48, 2100), (64, 30), (100, 60), (100, 2050),
                                 (200, 30), (200, 520)])
def test_matrices_that_are_not_finite(n, L, dtype):
    """A NaN or an infinity in one matrix: the status of the path the batch took
    before (the fused kernel's for small batches, the split path's for large ones),
    its neighbours untouched by it."""
    g = torch.Generator(device=DEV)
    g.manual_seed(7)
    b = torch.rand((L, n, n), generator=g, device=DEV, dtype=dtype) - 0.5
    a = (b + b.transpose(1, 2)).contiguous()
    good, gw, _ = eg.eigen_batch(a.clone())
    bad = [1, 7, 20]
    a[1, :, :] = float("nan")
    a[7, 5, 3] = float("nan")
    a[20, 4, 4] = float("inf")
    small = n not in (20,) and n < 65 and L < 2048 or (n == 20 and dtype == torch.float32 and L < 2048)
    if dtype == torch.float32 and n == 64:
        small = L < 1024
    z, w, info = eg.eigen_batch(a.clone())
    if n > 64:
        # the same statuses: 1 from the small batch's path, 0 from the large one's
        small = L < (2048 if dtype == torch.float32 and n <= 128 else 512)
        ok = [k for k in range(L) if k not in bad]
        assert torch.equal(z[ok], good[ok]) and torch.equal(w[ok], gw[ok]) and int(info[ok].abs().max()) == 0
        for k in bad:
            assert int(info[k]) == (1 if small else 0) and bool(torch.isnan(w[k]).any())
            assert bool(torch.isnan(z[k]).any()) or (small and torch.equal(z[k], a[k]))
        return
    zq, wq, iq = eg.eigen_batch(a.clone(), path="fused" if small else "split")
    ok = [k for k in range(L) if k not in bad]
    assert torch.equal(info, iq)
    assert torch.equal(z[ok], good[ok]) and torch.equal(w[ok], gw[ok])
    for k in bad:
        assert bool(torch.isnan(w[k]).any()) and bool(torch.isnan(wq[k]).any())
        assert torch.equal(torch.isnan(z[k]), torch.isnan(zq[k]))
        assert not small or torch.equal(z[k].nan_to_num(), a[k].nan_to_num())      # left as it was
