"""Statuses of the divide and conquer path against the QL routes'."""
import numpy as np
import pytest
import torch

import eigeng_batched as eg

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("n,L", [(20, 300), (20, 2100), (64, 300), (64, 2100)])
def test_warm_start_reports_what_it_cannot_solve(n, L):
    """Matrices whose Jacobi is cut short and whose tridiagonalisation underflows (entries
    of 1e-20 in FP32): reported in info and left as they were, in large batches too; the
    other matrices solved."""
    print(f"[warm status] n={n} L={L}", flush=True)
    rng = np.random.default_rng(n)
    b = rng.uniform(-1, 1, (L, n, n))
    a0 = ((b + b.transpose(0, 2, 1)) / 2).astype(np.float32)
    lost = np.arange(3, L, 97)
    a0[lost] *= np.float32(1e-20)
    a = torch.from_numpy(a0).to(DEV)
    q0 = torch.eye(n, device=DEV).expand(L, n, n).contiguous()
    z, w, info, _ = eg.eigen_batch_warm(a.clone(), q0, max_sweeps=1)
    torch.cuda.synchronize()
    assert bool((info[lost] > 0).all()) and torch.equal(z[lost], a[lost])
    ok = np.setdiff1d(np.arange(L), lost)
    assert int(info[ok].abs().max()) == 0
    v = z[ok].double()
    r = torch.linalg.matrix_norm(v @ a[ok].double() - w[ok].double().unsqueeze(2) * v)
    assert float((r / w[ok].double().abs().amax(1)).max()) <= 8 * n * 2.0 ** -23


def test_large_fp32_chunk_and_its_phases():
    """FP32 64 < n <= 128 in one chunk of more than 8192 matrices: the bits of a smaller
    batch, and of the call phase by phase."""
    n, L = 66, 9000
    g = torch.Generator(device=DEV)
    g.manual_seed(3)
    b = torch.rand((L, n, n), generator=g, device=DEV) - 0.5
    a = (b + b.transpose(1, 2)).contiguous()
    z, w, info = eg.eigen_batch(a.clone())
    z0, w0, _ = eg.eigen_batch(a[6000:].clone())
    ws = torch.empty(eg.bufsize(L, n, n, n, 4), dtype=torch.uint8, device=DEV)
    zp, wp = a.clone(), torch.empty_like(w)
    for ph in ("tri", "ql", "apply"):
        eg.eigen_batch(zp, w=wp, workspace=ws, phases=[ph])
    torch.cuda.synchronize()
    assert int(info.abs().max()) == 0
    assert torch.equal(z[6000:], z0) and torch.equal(w[6000:], w0)
    assert torch.equal(zp, z) and torch.equal(wp, w)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("n,L", [(8, 2100), (16, 2100), (20, 2100), (32, 3000), (48, 2100), (64, 2100), (100, 2100)])
def test_eigenvalues_after_the_second_phase(n, L, dtype):
    """The first two phases, together or one by one: eigenvalues and status, as after the
    QL recurrence, with a as it was; the third then stores the vectors."""
    print(f"[phases] n={n} L={L} {dtype}", flush=True)
    g = torch.Generator(device=DEV)
    g.manual_seed(n)
    b = torch.rand((L, n, n), generator=g, device=DEV, dtype=dtype) - 0.5
    a = (b + b.transpose(1, 2)).contiguous()
    z, w, _ = eg.eigen_batch(a.clone())
    ws = torch.empty(eg.bufsize(L, n, n, n, a.element_size()), dtype=torch.uint8, device=DEV)
    for phases in ([["tri", "ql"], ["apply"]], [["tri"], ["ql"], ["apply"]], [["tri"], ["ql", "apply"]]):
        zp, wp = a.clone(), torch.full_like(w, float("nan"))
        info = torch.full((L,), -7, dtype=torch.int32, device=DEV)
        for ph in phases:
            if ph == ["apply"]:
                assert torch.equal(wp, w) and torch.equal(zp, a) and int(info.abs().max()) == 0
            eg.eigen_batch(zp, w=wp, info=info, workspace=ws, phases=ph)
        assert torch.equal(wp, w) and torch.equal(zp, z) and int(info.abs().max()) == 0


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("n,L", [(8, 40), (16, 3000), (20, 40), (20, 600), (40, 40), (64, 2100), (65, 40), (100, 2100),
                                 (200, 40), (300, 8), (512, 4)])
def test_merges_that_fail_are_reported(n, L, dtype):
    """One evaluation a root (0x8000000 with 0x400): a matrix with roots to find is
    reported in info and left as it was, a diagonal one is solved."""
    print(f"[dc lost] n={n} L={L} {dtype}", flush=True)
    g = torch.Generator(device=DEV)
    g.manual_seed(n)
    b = torch.rand((L, n, n), generator=g, device=DEV, dtype=dtype) - 0.5
    a = (b + b.transpose(1, 2)).contiguous()
    a[1::2] = torch.diag_embed(torch.diagonal(a[1::2], dim1=1, dim2=2))
    z, w, info = eg.eigen_batch(a.clone(), solver=eg.IMTQL2 | 0x400, path="dc")
    torch.cuda.synchronize()
    assert bool((info[0::2] == 1).all()) and torch.equal(z[0::2], a[0::2])
    assert int(info[1::2].abs().max()) == 0
    assert torch.equal(w[1::2], torch.diagonal(a[1::2], dim1=1, dim2=2).sort(dim=1)[0])
    assert torch.equal(z[1::2].abs().sum(2), torch.ones_like(w[1::2]))


def ql_route(n, L, dtype):
    """A route of the QL recurrence with the outcome of the path a batch took without
    divide and conquer (extra bits keep it off that path): (path, extra solver bits)."""
    f32 = dtype == torch.float32
    if n <= 64:
        least = 1 if 16 <= n <= 32 and not f32 or 28 <= n <= 32 else 1024 if f32 and n >= 56 else 2048
        return ("split-lds", 0) if L >= least else ("fused", 0)
    if f32 and n <= 128:
        return ("split-reg128", 0) if L >= 2048 else ("fused", 0)
    if L < 512:
        return ("fused", 0)
    return ("split-ws", 0) if n <= 256 else ("split", 1 << 28)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("n,L", [(8, 40), (8, 3000), (12, 3000), (20, 40), (20, 3000), (30, 40), (48, 100), (48, 2100),
                                 (60, 1500), (64, 30), (64, 2100), (100, 60), (100, 2050), (200, 30), (200, 520),
                                 (300, 30)])
def test_statuses_of_matrices_that_are_not_finite(n, L, dtype):
    """A NaN or an infinity: the status of the QL route, NaN among the eigenvalues of both,
    and for n <= 64 the same eigenvectors written or left."""
    path, extra = ql_route(n, L, dtype)
    print(f"[dc status] n={n} L={L} {dtype} against {path}", flush=True)
    g = torch.Generator(device=DEV)
    g.manual_seed(7)
    b = torch.rand((L, n, n), generator=g, device=DEV, dtype=dtype) - 0.5
    a = (b + b.transpose(1, 2)).contiguous()
    bad = [1, 7, 20, 25]
    a[1] = float("nan")
    a[7, 5, 3] = float("nan")
    a[20, 4, 4] = float("inf")
    a[25, 6, 2] = -float("inf")
    z, w, info = eg.eigen_batch(a.clone())
    zq, wq, iq = eg.eigen_batch(a.clone(), solver=eg.IMTQL2 | extra, path=path)
    torch.cuda.synchronize()
    assert torch.equal(info, iq)
    assert bool(torch.isnan(w[bad]).any(1).all()) and bool(torch.isnan(wq[bad]).any(1).all())
    ok = [k for k in range(L) if k not in bad]
    assert bool(torch.isfinite(w[ok]).all()) and bool(torch.isfinite(z[ok]).all())
    if n <= 64:
        assert torch.equal(torch.isnan(z[bad]), torch.isnan(zq[bad]))
    if int(info[1]) != 0:
        assert torch.equal(z[bad].nan_to_num(), a[bad].nan_to_num())


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n", [9, 20, 33, 48, 64])
def test_ql_split_kernels_in_large_batches(n, dtype):
    """The separate QL kernels on batches that divide and conquer takes otherwise: with d
    and e in LDS, and in registers (TQL2, and the order of the iteration); the bounds are
    the reference checker's."""
    L = 2100
    print(f"[ql split] n={n} {np.dtype(dtype).name}", flush=True)
    rng = np.random.default_rng(n)
    b = rng.uniform(-1, 1, (L, n, n))
    a = torch.from_numpy(((b + b.transpose(0, 2, 1)) / 2).astype(dtype)).to(DEV)
    we = np.linalg.eigvalsh(a.cpu().numpy().astype(np.float64))
    eps = float(np.finfo(dtype).eps)
    tol = eps * (1023 if dtype == np.float64 else 31) * np.sqrt(n + 16.0) * np.abs(we).max(axis=1, keepdims=True)
    for kw in (dict(path="split-lds"), dict(path="split", solver=eg.TQL2), dict(path="split", unsorted=True)):
        z, w, info = eg.eigen_batch(a.clone(), **kw)
        assert int(info.abs().max()) == 0
        assert int(eg.check(a, w, z)[:, 3].max()) == 0
        assert (np.abs(np.sort(w.cpu().numpy().astype(np.float64), axis=1) - we) <= tol).all()
