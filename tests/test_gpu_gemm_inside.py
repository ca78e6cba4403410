"""Tiles of the batched product that lie inside it take unclamped loads: shapes on
both sides of that rule, every transposition, leading dimensions above the rows.

Bound: K products accumulated one after the other, on both sides: |error| <=
(2 K + 4) eps |A| |B|.
"""
import pytest
import torch

import eigeng_batched as eg

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("kind", [eg.GEMM_F64, eg.GEMM_F32])
@pytest.mark.parametrize("ta,tb", [(0, 0), (1, 0), (0, 1), (1, 1)])
@pytest.mark.parametrize("M,N,K", [(64, 64, 32), (64, 128, 96), (128, 64, 64), (65, 64, 32), (64, 66, 32), (64, 64, 33),
                                   (64, 64, 48), (130, 130, 160)])
def test_both_sides_of_the_rule(kind, ta, tb, M, N, K):
    print(f"[gemm] kind={kind} ta={ta} tb={tb} M={M} N={N} K={K}", flush=True)
    dt = torch.float64 if kind == eg.GEMM_F64 else torch.float32
    batch, pad = 5, 3
    g = torch.Generator().manual_seed(M + N + K)
    a = torch.randn((batch, M if ta else K, (K if ta else M) + pad), generator=g, dtype=dt)
    b = torch.randn((batch, K if tb else N, (N if tb else K) + pad), generator=g, dtype=dt)
    a[:, :, -pad:] = float("nan")
    b[:, :, -pad:] = float("nan")
    c = torch.full((batch, N, M + pad), -7.0, dtype=dt, device=DEV)
    rc = eg.gemm_raw(kind, ta, tb, M, N, K, 1.0, a.to(DEV), a.shape[2], a[0].numel(), b.to(DEV), b.shape[2],
                     b[0].numel(), 0.0, None, 0, 0, c, M + pad, c[0].numel(), batch)
    torch.cuda.synchronize()
    assert rc == 0
    c = c.cpu()
    assert bool((c[:, :, M:] == -7.0).all())
    av, bv = a[:, :, :-pad].double(), b[:, :, :-pad].double()
    op_a = av if ta else av.transpose(1, 2).contiguous()          # M x K
    op_b = bv if tb else bv.transpose(1, 2).contiguous()          # K x N
    ref, mag = op_a @ op_b, op_a.abs() @ op_b.abs()
    err = (c[:, :, :M].transpose(1, 2).double() - ref).abs()
    # the reference itself rounds in float64
    assert bool((err <= (2 * K + 4) * torch.finfo(dt).eps * mag).all())
