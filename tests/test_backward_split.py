"""The float32 one-pass backward of dense 64 x 64 blocks with its block groups
split into runs of whole float32 partial sums: groups of unequal length, a run
past the end, one and several states, both geometries (innermost axis a
bystander, or a target).

float32 sums run over at most 8 tiles of 32 orbits, so a dP entry is within
256 u (u = 2^-24) of sum |ybar| |x|, and one u for the result; xbar sums 64 products.
"""
import numpy as np
import pytest
import torch

from quantumsim_amd import _native as nat
from test_kernel_indexing import emulate_backward


@pytest.mark.parametrize('targets', [(1, 2, 4), (2, 6, 7)])
@pytest.mark.parametrize('blocks', [1, 3, 5])
def test_host_replay(targets, blocks, rng):
    n = 8 if targets == (2, 6, 7) else 9
    x, ybar = rng.standard_normal((2,) + (4,) * n)
    P = rng.standard_normal((64, 64))
    xbar, dp = emulate_backward(nat.QSV_F32, x, ybar, P, targets, blocks)
    mx, my = (np.moveaxis(a, targets, (0, 1, 2)).reshape(64, -1) for a in (x, ybar))
    got = np.moveaxis(xbar, targets, (0, 1, 2)).reshape(64, -1)
    assert np.allclose(got, P.T @ my, rtol=1e-12, atol=1e-11)
    assert np.allclose(dp, my @ mx.T, rtol=1e-12, atol=1e-10)


@pytest.mark.gpu
@pytest.mark.parametrize('targets', [(1, 4, 7), (5, 9, 10)])
@pytest.mark.parametrize('batch', [1, 3, 6])
def test_against_float64(targets, batch):
    from quantumsim_amd.autograd import _fused_backward_raw
    n = 11
    g = torch.Generator(device='cuda').manual_seed(batch)
    x, ybar = torch.randn((2, batch) + (4,) * n, device='cuda', generator=g)
    P = torch.randn((batch, 64, 64), device='cuda', generator=g) / 8
    print(targets, batch, flush=True)
    gx, gp = _fused_backward_raw(x.view(batch, -1), ybar.view(batch, -1), P, (4,) * n, targets)
    at = [t + 1 for t in targets]
    rest = [i for i in range(n + 1) if i not in at and i != 0]
    u = 2.0 ** -24
    for b in range(batch):
        mx, my, mg = (a[b].permute([i - 1 for i in at + rest]).reshape(64, -1).double()
                      for a in (x, ybar, gx.view(x.shape)))
        ref = my @ mx.t().contiguous()
        assert ((gp[b].double() - ref).abs() <= 257 * u * (my.abs() @ mx.abs().t().contiguous())
                ).all()
        Pt = P[b].double().t().contiguous()
        assert ((mg - Pt @ my).abs() <= 65 * u * (Pt.abs() @ my.abs())).all()
