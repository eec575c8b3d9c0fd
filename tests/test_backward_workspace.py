"""Workspace of the gradients of dense 64 x 64 blocks: what
qsv_ptm_grad_workspace_bytes names is enough for both backwards, for any caller
that sized its buffer by it, and the one-pass float32 backward uses more only
where it is given (qsv_batched_backward_workspace_bytes)."""
import numpy as np
import pytest
import torch

from quantumsim_amd import _native as nat

TILE_BYTES = 64 * 64 * 8


def _grad_bytes(batch, n, targets):
    return nat.lib().qsv_ptm_grad_workspace_bytes(batch, n, nat.i64([4] * n), 3,
                                                  nat.i32(targets), nat.i32([4] * 3))


def test_gradient_workspace():
    """64 blocks a state (csrc/qsv_grad.hip, kGrad64Blocks), in either type."""
    for n in (6, 8, 11, 12):
        for batch in (0, 1, 2, 6, 40):
            for targets in ([0, 1, 2], [n - 3, n - 2, n - 1]):
                assert _grad_bytes(batch, n, targets) == 64 * batch * TILE_BYTES


def test_backward_workspace():
    L = nat.lib()
    for n, batch in [(11, 1), (11, 6), (9, 40)]:
        ask = lambda code: L.qsv_batched_backward_workspace_bytes(
            code, batch, n, nat.i64([4] * n), 3, nat.i32([1, 4, 7]))
        assert ask(nat.QSV_F64) == _grad_bytes(batch, n, [1, 4, 7])
        assert ask(nat.QSV_F32) == max(1024, 64 * batch) * TILE_BYTES
    assert L.qsv_batched_backward_workspace_bytes(nat.QSV_F32, 1, 11, nat.i64([4] * 11), 3,
                                                  nat.i32([1, 4, 11])) < 0


@pytest.mark.gpu
@pytest.mark.parametrize('targets', [(1, 4, 7), (6, 9, 10)])
@pytest.mark.parametrize('batch', [1, 3])
def test_backward_in_any_workspace(targets, batch):
    """The smaller workspace and the larger one against float64."""
    L, n = nat.lib(), 11
    g = torch.Generator(device='cuda').manual_seed(batch)
    x, ybar = torch.randn((2, batch, 4 ** n), device='cuda', generator=g)
    P = torch.randn((batch, 64, 64), device='cuda', generator=g) / 8
    dims, tg = nat.i64([4] * n), nat.i32(targets)
    sizes = [_grad_bytes(batch, n, list(targets)),
             L.qsv_batched_backward_workspace_bytes(nat.QSV_F32, batch, n, dims, 3, tg)]
    at = [t + 1 for t in targets]
    order = [0] + at + [i for i in range(1, n + 1) if i not in at]
    mx, my = (a.view((batch,) + (4,) * n).permute(order).reshape(batch, 64, -1).double()
              for a in (x, ybar))
    u = 2.0 ** -24
    out = []
    for size in sizes:
        print(targets, batch, size, flush=True)
        ws = torch.empty(size, dtype=torch.uint8, device='cuda')
        gx, gp = torch.empty_like(x), torch.empty_like(P)
        nat.check(L.qsv_apply_ptm_batched_backward(
            nat.QSV_F32, x.data_ptr(), ybar.data_ptr(), gx.data_ptr(), batch, n, dims, 3, tg,
            P.data_ptr(), 64 * 64, gp.data_ptr(), 0, ws.data_ptr(), size,
            torch.cuda.current_stream().cuda_stream or None), 'backward')
        # float32 sums of at most 256 products, then float64, one rounding
        for b in range(batch):
            mxt = mx[b].t().contiguous()
            assert ((gp[b].double() - my[b] @ mxt).abs()
                    <= 257 * u * (my[b].abs() @ mxt.abs())).all()
        out.append(gx)
    assert torch.equal(*out)
    short = torch.empty(TILE_BYTES, dtype=torch.uint8, device='cuda')
    assert L.qsv_apply_ptm_batched_backward(
        nat.QSV_F32, x.data_ptr(), ybar.data_ptr(), gx.data_ptr(), batch, n, dims, 3, tg,
        P.data_ptr(), 64 * 64, gp.data_ptr(), 0, short.data_ptr(), TILE_BYTES, None) == -1


def test_gradient_blocks_of_many_small_states():
    """Launch shapes of the gradients of 1- and 2-qubit PTMs of many 7-qubit states:
    1024 orbits a block, fewer where few states leave the chip idle.  A float64
    state of two qubits' 1024 orbits is not split in two (512 states: 34.8 us
    against 28.5), in three it gains (340 states: 20.7 against 23.6); float32 gains
    from two (18.1 against 25.3)."""
    L = nat.lib()
    ask = lambda code, batch: L.qsv_ptm_grad_blocks(
        code, batch, 7, nat.i64([4] * 7), 2, nat.i32([0, 1]), nat.i32([4, 4]))
    for batch, f64, f32 in [(1, 16, 16), (128, 8, 8), (340, 3, 3), (400, 1, 2), (512, 1, 2),
                            (600, 1, 1)]:
        assert (ask(nat.QSV_F64, batch), ask(nat.QSV_F32, batch)) == (f64, f32), batch
