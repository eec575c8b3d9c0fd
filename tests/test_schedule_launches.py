"""The gate schedule's launches issued segment by segment from the library
(qsv_schedule_forward / _backward): the same bits as the single launches in the
same order, for every checkpoint interval, positions without gradients, empty
segments, states off the 16-byte grid, qutrits among the qubits and one state; the
ledger sees the same launches.
"""
import ctypes

import numpy as np
import pytest
import torch

from quantumsim_amd import _native as nat

SHAPES = [((4, 4, 4, 4, 4, 4), [(0, 1), (5,), (1, 2, 3), (3, 4, 5)]),
          ((9, 4, 9, 4), [(0, 1), (2,), (3, 1)])]


def test_gates_outside_the_steps_are_refused():
    L = nat.lib()
    rows = (nat.SchedPos * 1)()
    rows[0].k, rows[0].n_steps = 1, 2
    one = (ctypes.c_void_p * 2)(1, 1)
    cur = ctypes.c_int32(0)
    for gate in [(1, 0), (-1, 0), (0, 2), (0, -1)]:
        g = np.array(gate, dtype=np.int32)
        assert L.qsv_schedule_forward(nat.QSV_F32, 2, nat.i64([4, 4]), 1, rows, 1, 1,
                                      g.ctypes.data, 1, one, nat.SchedHook(), None) == -1
        assert L.qsv_schedule_backward(nat.QSV_F32, 2, nat.i64([4, 4]), 1, rows, 1, 1,
                                       g.ctypes.data, 1, one, one, one, 0, 1, 1,
                                       ctypes.byref(cur), nat.SchedHook(), None) == -1


def _case(shape, targets, B, dtype, skew, grad_steps):
    rng = np.random.default_rng(len(shape) + B)
    N = int(np.prod(shape))
    mk = lambda *s: torch.tensor(rng.standard_normal(s), dtype=dtype, device='cuda')
    dims = [int(np.prod([shape[q] for q in t])) for t in targets]
    steps = [(mk(3, B, D, D) / D ** 0.5).requires_grad_(g) for D, g in zip(dims, grad_steps)]
    x0 = mk(B * N + skew)[skew:].view(B, N).requires_grad_()
    P = len(targets)
    every = [(p, w) for w in range(3) for p in range(P)]
    if B == 1:
        segments = [(1, 1, []), (1, 0, every)]
    else:
        segments = [(B, B - 1, every[:P + 1]), (B - 1, B - 1, []), (B - 1, 1, every[P + 1:-1]),
                    (1, 0, every[-1:])]
    return x0, steps, segments, mk(B, N)


def _single_launches(x0, steps, targets, segments, shape, w):
    """Every gate by its own calls; the gradients the same way."""
    from quantumsim_amd.autograd import _apply_raw, _fused_backward_raw, _ptm_grad_raw
    dims = [[shape[q] for q in t] for t in targets]
    x, xs, finals = x0.detach(), [], torch.empty_like(w)
    with torch.no_grad():
        for active, nxt, gates in segments:
            for p, s in gates:
                xs.append(x)
                x = _apply_raw(x, steps[p][s], shape, targets[p], dims[p])
            finals[nxt:active] = x[nxt:]
            x = x[:nxt]
        grads = [torch.zeros_like(t) for t in steps]
        gy = torch.empty((0, w.shape[1]), dtype=w.dtype, device=w.device)
        for active, nxt, gates in reversed(segments):
            gy = torch.cat([gy, w[nxt:active]])
            for p, s in reversed(gates):
                xg, done = xs.pop(), None
                if steps[p].requires_grad and w.dtype == torch.float32:
                    done = _fused_backward_raw(xg, gy, steps[p][s], shape, targets[p],
                                               gp_out=grads[p][s])
                if done is not None:
                    gy = done[0]
                    continue
                if steps[p].requires_grad:
                    _ptm_grad_raw(xg, gy, shape, targets[p], dims[p], out=grads[p][s])
                gy = _apply_raw(gy, steps[p][s].transpose(1, 2), shape, targets[p], dims[p])
    return finals, gy, grads


@pytest.mark.gpu
@pytest.mark.parametrize('dtype', [torch.float32, torch.float64])
@pytest.mark.parametrize('B,k,skew,frozen', [(3, 1, 0, ()), (3, 2, 0, (0,)), (4, 3, 1, ()),
                                             (1, 5, 0, (1, 2)), (3, 100, 0, ())])
@pytest.mark.parametrize('shape,targets', SHAPES)
def test_same_bits_as_single_launches(shape, targets, B, k, skew, frozen, dtype):
    from quantumsim_amd.autograd import run_schedule
    from quantumsim_amd.ledger import Ledger
    x0, steps, segments, w = _case(shape, targets, B, dtype, skew,
                                   [p not in frozen for p in range(len(targets))])
    print(shape, B, k, skew, frozen, dtype, flush=True)
    inputs = [x0] + [t for t in steps if t.requires_grad]
    out = run_schedule(x0, steps, targets, segments, shape, k)
    got = torch.autograd.grad((out * w).sum(), inputs)
    ref, gx, grads = _single_launches(x0, steps, targets, segments, shape, w)
    assert torch.equal(out, ref)
    assert torch.equal(got[0], gx)
    for a, b in zip(got[1:], [g for g, t in zip(grads, steps) if t.requires_grad]):
        assert torch.equal(a, b)
    with Ledger(timed=False) as one:
        _single_launches(x0, steps, targets, segments, shape, w)
    with Ledger(timed=False) as led:
        torch.autograd.grad((run_schedule(x0, steps, targets, segments, shape, 1) * w).sum(),
                            inputs)
    assert {f: tuple(r[:2]) + (r[3],) for f, r in led.rows.items()} == \
        {f: tuple(r[:2]) + (r[3],) for f, r in one.rows.items()}
