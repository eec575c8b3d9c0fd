"""Gate schedules at the ends of what run_schedule takes: gates named by numbers
that no table holds, and segments in which no state runs."""
import ctypes

import numpy as np
import pytest
import torch

from quantumsim_amd import _native as nat
from quantumsim_amd.autograd import run_schedule


@pytest.mark.parametrize('gate', [(0, 2 ** 31), (0, 2 ** 33), (2 ** 33, 0), (0, -2 ** 33),
                                  (0, 2 ** 70), (0, 3), (1, 0), (-1, 0)])
def test_gates_beyond_the_steps_are_refused(gate):
    x0 = torch.zeros((2, 16))
    steps = [torch.zeros((3, 2, 4, 4))]
    with pytest.raises(ValueError, match='outside the steps'):
        run_schedule(x0, steps, [(0,)], [(2, 0, [(0, 0), gate])], (4, 4))


@pytest.mark.parametrize('gates', [[(0, 0, 1), (0, 1, 2)], [(0,), (1,)], [0, 0, 0, 1],
                                   [(0, 0), (0,)]])
def test_gates_that_are_no_pairs_are_refused(gates):
    """Six numbers are not three gates."""
    x0 = torch.zeros((2, 16))
    steps = [torch.zeros((3, 2, 4, 4))] * 3
    with pytest.raises((TypeError, ValueError)):
        run_schedule(x0, steps, [(0,)] * 3, [(2, 0, gates)], (4, 4))


@pytest.mark.parametrize('dtype', [nat.QSV_F32, nat.QSV_F64])
@pytest.mark.parametrize('fused', [0, 1])
def test_no_running_state(dtype, fused):
    """Segments without states launch nothing, gradients included; the adjoint's
    buffers change places gate by gate all the same."""
    L, n = nat.lib(), 7
    dims = nat.i64([4] * n)
    rows = (nat.SchedPos * 1)()
    r = rows[0]
    r.k, r.n_steps, r.fused, r.targets[:3] = 3, 3, fused, (1, 2, 4)
    r.ptm = r.ptm_t = r.grad_ptm = 4096
    r.step, r.state, r.workspace = 64 * 64, 64 * 64, 0
    gates = np.array([(0, 0), (0, 1), (0, 2)], dtype=np.int32)
    ptrs = (ctypes.c_void_p * 3)(4096, 4096, 8192)
    assert L.qsv_schedule_forward(dtype, n, dims, 1, rows, 0, 3, gates.ctypes.data, 4096, ptrs,
                                  nat.SchedHook(), None) == 0
    for every in (1, 2, 3):
        cur = ctypes.c_int32(7)
        assert L.qsv_schedule_backward(dtype, n, dims, 1, rows, 0, 3, gates.ctypes.data, every,
                                       ptrs, ptrs, ptrs, 0, 4096, 0, ctypes.byref(cur),
                                       nat.SchedHook(), None) == 0
        assert cur.value == 1


def test_schedule_without_positions_under_a_ledger():
    from quantumsim_amd.ledger import Ledger
    x0 = torch.ones((2, 16), requires_grad=True)
    with Ledger(timed=False):
        out = run_schedule(x0, [], [], [(2, 1, []), (1, 0, [])], (4, 4))
        gx, = torch.autograd.grad(out.sum(), [x0])
    assert torch.equal(out, x0) and torch.equal(gx, torch.ones_like(x0))
