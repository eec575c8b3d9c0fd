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
