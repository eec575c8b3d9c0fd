"""Rotation and damping PTMs of the layered circuits' parameters in one launch
(qsv_gate_params) against the tensor operations and their autograd.

A rotation entry is a chain of nine products of factors <= 1: 16 u apart at
most (u = 2^-53); a gradient entry sums at most 16 x 9 of them (64 u of the sum
of |dP|, pairwise cancellations included).  A damping entry is a few rounded
operations on numbers <= 1: 16 u.  Its gradients are three such terms times
2 t / T^2: 64 u of the sum of |dP| times that, the conditioning of 1 - gamma and
1 - lambda near 1 included.
"""
import ctypes

import numpy as np
import pytest
import torch

from quantumsim_amd import _native as nat
from quantumsim_amd import workloads as wl

U = 2.0 ** -53
T = wl.GATE_TIME * 1e6
SHAPES = [(1, 1, 1, 1), (3, 2, 3, 4), (2, 7, 8, 5), (5, 13, 13, 7), (1, 16, 16, 16), (4, 3, 3, 11)]


def _inputs(shape, device='cpu'):
    B, own, layers, n = shape
    rng = np.random.default_rng(sum(shape))
    mk = lambda a: torch.tensor(a, dtype=torch.float64, device=device)
    t1 = rng.uniform(20, 40, (B, n))
    return (mk(rng.uniform(0, 2 * np.pi, (B, own, n, 2))), mk(t1),
            mk(rng.uniform(0.4, 1.9, (B, n)) * t1),
            mk(rng.standard_normal((B, layers, n, 4, 4))), mk(rng.standard_normal((B, n, 4, 4))))


def _check(shape, rot, damp, grads, inputs):
    a, t1, t2, drot, ddamp = (x.cpu() for x in inputs)
    own, layers = shape[1], shape[2]
    leaves = [x.clone().requires_grad_() for x in (a, t1, t2)]
    rrot, rdamp = wl._gate_ptms_ops(*leaves, layers)
    ref = torch.autograd.grad((rrot, rdamp), leaves, (drot, ddamp))
    assert (rot.cpu() - rrot).abs().max() <= 16 * U
    assert (damp.cpu() - rdamp).abs().max() <= 16 * U
    bound = 64 * U * drot[:, :own].abs().sum((-2, -1))[..., None]
    assert ((grads[0].cpu() - ref[0]).abs() <= bound).all()
    for got, want, t in zip(grads[1:], ref[1:], (t1, t2)):
        bound = 64 * U * ddamp.abs().sum((-2, -1)) * 2 * T * (t1 ** -2 + t ** -2)
        assert ((got.cpu() - want).abs() <= bound).all()


@pytest.mark.parametrize('shape', SHAPES)
def test_host_replay(shape):
    B, own, layers, n = shape
    a, t1, t2, drot, ddamp = ins = _inputs(shape)
    coef, damp = a.new_empty((B, layers, n, 9)), torch.empty_like(ddamp)
    da, d1, d2 = (torch.full_like(x, float('nan')) for x in (a, t1, t2))
    terms = wl._rotation_terms(torch.device('cpu'))
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    nat.check(nat.lib().qsv_emulate_gate_params(
        B, layers, own, n, p(a), p(terms), p(coef), p(t1), p(t2), T, p(damp), p(drot), p(da),
        p(ddamp), p(d1), p(d2)), 'emulate_gate_params')
    _check(shape, (coef @ terms).reshape(drot.shape), damp, (da, d1, d2), ins)


@pytest.mark.gpu
@pytest.mark.parametrize('shape', SHAPES)
def test_device(shape):
    ins = _inputs(shape, 'cuda')
    # strided parameters are accepted
    a = ins[0].transpose(0, 1).contiguous().transpose(0, 1).requires_grad_()
    t1, t2 = ins[1].clone().requires_grad_(), ins[2].clone().requires_grad_()
    rot, damp = wl.gate_ptms(a, t1, t2, shape[2])
    grads = torch.autograd.grad((rot, damp), (a, t1, t2), ins[3:])
    _check(shape, rot.detach(), damp.detach(), grads, ins)


@pytest.mark.gpu
def test_second_derivative_and_single_precision():
    """A gradient that is differentiated again, parameters without gradients
    and float32 parameters go by the tensor operations' rules."""
    a, t1, t2, drot, ddamp = _inputs((2, 3, 4, 3), 'cuda')
    a.requires_grad_()
    assert not wl.gate_ptms(a, t1, t2)[1].requires_grad
    t1.requires_grad_()

    def second(f):
        rot, damp = f(a, t1, t2, 4)
        g, = torch.autograd.grad((rot, damp), a, (drot, ddamp), create_graph=True)
        return torch.autograd.grad((g ** 2).sum(), a)[0]
    got, want = second(wl.gate_ptms), second(wl._gate_ptms_ops)
    assert (got - want).abs().max() <= 1e-12 * want.abs().max()
    assert wl.gate_ptms(a.detach().float(), t1.detach().float(), t2.float())[0].dtype == torch.float32


@pytest.mark.gpu
def test_rates_without_kraus_operators_are_not_a_number():
    """T2 > 2 T1 and negative T1: not a number in every entry, as the Kraus
    sums give."""
    mk = lambda *v: torch.tensor([v], dtype=torch.float64, device='cuda')
    a = torch.zeros((1, 1, 3, 2), dtype=torch.float64, device='cuda')
    t1, t2 = mk(20., -3., 25.), mk(50., 10., 30.)
    damp = wl.gate_ptms(a, t1, t2)[1]
    ref = wl.damping_ptms(t1, t2)
    assert torch.equal(torch.isnan(damp), torch.isnan(ref))
