"""Every ordered pair of targets of the persistent circuits' in-place two-qubit
contraction (lanes and groups of orbits chosen by the targets' digits), at the
widths where groups, waves and lanes run out, one-qubit gates between them.

The PTMs are orthogonal, so |S| = 1 and |Y| = |w| throughout, and a gate adds
at most 17 units in the last place (sixteen products, the rounded PTM) times
the norm 4 of |P|: G gates leave 68 G u |w| on a population (|w| = 1) and on a
gradient entry, which is a product of the two.
"""
import numpy as np
import pytest
import torch

from oracle import bases as ob
from oracle.pauli_vector import PauliVectorNumpy
from quantumsim_amd import persistent

GATES = 12


def _program(n, rng):
    pairs = [(a, b) for a in range(n) for b in range(n) if a != b]
    rng.shuffle(pairs)
    circuits, pool, off = [], [], 0
    for i in range(0, len(pairs), GATES - 2):
        gates = []
        for targets in [(i % n,)] + [tuple(p) for p in pairs[i:i + GATES - 2]] + [(n - 1,)]:
            D = 4 ** len(targets)
            pool.append(np.linalg.qr(rng.standard_normal((D, D)))[0].ravel())
            gates.append((targets, off))
            off += D * D
        circuits.append((n, gates))
    return circuits, np.concatenate(pool)


@pytest.mark.parametrize('n', [2, 3, 4, 5, 7])
def test_all_pairs_on_the_host(n):
    rng = np.random.default_rng(n)
    circuits, pool = _program(n, rng)
    pops, _ = persistent.emulate(persistent.CircuitTable(circuits, pool.size), pool)
    ref = []
    for _, gates in circuits:
        o = PauliVectorNumpy([ob.general(2)] * n, force=True)
        for targets, off in gates:
            D = 4 ** len(targets)
            o.apply_ptm(pool[off:off + D * D].reshape([4] * (2 * len(targets))), *targets)
        ref.append(o.diagonal())
    assert np.abs(pops - np.concatenate(ref)).max() < 68 * GATES * 2.0 ** -53


@pytest.mark.gpu
@pytest.mark.parametrize('dtype,n', [(torch.float64, n) for n in (2, 3, 4, 5, 6)]
                         + [(torch.float32, n) for n in (2, 3, 4, 5, 6, 7)])
def test_all_pairs_on_the_gpu(dtype, n):
    rng = np.random.default_rng(n)
    circuits, pool = _program(n, rng)
    circuits.append((1, []))
    if n > 2:     # a narrower circuit beside it, and one without gates
        circuits.insert(0, (2, []))
    table = persistent.CircuitTable(circuits, pool.size, 'cuda')
    w = rng.standard_normal(table.pop_elems)
    ref, dref = persistent.emulate(table, pool, w)
    dev = torch.from_numpy(pool).cuda().requires_grad_()
    pops = persistent.run(dev, table, dtype)
    grad, = torch.autograd.grad(pops, dev, torch.from_numpy(w).cuda())
    tol = 68 * GATES * (2.0 ** -53 if dtype == torch.float64 else 2.0 ** -24)
    assert np.abs(pops.detach().cpu().numpy() - ref).max() < tol
    assert np.abs(grad.cpu().numpy() - dref).max() < 2 * tol * np.linalg.norm(w)
