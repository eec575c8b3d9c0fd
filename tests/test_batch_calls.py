"""CircuitBatch at the ends of what it takes: groups of circuits without layers,
and more circuits of one width than a grid's second axis holds."""
import numpy as np
import pytest
import torch

from quantumsim_amd import windows
from quantumsim_amd.autograd import cz_ptm
from quantumsim_amd.batch import CircuitBatch
from quantumsim_amd.workloads import damping_ptms, rotation_ptms


def _circuit(n, layers):
    g = np.random.default_rng(10 * n + layers)
    t1 = g.uniform(20, 40, n)
    return {'n': n, 'layers': layers, 'angles': g.uniform(0, 2 * np.pi, (layers, n, 2)),
            't1': t1, 't2': 0.5 * t1}


def _by_circuit(cb):
    out = {}
    for g, p in zip(cb.groups, cb.populations()):
        for b, i in enumerate(g.members):
            out[i] = p[b].detach()
    return [out[i] for i in sorted(out)]


@pytest.mark.gpu
@pytest.mark.parametrize('kw', [{}, {'fuse_qudits': 0}, {'block_kernel': False}])
@pytest.mark.parametrize('widths', [(4, 5), (8, 9)])
def test_circuits_without_layers(widths, kw):
    """A width all of whose circuits have no layer, beside one with layers."""
    if widths[0] == 8 and not kw:
        kw = {'persistent_kernel': True, 'block_kernel': False}
    cs = [_circuit(widths[0], 0), _circuit(widths[1], 3), _circuit(widths[0], 0)]
    got = _by_circuit(CircuitBatch(cs, dtype=torch.float64, **kw))
    for i in (0, 2):
        assert got[i][0] == 1 and got[i][1:].abs().max() == 0
    ref = _by_circuit(CircuitBatch(cs[1:2], dtype=torch.float64, **kw))
    assert torch.equal(got[1], ref[0])


@pytest.mark.parametrize('batch,n_windows', [(65537, 1), (1, 65537)])
def test_single_gates_of_many_circuits_and_windows(batch, n_windows):
    """The single gates of narrow circuits, replayed: D R of every layer."""
    g = np.random.default_rng(0)
    mk = lambda a: torch.tensor(a, dtype=torch.float64)
    rot = rotation_ptms(mk(g.uniform(0, 2 * np.pi, (batch, 2 * n_windows, 1, 2))))
    damp = damping_ptms(mk(g.uniform(20, 40, (batch, 1))), mk(g.uniform(10, 20, (batch, 1))))
    plan = windows.LayerGatePlan(1, n_windows, batch)
    out, _, _ = windows.emulate(plan, rot.numpy(), damp.numpy(),
                                np.ones((batch, n_windows), np.uint8),
                                cz_ptm(torch.device('cpu')).reshape(16, 16).numpy())
    ref = (damp[:, None] @ rot).numpy()                # [batch, layers, 1, 4, 4]
    for p, (_, D, off) in enumerate(plan.positions):
        got = out[off:off + n_windows * batch * 16].reshape(n_windows, batch, 4, 4)
        # four products of entries below 1
        np.testing.assert_allclose(got, ref[:, p::2, 0].transpose(1, 0, 2, 3), rtol=0,
                                   atol=8 * 2.0 ** -53)


@pytest.mark.gpu
def test_many_circuits_of_one_width():
    cs = [_circuit(1, 1 + i % 2) for i in range(65537)]
    cs[0], cs[-1] = _circuit(1, 3), _circuit(1, 4)
    got = _by_circuit(CircuitBatch(cs, dtype=torch.float64))
    for i in (0, 1, 2, 65535, 65536):
        assert torch.equal(got[i], _by_circuit(CircuitBatch([cs[i]], dtype=torch.float64))[0])


@pytest.mark.gpu
def test_a_circuit_of_many_layers():
    c = _circuit(1, 131073)
    got, = _by_circuit(CircuitBatch([c], dtype=torch.float64))
    mk = lambda a: torch.tensor(a, dtype=torch.float64)
    ptms = (damping_ptms(mk(c['t1'][None]), mk(c['t2'][None]))[0] @
            rotation_ptms(mk(c['angles']))).numpy()
    v = np.array([1.0, 0, 0, 0])
    for p in ptms[:, 0]:
        v = p @ v
    # each layer rounds four products; damping forgets all but the last few hundred
    # layers, which the bound does not use
    assert np.abs(got.cpu().numpy() / got.sum().item() - v[:2] / v[:2].sum()).max() <= \
        131073 * 8 * 2.0 ** -53
