"""CircuitBatch at the ends of what it takes: groups of circuits without layers,
and more circuits of one width than a grid's second axis holds."""
import numpy as np
import pytest
import torch

from quantumsim_amd.batch import CircuitBatch


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
