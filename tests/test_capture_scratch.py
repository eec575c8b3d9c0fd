"""Scratch memory of captured launches: a graph holds addresses, so the buffers
that its launches use may not be the caches' (which replace a buffer by a larger one
and give the old one back); they come from the graph's own pool."""
import pytest
import torch

from quantumsim_amd import autograd
from quantumsim_amd.pauli_vectors import hip


@pytest.mark.parametrize('get,bufs', [
    (lambda n: autograd._Workspace.get(torch.device('cpu'), n), autograd._Workspace._bufs),
    (lambda n: autograd._Workspace.get(torch.device('cpu'), n, 'schedule'),
     autograd._Workspace._bufs),
    (lambda n: hip._Scratch.get(torch.device('cpu'), 'ptm', n), hip._Scratch._bufs)])
def test_captured_launches_use_no_cached_buffer(monkeypatch, get, bufs):
    class Stream:
        cuda_stream = 77
    capturing = [False]
    monkeypatch.setattr(torch.cuda, 'current_stream', lambda device=None: Stream)
    monkeypatch.setattr(torch.cuda, 'is_current_stream_capturing', lambda: capturing[0])
    monkeypatch.setattr(hip, '_raw_stream', lambda device: 77)
    before = dict(bufs)
    try:
        eager = get(1000)
        assert get(500) is eager
        kept = dict(bufs)
        capturing[0] = True
        for size in (500, 1000, 5000):
            t = get(size)
            assert t is not eager and t.numel() >= size
        assert {k: id(v) for k, v in bufs.items()} == {k: id(v) for k, v in kept.items()}
        capturing[0] = False
        assert get(1000) is eager
    finally:
        bufs.clear()
        bufs.update(before)


@pytest.mark.gpu
def test_replay_after_the_cached_buffer_grew():
    """A captured gradient of small PTMs, then one that needs more scratch on the
    same stream, with whatever was given back written over."""
    g = torch.Generator(device='cuda').manual_seed(0)
    mk = lambda *s: torch.randn(s, device='cuda', generator=g)
    x, w = mk(3, 4 ** 6), mk(3, 4 ** 6)
    P = (mk(3, 16, 16) / 4).requires_grad_()
    step = lambda: torch.autograd.grad(
        (autograd.apply(x, P, (4,) * 6, (1, 3)) * w).sum(), [P])
    stream = torch.cuda.Stream()
    graph, stream, out = autograd.capture_step(step, stream=stream)
    ref = step()[0].clone()
    with torch.cuda.stream(stream):
        X, Q = mk(40, 4 ** 8), (mk(40, 64, 64) / 8).requires_grad_()
        torch.autograd.grad(autograd.apply(X, Q, (4,) * 8, (1, 3, 5)).sum(), [Q])
    torch.cuda.synchronize()
    for rep in range(3):
        with torch.cuda.stream(stream):
            junk = [torch.full((1 << k,), 0x7f, dtype=torch.uint8, device='cuda')
                    for k in range(9, 24) for _ in range(4)]
        torch.cuda.synchronize()
        kept = [j.clone() for j in junk]
        with torch.cuda.stream(stream):
            graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out[0], ref), rep
        for a, b in zip(junk, kept):           # and the replay wrote over no one's memory
            assert torch.equal(a, b), rep
        del junk, kept
