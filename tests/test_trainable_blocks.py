"""TrainableCircuit's blocks built by the library (workloads.TrainableCircuit
with blocks of three qubits): what the route keeps alive, and the calls it must
take or leave to the composed gates.  CPU tests run the launches' replays in
place of the kernels."""
import ctypes

import numpy as np
import pytest
import torch

from quantumsim_amd import _native as nat
from quantumsim_amd import windows
from quantumsim_amd.workloads import TrainableCircuit

# float64 products of at most eight 64 x 64 factors of row sums below 2
TOL = 8 * 64 * 2 * 2.0 ** -52


class _HostLib:
    """The library with the block kernels' launches replayed on host memory."""

    def __init__(self):
        self._lib = nat.lib()

    def __getattr__(self, name):
        return getattr(self._lib, name)

    def qsv_put(self, host, nbytes, dst, stream):
        ctypes.memmove(dst, host, nbytes)
        return 0

    def qsv_layer_blocks(self, dtype, n_pos, table, table_dev, batch, n, layers, rot, damp, cz,
                         out, out_elems, stream):
        p = lambda a: ctypes.cast(a, nat._c_f64p)
        return self._lib.qsv_emulate_layer_blocks(n_pos, table_dev, batch, n, layers, p(rot),
                                                  p(damp), p(cz), p(out), out_elems, None, None,
                                                  None)


@pytest.fixture
def host_lib(monkeypatch):
    lib = _HostLib()
    monkeypatch.setattr(nat, 'lib', lambda: lib)
    monkeypatch.setattr(windows, '_stream', lambda: None)


def _tensors(obj, seen=None):
    """Tensors reachable from an object's attributes and containers."""
    seen = set() if seen is None else seen
    if id(obj) in seen:
        return []
    seen.add(id(obj))
    if isinstance(obj, torch.Tensor):
        return [obj]
    if isinstance(obj, dict):
        return [t for kv in obj.items() for o in kv for t in _tensors(o, seen)]
    if isinstance(obj, (list, tuple, set)):
        return [t for o in obj for t in _tensors(o, seen)]
    return _tensors(vars(obj), seen) if hasattr(obj, '__dict__') else []


def _params(tc, sets, device='cpu'):
    return tc.initial_params(sets, seed=4, device=device, dtype=torch.float64)


def test_circuit_object_owns_no_device_memory(host_lib):
    """Captured launches hold device addresses: none of them may belong to the
    circuit, which the caller is free to drop or to use with other set counts."""
    tc = TrainableCircuit(n=5, layers=7)
    for sets in (1, 2):
        ang, t1, t2 = _params(tc, sets)
        got = tc._blocks(ang, t1, t2, torch.float64)
        ref = tc.gates(ang, t1, t2, 3)
        assert [g.targets for g in got] == [g.targets for g in ref]
        for a, b in zip(got, ref):
            assert (a.ptm - b.ptm).abs().max() <= TOL
    assert not _tensors(tc)


@pytest.mark.gpu
def test_captured_step_outlives_its_circuit():
    """Replays of a step whose circuit is gone, after nine other set counts and
    with the freed memory written over, equal the eager step."""
    from quantumsim_amd.autograd import capture_step

    def make():
        tc = TrainableCircuit(n=6, layers=8)
        params = [p.requires_grad_() for p in _params(tc, 4, 'cuda')]
        target = torch.full((4, 64), 1 / 64, dtype=torch.float64, device='cuda')

        def step():
            p = tc.populations(*params, torch.float32, checkpoint_every=4, fuse_qudits=3)
            return torch.autograd.grad(tc.kl(target, p).sum(), params)
        # the parameters and the target are the graph's inputs: the caller's to keep
        return capture_step(step) + ([g.clone() for g in step()], params, target)

    graph, stream, out, ref, *inputs = make()
    other = TrainableCircuit(n=6, layers=8)
    for sets in range(5, 14):
        other.populations(*_params(other, sets, 'cuda'), torch.float32, fuse_qudits=3)
    del other
    torch.cuda.synchronize()
    for rep in range(3):
        # whatever the allocator has back is handed out and written over
        junk = [torch.full((size,), 0x7f, dtype=torch.uint8, device='cuda')
                for size in (512, 2048, 4096, 8192, 1 << 16, 1 << 20) for _ in range(16)]
        torch.cuda.synchronize()
        del junk
        with torch.cuda.stream(stream):
            graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(out, ref):
            assert torch.equal(a, b), rep


@pytest.mark.parametrize('which', [(0, 1, 2), (0, -1, 1)])
def test_missing_rotation_set_is_refused(host_lib, which):
    """The layer map indexes the rotation sets on the device, where nothing
    checks it."""
    plan = windows.LayerBlockPlan(3, 3, 2)
    rot = torch.zeros((2, 2, 3, 4, 4), dtype=torch.float64)
    damp = torch.zeros((2, 3, 4, 4), dtype=torch.float64)
    cz = torch.zeros((16, 16), dtype=torch.float64)
    with pytest.raises(IndexError, match='rotation set'):
        windows.layer_blocks(rot, damp, plan, torch.float64, cz, which)


def test_fewer_rotation_sets_than_blocks(host_lib):
    tc = TrainableCircuit(n=4, layers=12, block=4, n_blocks=3)
    ang, t1, t2 = _params(tc, 2)
    for make in (lambda a: tc.gates(a, t1, t2, 3), lambda a: tc._blocks(a, t1, t2, torch.float64)):
        with pytest.raises(IndexError):
            make(ang[:, :2].contiguous())


@pytest.fixture
def gates_of(host_lib, monkeypatch):
    """The gates that populations() hands to run_circuit, on host tensors."""
    from quantumsim_amd import autograd
    seen = []

    def run_circuit(x0, gates, shape, checkpoint_every):
        seen.append(gates)
        return x0
    monkeypatch.setattr(autograd, 'run_circuit', run_circuit)
    monkeypatch.setattr(autograd, 'diagonal', lambda x, bases: x)
    # the library's route is for tensors on a device; the replay takes host ones
    monkeypatch.setattr(TrainableCircuit, '_on_device', staticmethod(lambda *t: True),
                        raising=False)

    def call(tc, ang, t1, t2):
        tc.populations(ang, t1, t2, torch.float64, fuse_qudits=3)
        return seen.pop()
    return call


def _same_gates(got, ref):
    assert [g.targets for g in got] == [g.targets for g in ref]
    for a, b in zip(got, ref):
        assert a.ptm.shape == b.ptm.shape
        # float64 products of up to 80 factors of row sums below 2, damped
        assert ((a.ptm - b.ptm).abs() <= 10 * TOL).all()


@pytest.mark.parametrize('n,layers', [(1, 9), (1, 40), (2, 6), (2, 40), (3, 5), (3, 40), (4, 40),
                                      (5, 0), (4, 1), (6, 12)])
def test_every_width_and_depth(gates_of, n, layers):
    """Few qubits put all the layers' gates into one block."""
    tc = TrainableCircuit(n=n, layers=layers)
    for sets in (0, 1, 3):
        p = _params(tc, sets)
        _same_gates(gates_of(tc, *p), tc.gates(*p, 3))


@pytest.mark.gpu
@pytest.mark.parametrize('n,layers', [(1, 40), (2, 6), (3, 5), (3, 40), (4, 40)])
def test_populations_of_few_qubits(n, layers):
    """Populations and gradients in blocks against one gate at a time, float64."""
    tc = TrainableCircuit(n=n, layers=layers)
    out = []
    for fuse in (3, 0):
        p = [t.requires_grad_() for t in _params(tc, 2, 'cuda')]
        pops = tc.populations(*p, torch.float64, fuse_qudits=fuse)
        w = torch.linspace(-1, 1, pops.numel(), dtype=torch.float64, device='cuda').view_as(pops)
        out.append([pops.detach()] + list(torch.autograd.grad((pops * w).sum(), p)))
    for a, b in zip(*out):
        # up to 2 x 40 applications, 64 products of entries below 2 each
        assert (a - b).abs().max().item() <= 80 * 64 * 2 * 2.0 ** -52 * max(1.0, b.abs().max().item())


def test_shared_and_wider_parameters(gates_of):
    """What the composition broadcasts or ignores: T1 and T2 or angles shared by
    the sets, parameters of more qubits, sets or layers of angles than are used."""
    tc = TrainableCircuit(n=4, layers=7)
    ang, t1, t2 = _params(tc, 3)
    wide = TrainableCircuit(n=5, layers=7, n_blocks=4)
    wang, w1, w2 = _params(wide, 3)
    for p in [(ang, t1[:1], t2[:1]), (ang[:1], t1, t2), (ang[:1], t1[:1], t2[:1]),
              (wang, w1, w2), (ang, w1, w2), (wang, t1, t2),
              (ang.transpose(0, 1).contiguous().transpose(0, 1), t1, t2)]:
        _same_gates(gates_of(tc, *p), tc.gates(*p, 3))


def test_overridden_gates_are_used(gates_of):
    """gates() is the circuit's definition: a subclass's or an instance's own is
    what populations() runs."""
    class Reversed(TrainableCircuit):
        def gates(self, ang, t1, t2, fuse_qudits=0):
            return super().gates(ang, t1, t2, fuse_qudits)[::-1]

    tc = Reversed(n=4, layers=7)
    p = _params(tc, 2)
    _same_gates(gates_of(tc, *p), tc.gates(*p, 3))
    tc = TrainableCircuit(n=4, layers=7)
    plain = tc.gates(*p, 3)
    tc.gates = lambda ang, t1, t2, fuse_qudits=0: plain[:2]
    _same_gates(gates_of(tc, *p), plain[:2])

    class Renamed(TrainableCircuit):         # the same gates: either route
        pass
    _same_gates(gates_of(Renamed(n=4, layers=7), *p), plain)


def test_gates_replaced_on_the_class_are_used(gates_of, monkeypatch):
    tc = TrainableCircuit(n=4, layers=7)
    p = _params(tc, 2)
    plain = tc.gates(*p, 3)
    monkeypatch.setattr(TrainableCircuit, 'gates',
                        lambda self, ang, t1, t2, fuse_qudits=0: plain[:2])
    _same_gates(gates_of(tc, *p), plain[:2])
