"""Circuits and layouts that fusion.apply_circuit's routes through the library must
leave alone or treat as the composition on the host does (quantumsim_amd.fusion)."""
import numpy as np
import pytest

from quantumsim_amd import _native as nat
from quantumsim_amd import fusion
from quantumsim_amd.fusion import CircuitPasses, _qubit_gates, fuse


class _Recorder:
    """Stands for a PauliVectorHIP of n qubits: keeps what is applied."""

    def __init__(self, n):
        self.n_qubits, self.dim_pauli = n, (4,) * n
        self.applied = []

    def apply_ptm(self, ptm, *qubits):
        self.applied.append((np.array(ptm), qubits))

    def run_passes(self, *arrays):
        return False


@pytest.fixture
def applied(monkeypatch):
    """What apply_circuit applies to a float32 vector of n qubits."""
    monkeypatch.setattr(fusion, '_native_circuit', lambda pv, gates: _qubit_gates(gates, pv.n_qubits))

    def call(n, gates, max_qudits=3):
        pv = _Recorder(n)
        count = fusion.apply_circuit(pv, gates, max_qudits)
        assert count == len(pv.applied)
        return pv.applied
    return call


@pytest.mark.parametrize('value', [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize('order', ['bad first', 'bad last', 'one qubit', 'same pair'])
def test_non_finite_ptms(applied, value, order):
    """0 * inf is not a number in every composed entry it enters, as in fuse()."""
    rng = np.random.default_rng(1)
    bad = rng.standard_normal((4,) * 4)
    bad[1, 1, 1, 1] = value
    diag = np.diag(rng.standard_normal(16)).reshape((4,) * 4)
    gates = {'bad first': [(bad, (0, 1)), (diag, (1, 2))],
             'bad last': [(diag, (1, 2)), (bad, (0, 1))],
             'one qubit': [(bad, (0, 1)), (np.diag(rng.standard_normal(4)), (1,))],
             'same pair': [(bad, (0, 1)), (diag, (0, 1))]}[order]
    with np.errstate(invalid='ignore'):
        ref = fuse(gates, [4] * 4, 3)
        got = applied(4, gates)
    assert [q for _, q in got] == [f.qudits for f in ref]
    for (p, _), f in zip(got, ref):
        np.testing.assert_array_equal(np.isnan(p), np.isnan(f.ptm))
        np.testing.assert_array_equal(np.isinf(p), np.isinf(f.ptm))


@pytest.mark.parametrize('max_qudits', [float('inf'), 2.5, 4.0])
def test_bound_of_any_number(applied, max_qudits):
    rng = np.random.default_rng(2)
    gates = [(rng.standard_normal((4,) * 4), (q, q + 1)) for q in (0, 2, 1)]
    ref = fuse(gates, [4] * 4, max_qudits)
    got = applied(4, gates, max_qudits)
    assert [q for _, q in got] == [f.qudits for f in ref]
    for (p, _), f in zip(got, ref):
        np.testing.assert_allclose(p, f.ptm, rtol=0, atol=1e-12)


def test_targets_of_any_iterable(applied):
    """Targets are read once, as fuse() reads them."""
    rng = np.random.default_rng(3)
    qs = [(0, 1), (2, 3), (1, 2)]
    ptms = [rng.standard_normal((4,) * 4) for _ in qs]
    ref = fuse(list(zip(ptms, qs)), [4] * 4, 3)
    for third in (rng.standard_normal((4,) * 4), rng.standard_normal((4,) * 6)):
        tail = tuple(range(third.ndim // 2))
        got = applied(4, iter([(p, iter(q)) for p, q in zip(ptms + [third], qs + [tail])]))
        ref = fuse(list(zip(ptms + [third], qs + [tail])), [4] * 4, 3)
        assert [q for _, q in got] == [f.qudits for f in ref]


@pytest.mark.parametrize('strides', [[128, 32, 8], [512, 128, 16], [32, 8, 2], [16, 8, 1]])
def test_strides_without_a_unit_axis_are_refused(strides):
    """The passes read pairs of neighbouring entries: the innermost axis has
    stride 1 (and no axis overlaps another)."""
    rng = np.random.default_rng(0)
    arrays = _qubit_gates([(rng.standard_normal((4,) * 4), (0, 1))], 3)
    with pytest.raises((NotImplementedError, ValueError)):
        CircuitPasses(3, strides, *arrays)


@pytest.mark.parametrize('n,pad_from', [(4, 2), (5, 2), (7, 3), (9, 5), (10, 4)])
def test_replay_of_padded_layouts(n, pad_from):
    """Axes from some on padded by 4 KB, as large vectors have them."""
    from test_circuit_passes import _apply, _circuit, _strides
    rng = np.random.default_rng(30 * n)
    for kind in ('brick', 'random'):
        gates = _circuit(n, kind, rng)
        x = rng.standard_normal((4,) * n)
        strides, extent = _strides(n, pad_from, 512)
        assert extent > x.size
        phys = np.full(extent, np.nan)
        view = np.lib.stride_tricks.as_strided(phys, x.shape, [8 * s for s in strides])
        view[...] = x
        plan = CircuitPasses(n, strides, *_qubit_gates(gates, n))
        nat.check(nat.lib().qsv_emulate_circuit(plan.handle, phys.ctypes.data_as(nat._c_f64p)),
                  'run')
        # 16 products and sums per gate, each within half an ulp of a norm that
        # the gates keep
        ref = _apply(x, gates)
        assert np.linalg.norm(view - ref) <= 32 * len(gates) * 2.0 ** -53 * np.linalg.norm(x)
        assert np.isnan(phys).sum() == extent - x.size


def _pairs(kind, n, count):
    m = n // 2
    pairs = {'triples': [(0, 1), (m, m + 1), (1, 2), (m + 1, m + 2)],
             'chain of triples': [t for b in range(0, n - 2, 3) for t in ((b, b + 1), (b + 1, b + 2))],
             'brick': [(q, q + 1) for p in (0, 1) for q in range(p, n - 1, 2)]}[kind]
    return [pairs[i % len(pairs)] for i in range(count)]


# ms a call on float64 vectors, in passes and in blocks of up to three qubits (14 and
# 15 qubits: 2 and 8 GB; 11 qubits: 32 MB)
@pytest.mark.parametrize('kind,n,count,passes_ms,blocks_ms', [
    ('triples', 14, 24, 4.19, 1.89), ('triples', 14, 200, 31.2, 2.94),
    ('triples', 15, 64, 40.2, 7.31), ('chain of triples', 15, 80, 50.8, 18.0),
    ('chain of triples', 14, 200, 31.2, 4.23), ('brick', 14, 60, 13.0, 28.2),
    ('brick', 15, 60, 57.1, 112.0), ('brick', 13, 60, 3.70, 7.49),
    ('triples', 11, 200, 1.07, 2.13), ('triples', 9, 64, 0.33, 0.74),
    ('triples', 13, 200, 8.24, 2.33), ('chain of triples', 9, 200, 0.85, 2.18)])
def test_many_gates_in_few_blocks_stay_blocks(monkeypatch, kind, n, count, passes_ms, blocks_ms):
    """A pass pays for every two-qubit gate, a dense block only once."""
    monkeypatch.setattr(fusion, '_native_circuit', lambda pv, gates: _qubit_gates(gates, pv.n_qubits))
    rng = np.random.default_rng(0)
    ptm = rng.standard_normal((4,) * 4)

    class Vector(_Recorder):
        def run_passes(self, ks, targets, ptms, worth=None):
            plan = CircuitPasses(n, [4 ** (n - 1 - q) for q in range(n)], ks, targets, ptms)
            self.taken = worth is None or worth(plan)
            return self.taken
    pv = Vector(n)
    fusion.apply_circuit(pv, [(ptm, t) for t in _pairs(kind, n, count)], 3)
    assert pv.taken == (passes_ms < blocks_ms)
    assert bool(pv.applied) != pv.taken


@pytest.mark.gpu
def test_circuit_without_gates_copies():
    import torch
    n = 3
    empty = np.zeros(0, dtype=np.int32)
    plan = CircuitPasses(n, [16, 4, 1], empty, empty, np.zeros(0))
    assert plan.passes == 0
    x = torch.randn(64, dtype=torch.float64, device='cuda')
    y = torch.zeros_like(x)
    plan.run(x.data_ptr(), y.data_ptr(), None, torch.cuda.current_stream().cuda_stream or None)
    torch.cuda.synchronize()
    assert torch.equal(x, y)


def _host_vector(n):
    """A float64 vector of n qubits without its device memory."""
    import torch
    from quantumsim_amd import bases
    from quantumsim_amd.pauli_vectors import PauliVectorHIP
    pv = PauliVectorHIP.__new__(PauliVectorHIP)
    pv.bases = [bases.general(2)] * n
    pv._shape, pv._dtype = (4,) * n, torch.float64
    return pv


@pytest.mark.parametrize('where', ['class', 'subclass', 'instance'])
def test_replaced_apply_ptm_sees_every_block(monkeypatch, where):
    """apply_circuit goes by the vector's apply_ptm wherever that is not the
    library's own."""
    from quantumsim_amd.pauli_vectors import PauliVectorHIP
    rng = np.random.default_rng(5)
    gates = [(rng.standard_normal((4,) * 4), (q, q + 1)) for q in (0, 2, 1)]
    assert fusion._native_circuit(_host_vector(4), gates) is not None
    seen = []
    pv = _host_vector(4)
    if where == 'class':
        monkeypatch.setattr(PauliVectorHIP, 'apply_ptm', lambda self, p, *q: seen.append(q))
    elif where == 'subclass':
        pv.__class__ = type('Sub', (PauliVectorHIP,),
                            {'apply_ptm': lambda self, p, *q: seen.append(q)})
    else:
        pv.apply_ptm = lambda p, *q: seen.append(q)
    monkeypatch.setattr(PauliVectorHIP, 'run_passes', lambda self, *a: True)
    count = fusion.apply_circuit(pv, gates, 3)
    assert count == len(seen) and seen == [f.qudits for f in fuse(gates, [4] * 4, 3)]
