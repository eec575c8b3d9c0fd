"""Circuits and layouts that fusion.apply_circuit's routes through the library must
leave alone or treat as the composition on the host does (quantumsim_amd.fusion)."""
import numpy as np
import pytest

from quantumsim_amd import fusion
from quantumsim_amd.fusion import _qubit_gates, fuse


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
