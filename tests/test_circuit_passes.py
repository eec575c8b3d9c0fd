"""Circuits applied in passes of several gates (fusion.apply_circuit,
csrc/qsv_slab.hip): the passes' replay on the CPU and the kernel on the GPU
against gate-by-gate application in float64; the block count against
fusion.fuse."""
import numpy as np
import pytest

from quantumsim_amd import _native as nat
from quantumsim_amd.fusion import CircuitPasses, QubitBlocks, _qubit_gates, apply_circuit, fuse


def _contraction(k, rng):
    """A random PTM of spectral norm 1: magnitudes stay within the vector's."""
    D = 4 ** k
    q, _ = np.linalg.qr(rng.standard_normal((D, D)))
    return q.reshape((4,) * (2 * k))


def _circuit(n, kind, rng):
    if kind == 'brick':
        gates = []
        for layer in range(5):
            gates += [(_contraction(1, rng), (q,)) for q in range(n)]
            gates += [(_contraction(2, rng), (q, q + 1)) for q in range(layer % 2, n - 1, 2)]
            gates += [(_contraction(1, rng), (q,)) for q in range(n)]
        return gates
    if kind == 'random':         # any pairs in either order, repeats, lone qubits
        gates = []
        for _ in range(5 * n):
            k = int(rng.integers(1, 3))
            q = rng.choice(n, k, replace=False)
            gates.append((_contraction(k, rng), tuple(int(t) for t in q)))
        return gates
    # single-qubit gates only, on some of the qubits
    return [(_contraction(1, rng), (q,)) for q in range(0, n, 2) for _ in range(2)]


def _apply(x, gates):
    n = x.ndim
    for p, qs in gates:
        k = len(qs)
        lo = list(range(n))
        for j, q in enumerate(qs):
            lo[q] = n + j
        x = np.einsum(p, [n + j for j in range(k)] + list(qs), x, list(range(n)), lo)
    return x


def _strides(n, pad_from, pad):
    st, acc = [0] * n, 1
    for q in reversed(range(n)):
        st[q] = acc + (pad if n - 1 - q >= pad_from else 0)
        acc = st[q] * 4
    return st, acc


@pytest.mark.parametrize('kind', ['brick', 'random', 'single'])
@pytest.mark.parametrize('n,pad_from', [(2, 99), (3, 99), (4, 99), (5, 99), (6, 99), (7, 99),
                                        (9, 99)])
def test_replay(n, pad_from, kind):
    rng = np.random.default_rng(10 * n + len(kind))
    gates = _circuit(n, kind, rng)
    x = rng.standard_normal((4,) * n)
    strides, extent = _strides(n, pad_from, 512)
    phys = np.zeros(extent)
    view = np.lib.stride_tricks.as_strided(phys, x.shape, [8 * s for s in strides])
    view[...] = x
    plan = CircuitPasses(n, strides, *_qubit_gates(gates, n))
    if n <= 6:
        assert plan.passes == 1               # the whole vector in one tile
    nat.check(nat.lib().qsv_emulate_circuit(plan.handle, phys.ctypes.data_as(nat._c_f64p)), 'run')
    ref = _apply(x, gates)
    # 16 products and sums per gate, each within half an ulp of a norm that
    # the gates keep
    eps = 2.0 ** -53
    assert np.linalg.norm(view - ref) <= 32 * len(gates) * eps * np.linalg.norm(x)


@pytest.mark.parametrize('max_qudits', [2, 3, 4])
@pytest.mark.parametrize('kind', ['brick', 'random', 'single'])
@pytest.mark.parametrize('n', [2, 5, 9])
def test_blocks(n, kind, max_qudits):
    """The library's blocks are fuse()'s: qubits, order and PTMs."""
    gates = _circuit(n, kind, np.random.default_rng(n))
    got = QubitBlocks(n, *_qubit_gates(gates, n), max_qudits)
    ref = fuse(gates, [4] * n, max_qudits)
    assert len(got) == len(ref)
    for (ptm, qubits), f in zip(got, ref):
        assert qubits == f.qudits
        # products of at most 5 n orthogonal PTMs of 256 columns
        np.testing.assert_allclose(ptm, f.ptm, rtol=0, atol=5 * n * 256 * 2.0 ** -53)


def test_refused_layouts_and_gates():
    rng = np.random.default_rng(0)
    gates = _circuit(4, 'brick', rng)
    strides, _ = _strides(4, 2, 1)            # runs that are no multiple of 64 bytes
    with pytest.raises(NotImplementedError):
        CircuitPasses(4, strides, *_qubit_gates(gates, 4))
    assert _qubit_gates(gates + [(_contraction(3, rng), (0, 1, 2))], 4) is None
    assert _qubit_gates([(_contraction(2, rng), (1, 1))], 4) is None
    assert _qubit_gates([(_contraction(1, rng), (4,))], 4) is None
    assert _qubit_gates([(np.eye(2), (0,))], 4) is None
    assert _qubit_gates([(np.eye(4, dtype=complex), (0,))], 4) is None


@pytest.mark.gpu
@pytest.mark.parametrize('dtype', ['float64', 'float32'])
@pytest.mark.parametrize('kind', ['brick', 'random', 'single'])
@pytest.mark.parametrize('n', [2, 3, 6, 7, 8, 11, 12])
def test_kernel(n, kind, dtype):
    import quantumsim_amd as qa
    from quantumsim_amd import bases
    rng = np.random.default_rng(20 * n + len(kind))
    gates = _circuit(n, kind, rng)
    x = rng.standard_normal((4,) * n)
    bs = [bases.general(2)] * n
    pv = qa.PauliVectorHIP(bs, x, force=True, dtype=dtype)
    before = pv.to_torch()
    x = before.cpu().numpy().astype(np.float64)
    count = apply_circuit(pv, gates, 3)
    assert count == len(fuse(gates, [4] * n, 3))
    ref = qa.PauliVectorHIP(bs, x, force=True, dtype='float64')
    for p, q in gates:
        ref.apply_ptm(p, *q)
    ref = ref.to_pv()
    got = pv.to_pv().astype(np.float64)
    # K = 16 products and sums per gate, each within half an ulp of the norm
    # that the gates keep, on both sides
    eps = 2.0 ** -53 if dtype == 'float64' else 2.0 ** -24
    assert np.linalg.norm(got - ref) <= 32 * len(gates) * eps * np.linalg.norm(x)
    # in passes, the vector handed out before is only read
    assert dtype == 'float32' or np.array_equal(before.cpu().numpy().astype(np.float64), x)
