"""Gate fusion: turn a gate list into fewer, denser PTM applications.

A circuit applied gate by gate reads and writes the whole Pauli vector once
per gate.  Runs of gates that together act on at most ``max_qudits``
qudits compose into one dense PTM (the reference builds such PTMs with
``_Chain.ptm``, quantumsim/operations/operation.py:610-623, and applies a
3-qubit one in test_operations.py:174-195), applied in a single pass: the
16x16 streaming kernel for 2 qudits, the MFMA kernel for 3-4 qubits.

The pass keeps several open blocks on disjoint qudit sets (gates on
disjoint qudits commute, so their blocks can stay open side by side).  A
gate touching open blocks joins the largest subset of them whose union with
its own qudits fits ``max_qudits`` (ties: the subset holding more gates);
the touched blocks left out are emitted first (they act on a qudit of the
gate, so they must precede it).  At the end every open block is emitted.
Square PTMs (same input and output dimension per qudit) only.

``apply_circuit`` runs qubit circuits without forming these blocks: in passes
over the vector that each apply several two-qubit gates from LDS.
"""
import itertools
import numpy as np

from . import _native as nat

__all__ = ['fuse', 'fuse_plan', 'FusedGate', 'embed_ptm', 'embed_ptm_batched', 'fuse_batched',
           'apply_circuit']


class FusedGate:
    """A dense PTM over ``qudits`` (ascending), layout (out..., in...);
    ``sources``: indices of the input gates it is the product of, in
    application order."""
    __slots__ = ('ptm', 'qudits', 'n_source', 'sources')

    def __init__(self, ptm, qudits, n_source, sources=()):
        self.ptm = ptm
        self.qudits = tuple(qudits)
        self.n_source = n_source
        self.sources = tuple(sources)

    def __iter__(self):          # (ptm, qudits) unpacking, like the inputs
        yield self.ptm
        yield self.qudits


def embed_ptm(ptm, qudits, block, dims):
    """PTM of ``ptm`` (acting on ``qudits`` in that order) as a square
    matrix over ``block`` (sorted), identity on the other block qudits."""
    k = len(qudits)
    pos = [block.index(q) for q in qudits]
    m = len(block)
    din = [dims[q] for q in block]
    p = np.asarray(ptm, dtype=np.float64).reshape([dims[q] for q in qudits] * 2)
    # einsum labels: output axes 0..m-1, input axes m..2m-1
    args = [p, [pos[j] for j in range(k)] + [m + pos[j] for j in range(k)]]
    for b in range(m):
        if b not in pos:
            args += [np.eye(din[b]), [b, m + b]]
    out = np.einsum(*args, list(range(2 * m)), optimize=True)
    D = int(np.prod(din))
    return out.reshape(D, D)


class _Block:
    __slots__ = ('qudits', 'mat', 'n', 'src')

    def __init__(self, qudits, mat, n, src):
        self.qudits = qudits      # sorted tuple
        self.mat = mat            # D x D in the block's qudit order
        self.n = n
        self.src = src            # source gate indices, application order


def _merge(blocks, dims):
    """Blocks on disjoint qudits -> one block (their PTMs commute)."""
    qs = tuple(sorted(q for b in blocks for q in b.qudits))
    mat = np.eye(int(np.prod([dims[q] for q in qs])))
    for b in blocks:
        mat = embed_ptm(b.mat.reshape([dims[q] for q in b.qudits] * 2), b.qudits, qs,
                        dims) @ mat
    return _Block(qs, mat, sum(b.n for b in blocks), [i for b in blocks for i in b.src])


def fuse(gates, dims, max_qudits=2):
    """Fuse ``gates`` = [(ptm, qudits), ...] on a vector with per-qudit Pauli
    dimensions ``dims``.  Returns a list of FusedGate whose sequential
    application equals that of ``gates``."""
    open_blocks = {}              # qudit -> block
    out = []

    def emit(b):
        shape = [dims[q] for q in b.qudits] * 2
        out.append(FusedGate(b.mat.reshape(shape), b.qudits, b.n, b.src))
        for q in b.qudits:
            del open_blocks[q]

    for gi, (ptm, qudits) in enumerate(gates):
        qudits = tuple(int(q) for q in qudits)
        p = np.asarray(ptm)
        k = len(qudits)
        if p.shape[:k] != p.shape[k:] or any(p.shape[j] != dims[q] for j, q in enumerate(qudits)):
            raise ValueError('fuse() needs square PTMs matching the qudit dimensions')
        touched = []
        for q in qudits:
            b = open_blocks.get(q)
            if b is not None and b not in touched:
                touched.append(b)
        # largest subset of the touched blocks that fits together with the gate
        best, best_key = (), None
        for r in range(len(touched), -1, -1):
            for sub in itertools.combinations(touched, r):
                u = set(qudits).union(*(b.qudits for b in sub))
                if len(u) > max_qudits and sub:
                    continue
                key = (len(u) if sub else 0, sum(b.n for b in sub))
                if best_key is None or key > best_key:
                    best, best_key = sub, key
        for b in touched:
            if b not in best:
                emit(b)
        union = set(qudits).union(*(b.qudits for b in best))
        qs = tuple(sorted(union))
        if best:
            base = _merge(list(best), dims) if len(best) > 1 else best[0]
            for b in best:
                for q in b.qudits:
                    open_blocks.pop(q, None)
            prev = base.mat
            if base.qudits != qs:
                prev = embed_ptm(prev.reshape([dims[q] for q in base.qudits] * 2),
                                 base.qudits, qs, dims)
            nb = _Block(qs, embed_ptm(p, qudits, qs, dims) @ prev, base.n + 1, base.src + [gi])
        else:
            nb = _Block(qs, embed_ptm(p, qudits, qs, dims), 1, [gi])
        for q in nb.qudits:
            open_blocks[q] = nb
    seen = []
    for b in open_blocks.values():
        if b not in seen:
            seen.append(b)
    for b in seen:
        emit(b)
    return out


_PLANS = {}
_EYES = {}


def fuse_plan(qudit_sets, dims, max_qudits=3):
    """The blocks ``fuse`` forms for gates on ``qudit_sets`` (the grouping
    depends only on which qudits the gates touch): [(block qudits, source
    gate indices in application order), ...].  Cached."""
    key = (tuple(tuple(int(q) for q in t) for t in qudit_sets), tuple(dims), max_qudits)
    plan = _PLANS.get(key)
    if plan is None:
        probe = [(np.eye(int(np.prod([dims[q] for q in t]))).reshape([dims[q] for q in t] * 2), t)
                 for t in key[0]]
        plan = [(f.qudits, f.sources) for f in fuse(probe, dims, max_qudits)]
        _PLANS[key] = plan
    return plan


def embed_ptm_batched(ptm, qudits, block, dims):
    """Torch form of ``embed_ptm`` for a batch: ptm [B, D, D] acting on
    ``qudits`` -> [B, Db, Db] over ``block`` (sorted), identity elsewhere."""
    import torch
    qudits, block = tuple(qudits), tuple(block)
    if qudits == block:
        return ptm
    k, m = len(qudits), len(block)
    pos = [block.index(q) for q in qudits]
    B = ptm.shape[0]
    p = ptm.reshape([B] + [dims[q] for q in qudits] * 2)
    # labels: batch 0, outputs 1..m, inputs m+1..2m
    ops = [p, [0] + [1 + pos[j] for j in range(k)] + [1 + m + pos[j] for j in range(k)]]
    for b in range(m):
        if b not in pos:
            key = (dims[block[b]], ptm.dtype, ptm.device)
            eye = _EYES.get(key)
            if eye is None:
                from .autograd import shared_constant
                eye = _EYES[key] = shared_constant(
                    torch.eye(key[0], dtype=ptm.dtype, device=ptm.device))
            ops += [eye, [1 + b, 1 + m + b]]
    out = torch.einsum(*ops, list(range(2 * m + 1)))
    D = int(np.prod([dims[q] for q in block]))
    return out.reshape(B, D, D)


def fuse_batched(gates, dims, max_qudits=3, plan=None):
    """Fuse batched gates (objects with ``.ptm`` [B or 1, D, D] torch
    tensors and ``.targets``) into dense blocks of up to ``max_qudits``
    qudits with torch ops, so autograd reaches the source PTMs.  ``plan``:
    [(block qudits, source indices in order), ...] to use instead of
    ``fuse_plan``'s.  Returns [(ptm [B, Db, Db], block qudits), ...] in
    application order."""
    if plan is None:
        plan = fuse_plan([g.targets for g in gates], dims, max_qudits)
    out = []
    for block, src in plan:
        mat = None
        for i in src:
            e = embed_ptm_batched(gates[i].ptm, gates[i].targets, block, dims)
            mat = e if mat is None else e @ mat
        out.append((mat, block))
    return out


class CircuitPasses:
    """A qubit circuit planned as passes over a float64 vector (qsv_circuit_*):
    ``ks``, ``targets`` (two per gate) and the concatenated float64 ``ptms``
    for a vector of n qubits with element strides ``strides``."""

    def __init__(self, n, strides, ks, targets, ptms):
        import ctypes
        self._lib = nat.lib()
        self.handle = None
        handle = ctypes.c_void_p()
        nat.check(self._lib.qsv_circuit_create(
            n, nat.i64(strides), len(ks), ks.ctypes.data_as(nat._c_i32p),
            targets.ctypes.data_as(nat._c_i32p), ptms.ctypes.data_as(nat._c_f64p),
            ctypes.byref(handle)), 'apply_circuit')
        self.handle = handle.value

    def __del__(self):
        if self.handle is not None:
            self._lib.qsv_circuit_destroy(self.handle)

    @property
    def passes(self):
        return self._lib.qsv_circuit_passes(self.handle)

    def table(self, device):
        """The blocks' tables on ``device``, copied from pinned memory on the
        current stream."""
        import torch
        n = self._lib.qsv_circuit_table_bytes(self.handle)
        host = torch.empty(max(n, 1), dtype=torch.uint8, pin_memory=True)
        nat.check(self._lib.qsv_circuit_table(self.handle, host.data_ptr()), 'apply_circuit')
        return host.to(device, non_blocking=True)

    def run(self, src, dst, table, stream):
        nat.check(self._lib.qsv_circuit_run(self.handle, src, dst, table, stream),
                  'apply_circuit')


class QubitBlocks:
    """``fuse`` for the circuits ``_qubit_gates`` takes, planned and composed
    in the library: the same blocks in the same order, PTMs equal to
    rounding.  Iterating composes one block at a time: (ptm, qubits).
    NotImplementedError for PTMs that are not finite (the library skips zeros
    where ``fuse`` makes 0 * inf a NaN)."""

    def __init__(self, n, ks, targets, ptms, max_qudits):
        import ctypes
        self._lib = nat.lib()
        self.handle = None
        handle = ctypes.c_void_p()
        nat.check(self._lib.qsv_circuit_blocks_create(
            n, len(ks), ks.ctypes.data_as(nat._c_i32p), targets.ctypes.data_as(nat._c_i32p),
            ptms.ctypes.data_as(nat._c_f64p), int(max_qudits), ctypes.byref(handle)), 'fuse')
        self.handle = handle.value

    def __del__(self):
        if self.handle is not None:
            self._lib.qsv_circuit_blocks_destroy(self.handle)

    def __len__(self):
        return self._lib.qsv_circuit_blocks_count(self.handle)

    def dearer_than(self, passes):
        """Whether a CircuitPasses of the same gates takes no longer
        (qsv_circuit_pays)."""
        return bool(self._lib.qsv_circuit_pays(passes.handle, self.handle))

    def __iter__(self):
        qubits = np.zeros(32, dtype=np.int32)
        for i in range(len(self)):
            k = nat.check(self._lib.qsv_circuit_block_qubits(
                self.handle, i, qubits.ctypes.data_as(nat._c_i32p)), 'fuse')
            ptm = np.empty((4,) * (2 * k))
            nat.check(self._lib.qsv_circuit_block_ptm(
                self.handle, i, ptm.ctypes.data_as(nat._c_f64p)), 'fuse')
            yield ptm, tuple(int(q) for q in qubits[:k])


def _qubit_gates(gates, n):
    """(ks, targets, ptms) arrays of a circuit of 1- and 2-qubit gates with
    real square PTMs on n qubits, or None if it holds any other gate."""
    ks, targets, ptms = [], [], []
    for ptm, qudits in gates:
        p = np.asarray(ptm)
        k = len(qudits)
        if k not in (1, 2) or p.shape != (4,) * (2 * k) or p.dtype.kind not in 'fiub':
            return None
        q = [int(t) for t in qudits]
        if min(q) < 0 or max(q) >= n or (k == 2 and q[0] == q[1]):
            return None
        ks.append(k)
        targets += q if k == 2 else (q[0], -1)
        ptms.append(p.reshape(-1))
    return (np.array(ks, dtype=np.int32), np.array(targets, dtype=np.int32),
            np.concatenate(ptms).astype(np.float64, copy=False))


def _native_circuit(pv, gates):
    """_qubit_gates' arrays where the library plans the circuit: a
    PauliVectorHIP of 2 to 16 qubits in full bases whose apply_ptm nobody
    replaced; else None."""
    from .pauli_vectors import hip
    if not isinstance(pv, hip.PauliVectorHIP) or \
            getattr(pv.apply_ptm, '__func__', None) is not hip._apply_ptm:
        return None
    n = pv.n_qubits
    if not 2 <= n <= 16 or pv.data_shape != (4,) * n or pv.dim_pauli != (4,) * n:
        return None
    return _qubit_gates(gates, n)


def apply_circuit(pv, gates, max_qudits=3):
    """Apply ``gates`` = [(ptm, qudits), ...] (PTMs in ``pv``'s bases) to the
    Pauli vector ``pv``, fused into blocks of up to ``max_qudits`` qudits
    (0 or 1: gate by gate).  Returns the number of blocks.

    On float64 vectors, circuits of 1- and 2-qubit gates on qubits in full
    bases run in passes that each apply several two-qubit blocks from LDS
    (csrc/qsv_slab.hip): the same product, rounded in another order.  Float32
    vectors keep the blocks, whose rounding the populations of a float32 run
    carry to their last digit; so do circuits of one block (one pass either
    way) or of few blocks of many gates (QubitBlocks.dearer_than), layouts
    without aligned runs and graph capture (the passes' tables are copied from
    host memory).  Any other circuit is fused by ``fuse``."""
    if max_qudits is None or max_qudits <= 1:
        for ptm, qudits in gates:
            pv.apply_ptm(np.asarray(ptm), *qudits)
        return len(gates)
    gates = list(gates)
    try:
        arrays = _native_circuit(pv, gates) if gates else None
    except TypeError:                # targets without a length: read once each
        gates = [(ptm, tuple(qudits)) for ptm, qudits in gates]
        arrays = _native_circuit(pv, gates)
    fused = None
    if arrays is not None:
        try:
            fused = QubitBlocks(pv.n_qubits, *arrays, min(max_qudits, pv.n_qubits))
        except NotImplementedError:
            pass
        else:
            if len(fused) > 1 and pv.run_passes(*arrays, fused.dearer_than):
                return len(fused)
    if fused is None:
        fused = fuse(gates, list(pv.dim_pauli), max_qudits)
    for ptm, qudits in fused:
        pv.apply_ptm(ptm, *qudits)
    return len(fused)
