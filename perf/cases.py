"""What the framework is timed on: calls a user's program makes, over the range of sizes it makes
them at.

A case is a dict of plain values; its "kind" names the program:

  gates    a noisy circuit on one Pauli vector, gate by gate (PauliVectorHIP.apply_ptm), populations
           at the end
  fused    the same circuits through the gate-fusion entry point (fusion.apply_circuit)
  measure  readout and projective measurement of one vector: meas_prob of every qubit, a projection
           of a copy, renormalize, the reduced state of two qubits, the diagonal
  qudits   the mixed qutrit / qubit program: random 2-qudit channels, readout, basis reduction,
           partial_trace and multitake
  batch    many circuits of different widths and depths, forward and adjoint (CircuitBatch.step)
  train    the trainable circuit's KL loss and its gradients (TrainableCircuit.populations)
  block    one differentiable PTM application on a batch of states, forward and backward
           (autograd.apply)
  qset     circuits of any qudit shapes together, forward and backward (circuit_set.CircuitSet)

PTMs, states and their references are built here from Kraus operators with plain numpy / torch in
64 bits; the framework's own code is only what ``run`` calls.
"""
import math
import random

import numpy as np
import torch

import quantumsim_amd as qa
from quantumsim_amd import bases
from quantumsim_amd.autograd import apply
from quantumsim_amd.batch import CircuitBatch
from quantumsim_amd.circuit_set import CircuitSet
from quantumsim_amd.fusion import apply_circuit
from quantumsim_amd.workloads import TrainableCircuit

DEV = 'cuda'
GATE_US = 0.02          # 20 ns gates; T1 and T2 in microseconds
DT = {'f64': torch.float64, 'f32': torch.float32}


def listed():
    return [
        # the smallest call: the six-qubit, 40-layer circuit with a random pairing per layer, 600
        # launches whose states stay in the caches (latency and host work of one call)
        dict(name='gates_6q_f64', kind='gates', n=6, layers=40, pairing='random', dtype='f64'),
        # two layers of the 14-qubit noisy brickwork circuit in float64 (2 GiB vector): 1- and
        # 2-qubit gates at every position, streamed from HBM
        dict(name='gates_14q_f64', kind='gates', n=14, layers=2, pairing='brickwork', dtype='f64'),
        # the same circuit as whole programs run it: fused, in both element types, and on an odd
        # number of qubits
        dict(name='fused_14q_f64', kind='fused', n=14, layers=10, pairing='brickwork', dtype='f64'),
        dict(name='fused_13q_f32', kind='fused', n=13, layers=20, pairing='brickwork', dtype='f32'),
        # readout and one projective measurement of a 12-qubit vector
        dict(name='measure_12q_f64', kind='measure', n=12, dtype='f64'),
        # ten qudits, six of them qutrits (9^6 4^4 entries): 81 x 81, 36 x 36 and 16 x 16 channels
        dict(name='qudits_10_f64', kind='qudits', qutrits=6, qubits=4, steps=3, dtype='f64'),
        # the batched sweep's narrow half (4-7 qubits, 20-80 layers) and its wide half (8-11)
        dict(name='batch_narrow_f32', kind='batch', circuits=192, n_lo=4, n_hi=7, l_lo=20, l_hi=80,
             dtype='f32'),
        dict(name='batch_wide_f32', kind='batch', circuits=24, n_lo=8, n_hi=11, l_lo=20, l_hi=80,
             dtype='f32'),
        # the 12-qubit, 40-layer, 96-parameter circuit, eight parameter sets
        dict(name='train_12q_f32', kind='train', n=12, layers=40, sets=8, dtype='f32'),
        # single dense 3-qubit blocks forward and backward: a middle position in float64, the
        # innermost qubits of an odd register in float32
        dict(name='block_10q_f64', kind='block', n=10, batch=32, targets='3,4,5', dtype='f64'),
        dict(name='block_11q_f32', kind='block', n=11, batch=32, targets='8,9,10', dtype='f32'),
        # leaky-qubit circuits: six qutrits, and three qutrits with three qubits, uneven depths
        dict(name='qset_f64', kind='qset', circuits=16, qutrits=6, gates=12, dtype='f64'),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    kind = rng.choice(['gates', 'fused', 'measure', 'qudits', 'batch', 'train', 'block', 'qset'])
    dtype = rng.choice(['f64', 'f32'])
    if kind in ('gates', 'fused'):
        n = rng.randint(4, 14 if kind == 'fused' else 13)
        # shallower as the vector grows: no more work than the listed largest
        most = 40 if n <= 10 else (20 if n <= 12 else 10)
        if kind == 'gates' and n > 10:
            most = 4
        return dict(kind=kind, n=n, layers=_log_int(rng, 2, most),
                    pairing=rng.choice(['random', 'brickwork']), dtype=dtype)
    if kind == 'measure':
        return dict(kind=kind, n=rng.randint(5, 12), dtype=dtype)
    if kind == 'qudits':
        return dict(kind=kind, qutrits=rng.randint(2, 5), qubits=rng.randint(1, 5),
                    steps=rng.randint(1, 4), dtype=dtype)
    if kind == 'batch':
        if rng.random() < 0.5:
            lo, hi, c = 4, 7, _log_int(rng, 16, 192)
        else:
            lo, hi, c = 7, 10, _log_int(rng, 4, 24)
        l_lo = rng.randint(5, 30)
        return dict(kind=kind, circuits=c, n_lo=lo, n_hi=rng.randint(lo + 1, hi), l_lo=l_lo,
                    l_hi=l_lo + rng.randint(5, 50), dtype=rng.choice(['f32', 'f32', 'f32', 'f64']))
    if kind == 'train':
        return dict(kind=kind, n=rng.randint(6, 11), layers=rng.choice([15, 20, 30, 40]),
                    sets=rng.randint(2, 16), dtype=rng.choice(['f32', 'f32', 'f64']))
    if kind == 'block':
        n, k = rng.randint(6, 11), rng.randint(1, 3)
        start = rng.randint(0, n - k)
        targets = list(range(start, start + k))
        if rng.random() < 0.3:                       # any qubits in any order
            targets = rng.sample(range(n), k)
        most = max(2, 32 * 4 ** (11 - n) // (2 if dtype == 'f64' else 1))
        return dict(kind=kind, n=n, batch=_log_int(rng, 2, min(most, 256)),
                    targets=','.join(str(t) for t in targets), dtype=dtype)
    return dict(kind=kind, circuits=rng.randint(2, 16), qutrits=rng.randint(2, 6),
                gates=rng.randint(3, 12), dtype=dtype)


# ------------------------------------------------------------------- physics, 64 bits
def _general(d):
    """|i><i|, then X_ij and Y_ij for j < i: the element order of bases.general."""
    out = []
    for i in range(d):
        m = np.zeros((d, d), complex)
        m[i, i] = 1
        out.append(m)
    r = math.sqrt(0.5)
    for i in range(d):
        for j in range(i):
            x, y = np.zeros((d, d), complex), np.zeros((d, d), complex)
            x[i, j] = x[j, i] = r
            y[i, j], y[j, i] = 1j * r, -1j * r
            out += [x, y]
    return np.array(out)


def _gell_mann3():
    """The generalised Gell-Mann matrices of a qutrit in row-major (i, j): bases.gell_mann(3)."""
    out = []
    r = math.sqrt(0.5)
    for i in range(3):
        for j in range(3):
            m = np.zeros((3, 3), complex)
            if i == j == 0:
                m = np.eye(3, dtype=complex) / math.sqrt(3)
            elif i == j:
                m[np.arange(i), np.arange(i)] = 1
                m[i, i] = -i
                m /= math.sqrt(i * (i + 1))
            elif i < j:
                m[i, j] = m[j, i] = r
            else:
                m[i, j], m[j, i] = 1j * r, -1j * r
            out.append(m)
    return np.array(out)


_Q2 = _general(2)


def _kron_basis(vs):
    out = np.ones((1, 1, 1), complex)
    for v in vs:
        out = np.einsum('xab,ycd->xyacbd', out, v).reshape(
            out.shape[0] * v.shape[0], out.shape[1] * v.shape[1], -1)
    return out


def _ptm(kraus, vin, vout=None):
    """P[x, y] = sum_k Re tr(P_x K_k P_y K_k^dag) over Kronecker bases, as a matrix."""
    bi = _kron_basis(vin)
    bo = bi if vout is None else _kron_basis(vout)
    m = sum(np.einsum('ab,ybc,dc->yad', k, bi, k.conj(), optimize=True) for k in kraus)
    return np.ascontiguousarray(
        (bo.reshape(len(bo), -1) @ m.transpose(0, 2, 1).reshape(len(bi), -1).T).real)


def _haar(d, g):
    q, r = np.linalg.qr(g.standard_normal((d, d)) + 1j * g.standard_normal((d, d)))
    return q * (np.diagonal(r) / np.abs(np.diagonal(r)))


def _channel(d, g, ops=4):
    z = g.standard_normal((ops * d, d)) + 1j * g.standard_normal((ops * d, d))
    return np.linalg.qr(z)[0].reshape(ops, d, d)


def _density(d, g):
    a = g.standard_normal((d, d)) + 1j * g.standard_normal((d, d))
    rho = a @ a.conj().T
    return rho / np.trace(rho).real


def _damping(t1, t2, t=GATE_US):
    ga = 1 - math.exp(-t / t1)
    la = 1 - math.exp(-2 * t * (1 / t2 - 0.5 / t1))
    a = [np.diag([1, math.sqrt(1 - ga)]), np.array([[0, math.sqrt(ga)], [0, 0]])]
    p = [np.diag([1, math.sqrt(1 - la)]), np.diag([0, math.sqrt(la)])]
    return _ptm(p, [_Q2]) @ _ptm(a, [_Q2])


def _noisy_circuit(n, layers, pairing, seed):
    """[(PTM, qubits)]: per layer a Haar-random unitary on every qubit, CZ on disjoint pairs,
    amplitude and phase damping of every qubit."""
    g = np.random.default_rng(seed)
    t1 = g.uniform(20, 40, n)
    damp = [_damping(t, g.uniform(10, t)) for t in t1]
    cz = _ptm([np.diag([1, 1, 1, -1])], [_Q2, _Q2]).reshape(4, 4, 4, 4)
    out = []
    for layer in range(layers):
        out += [(_ptm([_haar(2, g)], [_Q2]), (q,)) for q in range(n)]
        if pairing == 'random':
            p = g.permutation(n)
            pairs = [tuple(sorted((int(p[2 * i]), int(p[2 * i + 1])))) for i in range(n // 2)]
        else:
            pairs = [(q, q + 1) for q in range(layer % 2, n - 1, 2)]
        out += [(cz, pq) for pq in pairs] + [(damp[q], (q,)) for q in range(n)]
    return out


def _contract(x, p, qs):
    """The PTM matrix p on axes qs of the tensor x (torch, any shape)."""
    k = len(qs)
    x = torch.movedim(x, list(qs), list(range(k)))
    shape = x.shape
    din = math.prod(shape[:k])
    y = p @ x.reshape(din, -1)
    dout = [round(p.shape[0] ** (1 / k))] * k if p.shape[0] != din else list(shape[:k])
    return torch.movedim(y.reshape(dout + list(shape[k:])), list(range(k)), list(qs))


def _structure(c):
    """What a case's sizes leave open (which qudits meet, how deep each circuit is), the same for
    every seed."""
    text = ','.join('%s=%s' % (k, c[k]) for k in sorted(c) if k != 'name')
    return np.random.default_rng(list(text.encode()))


def _product_state(vs, dims, g):
    """A product of random one-qudit density matrices, expanded in the bases ``vs``."""
    x = np.ones(1)
    for v, d in zip(vs, dims):
        x = np.multiply.outer(x, np.einsum('xab,ba->x', v, _density(d, g)).real).reshape(-1)
    return torch.from_numpy(x).to(DEV).reshape([len(v) for v in vs])


def _diag64(x, vs):
    """Populations of the tensor x in the bases vs."""
    for q, v in enumerate(vs):
        c = torch.from_numpy(np.ascontiguousarray(np.diagonal(v, axis1=1, axis2=2).T.real)).to(x)
        x = torch.movedim(torch.tensordot(c, x, ([1], [q])), 0, q)
    return x


def _trace_out(x, vs, keep):
    for q in reversed(range(len(vs))):
        if q not in keep:
            t = torch.from_numpy(np.ascontiguousarray(np.trace(vs[q], axis1=1, axis2=2).real)).to(x)
            x = torch.tensordot(x, t, ([q], [0]))
    return x


# ---------------------------------------------------------------------- gates, fused
def _prepare_circuit(c, seed):
    circ = _noisy_circuit(c['n'], c['layers'], c['pairing'], seed)
    return dict(kind=c['kind'], n=c['n'], dtype=DT[c['dtype']], fused=c['kind'] == 'fused',
                gates=[(p.reshape([4] * (2 * len(q))), q) for p, q in circ])


def _run_circuit(s):
    pv = qa.PauliVectorHIP([bases.general(2)] * s['n'], force=True, dtype=s['dtype'])
    if s['fused']:
        apply_circuit(pv, s['gates'], 3)
    else:
        for p, q in s['gates']:
            pv.apply_ptm(p, *q)
    return pv.to_torch(), pv.diagonal(get_data=False)


def _exact_circuit(c, seed):
    x = torch.zeros([4] * c['n'], dtype=torch.float64, device=DEV)
    x.view(-1)[0] = 1
    one = {}
    for p, q in _noisy_circuit(c['n'], c['layers'], c['pairing'], seed):
        p = p.reshape(4 ** len(q), -1)
        if len(q) == 1:                          # merged until a pair needs the qubit
            one[q[0]] = p @ one.get(q[0], np.eye(4))
            continue
        p = p @ np.kron(one.pop(q[0], np.eye(4)), one.pop(q[1], np.eye(4)))
        x = _contract(x, torch.from_numpy(p).to(DEV), q)
    for q, p in one.items():
        x = _contract(x, torch.from_numpy(p).to(DEV), (q,))
    x = x.contiguous()
    return x, x[(slice(0, 2),) * c['n']].reshape(-1)


def _work_circuit(c):
    n, es = c['n'], 8 if c['dtype'] == 'f64' else 4
    N = 4 ** n
    if c['pairing'] == 'random':
        pairs = c['layers'] * (n // 2)
    else:
        pairs = sum(len(range(k % 2, n - 1, 2)) for k in range(c['layers']))
    if c['kind'] == 'fused':     # one call: the vector in and out, a pair's 16 x 16 product
        return dict(bytes=2 * N * es, flops=2 * 16 * N * pairs)
    ones = 2 * n * c['layers']   # each call leaves a whole vector behind
    return dict(bytes=(pairs + ones) * 2 * N * es, flops=2 * N * (16 * pairs + 4 * ones))


# -------------------------------------------------------------------------- measure
def _prepare_measure(c, seed):
    g = np.random.default_rng(seed)
    n = c['n']
    x = _product_state([_Q2] * n, [2] * n, g)
    # entangle it a little, so that the measured qubit says something about the others
    for q in range(0, n - 1, 2):
        x = _contract(x, torch.from_numpy(_ptm(_channel(4, g, 2), [_Q2, _Q2])).to(DEV), (q, q + 1))
    pv = qa.PauliVectorHIP([bases.general(2)] * n, x.contiguous(), force=True,
                           dtype=DT[c['dtype']])
    how = _structure(c)
    hit, keep = int(how.integers(n)), sorted(int(q) for q in how.choice(n, 2, replace=False))
    project = np.zeros((4, 4))
    project[0, 0] = 1
    return dict(kind='measure', pv=pv, hit=hit, keep=keep, project=project)


def _run_measure(s):
    pv = s['pv']
    probs = np.array([pv.meas_prob(q) for q in range(pv.n_qubits)])
    after = pv.copy()
    after.apply_ptm(s['project'], s['hit'])
    tr = after.renormalize()
    reduced = after.partial_trace(*s['keep'])
    return probs, float(tr), after.to_torch(), reduced.to_torch(), after.diagonal()


def _exact_measure(c, seed):
    s = _prepare_measure(c, seed)
    n, vs = c['n'], [_Q2] * c['n']
    x = s['pv'].to_torch().double().contiguous()
    d = _diag64(x, vs)
    probs = torch.stack([d.sum([a for a in range(n) if a != q]) for q in range(n)])
    y = _contract(x, torch.from_numpy(s['project']).to(DEV), (s['hit'],))
    tr = _diag64(y, vs).sum()
    y = (y / tr).contiguous()
    return (probs.cpu().numpy(), float(tr), y, _trace_out(y, vs, s['keep']).contiguous(),
            _diag64(y, vs).reshape(-1).cpu().numpy())


def _work_measure(c):
    N, es = 4 ** c['n'], 8 if c['dtype'] == 'f64' else 4
    return dict(bytes=2 * N * es + 2 ** c['n'] * 8, flops=N)


# --------------------------------------------------------------------------- qudits
_GM3 = _gell_mann3()
_D2 = _Q2[:2]
_SEL = np.eye(4)[:2]


def _qudit_program(c, seed):
    """Dimensions, starting state and steps; every step's PTM is in the bases the vector has then.
    The case alone says which qudits meet, the seed draws their channels and state."""
    g, how = np.random.default_rng(seed), _structure(c)
    dims = [3] * c['qutrits'] + [2] * c['qubits']
    how.shuffle(dims)
    n = len(dims)
    vs = [_GM3 if d == 3 else _Q2 for d in dims]
    x0 = _product_state(vs, dims, g)
    steps = []
    for _ in range(c['steps']):
        a, b = (int(q) for q in how.choice(n, 2, replace=False))
        full = [_GM3 if dims[q] == 3 else _Q2 for q in (a, b)]
        ptm = _ptm(_channel(dims[a] * dims[b], g), [vs[a], vs[b]], full)
        ptm = ptm.reshape([len(v) for v in full] + [len(vs[a]), len(vs[b])])
        vs[a], vs[b] = full
        hit = int(how.choice([q for q in range(n) if dims[q] == 2]))
        reduce_it = len(vs[hit]) == 4
        if reduce_it:
            vs[hit] = _D2
        keep = sorted(int(q) for q in how.choice(n, min(3, n), replace=False))
        take = [sorted(int(i) for i in how.choice(len(vs[q]), 2, replace=False)) for q in keep]
        steps.append(dict(pair=(a, b), ptm=ptm, hit=hit, reduce=reduce_it, keep=keep, take=take))
    return dims, x0, steps


def _prepare_qudits(c, seed):
    dims, x0, steps = _qudit_program(c, seed)
    return dict(kind='qudits', dims=dims, x0=x0.to(DT[c['dtype']]), steps=steps,
                dtype=DT[c['dtype']], full={3: bases.gell_mann(3), 2: bases.general(2)},
                diag2=bases.general(2).subbasis([0, 1]))


def _run_qudits(s):
    pv = qa.PauliVectorHIP([s['full'][d] for d in s['dims']], s['x0'], force=True,
                           dtype=s['dtype'])
    out = []
    for st in s['steps']:
        pv.apply_ptm(st['ptm'], *st['pair'])
        for q in st['pair']:
            pv.bases[q] = s['full'][s['dims'][q]]
        out.append(pv.meas_prob(st['hit']))
        if st['reduce']:
            pv.apply_ptm(_SEL, st['hit'])
            pv.bases[st['hit']] = s['diag2']
        part = pv.partial_trace(*st['keep'])
        out += [part.to_torch(), part.multitake(*st['take'])]
    return out + [pv.to_torch()]


def _exact_qudits(c, seed):
    dims, x0, steps = _qudit_program(c, seed)
    vs = [_GM3 if d == 3 else _Q2 for d in dims]
    x = x0.to(DT[c['dtype']]).double()
    out = []
    for st in steps:
        a, b = st['pair']
        da, db = st['ptm'].shape[:2]
        p = torch.from_numpy(st['ptm'].reshape(da * db, -1)).to(DEV)
        m = torch.movedim(x, (a, b), (0, 1))
        y = (p @ m.reshape(p.shape[1], -1)).reshape([da, db] + list(m.shape[2:]))
        x = torch.movedim(y, (0, 1), (a, b))
        for q in (a, b):
            vs[q] = _GM3 if dims[q] == 3 else _Q2
        h = st['hit']
        d = _diag64(x, vs)
        out.append(d.sum([q for q in range(len(dims)) if q != h]).cpu().numpy())
        if st['reduce']:
            x = x.narrow(h, 0, 2)
            vs[h] = _D2
        part = _trace_out(x, vs, st['keep']).contiguous()
        take = part
        for q, idx in enumerate(st['take']):
            take = take.index_select(q, torch.tensor(idx, device=DEV))
        out += [part, take.cpu().numpy()]
    return out + [x.contiguous()]


def _work_qudits(c):
    N, es = 9 ** c['qutrits'] * 4 ** c['qubits'], 8 if c['dtype'] == 'f64' else 4
    # per step at most: the vector through a pair's PTM and through the reduction
    return dict(bytes=c['steps'] * 3.5 * N * es, flops=c['steps'] * 2 * 81 * N)


# ---------------------------------------------------------------------------- batch
def _random_batch(c, seed):
    g, how = np.random.default_rng(seed), _structure(c)
    out = []
    for i in range(c['circuits']):
        # every width of the range, so that each case keeps its groups
        n = c['n_lo'] + i % (c['n_hi'] - c['n_lo'] + 1)
        layers = int(how.integers(c['l_lo'], c['l_hi'] + 1))
        t1 = g.uniform(20, 40, n)
        out.append(dict(n=n, layers=layers, angles=g.uniform(0, 2 * np.pi, (layers, n, 2)), t1=t1,
                        t2=np.array([g.uniform(10, t) for t in t1])))
    return out


def _prepare_batch(c, seed):
    cb = CircuitBatch(_random_batch(c, seed), dtype=DT[c['dtype']])
    return dict(kind='batch', cb=cb, weights=cb.random_weights(seed))


def _run_batch(s):
    loss, pops, grads = s['cb'].step(s['weights'])
    return loss.detach(), [p.detach() for p in pops], grads


def _rotations64(ang):
    """PTMs of RZ(b) RX(a) for angles [..., 2] -> [..., 4, 4]."""
    v = torch.from_numpy(_Q2).to(ang.device)
    a, b = ang[..., 0] / 2, ang[..., 1] / 2
    co, si = torch.cos(a).to(torch.complex128), torch.sin(a).to(torch.complex128)
    rx = torch.stack([torch.stack([co, -1j * si], -1), torch.stack([-1j * si, co], -1)], -2)
    rz = torch.exp(torch.stack([-1j * b, 1j * b], -1))
    u = rz[..., None] * rx
    m = torch.einsum('...ab,ybc,...dc->...yad', u, v, u.conj())
    return torch.einsum('xda,...yad->...xy', v, m).real


def _dampings64(t1, t2, t=GATE_US):
    """Closed form of amplitude then phase damping in the [0, 1, X, Y] basis."""
    e1 = torch.exp(-t / t1)
    e2 = torch.exp(-t * (1 / t2 - 0.5 / t1)) * torch.sqrt(e1)
    one, zero = torch.ones_like(e1), torch.zeros_like(e1)
    rows = [[one, 1 - e1, zero, zero], [zero, e1, zero, zero], [zero, zero, e2, zero],
            [zero, zero, zero, e2]]
    return torch.stack([torch.stack(r, -1) for r in rows], -2)


def _layered64(ang, t1, t2, depth):
    """Populations [B, 2^n] of the layered circuits: ang [B, L, n, 2], t1 / t2 [B, n], depth [B]."""
    B, L, n, _ = ang.shape
    rot, damp = _rotations64(ang), _dampings64(t1, t2)
    cz = torch.from_numpy(_ptm([np.diag([1, 1, 1, -1])], [_Q2, _Q2])).to(ang.device)
    eye = torch.eye(16, dtype=torch.float64, device=ang.device)
    x = torch.zeros((B, 4 ** n), dtype=torch.float64, device=ang.device)
    x[:, 0] = 1

    def kron(p, q):
        return torch.einsum('bij,bkl->bikjl', p, q).reshape(B, 16, 16)

    def at(m, x, q):                            # m [B, D, D] from qubit q on
        D = m.shape[-1]
        x = x.reshape(B, 4 ** q, D, -1).transpose(1, 2).reshape(B, D, -1)
        return (m @ x).reshape(B, D, 4 ** q, -1).transpose(1, 2).reshape(B, -1)
    for layer in range(L):
        on = (depth > layer)[:, None, None]
        paired = set()
        for q in range(layer % 2, n - 1, 2):
            paired |= {q, q + 1}
            m = kron(damp[:, q], damp[:, q + 1]) @ cz @ kron(rot[:, layer, q], rot[:, layer, q + 1])
            x = at(torch.where(on, m, eye), x, q)
        for q in range(n):
            if q not in paired:
                x = at(torch.where(on, damp[:, q] @ rot[:, layer, q], eye[:4, :4]), x, q)
    return x.reshape([B] + [4] * n)[(slice(None),) + (slice(0, 2),) * n].reshape(B, -1)


def _exact_batch(c, seed):
    circuits = _random_batch(c, seed)
    g = np.random.default_rng(seed)              # the weights' own stream
    by_n = {}
    for i, k in enumerate(circuits):
        by_n.setdefault(k['n'], []).append(i)
    loss, pops, grads = 0.0, [], []
    for n in sorted(by_n):
        who = sorted(by_n[n], key=lambda i: -circuits[i]['layers'])
        L = circuits[who[0]]['layers']
        w = torch.from_numpy(g.standard_normal((len(who), 2 ** n))).to(DEV)
        ang = np.zeros((len(who), L, n, 2))
        for r, i in enumerate(who):
            ang[r, :circuits[i]['layers']] = circuits[i]['angles']
        leaves = [torch.from_numpy(a).to(DEV) for a in (
            ang, np.array([circuits[i]['t1'] for i in who]),
            np.array([circuits[i]['t2'] for i in who]))]
        depth = torch.tensor([circuits[i]['layers'] for i in who], device=DEV)
        # as many circuits at a time as keep every gate's state in about 40 GB
        per = max(1, int(40e9 // (L * n * 4 ** n * 8)))
        got_p, got_g = [], []
        for lo in range(0, len(who), per):
            part = [t[lo:lo + per].clone().requires_grad_() for t in leaves]
            deep = int(depth[lo:lo + per].max())
            p = _layered64(part[0][:, :deep], part[1], part[2], depth[lo:lo + per])
            p = p / p.sum(-1, keepdim=True)
            one = (p * w[lo:lo + per]).sum()
            got_g.append(torch.autograd.grad(one, part))
            got_p.append(p.detach())
            loss += float(one.detach())
        pops.append(torch.cat(got_p))
        grads += [torch.cat([t[j] for t in got_g]) for j in range(3)]
    return torch.tensor(loss, dtype=torch.float64), pops, tuple(grads)


def _layer_flops(n, layers):
    """Multiply-adds x 2 of one pass of every pair's 16 x 16 and every lone qubit's 4 x 4 PTM."""
    f = 0
    for layer in range(layers):
        pairs = len(range(layer % 2, n - 1, 2))
        f += 2 * 4 ** n * (16 * pairs + 4 * (n - 2 * pairs))
    return f


def _work_batch(c):
    flops = by = 0
    for i in range(c['circuits']):
        n = c['n_lo'] + i % (c['n_hi'] - c['n_lo'] + 1)
        layers = (c['l_lo'] + c['l_hi']) // 2
        # forward, the adjoint's apply and the PTMs' gradient
        flops += 3 * _layer_flops(n, layers)
        by += 16 * (layers * n * 2 + 2 * n) + 16 * 2 ** n
    return dict(bytes=by, flops=flops)


# ---------------------------------------------------------------------------- train
def _train_inputs(c, seed):
    g = np.random.default_rng(seed)
    n, S = c['n'], c['sets']
    ang = g.uniform(0, 2 * np.pi, (S, 3, n, 2))
    t1 = g.uniform(20, 40, (S, n))
    t2 = 10 + (t1 - 10) * g.uniform(0, 1, (S, n))
    target = g.dirichlet(np.ones(2 ** n), S)
    return [torch.from_numpy(a).to(DEV) for a in (ang, t1, t2, target)]


def _prepare_train(c, seed):
    *params, target = _train_inputs(c, seed)
    return dict(kind='train', tc=TrainableCircuit(n=c['n'], layers=c['layers']), target=target,
                params=[p.requires_grad_() for p in params], dtype=DT[c['dtype']])


def _run_train(s):
    p = s['tc'].populations(*s['params'], s['dtype'], checkpoint_every=8, fuse_qudits=3)
    loss = s['tc'].kl(s['target'], p)
    grads = torch.autograd.grad(loss.sum(), s['params'])
    return (loss.detach(), p.detach()) + grads


def _exact_train(c, seed):
    *params, target = _train_inputs(c, seed)
    which = torch.tensor([(layer // 5) % 3 for layer in range(c['layers'])], device=DEV)
    got = []
    for i in range(c['sets']):
        part = [p[i:i + 1].clone().requires_grad_() for p in params]
        depth = torch.tensor([c['layers']], device=DEV)
        p = _layered64(part[0][:, which], part[1], part[2], depth)
        t = target[i:i + 1]
        loss = (t * (torch.log(t.clamp_min(1e-30)) - torch.log(p.clamp_min(1e-30)))).sum(-1)
        got.append((loss.detach(), p.detach()) + torch.autograd.grad(loss.sum(), part))
    return tuple(torch.cat(t) for t in zip(*got))


def _work_train(c):
    return dict(bytes=c['sets'] * (16 * (3 * c['n'] * 2 + 2 * c['n']) + 16 * 2 ** c['n']),
                flops=3 * c['sets'] * _layer_flops(c['n'], c['layers']))


# ---------------------------------------------------------------------------- block
def _block_inputs(c, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    targets = tuple(int(t) for t in c['targets'].split(','))
    D = 4 ** len(targets)
    dt = DT[c['dtype']]

    def normal(*shape):
        return torch.randn(shape, generator=g, device=DEV, dtype=dt)
    x, gy = normal(c['batch'], 4 ** c['n']), normal(c['batch'], 4 ** c['n'])
    return targets, x, normal(c['batch'], D, D) / math.sqrt(D), gy


def _prepare_block(c, seed):
    targets, x, ptm, gy = _block_inputs(c, seed)
    return dict(kind='block', x=x.requires_grad_(), ptm=ptm.requires_grad_(), gy=gy,
                targets=targets, shape=(4,) * c['n'])


def _run_block(s):
    y = apply(s['x'], s['ptm'], s['shape'], s['targets'])
    return (y.detach(),) + torch.autograd.grad(y, (s['x'], s['ptm']), s['gy'])


def _exact_block(c, seed):
    targets, x, ptm, gy = _block_inputs(c, seed)
    n, B, D = c['n'], c['batch'], 4 ** len(targets)
    at, front = [1 + t for t in targets], list(range(1, 1 + len(targets)))
    ys, gxs, gps = [], [], []
    for b in range(B):
        def mat(v):
            return torch.movedim(v[b].double().reshape([1] + [4] * n), at, front).reshape(D, -1)

        def back(m):
            return torch.movedim(m.reshape([1] + [4] * n), front, at).reshape(-1)
        xm, gm, p = mat(x), mat(gy), ptm[b].double()
        ys.append(back(p @ xm))
        gxs.append(back(p.T.contiguous() @ gm))
        gps.append(gm @ xm.T.contiguous())
    return torch.stack(ys), torch.stack(gxs), torch.stack(gps)


def _work_block(c):
    D = 4 ** len(c['targets'].split(','))
    N, es = c['batch'] * 4 ** c['n'], 8 if c['dtype'] == 'f64' else 4
    return dict(bytes=4 * N * es + 2 * c['batch'] * D * D * es, flops=3 * 2 * D * N)


# ----------------------------------------------------------------------------- qset
def _set_shapes(c):
    k = c['qutrits']
    return [[3] * k, ([3, 2] * 3)[:2 * max(1, (k + 1) // 2)]]


def _set_circuits(c, seed):
    """Half the circuits on qutrits alone, half on qutrits and qubits; those of one shape share
    their gate structure and differ in their channels and depth."""
    g, how = np.random.default_rng(seed), _structure(c)
    out = []
    vs = {3: _general(3), 2: _Q2}
    for half, dims in enumerate(_set_shapes(c)):
        n = len(dims)
        structure = []
        for i in range(c['gates']):
            q = int(how.integers(n))
            if n > 1 and i % 4 != 3:
                structure.append((q, (q + 1) % n))
            else:
                structure.append((q,))
        for r in range(half, c['circuits'], 2):
            depth = c['gates'] if r < 2 else int(how.integers(max(1, c['gates'] // 2), c['gates'] + 1))
            gates = []
            for t in structure[:depth]:
                d = math.prod(dims[q] for q in t)
                gates.append((_ptm(_channel(d, g, 2), [vs[dims[q]] for q in t]), t))
            out.append((dims, gates, g.standard_normal(math.prod(d * d for d in dims))))
    return out


def _prepare_qset(c, seed):
    circuits, ptms, weights = [], [], []
    for dims, gates, w in _set_circuits(c, seed):
        gs = [(torch.from_numpy(p).to(DEV).requires_grad_(), t) for p, t in gates]
        ptms += [p for p, _ in gs]
        weights.append(torch.from_numpy(w).to(DEV, DT[c['dtype']]))
        circuits.append(([bases.general(d) for d in dims], gs))
    return dict(kind='qset', cs=CircuitSet(circuits, dtype=DT[c['dtype']]), ptms=ptms,
                weights=weights)


def _run_qset(s):
    states = s['cs'].run()
    pops = s['cs'].populations(states)
    loss = sum((x * w).sum() for x, w in zip(states, s['weights']))
    loss = loss + sum((p * p).sum() for p in pops)
    grads = torch.autograd.grad(loss, s['ptms'])
    return ([x.detach() for x in states], [p.detach() for p in pops],
            torch.cat([t.reshape(-1) for t in grads]))


def _exact_qset(c, seed):
    states, pops, grads = [], [], []
    vs = {3: _general(3), 2: _Q2}
    for dims, gates, w in _set_circuits(c, seed):
        x = torch.zeros([d * d for d in dims], dtype=torch.float64, device=DEV)
        x.view(-1)[0] = 1
        ptms = [torch.from_numpy(p).to(DEV).requires_grad_() for p, _ in gates]
        for p, (_, t) in zip(ptms, gates):
            x = _contract(x, p, t)
        x = x.reshape(-1)
        p = _diag64(x.reshape([d * d for d in dims]), [vs[d] for d in dims]).reshape(-1)
        w = torch.from_numpy(w).to(DEV, DT[c['dtype']]).double()
        grads += torch.autograd.grad((x * w).sum() + (p * p).sum(), ptms)
        states.append(x.detach())
        pops.append(p.detach())
    return states, pops, torch.cat([t.reshape(-1) for t in grads])


def _work_qset(c):
    flops = by = 0
    for half, dims in enumerate(_set_shapes(c)):
        N = math.prod(d * d for d in dims)
        count = len(range(half, c['circuits'], 2))
        D = 81 if half == 0 else 36
        flops += count * 0.75 * c['gates'] * 3 * 2 * D * N
        by += count * 0.75 * c['gates'] * 2 * D * D * 8
    return dict(bytes=by, flops=flops)


# ------------------------------------------------------------------------------ api
_KINDS = {
    'gates': (_prepare_circuit, _run_circuit, _exact_circuit, _work_circuit),
    'fused': (_prepare_circuit, _run_circuit, _exact_circuit, _work_circuit),
    'measure': (_prepare_measure, _run_measure, _exact_measure, _work_measure),
    'qudits': (_prepare_qudits, _run_qudits, _exact_qudits, _work_qudits),
    'batch': (_prepare_batch, _run_batch, _exact_batch, _work_batch),
    'train': (_prepare_train, _run_train, _exact_train, _work_train),
    'block': (_prepare_block, _run_block, _exact_block, _work_block),
    'qset': (_prepare_qset, _run_qset, _exact_qset, _work_qset),
}


def prepare(case, seed):
    return _KINDS[case['kind']][0](case, seed)


def run(state):
    return _KINDS[state['kind']][1](state)


def exact(case, seed):
    return _KINDS[case['kind']][2](case, seed)


def work(case):
    return _KINDS[case['kind']][3](case)
