"""Dense blocks of brickwork windows built on the device in one launch.

A window is two consecutive layers of the layered noisy circuits of the
batched path (workloads.fused_layer_gates: per layer RX then RZ on every
qubit, CZ on the layer's brickwork bonds, amplitude + phase damping); its
gates are tiled into blocks of up to three qubits
(workloads.brickwork_window_plan).  ``window_blocks`` builds every block of
every window and circuit of a group from the per-qubit factors -- rotation
PTMs [B, 2 nw, n, 4, 4], damping PTMs [B, n, 4, 4] and the CZ PTM -- in ONE
kernel launch (qsv_window_blocks), and its backward maps the blocks'
gradients to those factors in one more (qsv_window_blocks_backward).  The
same products composed with torch ops (workloads.fused_layer_gates +
fusion.fuse_batched) take hundreds of small launches per group, forward and
backward.

No counterpart in the reference, which builds each operation's PTM on the
host (quantumsim/operations/operation.py:132-175, algebra.py:11-30).
"""
import numpy as np
import torch

from . import _native as nat
from .fusion import fuse_plan
from .workloads import brickwork_window_plan, layer_targets

__all__ = ['WBLOCK_DTYPE', 'WindowPlan', 'LayerGatePlan', 'LayerBlockPlan', 'window_blocks',
           'layer_blocks', 'emulate', 'emulate_layers']

WBLOCK_DTYPE = np.dtype([('nq', '<i4'), ('qubits', '<i4', 3), ('nf', '<i4'),
                         ('reserved', '<i4'), ('out_off', '<i8'), ('f_kind', '<i4', 4),
                         ('f_layer', '<i4', 4), ('f_slot0', '<i4', 4), ('f_slot1', '<i4', 4)])
assert WBLOCK_DTYPE.itemsize == 96


def _block_row(row, qs, gates, src, layer_of, off):
    """Fill one block-table row: qubits ``qs``, the gates ``src`` (indices of
    ``gates``' target tuples, in application order), output offset ``off``."""
    qs = tuple(int(q) for q in qs)
    if list(qs) != sorted(qs) or not 1 <= len(qs) <= 3 or not 1 <= len(src) <= 4:
        raise ValueError('block on qubits %s of %d gates' % (qs, len(src)))
    row['nq'] = len(qs)
    row['qubits'][:len(qs)] = qs
    row['nf'] = len(src)
    row['out_off'] = off
    for f, i in enumerate(src):
        t = gates[i]
        row['f_kind'][f] = len(t)
        row['f_layer'][f] = layer_of(i)
        row['f_slot0'][f] = qs.index(t[0])
        row['f_slot1'][f] = qs.index(t[1]) if len(t) == 2 else 0


def _to_device(table, device):
    return None if device is None else torch.from_numpy(table.view(np.uint8).copy()).to(device)


def _put(host, device):
    """A numpy array's bytes on ``device``, written by launches that carry them
    (qsv_put): a captured graph needs neither the array nor this tensor after."""
    out = torch.empty(host.nbytes, dtype=torch.uint8, device=device)
    nat.check(nat.lib().qsv_put(host.ctypes.data, host.nbytes, out.data_ptr(), _stream()), 'put')
    return out


class WindowPlan:
    """The block table of an n-qubit group with ``n_windows`` windows and
    ``batch`` circuits: per block position its qubits, factors (a lone qubit
    of layer l = kind 1, a bond of layer l = kind 2, in application order)
    and the offset of its [n_windows, batch, D, D] output."""

    def __init__(self, n, n_windows, batch, device=None):
        self.n, self.nw, self.batch = n, n_windows, batch
        ta, tb = layer_targets(n, 0), layer_targets(n, 1)
        gates = ta + tb
        plan = brickwork_window_plan(n)
        self.table = np.zeros(len(plan), WBLOCK_DTYPE)
        self.positions = []              # (block qubits, D, offset)
        off = 0
        for p, (qs, src) in enumerate(plan):
            D = 4 ** len(qs)
            _block_row(self.table[p], qs, gates, src, lambda i: 0 if i < len(ta) else 1, off)
            self.positions.append((tuple(qs), D, off))
            off += n_windows * batch * D * D
        self.out_elems = off
        self.device = device
        self.table_dev = _to_device(self.table, device)

    def host_ptr(self):
        return self.table.ctypes.data_as(nat.ctypes.c_void_p)


class LayerGatePlan(WindowPlan):
    """Every gate of a window a block of its own, in layer order: the PTMs of
    the layered circuit unfused (``positions`` as in WindowPlan)."""

    def __init__(self, n, n_windows, batch, device=None):
        self.n, self.nw, self.batch = n, n_windows, batch
        ta = layer_targets(n, 0)
        gates = ta + layer_targets(n, 1)
        self.table = np.zeros(len(gates), WBLOCK_DTYPE)
        self.positions = []
        off = 0
        for i, t in enumerate(gates):
            D = 4 ** len(t)
            _block_row(self.table[i], t, gates, [i], lambda i: 0 if i < len(ta) else 1, off)
            self.positions.append((tuple(t), D, off))
            off += n_windows * batch * D * D
        self.out_elems = off
        self.device = device
        self.table_dev = _to_device(self.table, device)


class LayerBlockPlan:
    """The fused blocks of a whole layered circuit of ``layers`` layers on n
    qubits (fusion.fuse_plan of its gates, blocks of up to three qubits) for
    ``batch`` parameter sets.  A block of more than four gates is built as
    two, in the last positions, and multiplied (``split``: block index ->
    (offset of the first part, of the second)).  Host memory only:
    layer_blocks writes the table to the device in every call, so that a
    captured step depends on no plan's lifetime.  ``device``: the only one the
    plan is used on (None: any).  NotImplementedError where a block holds more
    than eight gates (up to three qubits and a few layers on: all of them are one
    block), the split blocks differ in size, or there is nothing to build."""

    def __init__(self, n, layers, batch, device=None):
        self.n, self.layers, self.batch = n, layers, batch
        gates = [t for layer in range(layers) for t in layer_targets(n, layer)]
        layer_of = [layer for layer in range(layers) for _ in layer_targets(n, layer)]
        plan = fuse_plan(gates, [4] * n, 3)
        if any(len(src) > 8 for _, src in plan):
            raise NotImplementedError('a block of more than eight gates')
        whole = [k for k, (_, src) in enumerate(plan) if len(src) <= 4]
        split = [k for k, (_, src) in enumerate(plan) if len(src) > 4]
        if len({len(plan[k][0]) for k in split}) > 1:
            raise NotImplementedError('split blocks of several sizes')
        parts = [(k, plan[k][1]) for k in whole] + [(k, plan[k][1][:4]) for k in split] + \
                [(k, plan[k][1][4:]) for k in split]
        if not (1 <= len(parts) <= 65535 and 1 <= batch <= 65535):    # the launch's grid
            raise NotImplementedError('%d blocks for %d sets' % (len(parts), batch))
        self.table = np.zeros(len(parts), WBLOCK_DTYPE)
        self.blocks = [(tuple(qs), 4 ** len(qs)) for qs, _ in plan]
        self.offset = {}                 # whole block -> offset
        first, second = [], []           # offsets of the split blocks' parts
        off = 0
        for p, (k, src) in enumerate(parts):
            qs, D = self.blocks[k]
            _block_row(self.table[p], qs, gates, src, lambda i: layer_of[i], off)
            if p < len(whole):
                self.offset[k] = off
            else:
                (first if p < len(whole) + len(split) else second).append(off)
            off += batch * D * D
        self.split = split
        self.whole_elems = first[0] if split else off
        self.split_elems = second[0] - first[0] if split else 0
        self.split_D = self.blocks[split[0]][1] if split else 0
        self.out_elems = off
        self.device = device

    def host_ptr(self):
        return self.table.ctypes.data_as(nat.ctypes.c_void_p)


def _stream():
    s = torch.cuda.current_stream().cuda_stream
    return s if s else None


class _WindowBlocks(torch.autograd.Function):
    @staticmethod
    def forward(ctx, rot, damp, keep, plan, dtype, cz):
        rot = rot.detach().to(torch.float64).contiguous()
        damp = damp.detach().to(torch.float64).contiguous()
        out = torch.empty(plan.out_elems, dtype=dtype, device=rot.device)
        rc = nat.lib().qsv_window_blocks(
            nat.dtype_code(dtype), len(plan.table), plan.host_ptr(), plan.table_dev.data_ptr(),
            plan.batch, plan.nw, plan.n, rot.shape[1], rot.data_ptr(), damp.data_ptr(),
            keep.data_ptr(), cz.data_ptr(), out.data_ptr(), plan.out_elems, _stream())
        nat.check(rc, 'window_blocks')
        ctx.plan, ctx.dtype = plan, dtype
        ctx.save_for_backward(rot, damp, keep, cz)
        return tuple(out[off:off + plan.nw * plan.batch * D * D].view(plan.nw, plan.batch, D, D)
                     for _, D, off in plan.positions)

    @staticmethod
    def backward(ctx, *grads):
        rot, damp, keep, cz = ctx.saved_tensors
        plan = ctx.plan
        parts = []
        for g, (_, D, _) in zip(grads, plan.positions):
            n_el = plan.nw * plan.batch * D * D
            parts.append(torch.zeros(n_el, dtype=ctx.dtype, device=rot.device) if g is None
                         else g.to(ctx.dtype).reshape(-1))
        dout = torch.cat(parts)
        drot = torch.empty_like(rot)
        ddp = torch.empty((plan.batch, plan.nw, 2, plan.n, 4, 4), dtype=torch.float64,
                          device=rot.device)
        rc = nat.lib().qsv_window_blocks_backward(
            nat.dtype_code(ctx.dtype), len(plan.table), plan.host_ptr(),
            plan.table_dev.data_ptr(), plan.batch, plan.nw, plan.n, rot.shape[1],
            rot.data_ptr(), damp.data_ptr(), keep.data_ptr(), cz.data_ptr(), dout.data_ptr(),
            plan.out_elems, drot.data_ptr(), ddp.data_ptr(), _stream())
        nat.check(rc, 'window_blocks_backward')
        return drot, ddp.sum(dim=(1, 2)), None, None, None, None


def window_blocks(rot, damp, keep, plan, dtype, cz):
    """Blocks of every window: a tuple over block positions of [n_windows,
    batch, D, D] tensors in ``dtype`` (the layout run_schedule takes),
    differentiable with respect to ``rot`` [batch, >= 2 n_windows, n, 4, 4]
    and ``damp`` [batch, n, 4, 4] (float64).  ``keep`` [batch, n_windows]
    uint8: 0 where layer 2w + 1 is past the circuit's depth (the identity
    instead of its gates); ``cz``: the [16, 16] CZ PTM (float64)."""
    if rot.shape[0] != plan.batch or rot.shape[2] != plan.n or rot.shape[1] < 2 * plan.nw:
        raise ValueError('rotation PTMs of shape %s for %d circuits, %d windows, %d qubits'
                         % (tuple(rot.shape), plan.batch, plan.nw, plan.n))
    if tuple(damp.shape) != (plan.batch, plan.n, 4, 4):
        raise ValueError('damping PTMs of shape %s' % (tuple(damp.shape),))
    if keep.dtype != torch.uint8 or tuple(keep.shape) != (plan.batch, plan.nw) or \
            not keep.is_contiguous():
        raise ValueError('keep must be a contiguous uint8 [batch, n_windows] tensor')
    if cz.dtype != torch.float64 or cz.numel() != 256 or not cz.is_contiguous():
        raise ValueError('cz must be a contiguous float64 16 x 16 PTM')
    return _WindowBlocks.apply(rot, damp, keep, plan, dtype, cz)


class _LayerBlocks(torch.autograd.Function):
    @staticmethod
    def forward(ctx, rot, damp, which, plan, dtype, cz):
        # every layer's own rotations: the factors' gradients have one writer
        # per (layer, qubit)
        full, index = rot.detach(), None
        if which is not None:
            index = _put(np.array(which, dtype=np.int64), rot.device).view(torch.int64)
            full = full.index_select(1, index)
        full = full.contiguous()
        damp = damp.detach().contiguous()
        table = _put(plan.table, rot.device)
        out = torch.empty(plan.out_elems, dtype=torch.float64, device=rot.device)
        rc = nat.lib().qsv_layer_blocks(
            nat.QSV_F64, len(plan.table), plan.host_ptr(), table.data_ptr(), plan.batch,
            plan.n, plan.layers, full.data_ptr(), damp.data_ptr(), cz.data_ptr(), out.data_ptr(),
            plan.out_elems, _stream())
        nat.check(rc, 'layer_blocks')
        D, S = plan.split_D, plan.split_elems
        first = second = prod = None
        if S:
            first = out[plan.whole_elems:plan.whole_elems + S].view(-1, D, D)
            second = out[plan.whole_elems + S:].view(-1, D, D)
            prod = torch.bmm(second, first).to(dtype)
        whole = out[:plan.whole_elems].to(dtype)
        ctx.plan, ctx.dtype, ctx.n_rot = plan, dtype, rot.shape[1]
        saved = [full, damp, cz, table] + ([first, second] if S else []) + \
                ([index] if index is not None else [])
        ctx.parts = (bool(S), which is not None)
        ctx.save_for_backward(*saved)
        res = []
        for k, (_, d) in enumerate(plan.blocks):
            if k in plan.offset:
                off = plan.offset[k]
                res.append(whole[off:off + plan.batch * d * d].view(plan.batch, d, d))
            else:
                j = plan.split.index(k)
                res.append(prod[j * plan.batch:(j + 1) * plan.batch])
        return tuple(res)

    @staticmethod
    def backward(ctx, *grads):
        plan = ctx.plan
        saved = list(ctx.saved_tensors)
        full, damp, cz, table = saved[:4]
        has_split, has_which = ctx.parts

        def flat(k):
            d = plan.blocks[k][1]
            g = grads[k]
            return torch.zeros(plan.batch * d * d, dtype=ctx.dtype, device=full.device) \
                if g is None else g.to(ctx.dtype).reshape(-1)
        # dict order is the table's: whole blocks by offset
        parts = [torch.cat([flat(k) for k in plan.offset]).double()] if plan.offset else []
        if has_split:
            first, second = saved[4:6]
            g = torch.cat([flat(k) for k in plan.split]).double().view_as(first)
            parts.append(torch.bmm(second.transpose(1, 2).contiguous(), g).reshape(-1))
            parts.append(torch.bmm(g, first.transpose(1, 2).contiguous()).reshape(-1))
        dout = torch.cat(parts)
        dfull = torch.empty_like(full)
        ddp = torch.empty((plan.batch, plan.layers, plan.n, 4, 4), dtype=torch.float64,
                          device=full.device)
        rc = nat.lib().qsv_layer_blocks_backward(
            nat.QSV_F64, len(plan.table), plan.host_ptr(), table.data_ptr(), plan.batch,
            plan.n, plan.layers, full.data_ptr(), damp.data_ptr(), cz.data_ptr(), dout.data_ptr(),
            plan.out_elems, dfull.data_ptr(), ddp.data_ptr(), _stream())
        nat.check(rc, 'layer_blocks_backward')
        drot = dfull
        if has_which:
            # the layers' gradients summed per rotation set, as one product
            # with the 0/1 map (a fixed order)
            which = saved[-1]
            one = torch.nn.functional.one_hot(which, ctx.n_rot).to(torch.float64)   # [L, sets]
            drot = (dfull.flatten(2).transpose(1, 2) @ one).transpose(1, 2).reshape(
                full.shape[0], ctx.n_rot, plan.n, 4, 4)
        return drot, ddp.sum(dim=1), None, None, None, None


def layer_blocks(rot, damp, plan, dtype, cz, which=None):
    """The fused blocks of a layered circuit: [(PTMs [batch, D, D] in
    ``dtype``, qubits), ...] in application order, differentiable with
    respect to ``rot`` [batch, sets, n, 4, 4] (layer l uses set which[l]; None:
    one set per layer) and ``damp`` [batch, n, 4, 4], both float64.  The values
    of fusion.fuse_batched over workloads.fused_layer_gates, in two launches
    (one forward, one backward), the table's few and two small products.
    ``which``: host integers (a device tensor is read back first)."""
    sets = rot.shape[1]
    n_sets = plan.layers if which is None else sets
    if tuple(rot.shape) != (plan.batch, n_sets, plan.n, 4, 4) or \
            tuple(damp.shape) != (plan.batch, plan.n, 4, 4):
        raise ValueError('rotation PTMs of shape %s and damping PTMs of shape %s for %d sets, '
                         '%d qubits' % (tuple(rot.shape), tuple(damp.shape), plan.batch, plan.n))
    if rot.dtype != torch.float64 or damp.dtype != torch.float64:
        raise ValueError('rotation and damping PTMs must be float64')
    if which is not None:
        which = tuple(int(w) for w in (which.tolist() if hasattr(which, 'tolist') else which))
        if len(which) != plan.layers:
            raise ValueError('which must hold one rotation set per layer')
        for w in which:      # the device's index_select checks nothing
            if not 0 <= w < sets:
                raise IndexError('rotation set %d of %d' % (w, sets))
    if plan.device is not None and torch.device(plan.device).type != rot.device.type:
        raise ValueError('a plan for %s, rotation PTMs on %s' % (plan.device, rot.device))
    out = _LayerBlocks.apply(rot, damp, which, plan, dtype, cz)
    return [(m, qs) for m, (qs, _) in zip(out, plan.blocks)]


def emulate(plan, rot, damp, keep, cz, dout=None):
    """CPU replay of both kernels on numpy float64 arrays: (blocks flat,
    drot or None, ddamp_part or None)."""
    f64 = nat._c_f64p
    rot = np.ascontiguousarray(rot, dtype=np.float64)
    damp = np.ascontiguousarray(damp, dtype=np.float64)
    keep = np.ascontiguousarray(keep, dtype=np.uint8)
    cz = np.ascontiguousarray(cz, dtype=np.float64)
    out = np.zeros(plan.out_elems)
    drot = ddp = None
    if dout is not None:
        dout = np.ascontiguousarray(dout, dtype=np.float64)
        drot = np.full(rot.shape, np.nan)
        ddp = np.full((plan.batch, plan.nw, 2, plan.n, 4, 4), np.nan)
    rc = nat.lib().qsv_emulate_window_blocks(
        len(plan.table), plan.host_ptr(), plan.batch, plan.nw, plan.n, rot.shape[1],
        rot.ctypes.data_as(f64), damp.ctypes.data_as(f64),
        keep.ctypes.data_as(nat.ctypes.c_void_p), cz.ctypes.data_as(f64), out.ctypes.data_as(f64),
        plan.out_elems, None if dout is None else dout.ctypes.data_as(f64),
        None if drot is None else drot.ctypes.data_as(f64),
        None if ddp is None else ddp.ctypes.data_as(f64))
    nat.check(rc, 'emulate_window_blocks')
    return out, drot, ddp


def emulate_layers(plan, rot, damp, cz, dout=None):
    """CPU replay of the layer-block kernels on numpy float64 arrays, rot
    [batch, layers, n, 4, 4]: (parts flat, drot or None, ddamp_part or None)."""
    f64 = nat._c_f64p
    rot = np.ascontiguousarray(rot, dtype=np.float64)
    damp = np.ascontiguousarray(damp, dtype=np.float64)
    cz = np.ascontiguousarray(cz, dtype=np.float64)
    out = np.zeros(plan.out_elems)
    drot = ddp = None
    if dout is not None:
        dout = np.ascontiguousarray(dout, dtype=np.float64)
        drot = np.full(rot.shape, np.nan)
        ddp = np.full((plan.batch, plan.layers, plan.n, 4, 4), np.nan)
    rc = nat.lib().qsv_emulate_layer_blocks(
        len(plan.table), plan.host_ptr(), plan.batch, plan.n, plan.layers,
        rot.ctypes.data_as(f64), damp.ctypes.data_as(f64), cz.ctypes.data_as(f64),
        out.ctypes.data_as(f64), plan.out_elems, None if dout is None else dout.ctypes.data_as(f64),
        None if drot is None else drot.ctypes.data_as(f64),
        None if ddp is None else ddp.ctypes.data_as(f64))
    nat.check(rc, 'emulate_layer_blocks')
    return out, drot, ddp
