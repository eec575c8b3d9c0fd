"""Fused blocks of whole layered circuits and the unfused gates of windows
(quantumsim_amd.windows: LayerBlockPlan, LayerGatePlan), replayed on the CPU
and run on the GPU, against the torch composition (workloads.fused_layer_gates
+ fusion.fuse_batched) and torch autograd through it."""
import numpy as np
import pytest
import torch

from quantumsim_amd.autograd import Gate, cz_ptm
from quantumsim_amd.fusion import fuse_batched
from quantumsim_amd.windows import (LayerBlockPlan, LayerGatePlan, emulate, emulate_layers,
                                    layer_blocks)
from quantumsim_amd.workloads import damping_ptms, fused_layer_gates, rotation_ptms

# float64 products of at most eight 64 x 64 factors of row sums below 2
TOL = 8 * 64 * 2 * 2.0 ** -52


def _factors(n, sets, B, device='cpu'):
    rng = np.random.default_rng(17 * n + sets)
    mk = lambda a: torch.tensor(a, device=device, requires_grad=True)
    return (mk(rng.uniform(0, 2 * np.pi, (B, sets, n, 2))), mk(rng.uniform(20, 40, (B, n))),
            mk(rng.uniform(10, 20, (B, n))))


def _composed(rot, damp, n, which):
    gates = []
    for layer, s in enumerate(which):
        gates += fused_layer_gates(n, layer, rot[:, s], damp)
    return fuse_batched([Gate(g.ptm, g.targets) for g in gates], [4] * n, 3)


@pytest.mark.parametrize('n,layers', [(2, 3), (3, 1), (4, 15), (5, 7), (7, 4), (12, 6)])
def test_replay(n, layers):
    """n = 4 has blocks of five gates (built in two parts)."""
    B = 2
    ang, t1, t2 = _factors(n, layers, B)
    rot, damp = rotation_ptms(ang), damping_ptms(t1, t2)
    rot.retain_grad(), damp.retain_grad()
    ref = _composed(rot, damp, n, range(layers))
    plan = LayerBlockPlan(n, layers, B)
    assert (n == 4) == bool(plan.split) or n == 12
    cz = cz_ptm(torch.device('cpu')).reshape(16, 16).numpy()
    r, d = rot.detach().numpy(), damp.detach().numpy()
    out, _, _ = emulate_layers(plan, r, d, cz)
    rng = np.random.default_rng(5)
    ups = [rng.standard_normal(m.shape) for m, _ in ref]
    dout = np.zeros(plan.out_elems)
    D, S = plan.split_D, plan.split_elems
    for k, ((m, q), (qs, Dk)) in enumerate(zip(ref, plan.blocks)):
        assert q == qs
        n_el = B * Dk * Dk
        if k in plan.offset:
            got = out[plan.offset[k]:][:n_el].reshape(B, Dk, Dk)
            dout[plan.offset[k]:][:n_el] = ups[k].reshape(-1)
        else:
            o1 = plan.whole_elems + plan.split.index(k) * n_el
            first = out[o1:][:n_el].reshape(B, D, D)
            second = out[o1 + S:][:n_el].reshape(B, D, D)
            got = second @ first
            dout[o1:][:n_el] = (second.transpose(0, 2, 1) @ ups[k]).reshape(-1)
            dout[o1 + S:][:n_el] = (ups[k] @ first.transpose(0, 2, 1)).reshape(-1)
        np.testing.assert_allclose(got, m.detach().numpy(), rtol=0, atol=TOL)
    sum((m * torch.tensor(u)).sum() for (m, _), u in zip(ref, ups)).backward()
    _, drot, ddp = emulate_layers(plan, r, d, cz, dout)
    scale = max(1.0, float(rot.grad.abs().max()))
    np.testing.assert_allclose(drot, rot.grad.numpy(), rtol=0, atol=64 * TOL * scale)
    np.testing.assert_allclose(ddp.sum(1), damp.grad.numpy(), rtol=0,
                               atol=64 * layers * TOL * scale)


@pytest.mark.parametrize('n', [2, 3, 4, 7])
def test_gate_plan_replay(n):
    B, nw = 3, 2
    ang, t1, t2 = _factors(n, 2 * nw, B)
    rot, damp = rotation_ptms(ang).detach(), damping_ptms(t1, t2).detach()
    plan = LayerGatePlan(n, nw, B)
    cz = cz_ptm(torch.device('cpu')).reshape(16, 16).numpy()
    out, _, _ = emulate(plan, rot.numpy(), damp.numpy(), np.ones((B, nw), np.uint8), cz)
    for w in range(nw):
        ref = fused_layer_gates(n, 0, rot[:, 2 * w], damp) + \
            fused_layer_gates(n, 1, rot[:, 2 * w + 1], damp)
        assert len(ref) == len(plan.positions)
        for g, (t, D, off) in zip(ref, plan.positions):
            assert g.targets == t
            got = out[off + w * B * D * D:][:B * D * D].reshape(B, D, D)
            np.testing.assert_allclose(got, g.ptm.numpy(), rtol=0, atol=TOL)


@pytest.mark.gpu
@pytest.mark.parametrize('dtype', [torch.float64, torch.float32])
@pytest.mark.parametrize('n,layers', [(3, 1), (4, 15), (7, 20), (12, 40)])
def test_kernel(n, layers, dtype):
    B, which = 3, [(layer // 5) % 3 for layer in range(layers)]
    ang, t1, t2 = _factors(n, 3, B, 'cuda')
    rot, damp = rotation_ptms(ang), damping_ptms(t1, t2)
    ref = _composed(rot, damp, n, which)
    plan = LayerBlockPlan(n, layers, B, torch.device('cuda'))
    cz = cz_ptm(torch.device('cuda')).reshape(16, 16).contiguous()
    got = layer_blocks(rot, damp, plan, dtype, cz, torch.tensor(which, device='cuda'))
    eps = 0.0 if dtype == torch.float64 else 2.0 ** -24    # one rounding of entries below 2
    assert [q for _, q in got] == [q for _, q in ref]
    for (m, _), (r, _) in zip(got, ref):
        assert m.dtype == dtype and m.is_contiguous()
        assert (m.double() - r).abs().max().item() <= TOL + 2 * eps
    ups = [torch.randn(r.shape, dtype=torch.float64, device='cuda').to(dtype) for r, _ in ref]
    want = torch.autograd.grad(sum((r * u.double()).sum() for (r, _), u in zip(ref, ups)),
                               [ang, t1, t2], retain_graph=True)
    have = torch.autograd.grad([m for m, _ in got], [ang, t1, t2], ups)
    for a, b in zip(have, want):
        assert (a - b).abs().max().item() <= 64 * layers * TOL * max(1.0, b.abs().max().item())
