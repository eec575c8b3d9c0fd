"""Single gates of layered circuits built by the window kernels (positions of one
factor on one or two qubits: the small-LDS form), forward and backward, against
the host replay; the factors are products of a few numbers <= 1, so the sums of
at most 16 x 16 terms agree to 1e-13."""
import numpy as np
import pytest
import torch

from quantumsim_amd import windows as wd
from quantumsim_amd import workloads as wl
from quantumsim_amd.autograd import cz_ptm


@pytest.mark.gpu
@pytest.mark.parametrize('n,nw,batch', [(2, 1, 1), (3, 2, 3), (4, 3, 2), (7, 2, 5)])
def test_single_gates(n, nw, batch):
    rng = np.random.default_rng(n)
    mk = lambda a: torch.tensor(a, dtype=torch.float64, device='cuda')
    t1 = rng.uniform(20, 40, (batch, n))
    rot, damp = wl.gate_ptms(mk(rng.uniform(0, 6.28, (batch, 2 * nw, n, 2))), mk(t1),
                             mk(rng.uniform(10, t1)))
    rot, damp = rot.detach().requires_grad_(), damp.detach().requires_grad_()
    keep = torch.tensor(rng.integers(0, 2, (batch, nw)), dtype=torch.uint8, device='cuda')
    plan = wd.LayerGatePlan(n, nw, batch, torch.device('cuda'))
    cz = cz_ptm(torch.device('cuda')).reshape(16, 16).contiguous()
    print(n, nw, batch, flush=True)
    for dtype, tol in ((torch.float64, 1e-13), (torch.float32, 2e-7)):
        out = wd.window_blocks(rot, damp, keep, plan, dtype, cz)
        g = [torch.tensor(rng.standard_normal(tuple(m.shape)), dtype=dtype, device='cuda')
             for m in out]
        drot, ddamp = torch.autograd.grad(out, (rot, damp), g)
        flat = torch.cat([x.reshape(-1) for x in g]).double().cpu().numpy()
        ref, rrot, rdamp = wd.emulate(plan, rot.detach().cpu().numpy(),
                                      damp.detach().cpu().numpy(), keep.cpu().numpy(),
                                      cz.cpu().numpy(), flat)
        got = torch.cat([m.detach().reshape(-1) for m in out]).double().cpu().numpy()
        assert np.abs(got - ref).max() <= tol
        assert np.abs(drot.cpu().numpy() - rrot).max() <= 1e-12
        assert np.abs(ddamp.cpu().numpy() - rdamp.sum((1, 2))).max() <= 1e-12
