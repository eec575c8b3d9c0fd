"""Float32 64 x 64 applies of batches whose innermost axis is a bystander
(k_apply64d): the staging and stores replayed on the host against numpy, and on
the device the same bits as one PauliVectorHIP per state, at the fewest tiles,
odd tile counts, mixed dimensions and per-state or shared PTMs.
"""
import numpy as np
import pytest
import torch

from quantumsim_amd import _native as nat

GEOMS = [((4,) * 6, (0, 1, 2)), ((4,) * 6, (4, 1, 2)), ((4,) * 7, (5, 0, 3)),
         ((3, 4, 4, 2, 4, 4, 4), (4, 1, 2)), ((4, 4, 4, 3, 2, 4, 4), (1, 5, 0))]


@pytest.mark.parametrize('dims,targets', GEOMS)
@pytest.mark.parametrize('blocks', [0, 1, 3])
def test_host_replay(dims, targets, blocks, rng):
    x = rng.standard_normal(dims)
    P = rng.standard_normal((64, 64))
    y = np.zeros_like(x)
    f64 = nat._c_f64p
    nat.check(nat.lib().qsv_emulate_apply_ptm_vectors(
        nat.QSV_F32, x.ctypes.data_as(f64), y.ctypes.data_as(f64), len(dims), nat.i64(dims), 3,
        nat.i32(targets), P.ctypes.data_as(f64), blocks), 'emulate_apply_ptm_vectors')
    mx, my = (np.moveaxis(a, targets, (0, 1, 2)).reshape(64, -1) for a in (x, y))
    assert np.allclose(my, P @ mx, rtol=1e-12, atol=1e-11)


def test_other_geometries_are_refused(rng):
    x = rng.standard_normal((4,) * 6)
    P = np.zeros((64, 64))
    f64 = nat._c_f64p
    for dtype, dims, targets in ((nat.QSV_F64, (4,) * 6, (1, 2, 3)),
                                 (nat.QSV_F32, (4,) * 6, (3, 4, 5)),
                                 (nat.QSV_F32, (4,) * 5, (1, 2, 3))):
        assert nat.lib().qsv_emulate_apply_ptm_vectors(
            dtype, x.ctypes.data_as(f64), x.ctypes.data_as(f64), len(dims), nat.i64(dims), 3,
            nat.i32(targets), P.ctypes.data_as(f64), 0) == -3


@pytest.mark.gpu
@pytest.mark.parametrize('dims,targets', GEOMS + [((4,) * 8, (2, 0, 5)), ((4,) * 9, (1, 7, 4))])
def test_same_bits_as_single_states(dims, targets):
    import quantumsim_amd as qa
    from quantumsim_amd import bases
    from quantumsim_amd.autograd import _apply_raw
    if not all(d == 4 for d in dims):
        dims = tuple(4 if d == 3 else d for d in dims)      # bases of 2 or 4 entries
    rng = np.random.default_rng(len(dims))
    B = 3
    print(dims, targets, flush=True)
    x = rng.standard_normal((B,) + dims).astype(np.float32)
    P = (rng.standard_normal((B, 64, 64)) / 8).astype(np.float32)
    xd, Pd = torch.tensor(x.reshape(B, -1), device='cuda'), torch.tensor(P, device='cuda')
    own = _apply_raw(xd, Pd, dims, targets, [4, 4, 4]).cpu()
    shared = _apply_raw(xd, Pd[:1], dims, targets, [4, 4, 4]).cpu()
    full = [bases.general(2) if d == 4 else bases.general(2).subbasis([0, 1]) for d in dims]
    for b in range(B):
        for PP, y in ((P[b], own[b]), (P[0], shared[b])):
            v = qa.PauliVectorHIP(full, x[b].astype(np.float64), dtype=torch.float32)
            v.apply_ptm(PP.astype(np.float64).reshape((4,) * 6), *targets)
            assert torch.equal(y, v.to_torch().reshape(-1).cpu()), b
