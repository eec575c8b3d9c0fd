"""PTM sizes that go through the table kernel (neither inline nor dense 64 x
64 / 256 x 256), at the edges of its tiles: 16-row blocks, 96-column chunks,
one and several row shares, orbit counts around 16 and 32, targets in any
order and position.  On the CPU the kernel's replay, on the GPU the kernel,
both against einsum in float64."""
import ctypes
import math

import numpy as np
import pytest

from quantumsim_amd import _native as nat

CASES = [
    # (dims, targets, dims_out)
    ((17, 1), (0,), (17,)),              # one orbit
    ((16, 17), (0,), (17,)),             # 17 rows of 16 columns, 17 orbits
    ((31, 3, 5), (0,), (1,)),            # one row, 15 orbits
    ((2, 33, 16), (1,), (48,)),          # 32 orbits, whole row blocks
    ((9, 9, 4), (2, 0), (4, 9)),         # reversed targets
    ((4, 9, 9), (1, 2), (9, 9)),         # innermost targets
    ((9, 3, 9, 11), (0, 2), (9, 9)),     # 33 orbits in runs of 11
    ((95, 5), (0,), (97,)),              # below a chunk, above six row blocks
    ((96, 3), (0,), (96,)),
    ((97, 33), (0,), (96,)),             # a second chunk of one column
    ((193, 2), (0,), (3,)),              # three chunks
    ((9, 9, 2, 4), (3, 0, 1), (4, 9, 9)),  # 324 x 324
]


def _data(dims, targets, dout, dtype, batch):
    rng = np.random.default_rng(sum(dims) + 7 * len(targets))
    np_t = np.float64 if dtype == nat.QSV_F64 else np.float32
    din = [dims[t] for t in targets]
    x = rng.standard_normal((batch,) + dims).astype(np_t)
    p = rng.standard_normal([batch] + list(dout) + din).astype(np_t)
    return x, p


def _einsum(x, p, dims, targets):
    n, k = len(dims), len(targets)
    lo = list(range(n))
    for j, t in enumerate(targets):
        lo[t] = n + j
    return np.einsum(p, [n + j for j in range(k)] + list(targets), x, list(range(n)), lo,
                     optimize=True)


def _check(got, x, p, dims, targets, eps):
    """|error| <= (K + 2) eps sum |P| |x|: K products and sums, and the
    reference's own (float64) rounding."""
    ref = _einsum(x.astype(np.float64), p.astype(np.float64), dims, targets)
    mag = _einsum(np.abs(x).astype(np.float64), np.abs(p).astype(np.float64), dims, targets)
    K = math.prod(dims[t] for t in targets)
    assert got.shape == ref.shape
    assert np.all(np.abs(got - ref) <= (K + 2) * eps * mag + 1e-300)


@pytest.mark.parametrize('dtype', [nat.QSV_F64, nat.QSV_F32])
@pytest.mark.parametrize('dims,targets,dout', CASES)
def test_table_replay(dims, targets, dout, dtype):
    x, p = _data(dims, targets, dout, dtype, 1)
    x, p = x[0].astype(np.float64), p[0].astype(np.float64)
    shape = list(dims)
    for t, d in zip(targets, dout):
        shape[t] = d
    out = np.full(shape, np.nan)
    path = (ctypes.c_int32 * 1)()
    f = nat._c_f64p
    rc = nat.lib().qsv_emulate_apply_ptm(
        dtype, x.ctypes.data_as(f), out.ctypes.data_as(f), len(dims), nat.i64(dims), None, None,
        len(targets), nat.i32(targets), nat.i32(dout), p.ctypes.data_as(f), path)
    nat.check(rc, 'emulate')
    assert path[0] == 3
    _check(out, x, p, dims, targets, 2.0 ** -52)


@pytest.mark.gpu
@pytest.mark.parametrize('dtype', [nat.QSV_F64, nat.QSV_F32])
@pytest.mark.parametrize('dims,targets,dout', CASES)
def test_table_kernel(dims, targets, dout, dtype):
    import torch
    B = 3
    x, p = _data(dims, targets, dout, dtype, B)
    xd, pd = torch.from_numpy(x).cuda(), torch.from_numpy(p).cuda()
    shape = list(dims)
    for t, d in zip(targets, dout):
        shape[t] = d
    out = torch.full([B] + shape, float('nan'), dtype=xd.dtype, device='cuda')
    D = math.prod(dout) * math.prod(dims[t] for t in targets)
    rc = nat.lib().qsv_apply_ptm_batched(
        dtype, xd.data_ptr(), out.data_ptr(), B, len(dims), nat.i64(dims), len(targets),
        nat.i32(targets), nat.i32(dout), pd.data_ptr(), D,
        torch.cuda.current_stream().cuda_stream or None)
    nat.check(rc, 'apply')
    got = out.cpu().numpy()
    eps = 2.0 ** -52 if dtype == nat.QSV_F64 else 2.0 ** -23
    for b in range(B):
        _check(got[b], x[b], p[b], dims, targets, eps)
