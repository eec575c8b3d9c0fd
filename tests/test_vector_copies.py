"""Copies of a PauliVectorHIP made by the copy and pickle modules (deepcopy,
torch.save): what a vector keeps for its own calls must neither stop them nor
travel with them."""
import copy
import io
import pickle

import numpy as np
import pytest
import torch

from quantumsim_amd import bases
from quantumsim_amd.pauli_vectors.hip import PauliVectorHIP, physical_strides


def _vector(monkeypatch, stream):
    """A vector as its constructor and one apply_ptm leave it, on host tensors."""
    from quantumsim_amd.pauli_vectors import hip
    monkeypatch.setattr(hip, '_raw_stream', lambda device: stream)
    pv = PauliVectorHIP.__new__(PauliVectorHIP)
    pv.bases = [bases.general(2)] * 3
    pv._dtype, pv._device, pv._shape = torch.float64, torch.device('cpu'), (4, 4, 4)
    pv._pstr, extent = physical_strides(pv._shape, 8)
    pv._spare, pv._geo = None, (None,) * 4
    for _ in range(2):
        store = pv._take_spare(extent)
        store.zero_()
        if not hasattr(pv, '_store'):
            pv._store = None
        pv._swap_in(store, extent, pv._shape, pv._pstr)
    pv._geometry()
    return pv


def _copies(pv):
    yield copy.deepcopy(pv)
    yield pickle.loads(pickle.dumps(pv))
    f = io.BytesIO()
    torch.save(pv, f)
    f.seek(0)
    yield torch.load(f, weights_only=False)      # written above


def test_vectors_are_copied_and_saved(monkeypatch):
    pv = _vector(monkeypatch, stream=7)
    for new in _copies(pv):
        assert new.data_shape == (4, 4, 4) and torch.equal(new._store, pv._store)
        assert new._store is not pv._store
        dims, strides = new._geometry()
        assert list(dims) == [4, 4, 4] and list(strides) == list(pv._pstr)


def test_copies_do_not_take_over_the_home_stream(monkeypatch):
    """A copy's buffers belong to the stream that made the copy: until they are
    known to be of the current stream, their use there is marked."""
    pv = _vector(monkeypatch, stream=7)
    new = copy.deepcopy(pv)                     # as if made under another stream
    monkeypatch.setattr(torch.cuda, 'current_stream', lambda device=None: None)
    marked = []
    monkeypatch.setattr(torch.Tensor, 'record_stream', lambda t, s: marked.append(t))
    pv._used_here(pv._store, pv._spare)
    assert not marked                           # made on the stream that uses them
    new._used_here(new._store, new._spare)
    assert len(marked) == 2


@pytest.mark.gpu
def test_device_vectors_are_copied_and_saved():
    rng = np.random.default_rng(0)
    x = rng.standard_normal((4,) * 3)
    pv = PauliVectorHIP([bases.general(2)] * 3, x)
    p = rng.standard_normal((4,) * 4)
    pv.apply_ptm(p, 0, 2)
    ref = pv.copy()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        made = list(_copies(pv))
    torch.cuda.synchronize()
    ref.apply_ptm(p, 1, 2)
    for new in made:
        new.apply_ptm(p, 1, 2)
        assert np.array_equal(new.to_pv(), ref.to_pv())
