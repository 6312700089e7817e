"""hmx_matvec_noalloc with more than 16 right-hand sides: passes of 32 and 48 columns where
their plan fits the static scratch, 16-column passes where it does not, and the coarser
leaf pieces that an operator keeps where the finer ones would not fit.  Bit for bit equal
to hmx_matvec, whose columns do not depend on the width of a pass."""
import re

import numpy as np
import pytest

from helpers import uniform_points
from test_zz_no_alloc import _call, _cm

pytestmark = pytest.mark.gpu
N = 4096


@pytest.fixture(scope="module")
def hm(cuda):
    import hmatrixgpu as H
    pts = uniform_points(N, 33)
    X = H.ClusterTree(pts, max_points_per_leaf=64)
    return H.HMatrix(H.LaplaceKernel(pts), X, X, eta=2.0, eps=1e-6, storage=("f64", "f32", "bf16"))


def _both(hm, cuda, storage, io, nrhs):
    import torch
    from hmatrixgpu import _lib as L
    from hmatrixgpu.hmatrix import STORAGE
    dt = torch.float64 if io == "f64" else torch.float32
    x = _cm(torch, np.random.default_rng(nrhs).standard_normal((N, nrhs)), dt, cuda)
    ref, y = (_cm(torch, np.full((N, nrhs), v), dt, cuda) for v in (np.nan, -7.0))
    L.check(_call("hmx_matvec", hm, STORAGE[storage], x, ref))
    rc = _call("hmx_matvec_noalloc", hm, STORAGE[storage], x, y)
    torch.cuda.synchronize()
    return rc, y, ref


def _need(hm, cuda, monkeypatch, storage, io, nrhs=16):
    """Bytes of scratch of 16-column passes, from the refusal at a limit of 0."""
    from hmatrixgpu import _lib as L
    monkeypatch.setenv("HMX_NOALLOC_LIMIT", "0")
    rc, _, _ = _both(hm, cuda, storage, io, nrhs)
    monkeypatch.delenv("HMX_NOALLOC_LIMIT")
    assert rc == 8  # HMX_ERR_UNSUPPORTED
    return int(re.search(rb"needs (\d+) bytes", L.lib.hmx_last_error()).group(1))


@pytest.mark.parametrize("storage,io", [("f64", "f64"), ("f32", "f32"), ("bf16", "f32"), ("f32", "f64")])
@pytest.mark.parametrize("nrhs", [20, 40, 49, 97])
def test_wide_noalloc(hm, cuda, monkeypatch, storage, io, nrhs):
    import torch
    rc, y, ref = _both(hm, cuda, storage, io, nrhs)
    assert rc == 0 and torch.equal(y, ref) and bool(torch.all(torch.isfinite(y)))
    need = _need(hm, cuda, monkeypatch, storage, io, nrhs)
    monkeypatch.setenv("HMX_NOALLOC_LIMIT", str(need))  # what 16 columns take, and no more
    rc, y, ref = _both(hm, cuda, storage, io, nrhs)
    assert rc == 0 and torch.equal(y, ref)
    monkeypatch.setenv("HMX_NOALLOC_LIMIT", str(need - 1))
    rc, y, _ = _both(hm, cuda, storage, io, nrhs)
    assert rc == 8 and bool(torch.all(y == -7.0))


@pytest.mark.parametrize("storage,io", [("f64", "f64"), ("f32", "f32"), ("bf16", "f32")])
def test_finer_pieces_do_not_push_a_product_past_the_scratch(hm, cuda, monkeypatch, storage, io):
    import torch
    fine = _need(hm, cuda, monkeypatch, storage, io)
    monkeypatch.setenv("HMX_LEAF_MIN_PIECE", str(1 << 20))
    hm.materialize(storage)
    monkeypatch.delenv("HMX_LEAF_MIN_PIECE")
    coarse = _need(hm, cuda, monkeypatch, storage, io)
    assert coarse < fine
    _, _, ref = _both(hm, cuda, storage, io, 16)
    monkeypatch.setenv("HMX_NOALLOC_LIMIT", str(coarse))
    hm.materialize(storage)  # the finer pieces are given up
    rc, y, again = _both(hm, cuda, storage, io, 16)
    assert rc == 0 and torch.equal(y, ref) and torch.equal(again, ref)
    monkeypatch.setenv("HMX_NOALLOC_LIMIT", str(coarse - 1))
    hm.materialize(storage)  # neither fits: the finer ones stay
    monkeypatch.delenv("HMX_NOALLOC_LIMIT")
    assert _need(hm, cuda, monkeypatch, storage, io) == fine
    hm.materialize(storage)
