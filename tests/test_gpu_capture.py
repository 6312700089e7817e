"""Products recorded into a HIP graph: every replay, and the eager products between the
capture and the first replay, equal the product of an ordinary stream bit for bit."""
import ctypes as C

import numpy as np
import pytest

from helpers import uniform_points

pytestmark = pytest.mark.gpu
N = 600


@pytest.fixture(scope="module")
def hm(cuda):
    import hmatrixgpu as H
    pts = uniform_points(N, 93)
    X = H.ClusterTree(pts, max_points_per_leaf=30)
    return H.HMatrix(H.LaplaceKernel(pts), X, X, eta=2.0, eps=1e-6, storage=("f64", "f32", "bf16"))


def _cols(nrhs, io, dev, fill=None):
    import torch
    dt = torch.float64 if io == "f64" else torch.float32
    if fill is not None:
        return torch.full((nrhs, N), fill, dtype=dt, device=dev).t()
    a = np.random.default_rng(nrhs).standard_normal((nrhs, N))
    return torch.tensor(a, dtype=dt, device=dev).t()


def _nan_like(t):
    import torch
    return torch.full((t.shape[1], t.shape[0]), float("nan"), dtype=t.dtype, device=t.device).t()


def _leave_nans(hm, nbytes):
    """Free blocks of `nbytes` bytes that hold only NaN (in every storage type), so that a
    later allocation of that size does not start out as zeros."""
    from hmatrixgpu import _lib as L
    hip = L.lib  # the symbols of the HIP runtime that the library is bound to
    blocks = [C.c_void_p() for _ in range(16)]
    for p in blocks:
        assert hip.hipMalloc(C.byref(p), C.c_size_t(nbytes)) == 0
        assert hip.hipMemset(p, 0xff, C.c_size_t(nbytes)) == 0
    assert hip.hipDeviceSynchronize() == 0
    for p in blocks:
        assert hip.hipFree(p) == 0


@pytest.mark.parametrize("storage,io", [("f64", "f64"), ("f32", "f32"), ("bf16", "f32"), ("f32", "f64")])
@pytest.mark.parametrize("nrhs", [1, 4, 16, 40])
def test_first_product_of_a_stream_is_captured(hm, cuda, storage, io, nrhs):
    """A relaxed capture may allocate, so the first product of a stream can be a captured
    one.  The stream's scratch is ready for products that run before the graph does."""
    import torch
    import hmatrixgpu as H
    x, ref = _cols(nrhs, io, cuda), _cols(nrhs, io, cuda, 0.0)
    H.mul_(ref, hm, x, storage=storage)
    torch.cuda.synchronize()
    hm.release_scratch(all_streams=True)
    H.mul_(_cols(min(nrhs, 16), io, cuda, 0.0), hm, x[:, :16], storage=storage)
    torch.cuda.synchronize()
    nbytes = hm.scratch_usage()[0]  # what a capture allocates (no wide pass)
    hm.release_scratch(all_streams=True)
    s = torch.cuda.Stream(device=cuda)
    y, y2, z = (_cols(nrhs, io, cuda, 0.0) for _ in range(3))
    torch.cuda.synchronize()
    _leave_nans(hm, nbytes)
    graphs = []
    with torch.cuda.stream(s):
        for out in (y, y2):
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g, stream=s, capture_error_mode="relaxed"):
                H.mul_(out, hm, x, storage=storage)
            graphs.append(g)
        H.mul_(z, hm, x, storage=storage)
    torch.cuda.synchronize()
    assert torch.equal(z, ref)
    for _ in range(3):
        for g, out in reversed(list(zip(graphs, (y, y2)))):
            out.zero_()
            torch.cuda.synchronize()
            with torch.cuda.stream(s):
                g.replay()
                H.mul_(z, hm, x, storage=storage)
            torch.cuda.synchronize()
            assert torch.equal(out, ref) and torch.equal(z, ref)
    hm.release_scratch(all_streams=True)


@pytest.mark.parametrize("storage,io", [("f64", "f64"), ("f32", "f32"), ("bf16", "f32")])
@pytest.mark.parametrize("warm,captured", [(40, 16), (40, 20), (40, 5), (20, 16), (20, 40), (20, 97)])
def test_capture_after_a_wide_product(hm, cuda, storage, io, warm, captured):
    """A stream that has run a product of more than 16 columns can capture any other one of
    more than four: the wider scratch serves narrower passes, none is allocated."""
    import torch
    import hmatrixgpu as H
    xw, yw, refw = _cols(warm, io, cuda), _cols(warm, io, cuda, 0.0), _cols(warm, io, cuda, 0.0)
    x, y, ref = _cols(captured, io, cuda), _cols(captured, io, cuda, 0.0), _cols(captured, io, cuda, 0.0)
    H.mul_(refw, hm, xw, storage=storage)
    H.mul_(ref, hm, x, storage=storage)
    torch.cuda.synchronize()
    hm.release_scratch(all_streams=True)
    s = torch.cuda.Stream(device=cuda)
    with torch.cuda.stream(s):
        H.mul_(yw, hm, xw, storage=storage)
        torch.cuda.synchronize()
        held = hm.scratch_usage()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            H.mul_(y, hm, x, storage=storage)
    assert hm.scratch_usage() == held
    for _ in range(3):
        y.zero_()
        yw.zero_()
        torch.cuda.synchronize()
        with torch.cuda.stream(s):
            g.replay()
            H.mul_(yw, hm, xw, storage=storage)
        torch.cuda.synchronize()
        assert torch.equal(y, ref) and torch.equal(yw, refw)
    hm.release_scratch(all_streams=True)


@pytest.mark.parametrize("storage,io", [("f64", "f64"), ("f32", "f32"), ("bf16", "f32")])
@pytest.mark.parametrize("n", [3, 40, 901])
def test_widths_in_turn_on_one_stream(cuda, n, storage, io):
    """Passes of 48, 32 and 16 columns take turns in the same scratch, down to an operator
    with fewer rows than the padding (one dense block); what a pass leaves there does not
    reach the next one."""
    import torch
    import hmatrixgpu as H
    pts = uniform_points(n, 94)
    X = H.ClusterTree(pts, max_points_per_leaf=50)
    op = H.HMatrix(H.LaplaceKernel(pts), X, X, eta=2.0, eps=1e-6, storage=storage)
    dt = torch.float64 if io == "f64" else torch.float32
    rng = np.random.default_rng(n)
    held = None
    for nrhs in (48, 16, 32, 5, 40, 97, 17, 16, 48):
        x = torch.tensor(rng.standard_normal((nrhs, n)), dtype=dt, device=cuda).t()
        y, ref = (torch.full((nrhs, n), float("nan"), dtype=dt, device=cuda).t() for _ in range(2))
        torch.cuda.synchronize()
        H.mul_(y, op, x, storage=storage)
        held = held or op.scratch_usage()
        assert op.scratch_usage() == held
        s = torch.cuda.Stream(device=cuda)
        with torch.cuda.stream(s):
            H.mul_(ref, op, x, storage=storage)
        torch.cuda.synchronize()
        op.release_scratch(s)
        assert torch.equal(y, ref), nrhs
        assert bool(torch.all(torch.isfinite(y)))
        H.mul_(_nan_like(y), op, _nan_like(x), storage=storage)  # X and T rows of NaN
