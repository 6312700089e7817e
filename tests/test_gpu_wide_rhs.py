"""Products with more than 16 right-hand sides run in passes of 16, 32 or 48 columns.
A column's sums do not depend on the width of its pass, so every result equals the
product of at most 16 columns at a time bit for bit: both widths, their remainders,
several passes, every storage, 32- and 64-bit row addresses, a leading dimension larger
than the matrix, and a stream under capture (no scratch for a wide pass)."""
import numpy as np
import pytest

from helpers import uniform_points

pytestmark = pytest.mark.gpu
N = 1500


@pytest.fixture(scope="module")
def hm(cuda):
    import hmatrixgpu as H
    pts = uniform_points(N, 91)
    X = H.ClusterTree(pts, max_points_per_leaf=30)
    return H.HMatrix(H.LaplaceKernel(pts), X, X, eta=2.0, eps=1e-6, storage=("f64", "f32", "bf16"))


def _x(nrhs, io, dev, pad=0):
    import torch
    dt = torch.float64 if io == "f64" else torch.float32
    a = torch.tensor(np.random.default_rng(nrhs).standard_normal((nrhs, N + pad)), dtype=dt, device=dev)
    return a.t()[:N]


def _by16(H, hm, x, storage):
    import torch
    out = torch.empty((x.shape[1], N), dtype=x.dtype, device=x.device).t()
    for a in range(0, x.shape[1], 16):
        # at least five columns, so that the part runs on MFMA as well
        lo = max(0, min(a, x.shape[1] - 5))
        part = torch.empty((min(16, x.shape[1] - lo), N), dtype=x.dtype, device=x.device).t()
        H.mul_(part, hm, x[:, lo:lo + 16], storage=storage)
        out[:, lo:lo + 16] = part
    return out


@pytest.mark.parametrize("storage,io,offset", [("f64", "f64", 0), ("f32", "f32", 0), ("bf16", "f32", 0),
                                               ("f32", "f64", 0), ("f64", "f64", 1 << 25)])
def test_wide_equals_narrow(hm, cuda, monkeypatch, storage, io, offset):
    import torch
    import hmatrixgpu as H
    if offset:  # 2^25 unused rows of 128 bytes or more: S is 4 GiB or more
        monkeypatch.setenv("HMX_STAGING_ROW_OFFSET", str(offset))
        hm.materialize(storage)
    for nrhs in (17, 32, 33, 47, 48, 49, 64, 97):
        x = _x(nrhs, io, cuda, pad=nrhs % 3)
        y = torch.full((nrhs, N), float("nan"), dtype=x.dtype, device=cuda).t()
        H.mul_(y, hm, x, storage=storage)
        ref = _by16(H, hm, x, storage)
        torch.cuda.synchronize()
        assert torch.equal(y, ref), nrhs
    if offset:
        hm.release_scratch(all_streams=True)
        monkeypatch.delenv("HMX_STAGING_ROW_OFFSET")
        hm.materialize(storage)


def test_capture_without_wide_scratch(hm, cuda):
    """A stream that has run 16 columns can capture 40: the wide pass's scratch is not
    allocated under capture."""
    import torch
    import hmatrixgpu as H
    x = _x(40, "f32", cuda)
    y = torch.zeros((40, N), dtype=torch.float32, device=cuda).t()
    ref = _by16(H, hm, x, "f32")
    s = torch.cuda.Stream(device=cuda)
    s.wait_stream(torch.cuda.current_stream(cuda))
    with torch.cuda.stream(s):
        H.mul_(y[:, :16], hm, x[:, :16], storage="f32")
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            H.mul_(y, hm, x, storage="f32")
    for _ in range(3):
        y.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, ref)
        y2 = torch.empty_like(y)
        H.mul_(y2, hm, x, storage="f32")
        torch.cuda.synchronize()
        assert torch.equal(y2, ref)
