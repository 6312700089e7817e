"""Products with more than 16 right-hand sides without the memory for a wide pass: they
run in narrower passes with the same bits, and the refusal holds until the stream's
scratch is released."""
import numpy as np
import pytest

from helpers import uniform_points

pytestmark = pytest.mark.gpu
N = 1100


@pytest.fixture(scope="module")
def hm(cuda):
    import hmatrixgpu as H
    pts = uniform_points(N, 95)
    X = H.ClusterTree(pts, max_points_per_leaf=30)
    return H.HMatrix(H.LaplaceKernel(pts), X, X, eta=2.0, eps=1e-6, storage=("f64", "f32", "bf16"))


@pytest.mark.parametrize("storage,io", [("f64", "f64"), ("f32", "f32"), ("bf16", "f32")])
@pytest.mark.parametrize("nrhs", [20, 40, 97])
def test_refused_wide_scratch(hm, cuda, monkeypatch, storage, io, nrhs):
    import torch
    import hmatrixgpu as H
    dt = torch.float64 if io == "f64" else torch.float32
    x = torch.tensor(np.random.default_rng(nrhs).standard_normal((nrhs, N)), dtype=dt, device=cuda).t()

    def product(cols):
        y = torch.full((cols, N), float("nan"), dtype=dt, device=cuda).t()
        H.mul_(y, hm, x[:, :cols], storage=storage)
        torch.cuda.synchronize()
        return y

    held = {}
    for cols in (16, 20, 40):  # passes of 16, 32 and 48
        hm.release_scratch(all_streams=True)
        product(min(cols, nrhs))
        held[cols] = hm.scratch_usage()[0]
    hm.release_scratch(all_streams=True)
    ref = product(nrhs)
    full = hm.scratch_usage()[0]
    assert held[16] < held[20] and full == (held[20] if nrhs == 20 else held[40])
    # a limit below one pass width leaves the next narrower one
    for limit, want in ((0, held[16]), (held[20] - 1, held[16]), (held[20], held[20]), (full, full)):
        hm.release_scratch(all_streams=True)
        monkeypatch.setenv("HMX_WIDE_SCRATCH_LIMIT", str(limit))
        assert torch.equal(product(nrhs), ref)
        assert hm.scratch_usage()[0] == want
        monkeypatch.delenv("HMX_WIDE_SCRATCH_LIMIT")
        assert torch.equal(product(nrhs), ref)
        assert hm.scratch_usage()[0] == want  # remembered
    hm.release_scratch(all_streams=True)
    assert torch.equal(product(nrhs), ref)
    assert hm.scratch_usage()[0] == full
    hm.release_scratch(all_streams=True)
