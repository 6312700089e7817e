"""Far-field panels whose row groups are shared by the waves of a workgroup (one or two
row groups: four or two waves on their k-tiles), alone and with the short column chunks
that a far field of long, thin panels takes.  Checked against the oracle's product on the
exported layout, with the tolerances of test_gpu_finish.py (FP64 1e-12, FP32 2e-6)."""
import numpy as np
import pytest

import oracle_lib as O
from helpers import layout_ns, rel, uniform_points

pytestmark = pytest.mark.gpu


def _operator(kind, storage):
    import hmatrixgpu as H
    if kind == "cube":  # a few row groups per cluster, remainders of every size
        pts = uniform_points(1501, 17)
        K, leaf, eta, tol = H.LaplaceKernel(pts), 30, 2.0, 1e-6
    else:  # rank 3 or 4 in clusters of up to a quarter of the points
        n = 9001
        a = 2 * np.pi * np.arange(n) / n
        pts = np.stack([np.cos(a), np.sin(a), 0 * a])
        K, leaf, eta, tol = H.Log2DKernel(pts), 32, 1.5, 1e-5
    X = H.ClusterTree(pts, max_points_per_leaf=leaf)
    return H.HMatrix(K, X, X, eta=eta, eps=tol, storage=storage)


@pytest.mark.parametrize("kind", ["cube", "circle"])
def test_shared_row_groups(cuda, kind):
    import torch
    import hmatrixgpu as H
    hm = _operator(kind, ("f64", "f32"))
    lay = layout_ns(hm)
    rng = np.random.default_rng(8)
    for nrhs in (1, 4, 16, 40):
        x = rng.standard_normal((hm.n, nrhs))
        ref = np.stack([O.mul_layout(lay, x[:, c]) for c in range(nrhs)], 1)
        for st, dt, tol in (("f64", torch.float64, 1e-12), ("f32", torch.float32, 2e-6)):
            xt = torch.tensor(x, dtype=dt, device=cuda).t().contiguous().t()
            y = torch.full((nrhs, hm.m), float("nan"), dtype=dt, device=cuda).t()
            H.mul_(y, hm, xt, storage=st)
            y2 = torch.empty_like(y)
            H.mul_(y2, hm, xt, storage=st)
            torch.cuda.synchronize()
            assert torch.equal(y, y2)
            assert rel(y.cpu().numpy(), ref) <= tol, (nrhs, st)
