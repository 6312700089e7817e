"""Far fields of a few long, thin panels (points on a circle, rank 3 or 4) take column
chunks of 128 k-tiles, whose partial results k_reduce sums: 1,024 columns in FP64 (from
about 12,000 points on), 2,048 in FP32 (from about 25,000 on).  The widest cluster here has
5,002 (7,502) columns, one chunk of the default 8,192, so a reduce launch per pass shows
that the short chunks were taken.

Checked against the oracle's product on the exported layout.  A chunk's sums have at most
2,048 terms, whatever the number of points, so the tolerances are those of
test_gpu_far_split.py (FP64 1e-12, FP32 2e-6)."""
import numpy as np
import pytest

import oracle_lib as O
from helpers import layout_ns, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage,n,tol", [("f64", 20011, 1e-12), ("f32", 30011, 2e-6)])
def test_short_chunks_of_long_thin_panels(cuda, monkeypatch, storage, n, tol):
    import torch
    import hmatrixgpu as H
    a = 2 * np.pi * np.arange(n) / n
    pts = np.stack([np.cos(a), np.sin(a), 0 * a])
    X = H.ClusterTree(pts, max_points_per_leaf=32)
    hm = H.HMatrix(H.Log2DKernel(pts), X, X, eta=1.5, eps=1e-5, storage=storage)
    dt = torch.float64 if storage == "f64" else torch.float32
    lay = layout_ns(hm)
    widths = hm.V_block_indices[1] - hm.V_block_indices[0] + 1
    assert widths.max() <= 8192

    def product(x):
        nrhs = x.shape[1]
        xt = torch.tensor(x, dtype=dt, device=cuda).t().contiguous().t()
        y = torch.full((nrhs, n), float("nan"), dtype=dt, device=cuda).t()
        hm.profile(True)
        hm.profile_read()
        H.mul_(y, hm, xt, storage=storage)
        torch.cuda.synchronize()
        launches = hm.profile_read()[1]
        hm.profile(False)
        return y, int(launches[2]) - 1  # stage 2: reduce (if any) and finish

    rng = np.random.default_rng(9)
    for nrhs in (1, 4, 16, 40):
        x = rng.standard_normal((n, nrhs))
        ref = np.stack([O.mul_layout(lay, x[:, c]) for c in range(nrhs)], 1)
        y, reduces = product(x)
        assert reduces == 1, nrhs
        y2, _ = product(x)
        assert torch.equal(y, y2)
        assert rel(y.cpu().numpy(), ref) <= tol, nrhs
    monkeypatch.setenv("HMX_FAR_CHUNK", "8192")
    hm.materialize(storage)
    y, reduces = product(x)
    assert reduces == 0
    assert rel(y.cpu().numpy(), ref) <= tol
