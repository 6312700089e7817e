"""The leaf results' way into Y: summed by k_finish (items cut into 1 .. 64 pieces, target
rows that do not fill a workgroup, column groups past nrhs), or written by the leaf
kernel (no item cut).  Checked against the oracle's product on the exported layout:
both sum the same FP64 entries in another order, at most a few thousand terms per
row, so 1e-12 is 1e3 times the rounding of such a sum; FP32 storage adds 6e-8 per entry
and operand, and 2e-6 leaves a factor of ten."""
import numpy as np
import pytest

import oracle_lib as O
from helpers import layout_ns, rel, uniform_points

pytestmark = pytest.mark.gpu


def _build(n, storage, monkeypatch, min_piece):
    import hmatrixgpu as H
    if min_piece:
        monkeypatch.setenv("HMX_LEAF_MIN_PIECE", str(min_piece))
        monkeypatch.setenv("HMX_LEAF_PIECES", "1000000")
    else:
        monkeypatch.setenv("HMX_LEAF_PIECES", "0")
    pts = uniform_points(n, n)
    X = H.ClusterTree(pts, max_points_per_leaf=50)
    return H.HMatrix(H.LaplaceKernel(pts), X, X, eta=2.0, eps=1e-6, storage=storage)


def _cm(a, dtype, dev):
    import torch
    t = torch.tensor(a, dtype=dtype, device=dev)
    return t.t().contiguous().t() if t.dim() == 2 else t


@pytest.mark.parametrize("min_piece", [4096, 30000, 0])
@pytest.mark.parametrize("n", [65, 1000, 2501, 8300])
def test_pieces_and_direct_rows(cuda, monkeypatch, n, min_piece):
    import torch
    import hmatrixgpu as H
    hm = _build(n, ("f64", "f32"), monkeypatch, min_piece)
    lay = layout_ns(hm)
    rng = np.random.default_rng(5)
    for nrhs in (1, 3, 5, 16, 17):
        x = rng.standard_normal((n, nrhs) if nrhs > 1 else n)
        ref = (np.stack([O.mul_layout(lay, x[:, c]) for c in range(nrhs)], 1) if nrhs > 1
               else O.mul_layout(lay, x))
        for st, dt, tol in (("f64", torch.float64, 1e-12), ("f32", torch.float32, 2e-6),
                            ("f64", torch.float32, 2e-6)):
            xt = _cm(x, dt, cuda)
            y = torch.full_like(xt, float("nan"))
            H.mul_(y, hm, xt, storage=st)
            torch.cuda.synchronize()
            assert rel(y.cpu().numpy(), ref) <= tol, (nrhs, st, dt)


def test_batch_of_cut_and_uncut_members(cuda, monkeypatch):
    """Members with and without cut items in one launch equal their own products."""
    import torch
    import hmatrixgpu as H
    hms = [_build(n, ("f32",), monkeypatch, mp) for n, mp in ((300, 0), (2501, 30000), (65, 0))]
    rng = np.random.default_rng(6)
    Xs = [_cm(rng.standard_normal((h.n, 3)), torch.float32, cuda) for h in hms]
    for members in (hms, hms[:1]):
        xs = Xs[:len(members)]
        ys = [torch.full_like(x, float("nan")) for x in xs]
        ones = [torch.full_like(x, float("nan")) for x in xs]
        B = H.HMatrixBatch(members, storage="f32", nrhs=3)
        B.set_config(4, "tree")
        for _ in range(2):
            B.matvec(ys, xs)
        for h, x, y in zip(members, xs, ones):
            H.mul_(y, h, x, storage="f32")
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(ys, ones))
