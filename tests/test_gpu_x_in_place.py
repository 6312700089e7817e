"""Products with one right-hand side of a small operator read X in place instead of
gathering it.  The gather path (taken when Y overlaps X, or X has another type than the
sums) reads the same values in the same order, so both give the same bits: sizes on both
sides of the line, every storage, rectangular operators, degrees of freedom of the dipole
tensor, and y = x."""
import numpy as np
import pytest

from helpers import uniform_points

pytestmark = pytest.mark.gpu


def _op(kind, n):
    import hmatrixgpu as H
    tp = uniform_points(n, 21)
    if kind == "dipole":
        X = H.ClusterTree(tp, max_points_per_leaf=16, dims=3)
        return H.HMatrix(H.DipoleKernel(tp), X, X, eta=2.0, eps=1e-5, storage=("f64", "f32", "bf16"))
    sp = uniform_points(n + 333, 22) if kind == "rect" else tp
    T = H.ClusterTree(tp, max_points_per_leaf=30)
    S = T if sp is tp else H.ClusterTree(sp, max_points_per_leaf=30)
    return H.HMatrix(H.LaplaceKernel(tp, sp), T, S, eta=2.0, eps=1e-6, storage=("f64", "f32", "bf16"))


@pytest.mark.parametrize("kind,n", [("cube", 70), ("cube", 1501), ("cube", 2300), ("cube", 4096),
                                    ("rect", 2000), ("dipole", 400)])
def test_in_place_equals_gather(cuda, kind, n):
    import torch
    import hmatrixgpu as H
    hm = _op(kind, n)
    for st, dt in (("f64", torch.float64), ("f32", torch.float32), ("bf16", torch.float32)):
        x = torch.tensor(np.random.default_rng(3).standard_normal(hm.n), dtype=dt, device=cuda)
        x[5] = 0.0
        y = torch.full((hm.m,), float("nan"), dtype=dt, device=cuda)
        H.mul_(y, hm, x, storage=st)
        # Y overlapping the end of X: the product gathers X first
        buf = torch.zeros(hm.n + hm.m, dtype=dt, device=cuda)
        buf[:hm.n] = x
        ov = buf[hm.n - 8:hm.n - 8 + hm.m]
        H.mul_(ov, hm, buf[:hm.n], storage=st)
        torch.cuda.synchronize()
        assert torch.equal(ov, y), st
        if hm.m == hm.n:
            z = x.clone()
            H.mul_(z, hm, z, storage=st)
            torch.cuda.synchronize()
            assert torch.equal(z, y), st


def test_infinities_and_other_types(cuda):
    """An infinite entry of X reaches exactly the rows that the gather path gives it."""
    import torch
    import hmatrixgpu as H
    hm = _op("cube", 1501)
    x = torch.tensor(np.random.default_rng(4).standard_normal(hm.n), device=cuda)
    x[7] = float("inf")
    y = torch.empty_like(x)
    H.mul_(y, hm, x)
    z = x.clone()
    H.mul_(z, hm, z)
    torch.cuda.synchronize()
    assert torch.equal(torch.isfinite(y), torch.isfinite(z))
    assert torch.equal(torch.nan_to_num(y), torch.nan_to_num(z))
    xf = torch.tensor(np.random.default_rng(5).standard_normal(hm.n), dtype=torch.float32, device=cuda)
    a, b = torch.empty_like(xf), torch.empty(hm.m, dtype=torch.float64, device=cuda)
    H.mul_(a, hm, xf, storage="f64")           # FP32 vectors, FP64 sums: gathered
    H.mul_(b, hm, xf.double(), storage="f64")  # read in place
    torch.cuda.synchronize()
    assert torch.equal(a, b.float())
