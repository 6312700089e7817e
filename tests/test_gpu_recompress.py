"""GPU recompression against the host's, bit for bit (the layout's digests), over the rank
classes of its core kernel: cores of k <= 32, <= 40 and <= 64 in LDS (even and odd k, so
even and odd numbers of Jacobi pairs) and beyond in global memory; rectangular blocks."""
import numpy as np
import pytest

from helpers import uniform_points

pytestmark = pytest.mark.gpu


def _build(H, tp, sp, tol, aca, leaf):
    T = H.ClusterTree(tp, max_points_per_leaf=leaf)
    S = T if sp is tp else H.ClusterTree(sp, max_points_per_leaf=leaf)
    return H.HMatrix(H.LaplaceKernel(tp, sp), T, S, eta=2.0, eps=tol, storage=(), aca=aca)


@pytest.mark.parametrize("rect", [False, True])
def test_rank_classes_equal_host(cuda, rect):
    import hmatrixgpu as H
    # two bodies, one side length apart: their blocks are large and of high rank
    tp, sp = uniform_points(2000, 3), uniform_points(2600, 4)
    tp[0, 1000:] += 2.0
    sp[0, 1300:] += 2.0
    if not rect:
        sp = tp
    seen = set()
    for tol, leaf in ((1e-2, 40), (1e-5, 64), (1e-7, 64), (1e-8, 100), (1e-12, 100)):
        g, h = (_build(H, tp, sp, tol, a, leaf) for a in ("gpu", "host"))
        fg, fh = g.block_features(), h.block_features()
        assert np.array_equal(fg["aca_rank"], fh["aca_rank"])
        assert np.array_equal(fg["rank"], fh["rank"])
        assert g.checksum() == h.checksum(), tol
        seen |= set(fg["aca_rank"].tolist())
    print("[recompress] ACA+ ranks %d .. %d" % (min(seen), max(seen)), flush=True)
    for lo, hi in ((1, 32), (33, 40), (41, 64), (65, 10 ** 6)):
        got = [k for k in seen if lo <= k <= hi]
        assert any(k % 2 for k in got) and any(k % 2 == 0 for k in got), (lo, hi)
