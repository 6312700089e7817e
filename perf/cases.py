"""What the H-matrix engine is timed on: the products, builds and predictor training that a
user of the package runs, from the smallest operator to one of 100,000 points.

    listed()             the fixed cases
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  inputs and handles a program holds before the call
    run(state)           one pass through the public entry points, with its outputs
    work(case)           bytes and operations of a pass
    exact(case, seed)    the outputs in 64 bits, by direct sums

A case names a kind of call:

    product    mul_(result, H, x) on device tensors (mul!)
    host       mul_(result, H, x) on numpy arrays (mul! of an HMatrixCPU)
    batch      HMatrixBatch.matvec of independent H-matrices of uneven size
    build      HMatrix(...) with the GPU ACA+, and its first product
    predictor  RankPredictor: training, then prediction
"""
import math
import os
import sys
import types

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "hmatrixgpu.jl_amd"))
import hmatrixgpu as hm  # noqa: E402

ELEM = {"f64": 8, "f32": 4, "bf16": 2}


def listed():
    return [
        # the reference's own test problem: a 2-D log kernel on a circle; the smallest operator,
        # where only the launches of a call count
        {"name": "circle_1000_f64", "kind": "product", "kernel": "log2d", "n": 1000, "leaf": 32,
         "eta": 1.5, "tol": 1e-5, "storage": "f64", "nrhs": 1},
        # a small 1/r operator inside an iterative solver: one FP64 vector per call
        {"name": "cube_4096_f64", "kind": "product", "kernel": "laplace", "n": 4096, "leaf": 32,
         "eta": 2.0, "tol": 1e-6, "storage": "f64", "nrhs": 1},
        # the plain drop-in mul! at an ordinary size
        {"name": "cube_65536_f64", "kind": "product", "kernel": "laplace", "n": 65536, "leaf": 64,
         "eta": 2.0, "tol": 1e-6, "storage": "f64", "nrhs": 1},
        # three vector components at once (a field), FP32, an odd size
        {"name": "cube_20011_f32_3rhs", "kind": "product", "kernel": "laplace", "n": 20011,
         "leaf": 64, "eta": 2.0, "tol": 1e-6, "storage": "f32", "nrhs": 3},
        # many FP32 right-hand sides (the headline's form), the largest operator here
        {"name": "cube_100000_f32_16rhs", "kind": "product", "kernel": "laplace", "n": 100000,
         "leaf": 64, "eta": 2.0, "tol": 1e-6, "storage": "f32", "nrhs": 16},
        # the same in BF16 storage
        {"name": "cube_50000_bf16_16rhs", "kind": "product", "kernel": "laplace", "n": 50000,
         "leaf": 64, "eta": 2.0, "tol": 1e-6, "storage": "bf16", "nrhs": 16},
        # a block Krylov step: more right-hand sides than one MFMA tile, FP64
        {"name": "cube_16384_f64_40rhs", "kind": "product", "kernel": "laplace", "n": 16384,
         "leaf": 64, "eta": 2.0, "tol": 1e-6, "storage": "f64", "nrhs": 40},
        # the demagnetising field of 6000 moments: the 3 x 3 dipole tensor, FP64
        {"name": "dipole_6000_f64", "kind": "product", "kernel": "dipole", "n": 6000, "leaf": 32,
         "eta": 2.0, "tol": 1e-5, "storage": "f64", "nrhs": 1},
        # a vector in host memory through the drop-in for the reference's CPU type
        {"name": "host_16384_f64", "kind": "host", "kernel": "laplace", "n": 16384, "leaf": 64,
         "eta": 1.5, "tol": 1e-5, "storage": "f64", "nrhs": 1},
        # independent bodies of uneven size, four FP32 vectors each, one launch
        {"name": "batch_16_f32_4rhs", "kind": "batch", "kernel": "laplace", "count": 16,
         "nmin": 2048, "nmax": 16384, "leaf": 64, "eta": 2.0, "tol": 1e-6, "storage": "f32",
         "nrhs": 4},
        # an operator built anew (moved points) and applied once
        {"name": "build_32768_f64", "kind": "build", "kernel": "laplace", "n": 32768, "leaf": 64,
         "eta": 2.0, "tol": 1e-6, "storage": "f64", "nrhs": 1},
        # the rank predictor trained on a solver's block statistics and evaluated on them
        {"name": "predictor_60000", "kind": "predictor", "n": 60000, "batch": 4096, "epochs": 4},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the listed ranges: sizes spread over their logarithm, odd ones among them."""
    kind = rng.choice(["product"] * 7 + ["host", "batch", "build", "predictor"])
    if kind == "predictor":
        return {"kind": kind, "n": _log_int(rng, 3000, 60000),
                "batch": rng.choice([256, 1000, 4096]), "epochs": rng.randint(1, 4)}
    case = {"kind": kind, "kernel": "laplace", "leaf": rng.choice([32, 64, 100]),
            "eta": rng.choice([1.5, 2.0]), "tol": rng.choice([1e-4, 1e-5, 1e-6]),
            "storage": rng.choice(["f64", "f32", "bf16"])}
    if kind == "batch":
        case.update(count=rng.randint(3, 16), nmin=rng.choice([500, 1000, 2048]),
                    nmax=_log_int(rng, 4096, 16384), storage=rng.choice(["f64", "f32"]),
                    nrhs=rng.choice([1, 3, 4, 16]))
        return case
    if kind == "host":
        case.update(n=_log_int(rng, 1000, 16384), storage="f64", nrhs=rng.choice([1, 1, 4]))
        return case
    if kind == "build":
        case.update(n=_log_int(rng, 1500, 32768), storage=rng.choice(["f64", "f32"]), nrhs=1)
        return case
    case["kernel"] = rng.choice(["laplace"] * 5 + ["log2d", "dipole"])
    case["nrhs"] = rng.choice([1, 1, 1, rng.randint(2, 4), rng.randint(5, 16), 16,
                               rng.randint(17, 48)])
    hi = {"laplace": 50000 if case["nrhs"] <= 16 else 16384, "log2d": 20000, "dipole": 6000}
    lo = {"laplace": 1500, "log2d": 1000, "dipole": 500}
    case["n"] = _log_int(rng, lo[case["kernel"]], hi[case["kernel"]])
    if case["kernel"] != "laplace":
        case["nrhs"] = min(case["nrhs"], 4)
        case["leaf"] = 32
    return case


# ---- inputs ---------------------------------------------------------------------------

def _points(case, seed):
    """Coordinates (3 x n): a circle with a seeded phase, or uniform in the unit cube."""
    rng = np.random.default_rng(seed)
    if case["kernel"] == "log2d":
        a = 2 * math.pi * (np.arange(case["n"]) / case["n"] + rng.random())
        return np.stack([np.cos(a), np.sin(a), np.zeros_like(a)])
    return rng.random((case["n"], 3)).T.copy()


def _batch_points(case, seed):
    """Uneven bodies: sizes log-uniform and fixed by the case, so that every seed costs the
    same; points uniform in boxes with one side in [1, 8]."""
    sizes = np.random.default_rng(case["count"]).uniform(math.log(case["nmin"]),
                                                         math.log(case["nmax"]), case["count"])
    rng = np.random.default_rng(seed)
    out = []
    for s in sizes:
        side = np.ones(3)
        side[rng.integers(3)] = rng.uniform(1.0, 8.0)
        out.append((rng.random((int(round(math.exp(s))), 3)) * side).T.copy())
    return out


def _vectors(case, n, seed, io):
    """x ~ N(0, 1) on the device: a vector, or column-major n x nrhs."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    if case["nrhs"] == 1:
        return torch.randn(n, dtype=io, device="cuda", generator=g)
    return torch.randn((case["nrhs"], n), dtype=io, device="cuda", generator=g).t()


def _io(case):
    return torch.float64 if case["storage"] == "f64" else torch.float32


def _kernel(case, pts):
    return {"laplace": hm.LaplaceKernel, "log2d": hm.Log2DKernel,
            "dipole": hm.DipoleKernel}[case["kernel"]](pts)


def _dims(case):
    return 3 if case["kernel"] == "dipole" else 1


def _operator(case, pts, storage):
    X = hm.ClusterTree(pts, max_points_per_leaf=case["leaf"], dims=_dims(case))
    return hm.HMatrix(_kernel(case, pts), X, X, eta=case["eta"], eps=case["tol"],
                      flatten=case["kind"] != "host", storage=storage,
                      aca="host" if case["kernel"] == "log2d" else "gpu")


def _samples(case, seed):
    """Block features and ranks as block_features() reports them: logarithms of cluster sizes
    over distances, of the tolerance and of point counts, cluster shapes, and a rank that grows
    with them."""
    rng = np.random.default_rng(seed)
    n = case["n"]
    dist = rng.uniform(0.05, 1.5, (n, 1))
    diam = dist * rng.uniform(0.1, 1.0, (n, 2))
    tol = rng.choice([1e-4, 1e-6, 1e-8], (n, 1))
    count = np.exp(rng.uniform(math.log(16), math.log(8192), (n, 2)))
    shape = -rng.exponential(0.5, (n, 4))
    f = np.concatenate([np.log(diam / dist), np.log(tol * dist), np.log(count), shape], 1)
    rank = 2 - 1.1 * f[:, 2] * np.exp(0.35 * (f[:, 0] + f[:, 1])) + rng.normal(0, 0.5, n)
    return f.astype(np.float32), np.maximum(1, np.round(rank)).astype(np.float32)


def prepare(case, seed):
    s = types.SimpleNamespace(case=case)
    kind = case["kind"]
    if kind == "predictor":
        s.features, s.ranks = _samples(case, seed)
        s.seed = seed
        return s
    if kind == "batch":
        s.members = [_operator(case, p, (case["storage"],)) for p in _batch_points(case, seed)]
        s.x = [_vectors(case, h.n, seed + i, _io(case)) for i, h in enumerate(s.members)]
        s.y = [torch.empty_like(x) for x in s.x]
        s.batch = hm.HMatrixBatch(s.members, storage=case["storage"], nrhs=case["nrhs"],
                                  io="f64" if case["storage"] == "f64" else "f32")
        return s
    s.points = _points(case, seed)
    n = s.points.shape[1] * _dims(case)
    s.x = _vectors(case, n, seed, _io(case))
    if kind == "build":
        return s
    s.H = _operator(case, s.points, (case["storage"],))
    if kind == "host":
        s.x = np.asfortranarray(s.x.cpu().numpy())
        s.y = np.empty_like(s.x, order="F")
    else:
        s.y = torch.empty_like(s.x)
    return s


def run(s):
    kind = s.case["kind"]
    if kind in ("product", "host"):
        return hm.mul_(s.y, s.H, s.x, storage=s.case["storage"])
    if kind == "batch":
        return s.batch.matvec(s.y, s.x)
    if kind == "build":
        H = _operator(s.case, s.points, (s.case["storage"],))
        info = H.info()
        return {"y": H * s.x, "leaves": info["leaves"], "max_rank": info["max_rank"],
                "nnz_D": info["nnz_D"], "nnz_U": info["nnz_U"], "nnz_V": info["nnz_V"]}
    P = hm.RankPredictor(seed=s.seed)
    loss = P.train(s.features, s.ranks, epochs=s.case["epochs"], batch=s.case["batch"],
                   seed=s.seed)
    return {"loss": loss, "weights": P.params()["master"], "predicted": P.predict(s.features)}


# ---- work and exact values ---------------------------------------------------------------

def _entries(case, pts):
    """Stored entries of the H-matrix: the dense blocks of the block tree, and for each
    admissible block the smaller of its dense and its low-rank form at the mean rank that the
    kernel and tolerance give (and the sum of (m + n) k of the latter)."""
    X = hm.ClusterTree(pts, max_points_per_leaf=case["leaf"], dims=_dims(case))
    direct, approx = hm.BlockTree(X, X, eta=case["eta"]).lists()
    size = X.node_end - X.node_start
    digits = -math.log10(case["tol"])
    rank = {"laplace": 3.7 * digits, "log2d": 0.8 * digits, "dipole": 5.4 * digits}[case["kernel"]]

    def of(pairs):
        return size[pairs[:, 0]].astype(float), size[pairs[:, 1]].astype(float)

    dm, dn = of(direct)
    am, an = of(approx)
    low = (am + an) * rank
    entries = (dm * dn).sum() + np.minimum(am * an, low).sum()
    return float(entries), float(low.sum()), float(len(am)), rank


def work(case):
    kind = case["kind"]
    if kind == "predictor":
        w = 9 * 64 + 64 * 64 + 64
        return {"bytes": 44.0 * case["n"], "flops": (6.0 * case["epochs"] + 2) * w * case["n"]}
    sets = _batch_points(case, 1) if kind == "batch" else [_points(case, 1)]
    io = 8 if case["storage"] == "f64" else 4
    total = {"bytes": 0.0, "flops": 0.0}
    for pts in sets:
        entries, low, blocks, rank = _entries(case, pts)
        n = pts.shape[1] * _dims(case)
        total["bytes"] += ELEM[case["storage"]] * entries + 2.0 * n * case["nrhs"] * io
        total["flops"] += 2.0 * entries * case["nrhs"]
        if kind == "build":  # crosses, two QRs, the applications of Q, the core's SVD
            total["flops"] += low * rank * 8 + blocks * rank ** 3 * 20
    return total


def _direct(case, pts, x):
    """K x by direct sums in FP64."""
    P = torch.tensor(pts.T.copy(), dtype=torch.float64, device="cuda")
    x = x.double()
    n = P.shape[0]
    out = torch.zeros_like(x)
    step = max(1, (1 << 26) // n)
    for a in range(0, n, step):
        b = min(n, a + step)
        d = [P[a:b, None, c] - P[None, :, c] for c in range(3)]
        r2 = (d[0] * d[0] + d[1] * d[1]) + d[2] * d[2]
        if case["kernel"] == "laplace":
            K = torch.where(r2 == 0, 0.0, r2.rsqrt())
            out[a:b] = K @ x
        elif case["kernel"] == "log2d":
            r = r2.sqrt()
            K = torch.where(r < 1e-12, 1.0, (-0.5 / math.pi) * torch.log(r.clamp_min(1e-300)))
            out[a:b] = K @ x
        else:
            inv5 = torch.where(r2 == 0, 0.0, r2 ** -2.5) / (4 * math.pi)
            for i in range(3):
                for j in range(3):
                    K = (r2 * inv5 if i == j else 0.0) - 3 * d[i] * d[j] * inv5
                    out[3 * a + i:3 * b:3] += K @ x[j::3]
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "predictor":
        return None  # a training run has no value without its own roundings
    if kind == "batch":
        sets = _batch_points(case, seed)
        return [_direct(case, p, _vectors(case, p.shape[1], seed + i, _io(case)))
                for i, p in enumerate(sets)]
    pts = _points(case, seed)
    y = _direct(case, pts, _vectors(case, pts.shape[1] * _dims(case), seed, _io(case)))
    if kind == "build":
        return {"y": y}
    return y.cpu().numpy() if kind == "host" else y
