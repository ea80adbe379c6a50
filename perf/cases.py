"""Workloads of the library as its users run them: K-NN graphs of host and device arrays, the search of query points,
the partition by one tree and the export of a graph, over the sizes of the package's own checks, examples and benchmark
configurations.

A case is a dict of plain values.  `what` is the entry point:
  knn          RSFK.find_nearest_neighbors           numpy in, numpy out
  knn_device   capi.knn_forest_device                tensors in and out, rows start with the point itself
  ann          RSFK.find_nearest_neighbors_ann       numpy in, numpy out
  ann_device   capi.knn_ann_device                   tensors in and out, rows start empty
  tree         RSFK.cluster_by_sample_tree           numpy in, numpy out
  graph        gpu_rsfk.graph.symmetric_knn_graph    numpy in, numpy out
  graph_device capi.symmetrize_device                tensors in and out
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "gpu-rsfk_amd"))

from gpu_rsfk import RSFK, capi                      # noqa: E402
from gpu_rsfk.graph import symmetric_knn_graph       # noqa: E402

AUTO_TREES = 50      # what find_nearest_neighbors takes for n_trees = -1 at all sizes below


def listed():
    return [
        # the package's own first check (gpu_rsfk.test): a small matrix, two exploration passes; launches count
        dict(name="knn_check_3k", what="knn", data="uniform", N=3000, D=200, K=30, trees=10, least=-1, most=128, explore=2),
        # the smallest benchmark configuration: four trees with wide buckets
        dict(name="knn_plumbing_10k", what="knn", data="uniform", N=10000, D=32, K=16, trees=4, least=32, most=128, explore=-1),
        # the example script's default data set with the defaults of find_nearest_neighbors (50 trees, one pass)
        dict(name="knn_defaults_20k", what="knn", data="gmm64", N=20000, D=32, K=32, trees=-1, least=-1, most=-1, explore=-1),
        # an ordinary data set of odd sizes, rows longer than half a wavefront, exploration asked for
        dict(name="knn_ragged_123k", what="knn", data="normal", N=123457, D=37, K=45, trees=12, least=-1, most=-1, explore=1),
        # neighbours for t-SNE (three times a perplexity of 30) of sparse image-like rows
        dict(name="knn_sparse_70k", what="knn", data="sparse", N=70000, D=784, K=90, trees=10, least=-1, most=-1, explore=1),
        # the headline benchmark, points already on the GPU
        dict(name="knn_device_1m_d100", what="knn_device", data="uniform", N=1000000, D=100, K=32, trees=50, least=-1, most=-1, explore=1),
        # clustered high-dimensional points from host memory: a gigabyte goes in
        dict(name="knn_gmm_1m_d256", what="knn", data="gmm64", N=1000000, D=256, K=32, trees=20, least=-1, most=-1, explore=-1),
        # the largest: ten million short rows, buckets of up to 256
        dict(name="knn_device_10m_d32", what="knn_device", data="normal", N=10000000, D=32, K=32, trees=10, least=64, most=256, explore=1),
        # one tree as a clustering, the example of the reference's README
        dict(name="tree_10k_d2", what="tree", data="uniform", N=10000, D=2, least=256, most=1024),
        # a batch of query points against a small base set, defaults
        dict(name="ann_20k_q1k", what="ann", data="gmm64", N=20000, Q=1000, D=64, K=16, trees=-1, least=-1, most=-1),
        # as many query points as base points, on the GPU
        dict(name="ann_device_1m_q1m", what="ann_device", data="uniform", N=1000000, Q=1000000, D=100, K=32, trees=50, least=-1, most=-1),
        # the symmetrised graph a spectral or UMAP pipeline takes
        dict(name="graph_device_1m", what="graph_device", data="uniform", N=1000000, D=32, K=32),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    while True:
        what = rng.choice(["knn"] * 6 + ["knn_device"] * 5 + ["ann"] * 2 + ["ann_device"] * 2 + ["tree"] * 2 + ["graph"] + ["graph_device"] * 2)
        case = dict(what=what, N=_log(rng, 1000, 2000000), D=_log(rng, 2, 1024))
        N, D = case["N"], case["D"]
        case["data"] = rng.choice(["uniform", "normal", "gmm64"] + ["sparse"] * (D >= 64))
        if N * D > 1.5e8:
            continue
        if what == "tree":
            least = _log(rng, 16, max(17, min(1024, N // 8)))
            return dict(case, least=least, most=least * rng.choice([2, 3, 4]))
        case["K"] = K = _log(rng, 4, 128)
        if what in ("graph", "graph_device"):
            if N * K > 3.2e7 or K * 8 > N:
                continue
            return case
        case["trees"] = rng.choice([-1, _log(rng, 2, 50), _log(rng, 2, 50)])
        trees = AUTO_TREES if case["trees"] < 0 else case["trees"]
        case["least"] = case["most"] = -1
        if rng.random() < 0.3:
            case["least"] = rng.randint(K + 1, 2 * K + 16)
            case["most"] = case["least"] * rng.choice([2, 3, 4])
        wide = max(2 * (K + 1), case["most"])
        if wide * 6 > N:
            continue
        if what.startswith("knn"):
            case["explore"] = rng.choice([-1, 0, 1, 1, 2])
            passes = _passes(case)
            # (no dearer than the largest listed cases: pairs of the buckets, pairs of the exploration, side tests)
            if N * wide * D * trees + 0.6 * passes * N * K * K * D > 3e11 or N * trees > 5e7 or N * K * K * passes > 1e9:
                continue
            return case
        case["Q"] = _log(rng, 500, 1000000)
        if case["Q"] * wide * D * trees > 3e11 or N * trees > 5e7 or case["Q"] * trees > 5e7 or (N + case["Q"]) * D > 2e8:
            continue
        return case


def _passes(case):
    return case["explore"] if case["explore"] >= 0 else (1 if case["K"] <= 32 else 0)


def _bucket_limits(case):
    least = case["least"] if case["least"] >= 0 else case["K"] + 1
    return least, case["most"] if case["most"] >= 0 else 2 * least


def _points(kind, rows, D, gen):
    """float32 rows on the GPU: i.i.d. uniform or normal, 64 clusters, or four fifths zeros."""
    if kind == "normal":
        return torch.randn((rows, D), generator=gen, device="cuda")
    X = torch.rand((rows, D), generator=gen, device="cuda")
    if kind == "gmm64":
        centres = torch.rand((64, D), generator=gen, device="cuda")
        of = torch.randint(0, 64, (rows,), generator=gen, device="cuda")
        return X.normal_(0.0, 0.1, generator=gen).add_(centres[of])
    if kind == "sparse":
        keep = torch.rand((rows, D), generator=gen, device="cuda") < 0.2
        return X.neg_().add_(1.0).mul_(keep)          # non-zero values in (0, 1]
    return X


def prepare(case, seed):
    what, N, D = case["what"], case["N"], case["D"]
    gen = torch.Generator(device="cuda").manual_seed(1 if what.startswith("graph") else seed)
    on_host = not what.endswith("_device")
    s = dict(case=case, rsfk=RSFK(random_state=0))
    X = _points(case["data"], N + case.get("Q", 0), D, gen)
    s["X"], Q = X[:N], X[N:]
    if what.startswith("ann"):
        s["Q"] = Q.cpu().numpy() if on_host else Q.contiguous()
    if what in ("knn_device", "ann_device"):
        s["idx"] = torch.empty((case.get("Q", N), case["K"]), dtype=torch.int32, device="cuda")
        s["dist"] = torch.empty((case.get("Q", N), case["K"]), dtype=torch.float32, device="cuda")
        s["self"] = torch.arange(case.get("Q", N), dtype=torch.int32, device="cuda")
    if what.startswith("graph"):
        # a K-NN graph as a short build leaves it, its points numbered anew by the seed (the number of edges stays)
        K = case["K"]
        idx = torch.full((N, K), -1, dtype=torch.int32, device="cuda")
        dist = torch.full((N, K), float("inf"), device="cuda")
        idx[:, 0] = torch.arange(N, dtype=torch.int32, device="cuda")
        dist[:, 0] = 0.0
        torch.cuda.synchronize()
        capi.knn_forest_device(2, K, N, D, K + 1, 2 * (K + 1), 5000, 0, 0, 0, s["X"].data_ptr(), idx.data_ptr(), dist.data_ptr())
        del s["X"]
        number = torch.randperm(N, generator=gen.manual_seed(seed), device="cuda").to(torch.int32)
        row = torch.empty_like(number, dtype=torch.int64)
        row[number.long()] = torch.arange(N, device="cuda")
        idx, dist = idx[row], dist[row]
        idx = torch.where(idx >= 0, number[idx.clamp(min=0).long()], idx)
        s["idx"], s["dist"] = (idx.cpu().numpy(), dist.cpu().numpy()) if on_host else (idx, dist)
        if not on_host:
            s["indptr"] = torch.empty(N + 1, dtype=torch.int32, device="cuda")
            s["cols"] = torch.zeros(2 * N * K, dtype=torch.int32, device="cuda")
            s["vals"] = torch.zeros(2 * N * K, dtype=torch.float32, device="cuda")
    elif on_host:
        s["X"] = s["X"].cpu().numpy()
    if what == "tree":
        # where the program keeps the buckets: room for any partition into buckets of least..most points
        room = N // case["least"] + 2
        s["members"], s["sizes"] = np.full(room * case["most"], -1, np.int32), np.zeros(room, np.int32)
    return s


def run(s):
    c = s["case"]
    what, N, D = c["what"], c["N"], c["D"]
    if what == "tree":
        leaves, widest, members, sizes = s["rsfk"].cluster_by_sample_tree(s["X"], verbose=0, min_tree_children=c["least"], max_tree_children=c["most"])
        s["members"][:members.size] = members
        s["sizes"][:leaves] = sizes
        return leaves, widest, s["members"], s["sizes"]
    K = c["K"]
    if what == "knn":
        return s["rsfk"].find_nearest_neighbors(s["X"], K, n_trees=c["trees"], min_tree_children=c["least"], max_tree_children=c["most"], nn_exploring_factor=c["explore"])
    if what == "ann":
        return s["rsfk"].find_nearest_neighbors_ann(s["X"], s["Q"], K, n_trees=c["trees"], min_tree_children=c["least"], max_tree_children=c["most"])
    if what == "graph":
        return symmetric_knn_graph(s["idx"], s["dist"])
    if what == "graph_device":
        n = capi.symmetrize_device(s["idx"].data_ptr(), s["dist"].data_ptr(), N, K, True, s["indptr"].data_ptr(), s["cols"].data_ptr(), s["vals"].data_ptr(), s["cols"].numel())
        return s["indptr"], s["cols"][:n], s["vals"][:n]
    least, most = _bucket_limits(c)
    trees = c["trees"] if c["trees"] >= 0 else AUTO_TREES
    idx, dist = s["idx"], s["dist"]
    idx.fill_(-1)
    dist.fill_(float("inf"))
    if what == "ann_device":
        capi.knn_ann_device(trees, K, N, c["Q"], D, least, most, 5000, 0, 0, s["X"].data_ptr(), s["Q"].data_ptr(), idx.data_ptr(), dist.data_ptr())
        return idx, dist
    idx[:, 0] = s["self"]
    dist[:, 0] = 0.0
    capi.knn_forest_device(trees, K, N, D, least, most, 5000, 0, 0, _passes(c), s["X"].data_ptr(), idx.data_ptr(), dist.data_ptr())
    return idx, dist


def work(case):
    what, N, D = case["what"], case["N"], case["D"]
    if what == "tree":
        # one side test of a point per level of a balanced tree
        levels = max(1.0, math.log2(max(2.0, N / case["most"])))
        return dict(bytes=4 * N * D + 4 * N, flops=2.0 * N * D * levels)
    K = case["K"]
    if what.startswith("graph"):
        # the rows once; columns and values of about 1.5 entries per stored one
        return dict(bytes=8 * N * K + 4 * N + 12 * N * K, flops=0)
    least, most = _bucket_limits(case)
    trees = case["trees"] if case["trees"] >= 0 else AUTO_TREES
    wide = 0.7 * most                                   # mean bucket
    levels = max(1.0, math.log2(max(2.0, N / wide)))
    if what.startswith("ann"):
        Q = case["Q"]
        return dict(bytes=4 * (N + Q) * D + 8 * Q * K, flops=trees * D * (2.0 * (N + Q) * levels + 3.0 * Q * wide))
    # side tests, every pair of a bucket once, and per exploration pass a distance for every entry of a row
    return dict(bytes=4 * N * D + 8 * N * K, flops=trees * N * D * (2.0 * levels + 1.5 * wide) + 3.0 * _passes(case) * N * K * D)


def tolerance(case):
    # 32-bit sums; a pair of neighbours whose distances differ in the last bits may change places
    return "exact" if case["what"] == "tree" else dict(rel=1e-5, differ=1e-3)
