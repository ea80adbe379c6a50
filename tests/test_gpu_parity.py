"""GPU parity tests: the HIP library, called through its C ABI, against the CPU
oracle on the same seeded inputs.

Bar: the tree partition (integer work) must be identical; K-NN rows, sorted by
(distance, index), must hold bit-identical distances and identical indices, ties
included (library and oracle order a row by (distance, index), so no result
depends on the order in which candidates arrive).
"""
import os

import numpy as np
import pytest

from util import (assert_knn_equal, baseline_points, check_partition, exact_knn_numpy, recall, rows_have_no_duplicates,
                  sort_rows)

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _say(*a):
    print(*a, flush=True)


# ---------------------------------------------------------------------------
# tree build
# ---------------------------------------------------------------------------
@pytest.mark.parametrize("N,D,MIN,MAX,dist", [
    (1, 3, 2, 4, "u"), (5, 2, 2, 4, "u"), (40, 1, 3, 8, "u"), (700, 5, 9, 20, "u"),   # tail phase only
    (1024, 16, 33, 66, "u"), (1025, 16, 33, 66, "u"),                                  # around the wide/tail threshold
    (5000, 32, 33, 66, "u"), (30000, 100, 33, 66, "u"), (60000, 3, 64, 256, "n"),      # wide phase, several levels
    (20000, 33, 17, 34, "n"), (8000, 784, 91, 182, "sparse"),
])
@pytest.mark.parametrize("screen", ["auto", "q8", "bf16", "q8-256"])
def test_tree_partition_is_identical(gpu, orc, rng, monkeypatch, N, D, MIN, MAX, dist, screen):
    """screen: which low-precision copy the side tests are screened on (RSFK_TREE_SCREEN; "auto" chooses from the
    data).  The partition must be the one of the fp32 arithmetic whatever the screen.  "q8-256": the 8-bit screen with
    the subtrees below the wide levels finished by workgroups of 256 threads, as launches over many subtrees have it
    (RSFK_TAIL_BLOCK; the few subtrees of a test otherwise get workgroups of 1024)."""
    if screen == "q8-256":
        monkeypatch.setenv("RSFK_TREE_SCREEN", "q8")
        monkeypatch.setenv("RSFK_TAIL_BLOCK", "256")
    elif screen != "auto":
        monkeypatch.setenv("RSFK_TREE_SCREEN", screen)
    if dist == "u":
        X = rng.random((N, D), dtype=np.float32)
    elif dist == "n":
        X = rng.standard_normal((N, D)).astype(np.float32)
    else:
        X = np.where(rng.random((N, D)) < 0.8, 0.0, 1.0 - rng.random((N, D))).astype(np.float32)
    for seed in (0, 9):
        _say("tree", N, D, MIN, MAX, dist, seed)
        perm, ls, lz, st = orc.build_tree(X, MIN, MAX, 5000, seed)
        gperm, gls, glz, gst = gpu.build_tree(X, MIN, MAX, 5000, seed)
        check_partition(gperm, gls, glz, N)
        assert np.array_equal(gperm, perm)
        assert np.array_equal(gls, ls) and np.array_equal(glz, lz)
        assert list(gst) == [len(ls), st[0], st[1], st[2]]


# Nodes that are split in vain again and again (MIN at half of MAX), finished from the distances of their points: leaf limits
# on either side of the square / triangular distance matrix and at the largest node that fits, rows shorter than a
# staging step, D not a multiple of 4, a common offset and duplicated points (nothing but the exact test decides),
# a depth limit that falls inside a chain.
@pytest.mark.parametrize("N,D,MIN,MAX,kind,depth", [
    (4000, 5, 33, 66, "n", 5000), (3000, 1, 8, 16, "n", 5000), (3000, 37, 53, 106, "n", 5000), (3000, 37, 54, 108, "n", 5000),
    (5000, 12, 112, 224, "n", 5000), (3000, 100, 33, 66, "offset", 5000), (3000, 6, 20, 40, "dup", 400), (4000, 16, 33, 66, "n", 14),
    (2500, 260, 60, 120, "n", 5000),
])
@pytest.mark.parametrize("screen", ["q8", "bf16"])
def test_tree_nodes_split_in_vain(gpu, orc, rng, monkeypatch, N, D, MIN, MAX, kind, depth, screen):
    monkeypatch.setenv("RSFK_TREE_SCREEN", screen)
    X = rng.standard_normal((N, D)).astype(np.float32)
    if kind == "offset":
        X = (X * 1e-3 + 1000.0).astype(np.float32)
    if kind == "dup":
        X = X[rng.integers(0, N // 8, N)]
    for seed in (1, 2):
        _say("tree split in vain", N, D, MIN, MAX, kind, depth, seed)
        perm, ls, lz, st = orc.build_tree(X, MIN, MAX, depth, seed)
        gperm, gls, glz, gst = gpu.build_tree(X, MIN, MAX, depth, seed)
        assert np.array_equal(gperm, perm)
        assert np.array_equal(gls, ls) and np.array_equal(glz, lz)
        assert list(gst) == [len(ls), st[0], st[1], st[2]]


# More equal rows than a bucket holds, in nodes that are split until the depth limit: square and triangular distance matrix, all
# points in such groups or a few of them, zeros of either sign (equal coordinates of different bits), rows whose distances
# underflow to zero without being equal, equal rows that hold an infinity.
@pytest.mark.parametrize("N,D,MIN,MAX,kind", [(3000, 6, 20, 40, "groups"), (4000, 33, 17, 34, "some"), (3000, 12, 54, 108, "groups"),
                                              (3000, 7, 33, 66, "zeros"), (2500, 5, 20, 40, "underflow"), (2500, 64, 17, 34, "infinite"),
                                              (2500, 3, 60, 120, "some")])
@pytest.mark.parametrize("screen", ["q8", "bf16"])
def test_tree_nodes_of_equal_rows(gpu, orc, rng, monkeypatch, N, D, MIN, MAX, kind, screen):
    monkeypatch.setenv("RSFK_TREE_SCREEN", screen)
    g = MAX + MAX // 3
    X = rng.standard_normal((N, D)).astype(np.float32)
    m = N if kind == "groups" else N // 4
    X[:m] = np.repeat(X[:m // g + 1], g, axis=0)[:m]
    if kind == "zeros":
        X[:m] = np.where(rng.random((m, D)) < 0.5, np.float32(0.0), np.float32(-0.0))
    if kind == "underflow":
        X[:m] += (rng.standard_normal((m, D)) * 1e-25).astype(np.float32)
        X[: m // 2] = (rng.standard_normal((m // 2, D)) * 1e-25).astype(np.float32)
    if kind == "infinite":
        X[:m, 3] = np.inf
    X = X[rng.permutation(N)]
    for seed in (1, 2):
        _say("tree of equal rows", N, D, MIN, MAX, kind, seed)
        perm, ls, lz, st = orc.build_tree(X, MIN, MAX, 300, seed)
        gperm, gls, glz, gst = gpu.build_tree(X, MIN, MAX, 300, seed)
        assert np.array_equal(gperm, perm)
        assert np.array_equal(gls, ls) and np.array_equal(glz, lz)
        assert list(gst) == [len(ls), st[0], st[1], st[2]]


# Rows whose dot products overflow (all of them near the limit; a tenth of the rows far above the others), overflow in one
# factor only, lie just below and above where the 8-bit copy is given up, or are denormal: every kernel of the side tests (wide levels point by point and node by node, tail, chains).
@pytest.mark.parametrize("kind", ["near_overflow", "mixed", "spread", "below", "above", "denormal"])
@pytest.mark.parametrize("env", [dict(SCREEN="q8", PM="7"), dict(SCREEN="q8", PM="0"), dict(SCREEN="q8", PM="0", TAIL="256"), dict(SCREEN="bf16"),
                                 dict(SCREEN="bf16", TAIL="256")], ids=lambda e: "-".join(e.values()))
def test_tree_of_rows_whose_sums_leave_fp32(gpu, orc, rng, monkeypatch, kind, env):
    for name, var in (("SCREEN", "RSFK_TREE_SCREEN"), ("PM", "RSFK_PM_LEVELS"), ("TAIL", "RSFK_TAIL_BLOCK")):
        if name in env:
            monkeypatch.setenv(var, env[name])
    N, D, MIN, MAX, depth = 6000, 48, 17, 34, 60
    X = rng.standard_normal((N, D))
    most = 7.07e18 / np.sqrt(D) / np.abs(X).max()
    scale = {"near_overflow": 3e18, "below": 0.999 * most, "above": 1.001 * most, "denormal": 3e-22, "mixed": np.where(rng.random((N, 1)) < 0.1, 3e18, 1.0),
             "spread": 10.0 ** rng.uniform(-25, 37, (N, 1))}[kind]
    X = (X * scale).astype(np.float32)
    for seed in (1, 2):
        _say("tree beyond fp32", kind, env, seed)
        perm, ls, lz, st = orc.build_tree(X, MIN, MAX, depth, seed)
        gperm, gls, glz, gst = gpu.build_tree(X, MIN, MAX, depth, seed)
        assert np.array_equal(gperm, perm)
        assert np.array_equal(gls, ls) and np.array_equal(glz, lz)
        assert list(gst) == [len(ls), st[0], st[1], st[2]]


# The bound of the 8-bit rows goes with the largest error of a coordinate or with the root of their mean square, whichever is smaller: a column that
# dwarfs the others (1-norm and 2-norm of a normal nearly the same), coordinates that all lie halfway between two steps (every error as large
# as the largest), all but a few exact, ranges around where squares may underflow, and rows of one value.
@pytest.mark.parametrize("kind", ["column", "halfway", "few_off", "tiny", "tinier", "one_value"])
@pytest.mark.parametrize("D", [3, 48, 100, 260])
@pytest.mark.parametrize("env", [dict(PM="7"), dict(PM="0", TAIL="256")], ids=lambda e: "-".join(e.values()))
def test_tree_bounds_by_largest_and_mean_error(gpu, orc, rng, monkeypatch, kind, D, env):
    monkeypatch.setenv("RSFK_TREE_SCREEN", "q8")
    monkeypatch.setenv("RSFK_PM_LEVELS", env["PM"])
    if "TAIL" in env:
        monkeypatch.setenv("RSFK_TAIL_BLOCK", env["TAIL"])
    N, MIN, MAX = 6000, 17, 34
    X = rng.standard_normal((N, D))
    if kind == "column":
        X[:, 0] *= 1000.0
    if kind == "halfway":                                       # 0, 255 and values k + 1/2 of a scale that is 1
        X = rng.integers(0, 255, (N, D)) + 0.5
        X[:, 0], X[:, 1] = 0.0, 255.0
    if kind == "few_off":
        X = rng.integers(0, 256, (N, D)) + np.where(rng.random((N, D)) < 0.02, 0.49, 0.0)
        X[:, 0], X[:, 1] = 0.0, 255.0
    if kind in ("tiny", "tinier"):
        X *= 1e-12 if kind == "tiny" else 1e-18
    if kind == "one_value":
        X[: N // 2] = rng.standard_normal((N // 2, 1))
    X = X.astype(np.float32)
    _say("tree bounds", kind, D, env)
    perm, ls, lz, st = orc.build_tree(X, MIN, MAX, 300, 1)
    gperm, gls, glz, gst = gpu.build_tree(X, MIN, MAX, 300, 1)
    assert np.array_equal(gperm, perm)
    assert np.array_equal(gls, ls) and np.array_equal(glz, lz)


# The 8-bit copy is the screen while the largest rounding error of its coordinates is below six of bfloat16's mean one, however the errors spread: here
# all coordinates but two lie half a step off, where the bound by the mean square is 1.7 times that by the largest.  Between 0 and 255 the error
# is 0.5, and bfloat16's the mean of the coordinates / 256: 5.0 of it with coordinates of up to 43.5, 10 with up to 15.5.
@pytest.mark.parametrize("top,row_bytes", [(44, 128), (16, 256)])
def test_screen_is_chosen_by_the_largest_error(gpu, orc, rng, top, row_bytes):
    import gpu_rsfk
    N, D, K = 1500, 100, 8
    X = (rng.integers(0, top, (N, D)) + 0.5).astype(np.float32)
    X[:, 3], X[:, 70] = 0.0, 255.0
    _say("screen by the largest error", top)
    gi, gd = gpu_rsfk.RSFK(random_state=2).find_nearest_neighbors(X, K, n_trees=2, nn_exploring_factor=0)
    assert gpu.last_build_report()["tree_screen_row_bytes"] == row_bytes
    oi, od = orc.forest(X, K, 2, K + 1, 2 * (K + 1), 5000, 2, 0)
    assert_knn_equal(gi, gd, oi, od)


# Side tests of the wide levels by the 8-bit copy: rows of 64 bytes and of one line to several, whole or ending in half a line; chunks of any size; rows of NaN,
# equal rows, and a common offset that leaves every point to the exact test; rows whose hyperplane takes more than 48 KB of LDS.
@pytest.mark.parametrize("D", [1, 47, 48, 49, 111, 112, 113, 176, 240, 241, 305, 1100, 13001])
@pytest.mark.parametrize("kind", ["n", "nan", "dup", "offset"])
def test_tree_wide_levels_by_the_8_bit_copy(gpu, orc, rng, monkeypatch, D, kind):
    for name, v in (("SCREEN", "q8"), ("MID", "0"), ("SMALL", "64")):
        monkeypatch.setenv("RSFK_TREE_" + name, v)
    monkeypatch.setenv("RSFK_PM_LEVELS", "0")
    N, MIN, MAX = 5000 if D < 300 else 2500 if D < 2000 else 300, 17, 34
    X = rng.standard_normal((N, D)).astype(np.float32)
    if kind == "nan":
        X[rng.random(N) < 0.02, D // 2] = np.nan
    if kind == "dup":
        X[: N // 3] = X[0]
    if kind == "offset":
        X = (X * 1e-3 + 1000.0).astype(np.float32)
    _say("tree wide levels", D, kind)
    perm, ls, lz, st = orc.build_tree(X, MIN, MAX, 100, 5)
    gperm, gls, glz, gst = gpu.build_tree(X, MIN, MAX, 100, 5)
    assert np.array_equal(gperm, perm)
    assert np.array_equal(gls, ls) and np.array_equal(glz, lz)


# The middle phase in one, two and three launches: largest nodes of up to three times the tail's, of one point more, of up to four times as many and of one
# point more; nodes of a tree that stay above the tail's size after the last of them; many equal rows, whose nodes lose a few points at a time.
@pytest.mark.parametrize("N", [512, 513, 768, 769, 1024, 1025, 1100, 4000, 12000])
@pytest.mark.parametrize("D,kind", [(2, "n"), (40, "n"), (70, "n"), (300, "n"), (5, "dup")])
def test_tree_middle_phase_by_launches(gpu, orc, rng, monkeypatch, N, D, kind):
    for name, v in (("SCREEN", "q8"), ("SMALL", "256")):
        monkeypatch.setenv("RSFK_TREE_" + name, v)
    X = rng.standard_normal((N, D)).astype(np.float32)
    if kind == "dup":
        X[: N // 3] = X[0]
    _say("tree middle phase", N, D, kind)
    perm, ls, lz, st = orc.build_tree(X, 17, 34, 100, 5)
    gperm, gls, glz, gst = gpu.build_tree(X, 17, 34, 100, 5)
    assert np.array_equal(gperm, perm)
    assert np.array_equal(gls, ls) and np.array_equal(glz, lz)


# The forms of the tail and of the chain phase: leaf limits on either side of the sizes of the chain's matrix (nodes of up to 64, 128
# and 256 points, and none), rows on either side of the lanes that share one, many subtrees (nodes above `small` points are wide) and
# few; rows without distances (NaN, and a few far longer than the others), clusters within one node, the index that query points
# are routed by is covered by the tests of the search.
@pytest.mark.parametrize("N,D,MIN,MAX,small,kind", [
    (9000, 7, 20, 40, 2048, "n"), (9000, 7, 20, 41, 2048, "n"), (9000, 40, 56, 113, 2048, "n"), (9000, 40, 57, 114, 2048, "n"),
    (9000, 19, 96, 191, 2048, "n"), (9000, 19, 96, 255, 2048, "n"), (9000, 19, 128, 256, 2048, "n"), (9000, 32, 3, 6, 2048, "n"),
    (30000, 32, 17, 34, 80, "n"), (30000, 64, 17, 34, 80, "n"), (30000, 65, 17, 34, 80, "n"), (12000, 256, 33, 66, 2048, "n"),
    (8000, 257, 33, 66, 2048, "n"), (9000, 24, 33, 66, 2048, "nan"), (9000, 24, 33, 66, 2048, "far"), (9000, 24, 96, 192, 2048, "far"),
    (9000, 36, 33, 66, 2048, "clusters"), (9000, 36, 8, 16, 2048, "clusters"), (6000, 9, 5, 10, 2048, "dup"), (20000, 50, 4, 8, 500, "clusters"),
])
@pytest.mark.parametrize("screen", ["q8", "bf16"])
@pytest.mark.parametrize("subtrees", ["few", "many"])
def test_tree_forms_of_tail_and_chain(gpu, orc, rng, monkeypatch, N, D, MIN, MAX, small, kind, screen, subtrees):
    if subtrees == "many":                                      # nodes leave for the chain phase after splits in vain
        monkeypatch.setenv("RSFK_TAIL_BLOCK", "256")
    monkeypatch.setenv("RSFK_TREE_SCREEN", screen)
    monkeypatch.setenv("RSFK_TREE_SMALL", str(small))
    X = rng.standard_normal((N, D)).astype(np.float32)
    if kind == "nan":
        X[rng.random(N) < 0.01, 1] = np.nan
    if kind == "far":
        X[rng.random(N) < 0.02] *= np.float32(1e3)
    if kind == "dup":
        X[: N // 3] = X[0]
    if kind == "clusters":
        X = (10.0 * rng.standard_normal((40, D))[rng.integers(0, 40, N)] + 1e-3 * X).astype(np.float32)
    for seed in (1, 2):
        _say("tree forms", N, D, MIN, MAX, small, kind, screen, seed)
        perm, ls, lz, st = orc.build_tree(X, MIN, MAX, 300, seed)
        gperm, gls, glz, gst = gpu.build_tree(X, MIN, MAX, 300, seed)
        assert np.array_equal(gperm, perm)
        assert np.array_equal(gls, ls) and np.array_equal(glz, lz)
        assert list(gst) == [len(ls), st[0], st[1], st[2]]


@pytest.mark.parametrize("K", [3, 12])
def test_index_of_nodes_that_leave_the_tail(gpu, orc, rng, monkeypatch, K):
    """Many subtrees: the index that query points are routed by, where nodes leave for the chain phase after splits in vain."""
    import gpu_rsfk
    monkeypatch.setenv("RSFK_TAIL_BLOCK", "256")
    N, NQ, D = 20000, 1500, 30
    X = (10.0 * rng.standard_normal((50, D))[rng.integers(0, 50, N + NQ)] + 0.3 * rng.standard_normal((N + NQ, D))).astype(np.float32)
    X, Q = np.ascontiguousarray(X[:N]), np.ascontiguousarray(X[N:])
    _say("index, splits in vain", K)
    gi, gd = gpu_rsfk.RSFK(random_state=5).find_nearest_neighbors_ann(X, Q, K, n_trees=3)
    oi, od = orc.ann_forest(X, Q, K, 3, K + 1, 2 * (K + 1), 5000, 5)
    assert_knn_equal(gi, gd, oi, od)


# The middle phase: nodes it takes whole (N at most its largest), from the wide levels, of sizes around a thread's last entry, one that
# is barely larger than what the tail takes; equal rows (splits in vain up to the depth limit); leaf limits above the tail's nodes.
@pytest.mark.parametrize("N,D,MIN,MAX,small,mid,kind", [
    (1025, 5, 17, 34, 64, 12288, "n"), (12288, 3, 64, 256, 2048, 12288, "n"), (12289, 3, 64, 256, 2048, 12288, "n"), (30000, 32, 17, 34, 96, 1024, "n"),
    (30000, 64, 33, 66, 128, 4096, "n"), (12000, 65, 33, 66, 128, 1088, "n"), (9000, 257, 17, 34, 64, 2048, "n"), (15000, 16, 400, 1000, 200, 12288, "n"),
    (6000, 9, 5, 10, 64, 12288, "dup"), (5000, 4, 1, 3, 64, 12288, "n"),
])
def test_tree_middle_phase(gpu, orc, rng, monkeypatch, N, D, MIN, MAX, small, mid, kind):
    monkeypatch.setenv("RSFK_TREE_SCREEN", "q8")
    monkeypatch.setenv("RSFK_TREE_SMALL", str(small))
    monkeypatch.setenv("RSFK_TREE_MID", str(mid))
    X = rng.standard_normal((N, D)).astype(np.float32)
    if kind == "dup":
        X[: N // 3] = X[0]
    for depth in (200, 6):
        _say("tree middle phase", N, D, MIN, MAX, small, mid, kind, depth)
        perm, ls, lz, st = orc.build_tree(X, MIN, MAX, depth, 3)
        gperm, gls, glz, gst = gpu.build_tree(X, MIN, MAX, depth, 3)
        assert np.array_equal(gperm, perm)
        assert np.array_equal(gls, ls) and np.array_equal(glz, lz)
        assert list(gst) == [len(ls), st[0], st[1], st[2]]


def test_tree_edge_cases(gpu, orc, rng):
    # identical points: re-drawn until the depth limit, then one forced bucket
    X = np.ones((3000, 4), np.float32)
    _say("tree identical points")
    gperm, gls, glz, gst = gpu.build_tree(X, 5, 10, 30, 0)
    perm, ls, lz, st = orc.build_tree(X, 5, 10, 30, 0)
    assert list(glz) == [3000] == list(lz) and gst[1] == st[0] == 30
    # depth limits
    X = rng.random((5000, 6), dtype=np.float32)
    for depth in (1, 2, 5, 12):
        _say("tree depth limit", depth)
        g = gpu.build_tree(X, 5, 10, depth, 1)
        o = orc.build_tree(X, 5, 10, depth, 1)
        assert np.array_equal(g[0], o[0]) and np.array_equal(g[2], o[2]) and g[3][1] == o[3][0] <= depth
    # duplicated points mixed with distinct ones, N smaller than MIN
    X = np.repeat(rng.random((300, 3), dtype=np.float32), 7, axis=0)
    _say("tree duplicates")
    g = gpu.build_tree(X, 9, 20, 200, 4)
    o = orc.build_tree(X, 9, 20, 200, 4)
    assert np.array_equal(g[0], o[0]) and np.array_equal(g[2], o[2])
    X = rng.random((20, 3), dtype=np.float32)
    g = gpu.build_tree(X, 33, 66, 5000, 0)
    assert list(g[2]) == [20]


# Buckets of a point or two: the tail kernel's lists of nodes and buckets leave room for few hyperplanes, down to one at a time (long rows)
@pytest.mark.parametrize("N,D,MIN,MAX", [(45, 99, 2, 4), (3000, 49, 2, 4), (5000, 100, 2, 5), (2500, 784, 2, 4), (2100, 2050, 2, 9), (300, 11152, 2, 4),
                                         (2600, 240, 2, 3), (3000, 100, 1, 4)])
@pytest.mark.parametrize("screen", ["auto", "q8", "bf16", "q8-256"])
def test_tree_of_buckets_of_two(gpu, orc, rng, monkeypatch, N, D, MIN, MAX, screen):
    """A partition with the shortest buckets over rows of more than 48 dimensions == the oracle's."""
    if screen == "q8-256":
        monkeypatch.setenv("RSFK_TREE_SCREEN", "q8")
        monkeypatch.setenv("RSFK_TAIL_BLOCK", "256")
    elif screen != "auto":
        monkeypatch.setenv("RSFK_TREE_SCREEN", screen)
    X = rng.standard_normal((N, D)).astype(np.float32)
    X[rng.random(N) < 0.1] = X[0]
    for depth in (5000, 9):
        _say("tree of buckets of two", N, D, MIN, MAX, screen, depth)
        perm, ls, lz, st = orc.build_tree(X, MIN, MAX, depth, 3)
        gperm, gls, glz, gst = gpu.build_tree(X, MIN, MAX, depth, 3)
        assert np.array_equal(gperm, perm)
        assert np.array_equal(gls, ls) and np.array_equal(glz, lz)
        assert list(gst) == [len(ls), st[0], st[1], st[2]]


@pytest.mark.parametrize("N,NQ,D,K,T,mn,mx", [(45, 30, 99, 7, 6, 2, 4), (4000, 500, 64, 5, 4, 2, 4), (1500, 200, 300, 10, 3, 2, 5)])
def test_search_and_build_with_buckets_of_two(gpu, orc, rng, N, NQ, D, K, T, mn, mx):
    """The trees of a K-NN build and those that carry an index, with the shortest buckets."""
    import gpu_rsfk
    X, Q = rng.standard_normal((N, D)).astype(np.float32), rng.standard_normal((NQ, D)).astype(np.float32)
    r = gpu_rsfk.RSFK(random_state=4)
    _say("build and search with buckets of two", N, NQ, D, K, T)
    gi, gd = r.find_nearest_neighbors(X, K, n_trees=T, min_tree_children=mn, max_tree_children=mx, nn_exploring_factor=1, ensure_valid_indices=False)
    oi, od = orc.forest(X, K, T, mn, mx, 5000, 4, 1)
    assert_knn_equal(gi, gd, oi, od)
    gi, gd = r.find_nearest_neighbors_ann(X, Q, K, n_trees=T, min_tree_children=mn, max_tree_children=mx, ensure_valid_indices=False)
    oi, od = orc.ann_forest(X, Q, K, T, mn, mx, 5000, 4)
    assert_knn_equal(gi, gd, oi, od)


# ---------------------------------------------------------------------------
# bucket K-NN on a fixed partition
# ---------------------------------------------------------------------------
@pytest.mark.parametrize("N,D,K,MIN,MAX", [
    (2000, 32, 16, 17, 34), (3000, 100, 32, 33, 66), (3000, 33, 8, 100, 300), (1500, 7, 90, 91, 182),
    (1200, 1, 4, 5, 10), (2500, 3, 1, 2, 4), (2000, 130, 64, 65, 130), (1500, 20, 65, 66, 140),
    (1800, 12, 200, 201, 420), (4000, 256, 32, 33, 66), (1500, 784, 90, 91, 182), (2000, 30, 32, 400, 1024),
    (2500, 10, 300, 301, 620), (4200, 6, 700, 701, 1500), (1600, 40, 1024, 400, 900),
])
@pytest.mark.parametrize("kernel", ["direct", "direct_per_bucket", "direct_per_64", "pairs_in_parts", "gram", "screen"])
def test_bucket_knn_matches_oracle(gpu, orc, rng, monkeypatch, N, D, K, MIN, MAX, kernel):
    """kernel: "direct" = fp32 chains for every pair, the buckets the specialised kernels leave through the pair of
    kernels that evaluates every pair once and hands the distances on through memory; "pairs_in_parts" = the same with
    1 MB of that memory, so that a launch goes in many parts (RSFK_BUCKET_PAIRS_MB=1), and without the kernel that keeps
    a bucket's points in LDS (RSFK_BUCKET_ROWS=0); "direct_per_bucket" / "direct_per_64" = the tiled kernels that need
    no working memory (RSFK_BUCKET_PAIRS=0), a workgroup per bucket or per 64 members of a bucket
    (RSFK_BUCKET_STRIP=0 / 1), also without the kernel for resident buckets; "gram" = the kernel that bounds the pair
    matrix on the matrix cores first and runs the chains only for the pairs that may enter a row (RSFK_GRAM_FROM=0);
    "screen" = the same idea in the two-wavefront kernel for buckets of up to 64 points (RSFK_BUCKET_SCREEN=always;
    other buckets, and K > 64, take the direct kernels)."""
    if kernel in ("direct_per_bucket", "direct_per_64", "pairs_in_parts"):
        if MAX <= 72 and K <= 64:
            pytest.skip("no bucket of this shape reaches the tiled kernels")
        monkeypatch.setenv("RSFK_BUCKET_ROWS", "0")
        if kernel == "pairs_in_parts":
            monkeypatch.setenv("RSFK_BUCKET_PAIRS_MB", "1")
        else:
            monkeypatch.setenv("RSFK_BUCKET_PAIRS", "0")
            monkeypatch.setenv("RSFK_BUCKET_STRIP", "0" if kernel == "direct_per_bucket" else "1")
    if kernel == "gram":
        monkeypatch.setenv("RSFK_GRAM_FROM", "0")
    if kernel == "screen":
        if K > 64 or MIN > 64:
            pytest.skip("no bucket of this shape reaches the screened small-bucket kernel")
        monkeypatch.setenv("RSFK_BUCKET_SCREEN", "always")
    X = rng.random((N, D), dtype=np.float32)
    oi, od = orc.init_lists(N, K)
    gi, gd = orc.init_lists(N, K)
    for seed in (3, 4):
        _say("bucket_knn", N, D, K, MIN, MAX, seed)
        perm, ls, lz, _ = orc.build_tree(X, MIN, MAX, 5000, seed)
        orc.bucket_knn(X, K, perm, lz, oi, od, starts=ls)
        gpu.bucket_knn(X, K, perm, lz, gi, gd, starts=ls)
        assert_knn_equal(gi, gd, oi, od)
        assert rows_have_no_duplicates(gi)


@pytest.mark.parametrize("N,D,K,MIN,MAX", [
    (4000, 32, 32, 64, 256), (3000, 48, 20, 80, 200), (2500, 16, 64, 70, 250), (3000, 64, 8, 65, 128),
    (2600, 32, 5, 30, 256),
])
def test_bucket_knn_resident_rows_matches_oracle(gpu, orc, rng, N, D, K, MIN, MAX):
    """Buckets of 73..256 low-dimensional points go to the kernel that keeps a bucket's points in LDS.  Three trees on
    the same rows of normally distributed points: in the second and third most candidates are above the last slot of
    the row they are offered to, and many of the others are points the row already holds."""
    X = rng.standard_normal((N, D)).astype(np.float32)
    oi, od = orc.init_lists(N, K)
    gi, gd = orc.init_lists(N, K)
    for seed in (3, 4, 5):
        _say("bucket_knn resident rows", N, D, K, MIN, MAX, seed)
        perm, ls, lz, _ = orc.build_tree(X, MIN, MAX, 5000, seed)
        orc.bucket_knn(X, K, perm, lz, oi, od, starts=ls)
        gpu.bucket_knn(X, K, perm, lz, gi, gd, starts=ls)
        assert_knn_equal(gi, gd, oi, od)
        assert rows_have_no_duplicates(gi)


@pytest.mark.parametrize("K", [20, 64])
@pytest.mark.parametrize("data", ["continuous", "grid", "mixed"])
@pytest.mark.parametrize("start", ["self", "empty", "self_far", "other"])
def test_bucket_knn_rows_that_start_new(gpu, orc, rng, start, data, K):
    """A row that holds at most the point itself is filled by counting, for every candidate, the candidates below it;
    two candidates at the same distance send the row to the insertions instead.  Rows start with the point itself,
    empty, with the point itself at a distance that is not 0, or with one other point (then they are not new); the points
    are continuous (no equal distances), on a small grid (nothing but equal distances and duplicates) or both.  Buckets
    of up to 72 points, so that both shapes of the small-bucket kernel run; with K = 64 the first tree does not fill
    the rows and the second finds rows that are neither new nor full."""
    N, D = 3000, 6
    X = rng.random((N, D), dtype=np.float32)
    if data == "grid":
        X = rng.integers(0, 3, (N, D)).astype(np.float32)
    elif data == "mixed":
        some = rng.random(N) < 0.05
        X[some] = rng.integers(0, 2, (int(some.sum()), D)).astype(np.float32)
    oi = np.full((N, K), -1, np.int32)
    od = np.full((N, K), np.inf, np.float32)
    if start in ("self", "self_far"):
        oi[:, 0] = np.arange(N)
        od[:, 0] = 0.0 if start == "self" else 0.3
    elif start == "other":
        # the point's partner in the pairs (0, 1), (2, 3), ... at its distance (a row must not hold a wrong distance:
        # an index could then leave the row and come back with another one, and the result would depend on the order)
        ti, td = orc.init_lists(N, 2)
        orc.bucket_knn(X, 2, np.arange(N, dtype=np.int32), np.full(N // 2, 2, np.int32), ti, td,
                       starts=np.arange(0, N, 2, dtype=np.int32))
        first_is_self = ti[:, 0] == np.arange(N)
        oi[:, 0] = np.where(first_is_self, ti[:, 1], ti[:, 0])
        od[:, 0] = np.where(first_is_self, td[:, 1], td[:, 0])
    gi, gd = oi.copy(), od.copy()
    for seed in (3, 4):
        _say("bucket_knn new rows", start, data, K, seed)
        perm, ls, lz, _ = orc.build_tree(X, 21, 72, 5000, seed)
        orc.bucket_knn(X, K, perm, lz, oi, od, starts=ls)
        gpu.bucket_knn(X, K, perm, lz, gi, gd, starts=ls)
        assert_knn_equal(gi, gd, oi, od)
        assert rows_have_no_duplicates(gi)


@pytest.mark.parametrize("data", ["continuous", "grid", "mixed", "notfinite"])
@pytest.mark.parametrize("start", ["self", "empty", "self_far", "flt_max"])
@pytest.mark.parametrize("K,MIN,MAX", [(8, 40, 120), (32, 64, 256), (60, 61, 200), (64, 33, 190)])
def test_bucket_knn_resident_rows_merged_by_counting(gpu, orc, rng, K, MIN, MAX, start, data):
    """Buckets of 73..256 points whose rows are merged by counting: rows that are new, rows of which most points are in the bucket
    again (the same partition twice), rows that are neither new nor full, equal distances, duplicated points, points that are not
    finite, and rows too long for one wavefront to count.  Empty slots hold +inf, or FLT_MAX as the reference's CLI leaves them."""
    N, D = 4000, 5
    X = rng.standard_normal((N, D)).astype(np.float32)
    perm, ls, lz, _ = orc.build_tree(X, MIN, MAX, 5000, 3)
    parts = [(perm, ls, lz), (perm, ls, lz), orc.build_tree(X, MIN, MAX, 5000, 4)[:3]]
    if data == "grid":
        X = rng.integers(0, 3, (N, D)).astype(np.float32)
    elif data == "mixed":
        some = rng.random(N) < 0.1
        X[some] = rng.integers(0, 2, (int(some.sum()), D)).astype(np.float32)
    elif data == "notfinite":
        X[rng.integers(0, N, 30), rng.integers(0, D, 30)] = np.nan
        X[rng.integers(0, N, 30), 0] = np.inf
    oi = np.full((N, K), -1, np.int32)
    od = np.full((N, K), np.finfo(np.float32).max if start == "flt_max" else np.inf, np.float32)
    if start != "empty":
        oi[:, 0] = np.arange(N)
        od[:, 0] = 0.3 if start == "self_far" else 0.0
    gi, gd = oi.copy(), od.copy()
    for perm, ls, lz in parts:
        _say("bucket_knn by counting", K, MIN, MAX, start, data)
        orc.bucket_knn(X, K, perm, lz, oi, od, starts=ls)
        gpu.bucket_knn(X, K, perm, lz, gi, gd, starts=ls)
        assert_knn_equal(gi, gd, oi, od)
        assert rows_have_no_duplicates(gi)


def _in_order_without_holes(idx, dist):
    """Rows ascend, and no empty slot stands before a neighbour."""
    return not ((idx[:, :-1] < 0) & (idx[:, 1:] >= 0)).any() and (dist[:, :-1] <= dist[:, 1:]).all()


# rows counted by a wavefront (K + 4 at most 64) and longer ones; dimensions on both sides of the line between counting and insertions
@pytest.mark.parametrize("data", ["continuous", "mixed"])
@pytest.mark.parametrize("which", ["nearest", "any", "pairs"])
@pytest.mark.parametrize("K,MIN,MAX,D", [(8, 40, 120, 9), (8, 80, 200, 4), (32, 64, 256, 9), (32, 64, 256, 5), (50, 74, 190, 7), (60, 61, 200, 6), (64, 70, 190, 12)])
def test_bucket_knn_resident_rows_that_hold_one_other_point(gpu, orc, rng, K, MIN, MAX, D, which, data):
    """A row whose only entry is a neighbour (with its distance) from the bucket the row meets next: the candidate that is that neighbour must
    not be counted a second time.  The neighbour is the nearest, any other one of the bucket, or what a partition into pairs left in
    rows that began empty; a fifth of the rows holds the point itself alone, or nothing."""
    N = 4000
    X = rng.standard_normal((N, D)).astype(np.float32)
    if data == "mixed":
        some = rng.random(N) < 0.1
        X[some] = rng.integers(0, 2, (int(some.sum()), D)).astype(np.float32)
    perm, ls, lz, _ = orc.build_tree(X, MIN, MAX, 5000, 3)
    oi = np.full((N, K), -1, np.int32)
    od = np.full((N, K), np.inf, np.float32)
    parts = [(perm, ls, lz), orc.build_tree(X, MIN, MAX, 5000, 4)[:3]]
    if which == "pairs":
        parts.insert(0, (perm, np.arange(0, N, 2, dtype=np.int32), np.full(N // 2, 2, np.int32)))
    else:
        ti, td = np.full((N, MAX), -1, np.int32), np.full((N, MAX), np.inf, np.float32)
        orc.bucket_knn(X, MAX, perm, lz, ti, td, starts=ls)
        at = np.zeros(N, np.int64) if which == "nearest" else rng.integers(0, (ti >= 0).sum(1))
        order = np.lexsort((ti, td), axis=1)[np.arange(N), at]
        oi[:, 0], od[:, 0] = ti[np.arange(N), order], td[np.arange(N), order]
        alone, nothing = rng.random(N) < 0.1, rng.random(N) < 0.1
        oi[alone, 0], od[alone, 0] = np.flatnonzero(alone), 0.0
        oi[nothing, 0], od[nothing, 0] = -1, np.inf
    gi, gd = oi.copy(), od.copy()
    for perm, ls, lz in parts:
        _say("bucket_knn rows with one other point", K, MIN, MAX, D, which, data)
        orc.bucket_knn(X, K, perm, lz, oi, od, starts=ls)
        gpu.bucket_knn(X, K, perm, lz, gi, gd, starts=ls)
        assert_knn_equal(gi, gd, oi, od)
        assert rows_have_no_duplicates(gi)
        assert _in_order_without_holes(gi, gd)


@pytest.mark.parametrize("N,D,K,T", [(6000, 3, 32, 1), (6000, 9, 32, 1), (5000, 7, 45, 2), (4000, 6, 63, 1)])
def test_extra_tree_after_buckets_of_two(gpu, orc, rng, N, D, K, T):
    """Rows that begin empty and meet buckets of 2 to 4 points, then those of the extra tree of ensure_valid_indices: up to 3 (K + 1) points, so
    that rows of a single neighbour are offered a resident bucket."""
    import gpu_rsfk
    mn, mx = 2, 4
    X = rng.standard_normal((N, D)).astype(np.float32)
    r = gpu_rsfk.RSFK(random_state=4)
    for nnef in (0, 1):
        _say("extra tree", N, D, K, T, nnef)
        gi, gd = r.find_nearest_neighbors(X, K, n_trees=T, min_tree_children=mn, max_tree_children=mx, nn_exploring_factor=nnef,
                                          point_in_self_neigh=False)
        oi, od = orc.init_lists(N, K, self_in=False)
        oi, od = orc.forest(X, K, T, mn, mx, 5000, 4, nnef, knn_idx=oi, knn_dist=od)
        oi, od = orc.forest(X, K, 1, K + 1, 3 * (K + 1), 5000, 4, nnef, knn_idx=oi, knn_dist=od)
        assert_knn_equal(gi, gd, oi, od)
        assert _in_order_without_holes(gi, gd)


def test_bucket_knn_single_bucket_is_exact_knn(gpu, rng):
    """One bucket holding every point: the kernel must return exact K-NN."""
    for N, D, K in [(300, 8, 16), (700, 20, 32)]:
        _say("bucket_knn all-in-one", N, D, K)
        X = rng.random((N, D), dtype=np.float32)
        gi = np.full((N, K), -1, np.int32)
        gd = np.full((N, K), np.inf, np.float32)
        gi[:, 0] = np.arange(N)
        gd[:, 0] = 0
        gpu.bucket_knn(X, K, np.arange(N, dtype=np.int32), np.array([N], np.int32), gi, gd,
                       starts=np.array([0], np.int32))
        ti, td = exact_knn_numpy(X, K)
        si, sd = sort_rows(gi, gd)
        assert np.array_equal(np.sort(si, 1), np.sort(ti, 1))
        assert np.allclose(sd, td, rtol=1e-5, atol=1e-7)          # direct-difference path: 1e-5 relative


def test_bucket_knn_padded_matrix_ragged_and_empty(gpu, orc, rng):
    N, D, K = 1500, 10, 8
    X = rng.random((N, D), dtype=np.float32)
    perm, ls, lz, _ = orc.build_tree(X, 9, 40, 5000, 2)
    mc = int(lz.max())
    # padded matrix with two extra buckets of size 0 and 1 (never produce candidates)
    nb = len(lz) + 2
    padded = np.full((nb, mc), -1, np.int32)
    sizes = np.zeros(nb, np.int32)
    for b, (s, z) in enumerate(zip(ls, lz)):
        padded[b, :z] = perm[s:s + z]
        sizes[b] = z
    padded[nb - 1, 0] = 5
    sizes[nb - 1] = 1
    oi, od = orc.init_lists(N, K)
    gi, gd = orc.init_lists(N, K)
    orc.bucket_knn(X, K, padded.ravel(), sizes, oi, od, starts=None, stride=mc)
    _say("bucket_knn padded")
    gpu.bucket_knn(X, K, padded.ravel(), sizes, gi, gd, starts=None, stride=mc)
    assert_knn_equal(gi, gd, oi, od)
    # FLT_MAX instead of +inf in the empty slots (the reference's CLI initialisation)
    gi2 = np.full((N, K), -1, np.int32)
    gd2 = np.full((N, K), np.finfo(np.float32).max, np.float32)
    oi2, od2 = gi2.copy(), gd2.copy()
    orc.bucket_knn(X, K, perm, lz, oi2, od2, starts=ls)
    gpu.bucket_knn(X, K, perm, lz, gi2, gd2, starts=ls)
    assert_knn_equal(gi2, gd2, oi2, od2)
    # nothing to do
    gpu.bucket_knn(X, K, perm, np.zeros(0, np.int32), gi2, gd2, starts=np.zeros(0, np.int32))
    # bad ids are rejected on the host
    with pytest.raises(gpu.RsfkError):
        gpu.bucket_knn(X, K, np.array([0, 1, N], np.int32), np.array([3], np.int32), gi2, gd2,
                       starts=np.array([0], np.int32))


@pytest.mark.parametrize("memory_mb", [None, "1"])
def test_bucket_knn_padded_matrix_of_large_buckets(gpu, orc, rng, monkeypatch, memory_mb):
    """Buckets handed over as rows of a padded matrix (no table of starts) that reach the pair of kernels which passes
    a bucket's distances through working memory: all at once, and in parts of a few buckets (1 MB of that memory)."""
    if memory_mb:
        monkeypatch.setenv("RSFK_BUCKET_PAIRS_MB", memory_mb)
    N, D, K = 2600, 12, 70
    X = rng.random((N, D), dtype=np.float32)
    perm, ls, lz, _ = orc.build_tree(X, 71, 150, 5000, 8)
    mc = int(lz.max())
    nb = len(lz) + 1
    padded = np.full((nb, mc), -1, np.int32)
    sizes = np.zeros(nb, np.int32)                      # the bucket in the middle of the matrix is empty
    for b, (s, z) in enumerate(zip(ls, lz)):
        row = b if b < nb // 2 else b + 1
        padded[row, :z] = perm[s:s + z]
        sizes[row] = z
    oi, od = orc.init_lists(N, K)
    gi, gd = orc.init_lists(N, K)
    for _ in range(2):                                  # the second call finds rows that are full
        orc.bucket_knn(X, K, padded.ravel(), sizes, oi, od, starts=None, stride=mc)
        _say("bucket_knn padded, large buckets", memory_mb)
        gpu.bucket_knn(X, K, padded.ravel(), sizes, gi, gd, starts=None, stride=mc)
        assert_knn_equal(gi, gd, oi, od)


# ---------------------------------------------------------------------------
# exploration
# ---------------------------------------------------------------------------
@pytest.mark.parametrize("join", ["join", "plain", "staged"])
@pytest.mark.parametrize("N,D,K,self_in", [(3000, 32, 16, True), (2000, 100, 32, True), (1500, 5, 8, False),
                                           (1200, 9, 90, True), (900, 3, 1, True), (2500, 20, 40, True),
                                           (1300, 6, 200, True), (40, 7, 33, True), (5000, 130, 12, True),
                                           (2200, 24, 64, True), (1600, 300, 100, True), (2600, 48, 20, True),
                                           (3000, 200, 32, True), (1100, 6, 300, True), (800, 5, 520, False)])
def test_explore_matches_oracle(gpu, orc, rng, monkeypatch, N, D, K, self_in, join):
    """Both ways of enumerating the candidates: the join over the reversed graph (default; with partly empty
    rows and a large K its marks overflow the small set; K above about 45 then takes the merge kernel that puts a
    whole workgroup on a point, and the general kernel finishes what is left; rows of more than 128 dimensions have
    their candidates taken nearer lower bounds first, several hundred per point at 3000 x 200 with K = 32),
    the same with the reversed graph made by the builder for large graphs (RSFK_REV_STAGED=1: two scatters staged in
    LDS, rows assembled in LDS), and every point for itself (RSFK_EXPLORE_JOIN=0)."""
    if join == "plain":
        monkeypatch.setenv("RSFK_EXPLORE_JOIN", "0")
    if join == "staged":
        if K > 256:
            pytest.skip("rows of more than 256 neighbours never take the join")
        monkeypatch.setenv("RSFK_REV_STAGED", "1")
    X = rng.random((N, D), dtype=np.float32)
    oi, od = orc.init_lists(N, K, self_in=self_in)
    MIN = max(2, K // 2)                 # buckets smaller than K+1 leave some rows partly empty
    for seed in range(2):
        perm, ls, lz, _ = orc.build_tree(X, MIN, 2 * MIN + 3, 5000, seed)
        orc.bucket_knn(X, K, perm, lz, oi, od, starts=ls)
    gi, gd = oi.copy(), od.copy()
    for _ in range(2):
        _say("explore", N, D, K, self_in)
        orc.explore(X, K, oi, od)
        gpu.explore(X, K, gi, gd, 1)
        assert_knn_equal(gi, gd, oi, od)
        assert rows_have_no_duplicates(gi)
    if not self_in:
        assert not (gi == np.arange(N)[:, None]).any()


@pytest.mark.parametrize("N,D,K", [(6000, 20, 16), (3000, 48, 90), (20001, 6, 5)])
def test_explore_with_the_reversed_graph_by_tiles(gpu, orc, rng, monkeypatch, N, D, K):
    """RSFK_REV_STAGED=2: the builder of medium graphs, bins of one point to 32, more than a tile of entries per part."""
    monkeypatch.setenv("RSFK_REV_STAGED", "2")
    X = rng.random((N, D), dtype=np.float32)
    oi, od = orc.init_lists(N, K, self_in=True)
    perm, ls, lz, _ = orc.build_tree(X, K + 1, 2 * K + 2, 5000, 0)
    orc.bucket_knn(X, K, perm, lz, oi, od, starts=ls)
    gi, gd = oi.copy(), od.copy()
    _say("explore tiles", N, D, K)
    orc.explore(X, K, oi, od)
    gpu.explore(X, K, gi, gd, 1)
    assert_knn_equal(gi, gd, oi, od)


@pytest.mark.parametrize("N,D,K", [(70001, 6, 31), (66000, 20, 32), (9001, 12, 3), (5000, 40, 1), (700, 33, 32), (2000, 20, 45), (3000, 65, 31),
                                   (2300, 100, 32), (2500, 128, 20), (600, 110, 90)])
def test_explore_with_the_staged_reversed_graph(gpu, orc, rng, monkeypatch, N, D, K):
    """RSFK_REV_STAGED=1: marks put in place window by window (more than 2^21 of them, a last piece of any length, few), bars as 16-bit codes beside
    the entries and, with few neighbours, gathered; rows that are not full; points far out, whose rounding errors are large.  More than 32
    neighbours: marks stored one by one, and, by the workgroups of rows without codes, from the bars themselves."""
    monkeypatch.setenv("RSFK_REV_STAGED", "1")
    if K > 64:
        monkeypatch.setenv("RSFK_OPTIONAL_MB", "0")
    X = rng.random((N, D), dtype=np.float32)
    X[::97] *= 1000.0
    oi, od = orc.init_lists(N, K, self_in=True)
    perm, ls, lz, _ = orc.build_tree(X, K + 1, 2 * K + 2, 5000, 0)
    orc.bucket_knn(X, K, perm, lz, oi, od, starts=ls)
    if K > 2:
        far = np.argsort(od, axis=1)[::7, -(K // 2):]
        rows = np.arange(0, N, 7)[:, None]
        oi[rows, far], od[rows, far] = -1, np.inf
    gi, gd = oi.copy(), od.copy()
    for _ in range(2):
        _say("explore staged", N, D, K)
        orc.explore(X, K, oi, od)
        gpu.explore(X, K, gi, gd, 1)
        assert_knn_equal(gi, gd, oi, od)


@pytest.mark.parametrize("values", ["any", "whole", "near"])
@pytest.mark.parametrize("N,D,K", [(1500, 6, 1), (3000, 3, 32), (3000, 33, 33), (2500, 130, 31), (2000, 8, 64), (1500, 200, 64), (1800, 20, 65),
                                   (1500, 12, 128), (1500, 140, 90), (1600, 10, 200)])
def test_explore_batches_merged_by_rank(gpu, orc, rng, N, D, K, values):
    """Rows of one, two and four slots per lane, with and without the tile, a wavefront and a workgroup per point; few and many entering
    candidates; distances that are equal (whole numbers) or differ in the last bits."""
    X = rng.standard_normal((N, D)).astype(np.float32)
    if values == "whole":
        X = np.round(X * np.float32(1.2)).astype(np.float32)
    elif values == "near":
        X = (np.float32(1) + np.float32(2.0 ** -20) * np.round(X * 8)).astype(np.float32)
    oi, od = orc.init_lists(N, K, self_in=True)
    perm, ls, lz, _ = orc.build_tree(X, K + 1, 2 * K + 2, 5000, 0)
    orc.bucket_knn(X, K, perm, lz, oi, od, starts=ls)
    gi, gd = oi.copy(), od.copy()
    _say("explore by rank", N, D, K, values)
    for _ in range(2):                                          # (the second pass: few enter)
        orc.explore(X, K, oi, od)
        gpu.explore(X, K, gi, gd, 1)
        assert_knn_equal(gi, gd, oi, od)


# fewer points than shares of the list, one point in the last share, whole shares; a workgroup per point after it (K = 100)
@pytest.mark.parametrize("N,D,K,T", [(20, 4, 9, 3), (65, 3, 20, 4), (1025, 8, 32, 8), (4224, 6, 30, 6), (4500, 12, 100, 5)])
def test_explore_points_with_many_marks_are_handed_on(gpu, capi, orc, rng, N, D, K, T):
    """Clusters little larger than a row: the neighbours of a point's neighbours are its own, so that most points have more marks than
    the first launch has room for and go to the next one through a list kept in shares."""
    import torch
    X = (rng.standard_normal((max(1, N // (2 * K)), D))[rng.integers(0, max(1, N // (2 * K)), N)] * 20 + rng.standard_normal((N, D))).astype(np.float32)
    oi, od = orc.forest(X, K, T, K + 1, 2 * K + 2, 5000, 3, 2)
    gi, gd = orc.init_lists(N, K, self_in=True)
    dX, di, dd = (torch.from_numpy(a).cuda() for a in (X, gi, gd))
    _say("explore handed on", N, D, K, T)
    capi.knn_forest_device(T, K, N, D, K + 1, 2 * K + 2, 5000, 0, 3, 2, dX.data_ptr(), di.data_ptr(), dd.data_ptr())
    torch.cuda.synchronize()
    assert_knn_equal(di.cpu().numpy(), dd.cpu().numpy(), oi, od)


# both sides of every line between the joins: neighbours in one to seven groups of 32, whole and with one over; dimensions around the
# largest that stay in registers and around those from which a workgroup takes a point
@pytest.mark.parametrize("N,D,K", [(900, 128, 33), (900, 129, 33), (700, 64, 64), (700, 200, 64), (600, 201, 64), (500, 500, 40), (500, 501, 40), (700, 32, 65),
                                   (600, 98, 90), (600, 99, 90), (700, 90, 96), (600, 17, 97), (600, 28, 128), (600, 29, 128), (500, 16, 129), (400, 130, 200), (300, 698, 160), (300, 700, 160), (400, 411, 256)])
@pytest.mark.parametrize("data", ["normal", "notfinite", "no codes"])
def test_explore_join_of_rows_of_many_neighbours(gpu, orc, rng, monkeypatch, N, D, K, data):
    """A wavefront per 32 neighbours of a point, a wavefront per point, a workgroup per point, with and without room for the codes == the
    oracle, two passes."""
    if data == "no codes":
        monkeypatch.setenv("RSFK_OPTIONAL_MB", "0")
    X = rng.standard_normal((N, D)).astype(np.float32)
    perm, ls, lz, _ = orc.build_tree(X, K + 1, 2 * K + 2, 5000, 0)
    if data == "notfinite":
        X[3, D // 2] = np.nan
        X[N - 1, D - 1] = -np.inf
    oi, od = orc.init_lists(N, K, self_in=True)
    orc.bucket_knn(X, K, perm, lz, oi, od, starts=ls)
    gi, gd = oi.copy(), od.copy()
    _say("explore join", N, D, K, data)
    for _ in range(2):
        orc.explore(X, K, oi, od)
        gpu.explore(X, K, gi, gd, 1)
        assert_knn_equal(gi, gd, oi, od)


# rows shorter than what four lanes load, of whole pieces and not, of several steps; without codes and (more than 128 dimensions) with them; one and two
# slots per lane, few candidates per point
@pytest.mark.parametrize("quads", ["0", "1"])
@pytest.mark.parametrize("N,D,K", [(1500, 5, 9), (1500, 23, 24), (1300, 48, 18), (1200, 47, 33), (1200, 130, 31), (900, 208, 32), (800, 288, 45), (900, 70, 80), (700, 189, 12)])
def test_explore_reads_rows_by_one_lane_or_four(gpu, orc, rng, monkeypatch, N, D, K, quads):
    monkeypatch.setenv("RSFK_MERGE_QUADS", quads)
    if K > 64:
        monkeypatch.setenv("RSFK_OPTIONAL_MB", "0")
    X = rng.standard_normal((N, D)).astype(np.float32)
    perm, ls, lz, _ = orc.build_tree(X, K + 1, 2 * K + 2, 5000, 0)
    oi, od = orc.init_lists(N, K, self_in=True)
    orc.bucket_knn(X, K, perm, lz, oi, od, starts=ls)
    gi, gd = oi.copy(), od.copy()
    for _ in range(2):
        _say("explore rows", N, D, K, quads)
        orc.explore(X, K, oi, od)
        gpu.explore(X, K, gi, gd, 1)
        assert_knn_equal(gi, gd, oi, od)


# a wavefront for every 32 neighbours of a point, a workgroup for every point
@pytest.mark.parametrize("N,D,K", [(13430000, 2, 129), (16800000, 201, 64)])
def test_explore_of_more_points_than_a_launch_has_threads_for(gpu, N, D, K):
    """The kernels that the size would take need 2^32 threads and more, which a launch cuts off without an error (about 100 GB of device
    memory).  Every row holds the next point, so the exploration finds the one after that; coordinates are small integers, all
    distances exact."""
    import torch
    torch.cuda.empty_cache()
    gpu.lib().rsfk_release_workspace()
    if torch.cuda.mem_get_info()[0] < 160 << 30:
        pytest.skip("needs 160 GB of device memory")
    X = torch.randint(0, 16, (N, D), device="cuda", dtype=torch.float32)
    p = torch.arange(N, device="cuda")
    one, two = (p + 1) % N, (p + 2) % N
    d1 = torch.cat([((X[q] - X[(q + 1) % N]) ** 2).sum(1) for q in p.split(1 << 22)])
    d2 = torch.cat([((X[q] - X[(q + 2) % N]) ** 2).sum(1) for q in p.split(1 << 22)])
    idx = torch.full((N, K), -1, dtype=torch.int32, device="cuda")
    dist = torch.full((N, K), float("inf"), device="cuda")
    idx[:, 0] = one.int()
    dist[:, 0] = d1
    scratch = torch.empty((N, K), dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    _say("explore", N, D, K)
    gpu.explore_device(X.data_ptr(), N, D, K, idx.data_ptr(), dist.data_ptr(), scratch.data_ptr())
    del scratch
    first = (d1 < d2) | ((d1 == d2) & (one < two))
    assert torch.equal(idx[:, 0], torch.where(first, one, two).int()) and torch.equal(idx[:, 1], torch.where(first, two, one).int())
    assert torch.equal(dist[:, 0], torch.minimum(d1, d2)) and torch.equal(dist[:, 1], torch.maximum(d1, d2))
    assert bool((idx[:, 2] == -1).all()) and bool((idx[:, K - 1] == -1).all())
    del idx, dist, X
    torch.cuda.empty_cache()
    gpu.lib().rsfk_release_workspace()


def test_more_rows_than_a_launch_has_wavefronts_for(gpu):
    """67.2 million points, 2^32 threads with a wavefront for every row: graph export by flags and exploration without the reversed graph (which takes
    50 million).  Every row holds the next point, small integers for coordinates."""
    import torch
    N, D, K = 67200000, 2, 3
    torch.cuda.empty_cache()
    gpu.lib().rsfk_release_workspace()
    if torch.cuda.mem_get_info()[0] < 60 << 30:
        pytest.skip("needs 60 GB of device memory")
    X = torch.randint(0, 256, (N, D), device="cuda", dtype=torch.float32)
    p = torch.arange(N, device="cuda", dtype=torch.int32)
    one, two, before = (p + 1) % N, (p + 2) % N, (p - 1) % N
    d1, d2 = ((X[one] - X) ** 2).sum(1), ((X[two] - X) ** 2).sum(1)
    idx = torch.full((N, K), -1, dtype=torch.int32, device="cuda")
    dist = torch.full((N, K), float("inf"), device="cuda")
    idx[:, 0] = one
    dist[:, 0] = d1
    indptr = torch.empty(N + 1, dtype=torch.int32, device="cuda")
    cols = torch.empty((N, 2), dtype=torch.int32, device="cuda")
    vals = torch.empty((N, 2), device="cuda")
    torch.cuda.synchronize()
    _say("symmetrize", N, K)
    assert gpu.symmetrize_device(idx.data_ptr(), dist.data_ptr(), N, K, 1, indptr.data_ptr(), cols.data_ptr(), vals.data_ptr(), 2 * N) == 2 * N
    assert torch.equal(indptr, 2 * torch.arange(N + 1, device="cuda", dtype=torch.int32))
    swap = cols[:, 0] != one
    assert torch.equal(torch.where(swap, cols[:, 1], cols[:, 0]), one) and torch.equal(torch.where(swap, cols[:, 0], cols[:, 1]), before)
    assert torch.equal(torch.where(swap, vals[:, 1], vals[:, 0]), d1) and torch.equal(torch.where(swap, vals[:, 0], vals[:, 1]), d1[before])
    del indptr, cols, vals, swap
    scratch = torch.empty((N, K), dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    _say("explore", N, D, K)
    gpu.explore_device(X.data_ptr(), N, D, K, idx.data_ptr(), dist.data_ptr(), scratch.data_ptr())
    first = (d1 < d2) | ((d1 == d2) & (one < two))
    assert torch.equal(idx[:, 0], torch.where(first, one, two)) and torch.equal(idx[:, 1], torch.where(first, two, one))
    assert torch.equal(dist[:, 0], torch.minimum(d1, d2)) and torch.equal(dist[:, 1], torch.maximum(d1, d2))
    assert bool((idx[:, 2] == -1).all())
    del idx, dist, X, scratch
    torch.cuda.empty_cache()
    gpu.lib().rsfk_release_workspace()


@pytest.mark.parametrize("padded", [False, True])
def test_more_buckets_than_a_launch_has_threads_for(gpu, padded):
    """17 million buckets of two points, by a table of starts and as rows of a padded matrix."""
    import torch
    nb, D, K = 17000000, 2, 2
    N = 2 * nb
    torch.cuda.empty_cache()
    if torch.cuda.mem_get_info()[0] < 20 << 30:
        pytest.skip("needs 20 GB of device memory")
    X = torch.randint(0, 256, (N, D), device="cuda", dtype=torch.float32)
    ids = torch.arange(N, dtype=torch.int32, device="cuda")
    starts = 2 * torch.arange(nb, dtype=torch.int32, device="cuda")
    sizes = torch.full((nb,), 2, dtype=torch.int32, device="cuda")
    idx = torch.full((N, K), -1, dtype=torch.int32, device="cuda")
    dist = torch.full((N, K), float("inf"), device="cuda")
    torch.cuda.synchronize()
    _say("buckets of two", N, padded)
    gpu.bucket_knn_device(X.data_ptr(), N, D, K, ids.data_ptr(), 0 if padded else starts.data_ptr(), sizes.data_ptr(), nb, 2,
                          idx.data_ptr(), dist.data_ptr())
    assert torch.equal(idx[:, 0], ids ^ 1) and bool((idx[:, 1] == -1).all())
    assert torch.equal(dist[:, 0], ((X - X[(ids ^ 1).long()]) ** 2).sum(1)) and bool(torch.isinf(dist[:, 1]).all())


@pytest.mark.parametrize("values", ["far", "tiny", "huge", "outlier", "spread", "notfinite"])
@pytest.mark.parametrize("N,D,K", [(2500, 16, 8), (2500, 33, 32), (1500, 129, 20), (1500, 40, 70)])
def test_explore_screens_rows_of_any_magnitude(gpu, orc, rng, N, D, K, values):
    """The float16 copy of the join has one scale for all rows: points far from the origin, at the ends of the range of fp32 (squares
    that vanish or overflow), one row that sets the scale for all others, columns of very different size, rows that are not finite.
    The three kernels of the join (short rows, long rows, a workgroup per point)."""
    X = rng.standard_normal((N, D)).astype(np.float32)
    perm, ls, lz, _ = orc.build_tree(X, K + 1, 2 * K + 2, 5000, 0)
    if values == "far":
        X = (X + np.float32(3.0e4)).astype(np.float32)
    elif values == "tiny":
        X = (X * np.float32(1e-21)).astype(np.float32)
    elif values == "huge":
        X = (X * np.float32(2e18)).astype(np.float32)
    elif values == "outlier":
        X[7] = np.float32(1e12)
    elif values == "spread":
        X = (X * np.logspace(-9, 9, D)[None, :]).astype(np.float32)
    else:
        X[3, D // 2] = np.nan
        X[11, 0] = np.inf
        X[N - 1, D - 1] = -np.inf
        X[0, 1] = np.nan
    oi, od = orc.init_lists(N, K, self_in=True)
    orc.bucket_knn(X, K, perm, lz, oi, od, starts=ls)
    gi, gd = oi.copy(), od.copy()
    _say("explore magnitudes", N, D, K, values)
    for _ in range(2):
        orc.explore(X, K, oi, od)
        gpu.explore(X, K, gi, gd, 1)
        assert_knn_equal(gi, gd, oi, od)


@pytest.mark.parametrize("codes", [True, False])
@pytest.mark.parametrize("N,D,K,leaf,spread", [(1500, 10, 46, 47, 1.0), (2500, 70, 64, 20, 1.0), (4000, 33, 65, 66, 1.0), (1200, 6, 128, 129, 0.02),
                                               (5000, 12, 100, 60, 1.0), (3000, 20, 256, 257, 1.0), (2000, 5, 200, 70, 0.05), (9000, 64, 90, 91, 1.0)])
def test_explore_with_a_workgroup_per_point(gpu, orc, rng, monkeypatch, N, D, K, leaf, spread, codes):
    """Long rows: one and several slots per lane; rows that are full and rows that are not (small leaves: hundreds of candidates enter,
    several rounds, more candidates than the list takes); few distinct candidates among thousands of marks (small spread: 40 clusters);
    without the codes of the join (RSFK_OPTIONAL_MB=0: no memory for them)."""
    if not codes:
        monkeypatch.setenv("RSFK_OPTIONAL_MB", "0")
    X = rng.standard_normal((N, D)).astype(np.float32)
    if spread < 1.0:
        X = (X[rng.integers(0, 40, N)] + np.float32(spread) * X).astype(np.float32)
    oi, od = orc.init_lists(N, K, self_in=True)
    for seed in range(2):
        perm, ls, lz, _ = orc.build_tree(X, leaf, 2 * leaf, 5000, seed)
        orc.bucket_knn(X, K, perm, lz, oi, od, starts=ls)
    gi, gd = oi.copy(), od.copy()
    _say("explore workgroup", N, D, K, leaf, spread, codes)
    for _ in range(2):
        orc.explore(X, K, oi, od)
        gpu.explore(X, K, gi, gd, 1)
        assert_knn_equal(gi, gd, oi, od)


@pytest.mark.parametrize("codes", [True, False])
@pytest.mark.parametrize("D", [129, 161, 191, 192, 193, 225, 257, 288, 292])
@pytest.mark.parametrize("K", [31, 32, 33, 45, 63])
def test_explore_of_long_vectors(gpu, orc, rng, monkeypatch, D, K, codes):
    """More than 128 dimensions: with the join's codes up to 288 of them (192 where D is not a multiple of 4) are read without the tile,
    and points of many marks (here: a first tree of small leaves, 500 clustered points) go to a workgroup each where the set has
    2048 places (K >= 32) and K > 32 or D >= 192; without the codes neither."""
    if not codes:
        monkeypatch.setenv("RSFK_OPTIONAL_MB", "0")
    N = 1500
    X = rng.standard_normal((N, D)).astype(np.float32)
    X[:500] = (X[rng.integers(0, 10, 500)] + np.float32(0.05) * X[:500]).astype(np.float32)
    oi, od = orc.init_lists(N, K, self_in=True)
    for seed, leaf in enumerate((K // 2, K + 1)):
        perm, ls, lz, _ = orc.build_tree(X, leaf, 2 * leaf, 5000, seed)
        orc.bucket_knn(X, K, perm, lz, oi, od, starts=ls)
    gi, gd = oi.copy(), od.copy()
    _say("explore long vectors", D, K, codes)
    for _ in range(2):
        orc.explore(X, K, oi, od)
        gpu.explore(X, K, gi, gd, 1)
        assert_knn_equal(gi, gd, oi, od)


@pytest.mark.parametrize("D,K", [(192, 32), (129, 33), (400, 50)])
def test_forest_of_long_vectors_with_many_marks(gpu, orc, rng, D, K):
    """The same from a forest of two trees: the points that the small set is tried on first (more than 4,096 points in their order)."""
    import gpu_rsfk
    X = rng.standard_normal((5003, D)).astype(np.float32)
    _say("forest of long vectors", D, K)
    gi, gd = gpu_rsfk.RSFK(random_state=0).find_nearest_neighbors(X, K, n_trees=2, min_tree_children=K + 1, max_tree_children=2 * K + 2,
                                                                    nn_exploring_factor=1)
    oi, od, _ = orc.forest(X, K, 2, K + 1, 2 * K + 2, 5000, 0, 1, want_log=True)
    assert_knn_equal(gi, gd, oi, od)


# ---------------------------------------------------------------------------
# the whole call, through the entry points the Python package binds
# ---------------------------------------------------------------------------
def test_find_nearest_neighbors_small_plumbing_config(gpu, orc):
    """BASELINE config 1 through RSFK.find_nearest_neighbors."""
    import gpu_rsfk
    X = np.random.default_rng(0).random((10000, 32), dtype=np.float32)
    r = gpu_rsfk.RSFK(random_state=0)
    _say("forest C1")
    gi, gd = r.find_nearest_neighbors(X, 16, n_trees=4, min_tree_children=32, max_tree_children=128)
    oi, od, olog = orc.forest(X, 16, 4, 32, 128, 5000, 0, 1, want_log=True)
    assert_knn_equal(gi, gd, oi, od)
    ti, _ = orc.bruteforce(X, 16)
    assert abs(recall(ti, gi) - recall(ti, oi)) < 1e-9 and recall(ti, gi) > 0.35
    log = r.log_forest.data
    assert log["Tree Depth"] == [int(v) for v in olog[0:4]]
    assert log["Max Leaf Size"] == [int(v) for v in olog[4:8]]
    assert log["Min Leaf Size"] == [int(v) for v in olog[8:12]]
    assert log["Total Leaves"] == [int(v) for v in olog[12:16]]
    assert all(t > 0 for t in log["KNN Sets Updates"]) and r._last_search_time > 0
    # the phases that have a counterpart here carry their time: side tests, hyperplanes of the wide levels,
    # scatter (the reference's node update) and the kernel that finishes the small subtrees (its bucket creation)
    for name in ("Check Points Side Time", "Create Nodes Time", "Update Nodes Time", "Bucket Creation Time"):
        assert all(t > 0 for t in log[name]), name
        assert sum(log[name]) < sum(log["Total Tree Building Time"])
    assert (gi >= 0).all()


@pytest.mark.parametrize("N,D,K,T,kw", [
    (20000, 100, 32, 6, {}),
    (5000, 16, 8, 3, dict(min_tree_children=4, max_tree_children=9)),          # second call with K+1 .. 3(K+1)
    (6000, 24, 40, 3, dict(nn_exploring_factor=2)),
    (4000, 12, 10, 2, dict(point_in_self_neigh=False, nn_exploring_factor=0)),
    (9000, 12, 64, 6, dict(nn_exploring_factor=2)),     # rows of 64: the small set of the merge is tried on a sample first
    (4000, 10, 300, 2, dict(nn_exploring_factor=1)),                           # eight slots per lane
    (1400, 8, 520, 2, dict(nn_exploring_factor=1, min_tree_children=200, max_tree_children=500)),   # sixteen
])
@pytest.mark.parametrize("variant", ["default", "bucket_screen"])
def test_find_nearest_neighbors_matches_oracle(gpu, orc, rng, monkeypatch, N, D, K, T, kw, variant):
    import gpu_rsfk
    if variant == "bucket_screen":
        monkeypatch.setenv("RSFK_BUCKET_SCREEN", "100")     # every tree but the first through the screened small-bucket kernel
    X = rng.standard_normal((N, D)).astype(np.float32)
    r = gpu_rsfk.RSFK(random_state=17)
    _say("forest", N, D, K, T, kw)
    gi, gd = r.find_nearest_neighbors(X, K, n_trees=T, **kw)
    mn = kw.get("min_tree_children", K + 1)
    mx = kw.get("max_tree_children", 2 * mn)
    nnef = kw.get("nn_exploring_factor", 1 if K <= 32 else 0)
    oi, od = orc.init_lists(N, K, self_in=kw.get("point_in_self_neigh", True))
    orc.forest(X, K, T, mn, mx, 5000, 17, nnef, knn_idx=oi, knn_dist=od)
    if mn < K + 1:
        orc.forest(X, K, 1, K + 1, 3 * (K + 1), 5000, 17, nnef, knn_idx=oi, knn_dist=od)
    assert_knn_equal(gi, gd, oi, od)


@pytest.mark.parametrize("data", ["normal", "clusters", "offset", "equal", "huge", "tiny", "rows"])
@pytest.mark.parametrize("N,D,K,mn,mx", [(3000, 2, 5, 60, 128), (3100, 16, 64, 65, 192), (2900, 17, 32, 64, 256), (3000, 32, 32, 64, 256),
                                         (4000, 33, 1, 64, 160), (3000, 36, 64, 65, 256), (2500, 44, 40, 60, 192),
                                         (2600, 49, 33, 60, 128), (2400, 64, 63, 64, 128), (2300, 68, 20, 60, 128),
                                         (3000, 20, 16, 17, 40), (3000, 100, 32, 32, 64), (2500, 64, 1, 4, 10), (2500, 130, 31, 32, 64)])
@pytest.mark.parametrize("screen", ["rule", "always"])
def test_later_trees_bound_pairs_and_merge_by_turns(gpu, capi, orc, rng, monkeypatch, N, D, K, mn, mx, data, screen):
    """Buckets that fit into LDS whole, and of at most 64 points, pairs bounded on the matrix cores (any remainder of dimensions, tiles and rows; bounds that
    drop nothing, rows that differ by less than the bound, equal rows), slots found by counting: from the tree the rule says, and from
    the first one on (more candidates of a member than lanes).  "rows": the caller's rows hold neighbours already, in any order."""
    monkeypatch.setenv("RSFK_FOREST_MERGE", "0")
    if screen == "always":
        monkeypatch.setenv("RSFK_BUCKET_SCREEN", "always")
    X = rng.standard_normal((N, D)).astype(np.float32)
    if data == "clusters":
        X = (0.01 * X + 30 * rng.standard_normal((40, D)).astype(np.float32)[rng.integers(0, 40, N)]).astype(np.float32)
    elif data == "offset":
        X += np.float32(2000)
    elif data == "equal":
        X = np.round(X[rng.integers(0, N, N)] * np.float32(1.5)).astype(np.float32)
    elif data == "huge":
        X *= np.float32(2e18)
        X[:: 97] *= np.float32(1e-19)
    elif data == "tiny":
        X *= np.float32(1e-19)
        X[:: 97] *= np.float32(1e-19)
    T = 7
    _say("later trees, resident buckets", N, D, K, mn, mx, data, screen)
    gi, gd = orc.init_lists(N, K, self_in=True)
    if data == "rows":
        orc.forest(X, K, 1, mn, mx, 5000, 90, 0, knn_idx=gi, knn_dist=gd)
        order = np.argsort(rng.random((N, K)), axis=1)
        gi, gd = (np.ascontiguousarray(np.take_along_axis(v, order, axis=1)) for v in (gi, gd))
    oi, od = gi.copy(), gd.copy()
    log = np.zeros(16 * T + 2, np.float32)
    capi.lib().pymodule_rsfk_knn(T, K, N, D, mn, mx, 5000, 0, 3, 0, X.ctypes.data, gi.ctypes.data, gd.ctypes.data, log.ctypes.data)
    orc.forest(X, K, T, mn, mx, 5000, 3, 0, knn_idx=oi, knn_dist=od)
    assert_knn_equal(gi, gd, oi, od)


@pytest.mark.parametrize("N,D,K,mn,mx,T,together", [(204551, 4, 25, 50, 200, 50, True), (400000, 2, 32, 64, 256, 50, True),
                                                    (400000, 32, 32, 64, 256, 50, False), (400000, 32, 32, 64, 256, 6, True)])
def test_many_points_take_the_trees_together_by_rule(gpu, rng, N, D, K, mn, mx, T, together):
    import gpu_rsfk
    X = rng.random((N, D), dtype=np.float32)
    _say("trees together or not", N, D, K, mn, mx, T)
    gi, gd = gpu_rsfk.RSFK(random_state=1).find_nearest_neighbors(X, K, n_trees=T, min_tree_children=mn, max_tree_children=mx, nn_exploring_factor=0)
    named = set(name for _, _, names in gpu.last_build_report()["bucket_kernels"] for name in names)
    assert (named == {"k_forest_pairs + k_forest_merge"}) == together, named
    some = rng.integers(0, N, 200)
    assert np.allclose(gd[some], ((X[some][:, None] - X[gi[some]]) ** 2).sum(2), rtol=1e-5) and rows_have_no_duplicates(gi[some])


# (forms: the trees whose pairs the rule bounds first; "+" = as the tree before, ".." = anything, then mostly that, of 150 trees)
@pytest.mark.parametrize("N,D,K,mn,mx,offset,forms", [
    (6000, 8, 4, 5, 10, 0, "00+"),            # few points in a bucket: not while many of them are offered to a row
    (6000, 100, 4, 5, 10, 0, "00000..1"),     # ... but once hardly any are
    (6000, 100, 4, 5, 10, 300, "00000..0"),   # ... and the bound shows that
    (6000, 70, 5, 9, 18, 0, "00+"),           # ... more of them, but two chunks of dimensions
    (6000, 16, 8, 10, 20, 0, "001"),          # while a row still gets three offers
    (6000, 16, 16, 17, 34, 0, "001+"),
    (6000, 8, 16, 20, 60, 300, "0010+"),      # a bound that does not tell the points apart: once
    (6000, 70, 16, 20, 60, 300, "0010+"),
    (6000, 16, 16, 17, 34, 300, "0011"),      # ... in buckets whose pairs all fit into the list
    (6000, 16, 16, 20, 60, 0, "001+"),
])
def test_form_of_the_small_buckets_follows_its_rule(gpu, capi, orc, rng, monkeypatch, N, D, K, mn, mx, offset, forms):
    monkeypatch.setenv("RSFK_FOREST_MERGE", "0")
    X = (rng.random((N, D)) + offset).astype(np.float32)
    T = 150 if ".." in forms else 8
    _say("form of the small buckets", N, D, K, mn, mx, offset)
    gi, gd = orc.init_lists(N, K, self_in=True)
    oi, od = gi.copy(), gd.copy()
    log = np.zeros(16 * T + 2, np.float32)
    capi.lib().pymodule_rsfk_knn(T, K, N, D, mn, mx, 5000, 0, 5, 0, X.ctypes.data, gi.ctypes.data, gd.ctypes.data, log.ctypes.data)
    orc.forest(X, K, T, mn, mx, 5000, 5, 0, knn_idx=oi, knn_dist=od)
    assert_knn_equal(gi, gd, oi, od)
    took = "".join(str(v) for v in gpu.last_build_report()["bucket_screened"])
    want = forms[:-1] + forms[-2] * (T + 1 - len(forms)) if forms.endswith("+") else forms
    first, _, last = want.partition("..")
    assert took.startswith(first) and (last == "" or took[-20:].count(last) > 10), took


# The workloads of the benchmark configurations 3, 4 and 5 (clustered D=256; sparse D=784 with K=90 and one
# exploration pass, the only shape that runs the general bucket kernel with two slots per lane together with the
# workgroup-per-point exploration merge; standard normal D=32 with buckets of 64..256 points), as forest +
# exploration through the package against the oracle, at sizes the oracle finishes in seconds.
@pytest.mark.parametrize("config,N,K,T,kw", [
    ("c3", 24000, 32, 6, {}),
    ("c4", 9000, 90, 4, dict(nn_exploring_factor=1)),
    ("c5", 70000, 32, 5, dict(min_tree_children=64, max_tree_children=256)),
], ids=["config3_gmm64_d256_k32", "config4_sparse_d784_k90_explore", "config5_normal_d32_buckets64_256"])
@pytest.mark.parametrize("kernel", ["direct", "gram", "screen", "tiled"])
def test_baseline_config_workloads_match_oracle(gpu, orc, monkeypatch, config, N, K, T, kw, kernel):
    import gpu_rsfk
    if kernel == "tiled":
        if config != "c4":
            pytest.skip("no bucket of this configuration reaches the general kernel")
        monkeypatch.setenv("RSFK_BUCKET_PAIRS", "0")       # the forms of the general kernel that need no working memory
    if kernel == "gram":
        monkeypatch.setenv("RSFK_GRAM_FROM", "1")          # every tree but the first through the screened bucket kernel
    if kernel == "screen":
        if config != "c3":
            pytest.skip("no bucket of this configuration reaches the screened small-bucket kernel")
        monkeypatch.setenv("RSFK_BUCKET_SCREEN", "100")
    else:
        monkeypatch.setenv("RSFK_BUCKET_SCREEN", "never")
    X = baseline_points(config, N)
    r = gpu_rsfk.RSFK(random_state=0)
    _say("forest", config, N, X.shape[1], K, T, kw)
    gi, gd = r.find_nearest_neighbors(X, K, n_trees=T, **kw)
    mn = kw.get("min_tree_children", K + 1)
    mx = kw.get("max_tree_children", 2 * mn)
    nnef = kw.get("nn_exploring_factor", 1 if K <= 32 else 0)
    assert nnef == 1
    oi, od, olog = orc.forest(X, K, T, mn, mx, 5000, 0, nnef, want_log=True)
    assert_knn_equal(gi, gd, oi, od)
    assert rows_have_no_duplicates(gi) and (gi >= 0).all()
    log = r.log_forest.data
    assert log["Total Leaves"] == [int(v) for v in olog[3 * T:4 * T]]
    assert log["Max Leaf Size"] == [int(v) for v in olog[1 * T:2 * T]]


# size-independent properties of the same three workloads at their full sizes
@pytest.mark.parametrize("config,N,K,T,mn,mx", [
    ("c3", 1000000, 32, 4, 33, 66),
    ("c4", 70000, 90, 10, 91, 182),
    ("c5", 10000000, 32, 3, 64, 256),
], ids=["config3_full_size", "config4_full_size", "config5_full_size"])
def test_baseline_config_properties_at_full_size(gpu, orc, config, N, K, T, mn, mx):
    import torch
    X = baseline_points(config, N)
    D = X.shape[1]
    dX = torch.from_numpy(X).cuda()
    idx = torch.full((N, K), -1, dtype=torch.int32, device="cuda")
    idx[:, 0] = torch.arange(N, dtype=torch.int32, device="cuda")
    dist = torch.full((N, K), float("inf"), dtype=torch.float32, device="cuda")
    dist[:, 0] = 0
    log = np.zeros(16 * T + 2, np.float32)
    _say("full size forest", config, N, D, K, T)
    gpu.knn_forest_device(T, K, N, D, mn, mx, 5000, 0, 0, 0, dX.data_ptr(), idx.data_ptr(), dist.data_ptr(), log)
    torch.cuda.synchronize()
    assert (log[1 * T:2 * T] <= mx).all() and (log[2 * T:3 * T] >= mn).all()
    assert (log[3 * T:4 * T] >= N / mx).all() and (log[3 * T:4 * T] <= N / mn).all()
    before = dist.max(1).values.clone()
    assert bool((idx >= 0).all()) and bool((idx < N).all())
    assert bool((dist[:, 1:] >= dist[:, :-1]).all())                 # rows come back ascending
    srt = torch.sort(idx, dim=1).values
    assert not bool((srt[:, 1:] == srt[:, :-1]).any())               # no point twice in a row
    del srt
    rng = np.random.default_rng(3)
    rows = rng.choice(N, 150, replace=False)
    hi, hd = idx[torch.from_numpy(rows).cuda()].cpu().numpy(), dist[torch.from_numpy(rows).cuda()].cpu().numpy()
    for r_, p in enumerate(rows):
        for k in range(0, K, 7):
            assert hd[r_, k] == orc.sqdist(X[p], X[hi[r_, k]])       # stored distance = distance of the stored neighbour
    # one exploration pass: the row maximum only falls, and sampled rows are what the oracle's rule gives from the
    # same graph (the K smallest (distance, index) of the old row and the neighbours of the old neighbours)
    old = idx.clone()
    scratch = torch.empty((N, K), dtype=torch.int32, device="cuda")
    _say("full size explore", config)
    gpu.explore_device(dX.data_ptr(), N, D, K, idx.data_ptr(), dist.data_ptr(), scratch.data_ptr())
    torch.cuda.synchronize()
    assert bool((dist.max(1).values <= before).all())
    for p in rows[:40]:
        orow = old[int(p)].cpu().numpy()
        cand = np.unique(np.concatenate([orow, old[torch.from_numpy(orow).long().cuda()].cpu().numpy().ravel()]))
        d = np.array([orc.sqdist(X[c], X[p]) for c in cand], np.float32)
        order = np.lexsort((cand, d))[:K]
        assert np.array_equal(idx[int(p)].cpu().numpy(), cand[order])
        assert np.array_equal(dist[int(p)].cpu().numpy(), d[order])


def test_reference_package_smoke_tests(gpu):
    """The two live smoke tests of the reference package (RSFK.py:841-903)."""
    import gpu_rsfk
    np.random.seed(0)
    _say("package test()")
    gpu_rsfk.test()


def test_cluster_by_sample_tree(gpu, orc, rng):
    import gpu_rsfk
    N, D = 4096, 99
    X = rng.random((N, D), dtype=np.float32)
    r = gpu_rsfk.RSFK(random_state=5)
    _say("cluster_by_sample_tree")
    total_leaves, max_child, nodes_buckets, bucket_sizes = r.cluster_by_sample_tree(
        X, min_tree_children=N // 30, max_tree_children=3 * (N // 30), verbose=0)
    perm, ls, lz, st = orc.build_tree(X, N // 30, 3 * (N // 30), 5000, 5)
    assert total_leaves == len(lz) and max_child == lz.max()
    assert nodes_buckets.shape == (total_leaves * max_child,) and np.array_equal(bucket_sizes, lz)
    nb = nodes_buckets.reshape(total_leaves, max_child)
    for b in range(total_leaves):
        assert np.array_equal(nb[b, :lz[b]], perm[ls[b]:ls[b] + lz[b]])
        assert (nb[b, lz[b]:] == -1).all()
    assert np.array_equal(np.sort(nb[nb >= 0]), np.arange(N))
    raw = r.cluster_by_sample_tree(X, min_tree_children=64, max_tree_children=256, verbose=0, numpy_result_format=False)
    assert raw[0].value > 0 and raw[1].value <= 256


def test_golden_vectors(gpu):
    g = np.load(os.path.join(ROOT, "tests", "golden", "small_knng.npz"))
    N, D, K, MIN, MAX, seed = [int(v) for v in g["params"]]
    X = g["X"]
    _say("golden")
    perm, ls, lz, st = gpu.build_tree(X, MIN, MAX, 5000, seed)
    assert np.array_equal(perm, g["perm"]) and np.array_equal(ls, g["leaf_start"]) and np.array_equal(lz, g["leaf_size"])
    gi = np.full((N, K), -1, np.int32)
    gd = np.full((N, K), np.inf, np.float32)
    gi[:, 0] = np.arange(N)
    gd[:, 0] = 0
    gpu.bucket_knn(X, K, perm, lz, gi, gd, starts=ls)
    assert_knn_equal(gi, gd, g["bucket_idx"], g["bucket_dist"])
    import gpu_rsfk
    fi, fd = gpu_rsfk.RSFK(seed).find_nearest_neighbors(X, K, n_trees=3, min_tree_children=MIN, max_tree_children=MAX)
    assert_knn_equal(fi, fd, g["forest_idx"], g["forest_dist"])
    qi, qd = gpu_rsfk.RSFK(seed).find_nearest_neighbors_ann(X, g["Q"], K, n_trees=3, min_tree_children=MIN,
                                                            max_tree_children=MAX, ensure_valid_indices=False)
    assert_knn_equal(qi, qd, g["ann_idx"], g["ann_dist"])
    indptr, cols, vals = gpu_rsfk.symmetric_knn_graph(g["forest_idx"], g["forest_dist"], drop_self=True)
    assert np.array_equal(indptr, g["csr_indptr"]) and np.array_equal(cols, g["csr_indices"])
    assert np.array_equal(vals, g["csr_data"])


# ---------------------------------------------------------------------------
# size-independent properties at a size the oracle is not run on
# ---------------------------------------------------------------------------
def test_properties_at_scale(gpu, orc):
    import torch
    N, D, K, T = 1000000, 100, 32, 8             # BASELINE config 2 at its full size
    rng = np.random.default_rng(0)
    X = rng.random((N, D), dtype=np.float32)
    dX = torch.from_numpy(X).cuda()
    idx = torch.full((N, K), -1, dtype=torch.int32, device="cuda")
    idx[:, 0] = torch.arange(N, dtype=torch.int32, device="cuda")
    dist = torch.full((N, K), float("inf"), dtype=torch.float32, device="cuda")
    dist[:, 0] = 0
    log = np.zeros(16 * T + 2, np.float32)
    _say("scale forest")
    gpu.knn_forest_device(T, K, N, D, K + 1, 2 * (K + 1), 5000, 0, 0, 0, dX.data_ptr(), idx.data_ptr(), dist.data_ptr(), log)
    torch.cuda.synchronize()
    gi, gd = idx.cpu().numpy(), dist.cpu().numpy()
    assert (gi >= 0).all() and (gi < N).all()
    assert rows_have_no_duplicates(gi)
    leaves = log[3 * T:4 * T]
    assert (log[1 * T:2 * T] <= 2 * (K + 1)).all() and (log[2 * T:3 * T] >= K + 1).all()
    assert (leaves >= N / (2 * (K + 1))).all() and (leaves <= N / (K + 1)).all()
    # stored distances are the distances of the stored neighbours
    rows = rng.choice(N, 300, replace=False)
    for p in rows:
        for k in range(0, K, 5):
            assert gd[p, k] == orc.sqdist(X[p], X[gi[p, k]])
    # one more identical forest cannot change anything (idempotence of the set update)
    before = gd.max(1).copy()
    _say("scale forest again")
    gpu.knn_forest_device(T, K, N, D, K + 1, 2 * (K + 1), 5000, 0, 0, 0, dX.data_ptr(), idx.data_ptr(), dist.data_ptr(), log)
    torch.cuda.synchronize()
    gi2, gd2 = idx.cpu().numpy(), dist.cpu().numpy()
    si, sd = sort_rows(gi, gd)
    si2, sd2 = sort_rows(gi2, gd2)
    assert np.array_equal(sd, sd2) and np.array_equal(si, si2)
    # exploration only lowers the row maximum, and the oracle agrees on a sample of rows
    scratch = torch.empty((N, K), dtype=torch.int32, device="cuda")
    _say("scale explore")
    gpu.explore_device(dX.data_ptr(), N, D, K, idx.data_ptr(), dist.data_ptr(), scratch.data_ptr())
    torch.cuda.synchronize()
    gi3, gd3 = idx.cpu().numpy(), dist.cpu().numpy()
    assert (gd3.max(1) <= before).all()
    assert rows_have_no_duplicates(gi3)
    # the oracle's exploration of a sample of rows, from the same graph: row p after the pass = the K smallest
    # (distance, index) of its old row and the neighbours of its old neighbours
    for p in rng.choice(N, 200, replace=False):
        cand = np.unique(np.concatenate([gi2[p], gi2[gi2[p]].ravel()]))
        cand = cand[cand != p] if p not in gi2[p] else cand
        d = np.array([orc.sqdist(X[c], X[p]) for c in cand], np.float32)
        order = np.lexsort((cand, d))[:K]
        assert np.array_equal(gi3[p], cand[order]) and np.array_equal(gd3[p], d[order])


# ---------------------------------------------------------------------------
# inputs chosen to stress the bfloat16 screens (tree side test, exploration)
# ---------------------------------------------------------------------------
def _hard_inputs(rng, kind, N, D):
    if kind == "offset":          # large common offset: bfloat16 keeps almost nothing of the differences
        return (1000.0 + rng.random((N, D))).astype(np.float32)
    if kind == "grid":            # coarse lattice: many points exactly on bisecting hyperplanes, many equal distances
        return rng.integers(0, 4, size=(N, D)).astype(np.float32)
    if kind == "tiny":            # values near the bottom of the normal range
        return (rng.random((N, D)) * 1e-30).astype(np.float32)
    if kind == "mixed":           # wildly different scales per dimension, both signs
        scale = np.logspace(-6, 6, D).astype(np.float32)
        return (rng.standard_normal((N, D)) * scale).astype(np.float32)
    if kind == "clusters":        # tight clusters: candidate distances crowd around the row maximum
        centres = rng.random((20, D))
        return (centres[rng.integers(20, size=N)] + 1e-3 * rng.standard_normal((N, D))).astype(np.float32)
    raise ValueError(kind)


@pytest.mark.parametrize("variant", ["default", "bucket_screen", "bucket_gram"])
@pytest.mark.parametrize("kind", ["offset", "grid", "tiny", "mixed", "clusters"])
def test_screens_never_change_a_result(gpu, orc, rng, monkeypatch, kind, variant):
    """The bfloat16 screens only skip work whose outcome is certain: trees, bucket K-NN and exploration on inputs
    that defeat a 8-bit mantissa must still be identical to the fp32 oracle.  "bucket_screen" also switches the
    buckets of up to 64 points to the two-wavefront kernel that bounds the pair matrix on the matrix cores
    (RSFK_BUCKET_SCREEN=always: every tree and the stage-level call), "bucket_gram" all buckets to the tiled kernel that
    does the same (RSFK_GRAM_FROM=0)."""
    import gpu_rsfk
    if variant == "bucket_screen":
        monkeypatch.setenv("RSFK_BUCKET_SCREEN", "always")
    if variant == "bucket_gram":
        monkeypatch.setenv("RSFK_GRAM_FROM", "0")
    N, D, K = 6000, 24, 10
    X = _hard_inputs(rng, kind, N, D)
    perm, ls, lz, st = orc.build_tree(X, K + 1, 2 * (K + 1), 300, 2)
    for screen in ("q8", "bf16"):
        _say("hard tree", kind, screen)
        monkeypatch.setenv("RSFK_TREE_SCREEN", screen)
        gperm, gls, glz, gst = gpu.build_tree(X, K + 1, 2 * (K + 1), 300, 2)
        assert np.array_equal(gperm, perm) and np.array_equal(glz, lz)
    monkeypatch.delenv("RSFK_TREE_SCREEN")
    _say("hard forest", kind)
    r = gpu_rsfk.RSFK(random_state=2)
    gi, gd = r.find_nearest_neighbors(X, K, n_trees=3, max_tree_depth=300, nn_exploring_factor=2)
    oi, od = orc.forest(X, K, 3, K + 1, 2 * (K + 1), 300, 2, 2)
    assert_knn_equal(gi, gd, oi, od)          # "grid": equal distances everywhere, ties go to the smaller index
    assert rows_have_no_duplicates(gi)


@pytest.mark.parametrize("K,mn,mx,env,expected", [
    (16, 17, 34, {}, ["k_bucket_knn_auto"]),
    (16, 17, 34, {"RSFK_BUCKET_SCREEN": "never"}, ["k_bucket_knn_auto"]),
    (16, 17, 34, {"RSFK_BUCKET_SCREEN": "always"}, ["k_bucket_knn_auto"]),
    (16, 40, 100, {}, ["k_bucket_knn_auto", "k_bucket_knn_small<72>", "k_bucket_knn_rows"]),
    (90, 91, 182, {}, ["k_bucket_pairs + k_bucket_merge_pairs"]),
    (90, 91, 182, {"RSFK_BUCKET_PAIRS": "0"}, ["k_bucket_knn<per 64 members>"]),
    (90, 91, 182, {"RSFK_BUCKET_PAIRS": "0", "RSFK_BUCKET_STRIP": "0"}, ["k_bucket_knn<per bucket>"]),
    (90, 91, 182, {"RSFK_GRAM_FROM": "1"}, ["k_bucket_pairs + k_bucket_merge_pairs", "k_bucket_knn_gram"]),
])
def test_report_of_a_build_names_what_ran(gpu, rng, monkeypatch, K, mn, mx, env, expected):
    """rsfk_last_build_report: the kernels every tree's buckets went to, the counts the algorithmic bytes are made of
    and the seconds of the three steps, for the build that has just run."""
    import gpu_rsfk
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    N, D, T = 6000, 20, 3
    X = rng.random((N, D), dtype=np.float32)
    r = gpu_rsfk.RSFK(random_state=4)
    _say("report of a build", K, mn, mx, env)
    r.find_nearest_neighbors(X, K, n_trees=T, min_tree_children=mn, max_tree_children=mx, nn_exploring_factor=1)
    rep = gpu.last_build_report()
    assert (rep["N"], rep["D"], rep["K"], rep["n_trees"]) == (N, D, K, T)
    runs = rep["bucket_kernels"]
    assert runs[0][0] == 0 and runs[-1][1] == T - 1
    assert all(runs[i][1] + 1 == runs[i + 1][0] for i in range(len(runs) - 1))
    named = set(name for _, _, names in runs for name in names)
    assert named == set(expected), named
    assert len(rep["bucket_pair_share"]) == T and len(rep["bucket_screened"]) == T
    if "RSFK_BUCKET_SCREEN" in env:                     # the form of the kernel the trees took
        assert rep["bucket_screened"] == [1 if env["RSFK_BUCKET_SCREEN"] == "always" else 0] * T
    assert rep["tree_points_tested"] >= N * T and 0 <= rep["tree_points_undecided"] <= rep["tree_points_tested"]
    assert rep["explore_passes"] == 1 and rep["explore_exact_distances"] > 0
    assert rep["tree_seconds"] > 0 and rep["bucket_seconds"] > 0 and rep["explore_seconds"] > 0


def test_workspace_is_reused_and_can_be_released(gpu, rng):
    """Device buffers are kept between calls; releasing them changes nothing but the next call's allocations."""
    import gpu_rsfk
    from gpu_rsfk import capi
    X = rng.random((5000, 20), dtype=np.float32)
    a = gpu_rsfk.RSFK(random_state=4).find_nearest_neighbors(X, 12, n_trees=3)
    b = gpu_rsfk.RSFK(random_state=4).find_nearest_neighbors(X, 12, n_trees=3)      # served from the kept buffers
    capi.lib().rsfk_release_workspace()
    c = gpu_rsfk.RSFK(random_state=4).find_nearest_neighbors(X, 12, n_trees=3)
    for r in (b, c):
        assert_knn_equal(r[0], r[1], a[0], a[1])


def test_rows_come_back_sorted_and_unsorted_input_is_accepted(gpu, orc, rng):
    """Rows handed in unsorted (the reference keeps them unordered) are merged correctly; rows come back ascending."""
    N, D, K = 3000, 12, 16
    X = rng.random((N, D), dtype=np.float32)
    oi, od = orc.forest(X, K, 2, nnef=0, seed=3)              # oracle rows are in arrival order (unsorted)
    assert (np.diff(od, axis=1) < 0).any()
    gi, gd = oi.copy(), od.copy()
    perm, ls, lz, _ = orc.build_tree(X, K + 1, 2 * (K + 1), 5000, 77)
    orc.bucket_knn(X, K, perm, lz, oi, od, starts=ls)
    _say("unsorted rows in")
    gpu.bucket_knn(X, K, perm, lz, gi, gd, starts=ls)
    assert_knn_equal(gi, gd, oi, od)
    changed = (np.sort(gi, 1) != np.sort(oi.copy(), 1)).any(1)     # rows identical as sets
    assert not changed.any()
    gi2, gd2 = gi.copy(), gd.copy()
    gpu.explore(X, K, gi2, gd2, 1)
    assert (np.diff(gd2, axis=1) >= 0).all()                       # every row ascending after a full pass


# ---------------------------------------------------------------------------
# query-set search
# ---------------------------------------------------------------------------
@pytest.mark.parametrize("N,NQ,D,MIN,MAX,dist", [
    (6000, 2500, 24, 9, 18, "normal"),
    (5000, 1, 130, 33, 66, "normal"),
    (3000, 777, 3, 5, 11, "grid"),           # many points on a hyperplane and duplicated points
    (20000, 4000, 64, 33, 66, "uniform"),
])
def test_queries_reach_the_leaf_the_oracle_routes_them_to(gpu, orc, rng, N, NQ, D, MIN, MAX, dist):
    """One tree and a row longer than any bucket: the row of a query is then exactly the bucket it was routed to."""
    import gpu_rsfk
    if dist == "grid":
        X = rng.integers(0, 6, (N, D)).astype(np.float32)
        Q = rng.integers(0, 6, (NQ, D)).astype(np.float32)
    elif dist == "uniform":
        X = rng.random((N, D), dtype=np.float32)
        Q = X[rng.permutation(N)[:NQ]].copy()           # queries that are base points: always on their own side
        Q[::2] += rng.standard_normal((len(Q[::2]), D)).astype(np.float32) * 0.01
    else:
        X = rng.standard_normal((N, D)).astype(np.float32)
        Q = rng.standard_normal((NQ, D)).astype(np.float32)
    perm, qs, qz = orc.route_queries(X, Q, MIN, MAX, 5000, 5)
    K = max(MAX, int(qz.max()))              # identical points cannot be split: such buckets stay above MAX
    assert (qz >= 1).all() and K <= 256
    r = gpu_rsfk.RSFK(random_state=5)
    _say("route", N, NQ, D, MIN, MAX, dist, K)
    gi, gd = r.find_nearest_neighbors_ann(X, Q, K, n_trees=1, min_tree_children=MIN, max_tree_children=MAX,
                                          ensure_valid_indices=False)
    for q in range(NQ):
        want = np.sort(perm[qs[q]:qs[q] + qz[q]])
        got = np.sort(gi[q][gi[q] >= 0])
        assert np.array_equal(got, want), (q, got, want)
    fin = gi >= 0
    assert np.isinf(gd[~fin]).all()
    d64 = ((X[gi[fin]].astype(np.float64) - np.repeat(Q, fin.sum(1), axis=0)) ** 2).sum(1)
    assert np.allclose(gd[fin], d64, rtol=1e-5, atol=1e-6)


@pytest.mark.parametrize("N,NQ,D,K,T,kw", [
    (20000, 3000, 100, 32, 5, {}),
    (8000, 1500, 18, 8, 3, dict(min_tree_children=4, max_tree_children=9)),    # second call with K+1 .. 3(K+1)
    (9000, 500, 50, 100, 3, {}),
    (7000, 2000, 33, 200, 2, dict(min_tree_children=40, max_tree_children=90, ensure_valid_indices=False)),
    (300, 50, 7, 5, 4, {}),
    (6000, 800, 12, 300, 2, {}),
    (5000, 300, 9, 700, 2, {}),
])
def test_find_nearest_neighbors_ann_matches_oracle(gpu, orc, rng, N, NQ, D, K, T, kw):
    import gpu_rsfk
    X = rng.standard_normal((N, D)).astype(np.float32)
    Q = rng.standard_normal((NQ, D)).astype(np.float32)
    r = gpu_rsfk.RSFK(random_state=23)
    _say("ann", N, NQ, D, K, T, kw)
    gi, gd = r.find_nearest_neighbors_ann(X, Q, K, n_trees=T, **kw)
    mn = kw.get("min_tree_children", K + 1)
    mx = kw.get("max_tree_children", 2 * mn)
    oi, od = orc.ann_forest(X, Q, K, T, mn, mx, 5000, 23)
    if kw.get("ensure_valid_indices", True) and mn < K + 1:
        orc.ann_forest(X, Q, K, 1, K + 1, 3 * (K + 1), 5000, 23, q_idx=oi, q_dist=od)
    assert gi.shape == (NQ, K) and gi.dtype == np.int32 and gd.dtype == np.float32
    assert_knn_equal(gi, gd, oi, od)
    assert rows_have_no_duplicates(gi)
    assert r._last_search_time > 0


# one query; one tree more than the wavefronts take in turn; buckets on both sides of 64 and 128; rows of one, two and
# more slots per lane; rows that end inside a 16-byte piece; more trees than go together; rows read by four lanes (from 129 dimensions on, and of 53) and by one
@pytest.mark.parametrize("N,NQ,D,K,T,mn,mx", [(300, 1, 1, 1, 2, 3, 6), (2000, 37, 33, 64, 5, 65, 65 * 2), (1500, 300, 64, 65, 9, 66, 128),
                                              (900, 130, 31, 16, 3, 17, 64), (700, 65, 100, 300, 4, 301, 700), (4000, 90, 7, 5, 70, 6, 12),
                                              (50, 20, 12, 8, 6, 60, 120), (1200, 33, 260, 20, 8, 21, 65), (5300, 60, 53, 30, 9, 31, 62),
                                              (700, 40, 129, 70, 3, 71, 150)])
@pytest.mark.parametrize("data", ["normal", "ties", "tiny"])
def test_ann_trees_together_match_oracle(gpu, capi, orc, rng, monkeypatch, N, NQ, D, K, T, mn, mx, data):
    """All trees of a query in one workgroup == one tree after the other == the oracle, also into rows that hold something."""
    import torch
    if data == "ties":          # points on the hyperplanes: sides that the rounded hyperplanes cannot decide
        draw = lambda n: rng.integers(0, 3, (n, D)).astype(np.float32)
    else:                       # "tiny": squares of rounding errors underflow
        draw = lambda n: (rng.standard_normal((n, D)) * (1e-18 if data == "tiny" else 1.0)).astype(np.float32)
    X, Q = draw(N), draw(NQ)
    dX, dQ = torch.from_numpy(X).cuda(), torch.from_numpy(Q).cuda()
    oi, od = orc.ann_forest(X, Q, K, T, mn, mx, 5000, 5)
    orc.ann_forest(X, Q, K, 2, mn, mx, 5000, 77, q_idx=oi, q_dist=od)
    for form in ("0", "1", "low"):                        # "low": one after the other, routed by the rounded hyperplanes
        monkeypatch.setenv("RSFK_ANN_FOREST", "1" if form == "1" else "0")
        monkeypatch.setenv("RSFK_ANN_ROUTE_LOW", "1" if form == "low" else "0")
        idx = torch.full((NQ, K), -1, dtype=torch.int32, device="cuda")
        dist = torch.full((NQ, K), float("inf"), dtype=torch.float32, device="cuda")
        _say("ann together", N, NQ, D, K, T, mn, mx, data, form)
        for trees, seed in ((T, 5), (2, 77)):
            capi.knn_ann_device(trees, K, N, NQ, D, mn, mx, 5000, 0, seed, dX.data_ptr(), dQ.data_ptr(), idx.data_ptr(), dist.data_ptr())
        torch.cuda.synchronize()
        assert_knn_equal(idx.cpu().numpy(), dist.cpu().numpy(), oi, od)


@pytest.mark.parametrize("N,D,K,T", [(3000, 200, 8, 8), (4000, 37, 70, 6)])
def test_ann_batches_take_the_form_their_buckets_ask_for(gpu, capi, orc, rng, monkeypatch, N, D, K, T):
    """Half of the points are equal, so that every tree has one bucket far above the leaf limit; the number of queries is such
    that batches with a larger one are searched tree by tree and the others together, in one call, into rows not in order."""
    import torch
    monkeypatch.setenv("RSFK_TREE_BATCH", "2")
    X = rng.standard_normal((N, D)).astype(np.float32)
    X[: N // 2] = X[0]
    X = X[rng.permutation(N)]
    widest = [orc.build_tree(X, K + 1, 2 * K + 2, 30, 5 + t)[2].max() for t in range(T)]
    line = np.median([max(widest[t:t + 2]) for t in range(0, T, 2)])
    NQ = int(1.2e5 * N / (D * line))
    Q = rng.standard_normal((NQ, D)).astype(np.float32)
    Q[: NQ // 3] = X[rng.integers(0, N, NQ // 3)]
    assert min(widest) > 1024 and NQ * (2 * K + 2) * D < 5e7
    idx = np.full((NQ, K), -1, np.int32)
    dist = np.full((NQ, K), np.inf, np.float32)
    orc.ann_forest(X, Q, K, 1, K + 1, 2 * K + 2, 30, 99, q_idx=idx, q_dist=dist)
    idx, dist = np.ascontiguousarray(idx[:, ::-1]), np.ascontiguousarray(dist[:, ::-1])
    di, dd, dX, dQ = (torch.from_numpy(a).cuda() for a in (idx, dist, X, Q))
    orc.ann_forest(X, Q, K, T, K + 1, 2 * K + 2, 30, 5, q_idx=idx, q_dist=dist)
    _say("ann batches", N, NQ, D, K, T, widest)
    capi.knn_ann_device(T, K, N, NQ, D, K + 1, 2 * K + 2, 30, 0, 5, dX.data_ptr(), dQ.data_ptr(), di.data_ptr(), dd.data_ptr())
    torch.cuda.synchronize()
    assert_knn_equal(di.cpu().numpy(), dd.cpu().numpy(), idx, dist)


# the dimensions whose bounds are made from float16 copies, whole and ragged; one and two blocks of members, their remainders, and more; items of
# one query, of 32 and more; few pairs that wait until the end and many
@pytest.mark.parametrize("N,NQ,D,K,T,mn,mx", [(700, 900, 97, 64, 4, 65, 130), (2000, 2500, 100, 32, 6, 33, 66), (600, 333, 101, 5, 7, 6, 12), (40, 1, 104, 3, 3, 50, 100),
                                              (1500, 1200, 112, 1, 5, 32, 64), (400, 65, 113, 10, 3, 150, 300), (900, 1000, 128, 20, 4, 21, 33)])
@pytest.mark.parametrize("data", ["normal", "ties", "offset", "huge", "apart"])
def test_ann_screened_by_copies_matches_oracle(gpu, capi, orc, rng, monkeypatch, N, NQ, D, K, T, mn, mx, data):
    """The bucket step that bounds the pairs by float16 copies == the oracle, also into rows that hold something, with queries that the
    copies' range does not hold, and without the memory for the copies."""
    import torch
    draw = {"normal": lambda n: rng.standard_normal((n, D)), "ties": lambda n: rng.integers(0, 3, (n, D)),
            "offset": lambda n: rng.standard_normal((n, D)) * 1e-2 + 300.0,
            "huge": lambda n: rng.standard_normal((n, D)) * np.where(rng.random((n, 1)) < 0.1, 3e18, 1.0),
            "apart": lambda n: rng.standard_normal((n, D)) * (1.0 if n == N else np.where(rng.random((n, 1)) < 0.3, 1e5, 2.0))}[data]
    X, Q = draw(N).astype(np.float32), draw(NQ).astype(np.float32)
    dX, dQ = torch.from_numpy(X).cuda(), torch.from_numpy(Q).cuda()
    oi, od = orc.ann_forest(X, Q, K, T, mn, mx, 5000, 5)
    orc.ann_forest(X, Q, K, 2, mn, mx, 5000, 77, q_idx=oi, q_dist=od)
    monkeypatch.setenv("RSFK_ANN_FOREST", "0")
    monkeypatch.setenv("RSFK_ANN_SCREEN", "always")
    for optional in (None, "0"):
        if optional is not None:
            monkeypatch.setenv("RSFK_OPTIONAL_MB", optional)
        idx = torch.full((NQ, K), -1, dtype=torch.int32, device="cuda")
        dist = torch.full((NQ, K), float("inf"), dtype=torch.float32, device="cuda")
        _say("ann screened by copies", N, NQ, D, K, T, mn, mx, data, optional)
        for trees, seed in ((T, 5), (2, 77)):
            capi.knn_ann_device(trees, K, N, NQ, D, mn, mx, 5000, 0, seed, dX.data_ptr(), dQ.data_ptr(), idx.data_ptr(), dist.data_ptr())
        torch.cuda.synchronize()
        assert_knn_equal(idx.cpu().numpy(), dist.cpu().numpy(), oi, od)


# calls whose early screened trees bound the pairs by the fp32 rows and whose late ones by the copies: from 256 MB and from 640 MB of rows on
@pytest.mark.parametrize("N,NQ,D,K,T", [(300000, 500001, 97, 10, 30), (700001, 900000, 104, 6, 14)])
def test_ann_screened_by_fp32_rows_then_by_copies(gpu, capi, monkeypatch, N, NQ, D, K, T):
    """== the search without room for copies (which the oracle has confirmed at small sizes)."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(3)
    X, Q = torch.randn(N, D, device="cuda", generator=g), torch.randn(NQ, D, device="cuda", generator=g)
    out = []
    for room in (None, "0"):
        if room is not None:
            monkeypatch.setenv("RSFK_OPTIONAL_MB", room)
        idx = torch.full((NQ, K), -1, dtype=torch.int32, device="cuda")
        dist = torch.full((NQ, K), float("inf"), device="cuda")
        torch.cuda.synchronize()
        _say("ann screened twice", N, NQ, D, K, T, room)
        capi.knn_ann_device(T, K, N, NQ, D, K + 1, 2 * K + 2, 5000, 0, 3, X.data_ptr(), Q.data_ptr(), idx.data_ptr(), dist.data_ptr())
        out.append((idx, dist))
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])


# Workgroups with many items each, as they have them from about 16,384 items (a million queries) on: the items that follow an item are looked up while it is
# worked on, and pairs of several items wait for each other.  Buckets of few members and queries (a pair or two of an item are
# left, so that tens of items wait together), items of 32 queries and more than one block of members, items between these; one workgroup,
# fewer than items, and as many as items of a tree or more.
@pytest.mark.parametrize("N,NQ,D,K,T,mn,mx", [(3000, 2500, 97, 4, 5, 3, 6), (1200, 1600, 100, 32, 6, 33, 66), (500, 900, 128, 64, 4, 100, 200), (900, 700, 113, 1, 6, 9, 18),
                                              (60, 200, 104, 7, 3, 8, 60)])
@pytest.mark.parametrize("data", ["normal", "ties", "huge"])
def test_ann_screened_by_copies_with_many_items_per_workgroup(gpu, capi, orc, rng, monkeypatch, N, NQ, D, K, T, mn, mx, data):
    """The bucket step that bounds the pairs by float16 copies, from one workgroup for all items to one for each == the oracle."""
    import torch
    draw = {"normal": lambda n: rng.standard_normal((n, D)), "ties": lambda n: rng.integers(0, 3, (n, D)),
            "huge": lambda n: rng.standard_normal((n, D)) * np.where(rng.random((n, 1)) < 0.1, 3e18, 1.0)}[data]
    X, Q = draw(N).astype(np.float32), draw(NQ).astype(np.float32)
    dX, dQ = torch.from_numpy(X).cuda(), torch.from_numpy(Q).cuda()
    oi, od = orc.ann_forest(X, Q, K, T, mn, mx, 5000, 5)
    monkeypatch.setenv("RSFK_ANN_FOREST", "0")
    monkeypatch.setenv("RSFK_ANN_SCREEN", "always")
    for groups in (1, 3, 50):
        monkeypatch.setenv("RSFK_ANN_SCREEN_GROUPS", str(groups))
        idx = torch.full((NQ, K), -1, dtype=torch.int32, device="cuda")
        dist = torch.full((NQ, K), float("inf"), dtype=torch.float32, device="cuda")
        _say("ann screened by copies, items per workgroup", N, NQ, D, K, T, mn, mx, data, groups)
        capi.knn_ann_device(T, K, N, NQ, D, mn, mx, 5000, 0, 5, dX.data_ptr(), dQ.data_ptr(), idx.data_ptr(), dist.data_ptr())
        torch.cuda.synchronize()
        assert_knn_equal(idx.cpu().numpy(), dist.cpu().numpy(), oi, od)


# one query, and the sizes around a wavefront's 64; every number of 16-dimension steps, rows that end inside one; trees that end within
# the first seven levels (the first one at its root) and go on below; queries in no tree's cloud
@pytest.mark.parametrize("N,NQ,D,K,T,mn,mx", [(40, 1, 3, 5, 3, 50, 100), (300, 63, 1, 4, 5, 5, 11), (2500, 64, 16, 3, 6, 4, 9), (5000, 65, 17, 2, 9, 3, 6),
                                              (1500, 500, 37, 8, 4, 9, 18), (2000, 257, 64, 16, 3, 17, 64), (6000, 129, 65, 5, 4, 6, 12), (900, 300, 81, 6, 3, 7, 14),
                                              (3000, 1000, 100, 4, 5, 5, 10), (1200, 100, 112, 4, 4, 5, 10), (4000, 200, 128, 10, 3, 11, 22)])
@pytest.mark.parametrize("data", ["normal", "ties", "tiny", "offset", "huge", "apart"])
def test_ann_first_levels_of_all_trees_match_oracle(gpu, capi, orc, rng, monkeypatch, N, NQ, D, K, T, mn, mx, data):
    """Queries that take the first seven levels by rounded hyperplanes on the matrix cores, then the others exactly, by rounded ones, and
    without the memory for either == the oracle."""
    import torch
    draw = {"normal": lambda n: rng.standard_normal((n, D)), "ties": lambda n: rng.integers(0, 3, (n, D)),
            "tiny": lambda n: rng.standard_normal((n, D)) * 1e-18, "offset": lambda n: rng.standard_normal((n, D)) * 1e-2 + 300.0,
            "huge": lambda n: rng.standard_normal((n, D)) * np.where(rng.random((n, 1)) < 0.1, 3e18, 1.0),
            "apart": lambda n: rng.standard_normal((n, D)) * (1.0 if n == N else 1e6) + (0.0 if n == N else -70.0)}[data]
    X, Q = draw(N).astype(np.float32), draw(NQ).astype(np.float32)
    dX, dQ = torch.from_numpy(X).cuda(), torch.from_numpy(Q).cuda()
    oi, od = orc.ann_forest(X, Q, K, T, mn, mx, 5000, 5)
    monkeypatch.setenv("RSFK_ANN_FOREST", "0")
    monkeypatch.setenv("RSFK_ANN_TOP", "1")
    for low, optional in (("0", None), ("1", None), ("1", "0")):
        monkeypatch.setenv("RSFK_ANN_ROUTE_LOW", low)
        if optional is not None:
            monkeypatch.setenv("RSFK_OPTIONAL_MB", optional)
        idx = torch.full((NQ, K), -1, dtype=torch.int32, device="cuda")
        dist = torch.full((NQ, K), float("inf"), dtype=torch.float32, device="cuda")
        _say("ann first levels", N, NQ, D, K, T, mn, mx, data, low, optional)
        capi.knn_ann_device(T, K, N, NQ, D, mn, mx, 5000, 0, 5, dX.data_ptr(), dQ.data_ptr(), idx.data_ptr(), dist.data_ptr())
        torch.cuda.synchronize()
        assert_knn_equal(idx.cpu().numpy(), dist.cpu().numpy(), oi, od)


# items of fewer and of more than 32 queries; buckets on both sides of 32 and 64 members; rows that end inside a step and inside
# a 16-byte piece; distances that overflow, a common offset that leaves the bounds useless, equal distances
@pytest.mark.parametrize("N,NQ,D,K,T,mn,mx", [(500, 900, 16, 64, 5, 65, 130), (3000, 2500, 100, 32, 6, 33, 66), (700, 333, 31, 5, 9, 6, 12),
                                              (400, 65, 3, 10, 4, 200, 400), (900, 64, 33, 1, 3, 32, 64), (600, 1000, 130, 20, 4, 21, 33)])
@pytest.mark.parametrize("data", ["normal", "ties", "offset", "huge"])
def test_ann_screened_buckets_match_oracle(gpu, capi, orc, rng, monkeypatch, N, NQ, D, K, T, mn, mx, data):
    """The bucket step that bounds the pairs on the matrix cores first (from the second tree on) == the oracle, also into rows
    that hold something and are not in order."""
    import torch
    draw = {"normal": lambda n: rng.standard_normal((n, D)), "ties": lambda n: rng.integers(0, 3, (n, D)),
            "offset": lambda n: rng.standard_normal((n, D)) * 1e-2 + 300.0,
            "huge": lambda n: rng.standard_normal((n, D)) * np.where(rng.random((n, 1)) < 0.1, 3e18, 1.0)}[data]
    X, Q = draw(N).astype(np.float32), draw(NQ).astype(np.float32)
    dX, dQ = torch.from_numpy(X).cuda(), torch.from_numpy(Q).cuda()
    oi, od = orc.ann_forest(X, Q, K, T, mn, mx, 5000, 5)
    monkeypatch.setenv("RSFK_ANN_FOREST", "0")
    monkeypatch.setenv("RSFK_ANN_SCREEN", "always")
    monkeypatch.setenv("RSFK_ANN_ROUTE_LOW", "1")
    idx = torch.full((NQ, K), -1, dtype=torch.int32, device="cuda")
    dist = torch.full((NQ, K), float("inf"), dtype=torch.float32, device="cuda")
    _say("ann screened", N, NQ, D, K, T, mn, mx, data)
    capi.knn_ann_device(T, K, N, NQ, D, mn, mx, 5000, 0, 5, dX.data_ptr(), dQ.data_ptr(), idx.data_ptr(), dist.data_ptr())
    torch.cuda.synchronize()
    assert_knn_equal(idx.cpu().numpy(), dist.cpu().numpy(), oi, od)
    idx, dist = idx.flip(1).contiguous(), dist.flip(1).contiguous()
    orc.ann_forest(X, Q, K, 2, mn, mx, 5000, 77, q_idx=oi, q_dist=od)
    capi.knn_ann_device(2, K, N, NQ, D, mn, mx, 5000, 0, 77, dX.data_ptr(), dQ.data_ptr(), idx.data_ptr(), dist.data_ptr())
    torch.cuda.synchronize()
    assert_knn_equal(idx.cpu().numpy(), dist.cpu().numpy(), oi, od)


@pytest.mark.parametrize("D", [1, 2, 3, 4, 5, 7, 36, 37, 39, 130])
@pytest.mark.parametrize("shift", [0, 1, 2, 3])
def test_rows_that_begin_at_any_float(gpu, capi, orc, rng, monkeypatch, D, shift):
    """Rows of any length at any multiple of four bytes, the last one at the end of its allocation: forest with exploration (both
    forms of the bucket step) and query-set search == the oracle."""
    import torch
    N, NQ, K, T, mn, mx = 1500, 400, 12, 5, 13, 80
    X, Q = rng.standard_normal((N, D)).astype(np.float32), rng.standard_normal((NQ, D)).astype(np.float32)
    oi, od = orc.forest(X, K, T, mn, mx, 5000, 3, 1)
    ai, ad = orc.ann_forest(X, Q, K, T, mn, mx, 5000, 3)
    put = lambda A: torch.cat([torch.full((shift,), 1e9), torch.from_numpy(A).flatten()]).cuda()[shift:]
    dX, dQ = put(X), put(Q)
    assert dX.data_ptr() % 16 == 4 * shift
    _say("rows at any float", D, shift)
    for form in ("0", "1"):
        monkeypatch.setenv("RSFK_FOREST_MERGE", form)
        monkeypatch.setenv("RSFK_ANN_FOREST", form)
        monkeypatch.setenv("RSFK_ANN_SCREEN", "always")
        idx = torch.full((N, K), -1, dtype=torch.int32, device="cuda")
        dist = torch.full((N, K), float("inf"), dtype=torch.float32, device="cuda")
        idx[:, 0] = torch.arange(N, dtype=torch.int32, device="cuda")
        dist[:, 0] = 0.0
        torch.cuda.synchronize()
        capi.knn_forest_device(T, K, N, D, mn, mx, 5000, 0, 3, 1, dX.data_ptr(), idx.data_ptr(), dist.data_ptr())
        assert_knn_equal(idx.cpu().numpy(), dist.cpu().numpy(), oi, od)
        idx = torch.full((NQ, K), -1, dtype=torch.int32, device="cuda")
        dist = torch.full((NQ, K), float("inf"), dtype=torch.float32, device="cuda")
        torch.cuda.synchronize()
        capi.knn_ann_device(T, K, N, NQ, D, mn, mx, 5000, 0, 3, dX.data_ptr(), dQ.data_ptr(), idx.data_ptr(), dist.data_ptr())
        assert_knn_equal(idx.cpu().numpy(), dist.cpu().numpy(), ai, ad)


def test_ann_device_entry_point_merges_into_given_rows(gpu, capi, orc, rng):
    """Device-resident call, twice with different seeds on the same rows == the oracle doing the same."""
    import torch
    N, NQ, D, K = 12000, 2048, 40, 16
    X = rng.standard_normal((N, D)).astype(np.float32)
    Q = rng.standard_normal((NQ, D)).astype(np.float32)
    dX, dQ = torch.from_numpy(X).cuda(), torch.from_numpy(Q).cuda()
    idx = torch.full((NQ, K), -1, dtype=torch.int32, device="cuda")
    dist = torch.full((NQ, K), float("inf"), dtype=torch.float32, device="cuda")
    log = np.zeros(16 * 3 + 2, np.float32)
    _say("ann device", N, NQ, D, K)
    capi.knn_ann_device(3, K, N, NQ, D, K + 1, 2 * K + 2, 5000, 0, 7, dX.data_ptr(), dQ.data_ptr(),
                        idx.data_ptr(), dist.data_ptr(), log)
    capi.knn_ann_device(2, K, N, NQ, D, K + 1, 2 * K + 2, 5000, 0, 100, dX.data_ptr(), dQ.data_ptr(),
                        idx.data_ptr(), dist.data_ptr())
    torch.cuda.synchronize()
    oi, od = orc.ann_forest(X, Q, K, 3, K + 1, 2 * K + 2, 5000, 7)
    orc.ann_forest(X, Q, K, 2, K + 1, 2 * K + 2, 5000, 100, q_idx=oi, q_dist=od)
    assert_knn_equal(idx.cpu().numpy(), dist.cpu().numpy(), oi, od)
    assert (log[9:12] > 0).all() and log[48] > 0          # Total Leaves per tree, total seconds
    # the recorded index must not change the partition a plain tree build gives
    perm, ls, lz, st = capi.build_tree(X, K + 1, 2 * K + 2, 5000, 7)
    operm, ostarts, osizes, ost = orc.build_tree(X, K + 1, 2 * K + 2, 5000, 7)
    assert np.array_equal(perm, operm) and np.array_equal(lz, osizes) and int(log[9]) == len(osizes)
    # no queries: nothing to do, nothing touched
    capi.knn_ann_device(2, K, N, 0, D, K + 1, 2 * K + 2, 5000, 0, 1, dX.data_ptr(), dQ.data_ptr(),
                        idx.data_ptr(), dist.data_ptr())


def test_ann_recall_rises_with_the_number_of_trees(gpu, rng):
    import gpu_rsfk
    N, NQ, D, K = 30000, 2000, 16, 10
    X = rng.random((N, D), dtype=np.float32)
    Q = rng.random((NQ, D), dtype=np.float32)
    d2 = (Q ** 2).sum(1)[:, None] - 2.0 * Q @ X.T + (X ** 2).sum(1)[None, :]
    true = np.argsort(d2, axis=1)[:, :K]
    r = gpu_rsfk.RSFK(random_state=1)
    rec = []
    for T in (1, 8, 40):
        gi, _ = r.find_nearest_neighbors_ann(X, Q, K, n_trees=T)
        rec.append(np.mean([len(set(gi[q]) & set(true[q])) / K for q in range(NQ)]))
    _say("ann recall", rec)
    assert rec[0] < rec[1] < rec[2] and rec[2] > 0.5


@pytest.mark.parametrize("N,mn,mx", [(40, 3, 6), (3000, 3, 6), (4000, 4, 9), (9000, 3, 7), (21000, 2, 5), (70000, 2, 4)])
def test_queries_are_counted_whatever_the_records(gpu, capi, orc, rng, monkeypatch, N, mn, mx):
    """Counters of the buckets a line apart, closer, and side by side (from few to many records of a tree), one tree after the other."""
    monkeypatch.setenv("RSFK_ANN_FOREST", "0")
    D, K, T, NQ = 3, 4, 3, 2500
    X, Q = rng.random((N, D), dtype=np.float32), rng.random((NQ, D), dtype=np.float32)
    Q[:1500] = Q[0]                                             # (most of them reach one bucket)
    qi, qd = np.full((NQ, K), -1, np.int32), np.full((NQ, K), np.inf, np.float32)
    _say("queries by records", N, mn, mx)
    log = np.zeros(16 * T + 2, np.float32)
    capi.lib().pymodule_rsfk_knn_ann(T, K, N, NQ, D, mn, mx, 5000, 0, 11, 0, X.ctypes.data, Q.ctypes.data, qi.ctypes.data, qd.ctypes.data, log.ctypes.data)
    oi, od = orc.ann_forest(X, Q, K, T, mn, mx, 5000, 11)
    assert_knn_equal(qi, qd, oi, od)


# ---------------------------------------------------------------------------
# symmetrised graph export
# ---------------------------------------------------------------------------
@pytest.mark.parametrize("N,K,drop_self", [(5000, 16, True), (3000, 100, False), (2000, 200, True), (1, 3, False),
                                           (700, 1, True), (900, 300, True), (700, 1000, False)])
def test_symmetric_graph_matches_oracle(gpu, orc, rng, N, K, drop_self):
    import gpu_rsfk
    idx = np.stack([rng.permutation(max(N, K + 1))[:K] for _ in range(N)]).astype(np.int32)
    idx[idx >= N] = -1                                           # only when N <= K: empty slots
    idx[:, 0] = np.arange(N)                                     # the point itself first, as the forest stores it
    for p in range(N):
        dup = np.flatnonzero(idx[p, 1:] == p) + 1
        idx[p, dup] = -1
    idx[rng.random((N, K)) < 0.02] = -1
    val = rng.random((N, K)).astype(np.float32)
    _say("symmetrize", N, K, drop_self)
    gp, gc, gv = gpu_rsfk.symmetric_knn_graph(idx, val, drop_self=drop_self)
    op, oc, ov = orc.symmetrize(idx, val, drop_self=drop_self)
    assert np.array_equal(gp, op) and np.array_equal(gc, oc)
    assert np.array_equal(gv, ov)          # a stored edge keeps its own value, an added one the value of its source
    gp2, gc2, gv2 = gpu_rsfk.symmetric_knn_graph(idx, None, drop_self=drop_self)
    assert np.array_equal(gp2, op) and np.array_equal(gc2, oc) and (gv2 == 0).all()


# Rows as unions of the stored neighbours and the reversed entries: rows of one, two and four entries per lane, rows that
# go to a workgroup (points that very many others store), rows of more candidates than that takes (the other form),
# empty rows, with and without the point itself.
@pytest.mark.parametrize("N,K,hubs,drop_self", [(900, 5, 0, True), (3000, 20, 3, False), (5000, 33, 40, True), (6000, 90, 200, True),
                                                (9000, 12, 1, True), (1500, 300, 5, False), (12000, 3, 2, True)])
def test_symmetric_graph_with_hubs_matches_oracle(gpu, orc, rng, monkeypatch, N, K, hubs, drop_self):
    import gpu_rsfk
    monkeypatch.setenv("RSFK_GRAPH_FLAGS", "0")
    idx = np.stack([rng.choice(N, K, replace=False) for _ in range(N)]).astype(np.int32)
    for h in range(hubs):                                       # a point most others store, in slot h (unless they do already)
        put = (rng.random(N) < 0.3 + 0.7 / (h + 1)) & ~(idx == h).any(1)
        idx[put, h % K] = h
    idx[rng.random((N, K)) < 0.05] = -1
    idx[N // 2:N // 2 + 20] = -1
    a, b = np.minimum(idx, np.arange(N)[:, None]).astype(np.int64), np.maximum(idx, np.arange(N)[:, None])
    val = ((a * 7919 + b * 104729) % 10007).astype(np.float32)  # one value per pair
    _say("symmetrize with hubs", N, K, hubs, drop_self)
    gp, gc, gv = gpu_rsfk.symmetric_knn_graph(idx, val, drop_self=drop_self)
    op, oc, ov = orc.symmetrize(idx, val, drop_self=drop_self)
    assert np.array_equal(gp, op) and np.array_equal(gc, oc) and np.array_equal(gv, ov)


# The forms of the row lengths and rows: four, two and one point per wavefront (K up to 32, 64 and beyond), stored neighbours as a table
# or as they are (K above 128), a last wavefront with points beyond N, rows on either side of what a wavefront takes together, hubs; the
# reversed graph by tiles (RSFK_REV_STAGED=2) and entry by entry.
@pytest.mark.parametrize("N,K,hubs", [(4001, 1, 0), (4003, 31, 2), (4001, 32, 0), (3001, 33, 2), (3001, 64, 0), (2999, 65, 3), (3001, 128, 0), (2801, 129, 2),
                                      (40000, 8, 5)])
@pytest.mark.parametrize("staged", ["0", "2"])
def test_symmetric_graph_forms(gpu, orc, rng, monkeypatch, N, K, hubs, staged):
    import gpu_rsfk
    monkeypatch.setenv("RSFK_GRAPH_FLAGS", "0")
    monkeypatch.setenv("RSFK_REV_STAGED", staged)
    idx = ((np.arange(N)[:, None] + np.cumsum(rng.integers(1, 4, (N, K)), axis=1)) % N).astype(np.int32)
    back = rng.random((N, K)) < 0.5                             # (half of the neighbours on the other side: mutual edges)
    idx = np.where(back, (2 * np.arange(N)[:, None] - idx) % N, idx).astype(np.int32)
    for p in range(N):
        if len(np.unique(idx[p])) < K:
            idx[p] = (p + 1 + np.arange(K)) % N
    for h in range(hubs):
        put = (rng.random(N) < (0.02, 0.2, 0.7)[h % 3]) & ~(idx == h).any(1)
        idx[put, h % K] = h
    idx[rng.random((N, K)) < 0.02] = -1
    a, b = np.minimum(idx, np.arange(N)[:, None]).astype(np.int64), np.maximum(idx, np.arange(N)[:, None])
    val = ((a * 7919 + b * 104729) % 10007).astype(np.float32)  # one value per pair
    _say("symmetrize forms", N, K, hubs, staged)
    gp, gc, gv = gpu_rsfk.symmetric_knn_graph(idx, val, drop_self=True)
    op, oc, ov = orc.symmetrize(idx, val, drop_self=True)
    assert np.array_equal(gp, op) and np.array_equal(gc, oc) and np.array_equal(gv, ov)


# The reversed graph in one launch (RSFK_REV_STAGED=3): a point per workgroup and many, a last workgroup with few, entries that are no multiple of four,
# hubs with more entries than a workgroup keeps.
@pytest.mark.parametrize("N,K,hubs", [(100, 7, 1), (257, 3, 0), (4003, 31, 2), (40000, 8, 5), (16500, 127, 0), (65537, 1, 0)])
def test_symmetric_graph_of_one_launch(gpu, orc, rng, monkeypatch, N, K, hubs):
    test_symmetric_graph_forms(gpu, orc, rng, monkeypatch, N, K, hubs, "3")


# Points per wavefront by the points and the neighbours: two and four with rows of many neighbours, on either side of the lines.
@pytest.mark.parametrize("N,K,hubs", [(31999, 32, 0), (32003, 32, 2), (31003, 31, 0), (15999, 32, 0), (16001, 32, 2), (16497, 33, 0), (16503, 33, 3), (32003, 64, 2)])
def test_symmetric_graph_points_per_wavefront(gpu, orc, rng, monkeypatch, N, K, hubs):
    import gpu_rsfk
    monkeypatch.setenv("RSFK_GRAPH_FLAGS", "0")
    idx = ((np.arange(N)[:, None] + np.cumsum(rng.integers(1, 4, (N, K)), axis=1)) % N).astype(np.int32)
    back = rng.random((N, K)) < 0.5
    idx = np.where(back, (2 * np.arange(N)[:, None] - idx) % N, idx).astype(np.int32)
    same = (np.diff(np.sort(idx, axis=1), axis=1) == 0).any(1)
    idx[same] = (np.flatnonzero(same)[:, None] + 1 + np.arange(K)) % N
    for h in range(hubs):
        put = (rng.random(N) < (0.005, 0.02, 0.3)[h % 3]) & ~(idx == h).any(1)
        idx[put, h % K] = h
    idx[rng.random((N, K)) < 0.02] = -1
    a, b = np.minimum(idx, np.arange(N)[:, None]).astype(np.int64), np.maximum(idx, np.arange(N)[:, None])
    val = ((a * 7919 + b * 104729) % 10007).astype(np.float32)  # one value per pair
    _say("symmetrize, points per wavefront", N, K, hubs)
    gp, gc, gv = gpu_rsfk.symmetric_knn_graph(idx, val, drop_self=True)
    op, oc, ov = orc.symmetrize(idx, val, drop_self=True)
    assert np.array_equal(gp, op) and np.array_equal(gc, oc) and np.array_equal(gv, ov)


@pytest.mark.parametrize("N,lead", [(16384, 0), (16385, 0), (16385, 4), (140000, 1020), (140001, 4092)])
def test_results_into_fresh_pages(gpu, capi, rng, N, lead):
    """Result arrays of up to 4 MiB and of more, anywhere on pages that do not exist yet: the results, and nothing beside them."""
    import mmap
    K, D = 32, 4
    X = rng.standard_normal((N, D)).astype(np.float32)
    nk = N * K
    want_idx, want_dist = np.zeros((N, K), np.int32), np.zeros((N, K), np.float32)
    want_dist += 1.0                                            # (present pages)
    log = np.zeros(64, np.float32)
    _say("results into fresh pages", N, lead)
    call = capi.lib().rsfk_knn_forest_fresh_host
    args = (1, K, N, D, K + 1, 3 * K, 5000, 0, 5, 0, 1)
    assert call(*args, X.ctypes.data, want_idx.ctypes.data, want_dist.ctypes.data, log.ctypes.data) == 0
    maps = [np.frombuffer(mmap.mmap(-1, lead + 4 * nk + 8192), np.uint8) for _ in range(2)]
    assert call(*args, X.ctypes.data, maps[0].ctypes.data + lead, maps[1].ctypes.data + lead, log.ctypes.data) == 0
    for m, want in zip(maps, (want_idx, want_dist)):
        assert np.array_equal(m[lead:lead + 4 * nk].view(want.dtype), want.ravel())
        assert not m[:lead].any() and not m[lead + 4 * nk:].any()


@pytest.mark.parametrize("N,K,hubs,optional", [(4100, 2, 1, None), (4200, 1, 1, None), (20000, 9, 60, None), (30000, 4, 3, None), (30000, 4, 3, "0")])
def test_rows_of_hubs_match_oracle(gpu, capi, orc, rng, monkeypatch, N, K, hubs, optional):
    """Rows of more candidates than a workgroup sorts (just above 4,096, several hubs, several shares of R(p) per hub), into
    arrays of the caller, with and without values, and the count alone; without room for the hubs' entries the other form."""
    import torch
    if optional is not None:
        monkeypatch.setenv("RSFK_OPTIONAL_MB", optional)
    idx = rng.integers(0, N, (N, K)).astype(np.int32)
    idx[:, 0] = rng.permutation(hubs)[np.minimum(rng.geometric(0.3, N) - 1, hubs - 1)] if hubs > 1 else 0
    for k in range(1, K):                                       # (a row must not hold a point twice)
        idx[(idx[:, :k] == idx[:, k:k + 1]).any(1), k] = -1
    idx[:hubs, 0] = -1
    a, b = np.minimum(idx, np.arange(N)[:, None]).astype(np.int64), np.maximum(idx, np.arange(N)[:, None])
    val = ((a * 7919 + b * 104729) % 10007).astype(np.float32)
    _say("rows of hubs", N, K, hubs, optional)
    op, oc, ov = orc.symmetrize(idx, val, drop_self=True)
    assert np.diff(op).max() > 4090
    di, dd = torch.from_numpy(idx).cuda(), torch.from_numpy(val).cuda()
    for dist in (dd.data_ptr(), 0):
        indptr = torch.zeros(N + 1, dtype=torch.int32, device="cuda")
        assert capi.symmetrize_device(di.data_ptr(), dist, N, K, True, indptr.data_ptr(), 0, 0, 0) == len(oc)
        cols = torch.full((len(oc),), -1, dtype=torch.int32, device="cuda")
        vals = torch.full((len(oc),), -1.0, device="cuda")
        assert capi.symmetrize_device(di.data_ptr(), dist, N, K, True, indptr.data_ptr(), cols.data_ptr(), vals.data_ptr(), len(oc)) == len(oc)
        torch.cuda.synchronize()
        assert np.array_equal(indptr.cpu().numpy(), op) and np.array_equal(cols.cpu().numpy(), oc)
        assert np.array_equal(vals.cpu().numpy(), ov if dist else np.zeros_like(ov))


def test_without_the_optional_working_memory(gpu, orc, rng, monkeypatch):
    """Nothing but speed depends on the blocks a call can do without: with none of them (RSFK_OPTIONAL_MB=0) the export, the
    build and the query-set search take their other forms and give the same results."""
    import gpu_rsfk
    monkeypatch.setenv("RSFK_OPTIONAL_MB", "0")
    N, D, K, T = 4000, 19, 70, 4
    X, Q = rng.standard_normal((N, D)).astype(np.float32), rng.standard_normal((50, D)).astype(np.float32)
    r = gpu_rsfk.RSFK(random_state=3)
    _say("no optional memory: build")
    gi, gd = r.find_nearest_neighbors(X, K, n_trees=T, nn_exploring_factor=1)
    oi, od = orc.forest(X, K, T, K + 1, 2 * (K + 1), 5000, 3, 1)
    assert_knn_equal(gi, gd, oi, od)
    assert ["k_forest_pairs + k_forest_merge"] not in [k[2] for k in gpu.last_build_report()["bucket_kernels"]]
    _say("no optional memory: queries")
    qi, qd = r.find_nearest_neighbors_ann(X, Q, K, n_trees=T)
    oi, od = orc.ann_forest(X, Q, K, T, K + 1, 2 * (K + 1), 5000, 3)
    assert_knn_equal(qi, qd, oi, od)
    _say("no optional memory: graph")
    gp, gc, gv = gpu_rsfk.symmetric_knn_graph(gi, gd)
    op, oc, ov = orc.symmetrize(gi, gd, drop_self=True)
    assert np.array_equal(gp, op) and np.array_equal(gc, oc) and np.array_equal(gv, ov)


def test_symmetric_graph_of_a_built_graph(gpu, capi, orc, rng):
    """On a graph the library built (one distance value per pair) the export equals the oracle's bit for bit; device
    entry point with the two-call protocol (count, then fill)."""
    import torch
    import gpu_rsfk
    N, D, K = 30000, 20, 12
    X = rng.standard_normal((N, D)).astype(np.float32)
    gi, gd = gpu_rsfk.RSFK(random_state=2).find_nearest_neighbors(X, K, n_trees=6)
    op, oc, ov = orc.symmetrize(gi, gd, drop_self=True)
    di, dd = torch.from_numpy(gi).cuda(), torch.from_numpy(gd).cuda()
    indptr = torch.empty(N + 1, dtype=torch.int32, device="cuda")
    _say("symmetrize device", N, K)
    nnz = capi.symmetrize_device(di.data_ptr(), dd.data_ptr(), N, K, True, indptr.data_ptr(), 0, 0, 0)
    assert nnz == len(oc) and N * (K - 1) <= nnz <= 2 * N * (K - 1)
    cols = torch.empty(nnz, dtype=torch.int32, device="cuda")
    vals = torch.empty(nnz, dtype=torch.float32, device="cuda")
    assert capi.symmetrize_device(di.data_ptr(), dd.data_ptr(), N, K, True, indptr.data_ptr(), cols.data_ptr(),
                                  vals.data_ptr(), nnz) == nnz
    torch.cuda.synchronize()
    assert np.array_equal(indptr.cpu().numpy(), op) and np.array_equal(cols.cpu().numpy(), oc)
    assert np.array_equal(vals.cpu().numpy(), ov)
    with pytest.raises(RuntimeError, match="too small"):
        capi.symmetrize_device(di.data_ptr(), dd.data_ptr(), N, K, True, indptr.data_ptr(), cols.data_ptr(),
                               vals.data_ptr(), nnz - 1)
    S = gpu_rsfk.symmetric_knn_graph(gi, gd, as_scipy=True)
    assert S.shape == (N, N) and (abs(S - S.T)).nnz == 0 and S.diagonal().sum() == 0


@pytest.mark.parametrize("self_in", [True, False])
def test_rows_made_on_the_device_equal_uploaded_rows(gpu, rng, self_in):
    """find_nearest_neighbors lets the library make the initial rows; the reference's entry point with the rows
    uploaded must give the same arrays."""
    import gpu_rsfk
    N, D, K, T = 9000, 20, 12, 3
    X = rng.standard_normal((N, D)).astype(np.float32)
    r = gpu_rsfk.RSFK(random_state=4)
    _say("fresh rows", self_in)
    gi, gd = r.find_nearest_neighbors(X, K, n_trees=T, point_in_self_neigh=self_in)
    hi = np.full((N, K), -1, np.int32)
    hd = np.full((N, K), np.inf, np.float32)
    if self_in:
        hi[:, 0] = np.arange(N, dtype=np.int32)
        hd[:, 0] = 0.0
    log = np.zeros(16 * T + 2, np.float32)
    r._lib.pymodule_rsfk_knn(T, K, N, D, K + 1, 2 * K + 2, 5000, 0, 4, 1, X, hi, hd, log)
    assert np.array_equal(gd, hd)
    assert_knn_equal(gi, gd, hi, hd)


@pytest.mark.parametrize("N,D,K", [(1500, 9000, 8), (1200, 20000, 6)])
def test_very_long_rows(gpu, orc, rng, N, D, K):
    """Rows far beyond what the LDS-resident fast paths take: the kernels with smaller working sets take over and the
    lists stay those of the oracle (forest with one exploration pass, and the query-set search)."""
    import gpu_rsfk
    X = rng.standard_normal((N, D)).astype(np.float32)
    r = gpu_rsfk.RSFK(random_state=3)
    _say("long rows", N, D, K)
    gi, gd = r.find_nearest_neighbors(X, K, n_trees=1)
    oi, od = orc.forest(X, K, 1, K + 1, 2 * K + 2, 5000, 3, 1)
    assert_knn_equal(gi, gd, oi, od)
    Q = rng.standard_normal((200, D)).astype(np.float32)
    ai, ad = r.find_nearest_neighbors_ann(X, Q, K, n_trees=1)
    qi, qd = orc.ann_forest(X, Q, K, 1, K + 1, 2 * K + 2, 5000, 3)
    assert_knn_equal(ai, ad, qi, qd)


def test_points_with_nan_coordinates(gpu, orc, rng):
    """A NaN distance is below no row maximum: such points keep only themselves, nobody holds them, and the rest of
    the graph is the oracle's (same trees: a NaN side test sends the point left in both)."""
    import gpu_rsfk
    N, D, K, T = 6000, 10, 8, 3
    X = rng.standard_normal((N, D)).astype(np.float32)
    bad = np.arange(0, N, 7)
    X[bad] = np.nan
    _say("nan rows")
    gi, gd = gpu_rsfk.RSFK(random_state=3).find_nearest_neighbors(X, K, n_trees=T)
    oi, od = orc.init_lists(N, K, self_in=True)
    orc.forest(X, K, T, K + 1, 2 * K + 2, 5000, 3, 1, knn_idx=oi, knn_dist=od)
    assert not np.isnan(gd).any() and not np.isnan(od).any()
    assert (gi[bad, 0] == bad).all() and (gi[bad, 1:] == -1).all()
    assert_knn_equal(gi, gd, oi, od)


@pytest.mark.parametrize("K,D", [(8, 24), (5, 32), (20, 16)])
def test_points_with_nan_coordinates_in_large_buckets(gpu, orc, rng, K, D):
    """The same rule in the kernel that keeps a bucket's points in LDS (buckets of 80..256 low-dimensional points),
    with a third of the points NaN and K small: in the first two trees of a build nearly every candidate of a member
    is below its row's last slot, so the step that drops candidates by a histogram of their distances runs, and it
    must see the candidates with a NaN distance as absent."""
    import gpu_rsfk
    N, T = 9000, 3
    X = rng.standard_normal((N, D)).astype(np.float32)
    bad = np.arange(0, N, 3)
    X[bad, rng.integers(0, D, size=len(bad))] = np.nan
    _say("nan rows, large buckets", K, D)
    gi, gd = gpu_rsfk.RSFK(random_state=5).find_nearest_neighbors(X, K, n_trees=T, min_tree_children=80,
                                                                  max_tree_children=256, nn_exploring_factor=0)
    oi, od = orc.init_lists(N, K, self_in=True)
    orc.forest(X, K, T, 80, 256, 5000, 5, 0, knn_idx=oi, knn_dist=od)
    assert not np.isnan(gd).any() and not np.isnan(od).any()
    assert (gi[bad, 0] == bad).all() and (gi[bad, 1:] == -1).all()
    assert_knn_equal(gi, gd, oi, od)


def test_middle_phase_needs_one_more_list_of_nodes(gpu, monkeypatch):
    """The number of trees built together is chosen by an estimate with one list of nodes (48 bytes for each bucket there may be) for the middle phase;
    what its later launches take is a few kilobytes."""
    import torch
    N, D, K, T, MIN = 40000, 4, 4, 50, 2
    X = torch.rand((N, D), device="cuda")
    held = {}
    for mid in ("0", None, "0", None):                     # (the first calls also load the kernels)
        if mid is None:
            monkeypatch.delenv("RSFK_TREE_MID")
        else:
            monkeypatch.setenv("RSFK_TREE_MID", mid)
        idx = dist = None
        gpu.lib().rsfk_release_workspace()
        idx = torch.full((N, K), -1, dtype=torch.int32, device="cuda")
        dist = torch.full((N, K), float("inf"), device="cuda")
        torch.cuda.synchronize()
        before = torch.cuda.mem_get_info()[0]
        _say("memory of the middle phase", mid)
        gpu.knn_forest_device(T, K, N, D, MIN, 2 * MIN, 5000, 0, 0, 0, X.data_ptr(), idx.data_ptr(), dist.data_ptr())
        held[mid] = before - torch.cuda.mem_get_info()[0]
    assert held[None] - held["0"] <= 48 * T * (N // MIN + 2) + (8 << 20), held


def test_forest_in_several_batches(gpu, orc, rng, monkeypatch):
    """Trees are built a batch at a time (all at once when memory allows); two per batch must give the same graph,
    for the K-NN graph (buckets of both kinds, so both streams of the bucket step are in use) and the query search."""
    import gpu_rsfk
    monkeypatch.setenv("RSFK_TREE_BATCH", "2")
    N, D, K, T = 30000, 20, 32, 5
    X = rng.standard_normal((N, D)).astype(np.float32)
    Q = rng.standard_normal((2000, D)).astype(np.float32)
    r = gpu_rsfk.RSFK(random_state=9)
    _say("batches")
    gi, gd = r.find_nearest_neighbors(X, K, n_trees=T)
    oi, od = orc.forest(X, K, T, K + 1, 2 * K + 2, 5000, 9, 1)
    assert_knn_equal(gi, gd, oi, od)
    assert r.log_forest.data["Total Leaves"] == [len(orc.build_tree(X, K + 1, 2 * K + 2, 5000, 9 + t)[2]) for t in range(T)]
    ai, ad = r.find_nearest_neighbors_ann(X, Q, K, n_trees=T)
    qi, qd = orc.ann_forest(X, Q, K, T, K + 1, 2 * K + 2, 5000, 9)
    assert_knn_equal(ai, ad, qi, qd)


def _random_case(seed):
    g = np.random.default_rng(1000 + seed)
    N = int(g.choice([37, 150, 700, 1300, 2600, 5200, 9000]))
    D = int(g.choice([1, 2, 3, 7, 16, 31, 32, 33, 64, 65, 100, 129, 257]))
    K = int(g.choice([1, 2, 5, 8, 16, 31, 32, 33, 48, 64, 65, 100]))
    T = int(g.integers(1, 5))
    MIN = int(g.choice([K + 1, max(2, K // 2), K + 7, 2 * K + 3]))
    MAX = int(2 * MIN + g.choice([0, 1, 5, MIN]))
    nnef = int(g.integers(0, 3))
    kind = str(g.choice(["normal", "uniform", "grid", "clusters"]))
    if kind == "normal":
        X = g.standard_normal((N, D))
    elif kind == "uniform":
        X = g.random((N, D)) * 100.0 - 30.0
    elif kind == "grid":
        X = g.integers(0, 4, (N, D)).astype(np.float64)          # many equal distances and duplicated points
    else:
        X = g.standard_normal((8, D))[g.integers(0, 8, N)] * 5.0 + 0.05 * g.standard_normal((N, D))
    return X.astype(np.float32), K, T, MIN, MAX, nnef, kind


@pytest.mark.parametrize("seed", range(24))
def test_random_shapes_match_oracle(gpu, orc, seed):
    """Seeded random shapes, bucket limits, numbers of exploration passes and kinds of data: K-NN graph, query-set
    search and graph export against the oracle.  On the grid data almost every distance is tied with others and
    points are duplicated: rows must still be identical, since ties are broken by index everywhere."""
    import gpu_rsfk
    X, K, T, MIN, MAX, nnef, kind = _random_case(seed)
    N, D = X.shape
    _say("random case", seed, N, D, K, T, MIN, MAX, nnef, kind)
    r = gpu_rsfk.RSFK(random_state=seed)
    gi, gd = r.find_nearest_neighbors(X, K, n_trees=T, min_tree_children=MIN, max_tree_children=MAX,
                                      nn_exploring_factor=nnef, ensure_valid_indices=False)
    oi, od = orc.forest(X, K, T, MIN, MAX, 5000, seed, nnef)
    assert_knn_equal(gi, gd, oi, od)
    assert rows_have_no_duplicates(gi)
    Q = X[::3] + np.float32(0.125)
    ai, ad = r.find_nearest_neighbors_ann(X, Q, K, n_trees=T, min_tree_children=MIN, max_tree_children=MAX,
                                          ensure_valid_indices=False)
    qi, qd = orc.ann_forest(X, Q, K, T, MIN, MAX, 5000, seed)
    assert_knn_equal(ai, ad, qi, qd)
    ip, cc, vv = gpu_rsfk.symmetric_knn_graph(gi, gd, drop_self=bool(seed & 1))
    op, oc, ov = orc.symmetrize(gi, gd, drop_self=bool(seed & 1))
    assert np.array_equal(ip, op) and np.array_equal(cc, oc) and np.array_equal(vv, ov)


@pytest.mark.parametrize("N,D,K,nnef", [(1500, 3, 400, 1), (2400, 2, 1024, 0)])
def test_rows_of_many_neighbours_on_tied_data(gpu, orc, N, D, K, nnef):
    """Rows of more than 256 neighbours (eight and sixteen slots per lane) on grid data, where most distances are tied
    and points are duplicated: graph (with an exploration pass in the smaller case), query-set search and graph export."""
    import gpu_rsfk
    g = np.random.default_rng(K)
    X = g.integers(0, 6, (N, D)).astype(np.float32)
    _say("many neighbours, tied data", N, D, K)
    r = gpu_rsfk.RSFK(random_state=5)
    gi, gd = r.find_nearest_neighbors(X, K, n_trees=2, min_tree_children=K // 2, max_tree_children=K + 50,
                                      nn_exploring_factor=nnef, ensure_valid_indices=False)
    oi, od = orc.forest(X, K, 2, K // 2, K + 50, 5000, 5, nnef)
    assert_knn_equal(gi, gd, oi, od)
    assert rows_have_no_duplicates(gi)
    Q = X[::5] + np.float32(0.25)
    ai, ad = r.find_nearest_neighbors_ann(X, Q, K, n_trees=2, min_tree_children=K // 2, max_tree_children=K + 50,
                                          ensure_valid_indices=False)
    qi, qd = orc.ann_forest(X, Q, K, 2, K // 2, K + 50, 5000, 5)
    assert_knn_equal(ai, ad, qi, qd)
    ip, cc, vv = gpu_rsfk.symmetric_knn_graph(gi, gd, drop_self=True)
    op, oc, ov = orc.symmetrize(gi, gd, drop_self=True)
    assert np.array_equal(ip, op) and np.array_equal(cc, oc) and np.array_equal(vv, ov)


# Buckets of several trees at once (k_forest_pairs + k_forest_merge): one, two and four candidates per lane, rows of one
# and two slots per lane, new rows with and without the point itself, buckets just above a tile, K at the rank limits,
# duplicated points (equal distances leave the ranking to the insertions), more trees than are in flight.
@pytest.mark.parametrize("N,D,K,T,mn,mx,nnef,self_in,dup", [
    (700, 5, 4, 4, 5, 12, 0, True, False),
    (3001, 33, 31, 11, 32, 66, 1, True, False),
    (2500, 20, 64, 5, 65, 130, 0, False, False),
    (4000, 8, 40, 6, 70, 250, 0, True, False),
    (2000, 12, 100, 7, 101, 256, 0, True, False),
    (1500, 7, 200, 4, 60, 140, 0, True, False),
    (2600, 3, 16, 8, 17, 40, 2, True, True),
    (1800, 4, 20, 5, 80, 200, 0, False, True),
])
def test_buckets_of_several_trees_at_once_match_oracle(gpu, orc, rng, monkeypatch, N, D, K, T, mn, mx, nnef, self_in, dup):
    import gpu_rsfk
    monkeypatch.setenv("RSFK_FOREST_MERGE", "1")
    X = rng.standard_normal((N, D)).astype(np.float32)
    if dup:
        X[N // 2:] = X[:N - N // 2]
    _say("several trees at once", N, D, K, T, mn, mx)
    gi, gd = gpu_rsfk.RSFK(random_state=3).find_nearest_neighbors(
        X, K, n_trees=T, min_tree_children=mn, max_tree_children=mx, nn_exploring_factor=nnef, point_in_self_neigh=self_in,
        ensure_valid_indices=False)
    assert gpu.last_build_report()["bucket_kernels"] == [[0, T - 1, ["k_forest_pairs + k_forest_merge"]]]
    oi, od = orc.init_lists(N, K, self_in=self_in)
    orc.forest(X, K, T, mn, mx, 5000, 3, nnef, knn_idx=oi, knn_dist=od)
    assert_knn_equal(gi, gd, oi, od)
