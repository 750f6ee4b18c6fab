"""Local maxima where the selection can go wrong: rows around the 64-column and
16-row tiles, values that share their leading bits, more equal values than a
workgroup sorts, non-finite values, more grids than one launch takes; against
the oracle's scan (ties by scan order) or, for NaN, the definition itself."""
import numpy as np
import pytest

import oracle
from partapp_amd.api import find_local_max

pytestmark = pytest.mark.gpu


def got_tuples(a):
    return [(int(r["d"]), int(r["x"]), int(r["y"]), float(r["score"])) for r in a]


def ref_tuples(g, max_n):
    return [(int(d), int(x), int(y), float(np.float32(v))) for d, x, y, v in oracle.find_local_max(g, max_n)]


def check(g, max_n, gpu):
    import torch
    assert got_tuples(find_local_max(torch.from_numpy(g).to(gpu), max_n)) == ref_tuples(g, max_n)


@pytest.mark.parametrize("shape", [(1, 1, 1), (2, 1, 70), (2, 70, 1), (3, 15, 63), (3, 16, 64), (3, 17, 65), (2, 33, 129)])
@pytest.mark.parametrize("max_n", [20, 4096])
def test_tile_edges(gpu, shape, max_n):
    check(np.random.default_rng(sum(shape)).normal(0, 1, shape).astype(np.float32), max_n, gpu)


@pytest.mark.parametrize("kind", ["one_bin", "two_ulps", "negative", "mixed_sign"])
def test_shared_leading_bits(gpu, kind):
    rng = np.random.default_rng(sum(map(ord, kind)))
    shape = (4, 130, 200)  # some 9000 maxima
    if kind == "one_bin":
        g = 16.0 + 0.5 * rng.random(shape)
    elif kind == "two_ulps":  # 1024 values: hundreds of ties at the threshold
        g = np.float32(1.0) + rng.integers(0, 1024, shape) * np.float32(2.0 ** -23)
    elif kind == "negative":
        g = -100.0 + 5.0 * rng.random(shape)
    else:
        g = rng.normal(0, 1e-20, shape)
    for max_n in (1, 1000, 4096):
        check(g.astype(np.float32), max_n, gpu)


def test_more_ties_than_a_workgroup_sorts(gpu):
    g = np.full((1, 100, 131), -1e6, dtype=np.float32)  # 13100 equal maxima
    check(g, 100, gpu)
    g[0, 50, 60] = 3.0
    check(g, 100, gpu)


def test_infinities(gpu):
    rng = np.random.default_rng(3)
    g = rng.normal(0, 1, (3, 40, 80)).astype(np.float32)
    g.flat[::97] = np.inf
    g.flat[5::89] = -np.inf
    check(g, 30, gpu)
    check(g, 4000, gpu)


def test_nan_points(gpu):
    # a NaN is greater than nothing and nothing is greater than it: in one slice it is kept
    # and its neighbours are judged without it
    import torch
    g = np.arange(20 * 70, dtype=np.float32).reshape(1, 20, 70)
    g[0, 7, 31] = np.nan
    r = find_local_max(torch.from_numpy(g).to(gpu), 100)
    assert [(int(a["d"]), int(a["x"]), int(a["y"])) for a in r] == [(0, 31, 7), (0, 69, 19)]


def test_more_grids_than_a_launch(gpu):
    import torch
    rng = np.random.default_rng(9)
    gs = [rng.normal(0, 1, (2, 5 + i % 7, 9 + i % 60)).astype(np.float32) for i in range(97)]
    res = find_local_max([torch.from_numpy(g).to(gpu) for g in gs], 25)
    for g, r in zip(gs, res):
        assert got_tuples(r) == ref_tuples(g, 25)
