"""Local maxima of grids whose values share more leading bits than the first
threshold looks at: values near LOG_ZERO, few distinct values, plateaus, in
grids of any sign, and more grids than one set of launches takes; against the
oracle's scan (ties by scan order)."""
import numpy as np
import pytest

import oracle
from partapp_amd.api import find_local_max

pytestmark = pytest.mark.gpu


def got(g, max_n, gpu):
    import torch
    r = find_local_max(torch.from_numpy(g).to(gpu), max_n)
    return [(int(a["d"]), int(a["x"]), int(a["y"]), float(a["score"])) for a in r]


def ref(g, max_n):
    return [(int(d), int(x), int(y), float(np.float32(v))) for d, x, y, v in oracle.find_local_max(g, max_n)]


def grid(kind):
    rng = np.random.default_rng(sum(map(ord, kind)))
    shape = (4, 250, 300)  # some 25000 maxima of noise
    if kind == "near_log_zero":    # spacing 1/16: all in one 22-bit bin, tens to a value
        return rng.normal(-1e6, 4, shape)
    if kind == "some_live":        # a few hundred above, the rest as before
        g = rng.normal(-1e6, 4, shape)
        g[1, ::16, ::20] = rng.normal(-3, 1, g[1, ::16, ::20].shape)
        return g
    if kind == "six_values":       # thousands to a value
        return -1e6 + rng.integers(0, 6, shape)
    if kind == "two_planes":       # a plateau in every other slice, none of whose neighbours reach it
        g = np.zeros(shape)
        g[::2] = 1.0
        g[0, 100:110, 50:60] = rng.random((10, 10)) + 1.0
        return g
    if kind == "negative_plane":
        g = np.full((1,) + shape[1:], -2.5)
        g[0, 7, 5:300:7] = -2.25
        return g
    g = np.full((1,) + shape[1:], np.inf)  # infinite_plane
    return g


@pytest.mark.parametrize("kind", ["near_log_zero", "some_live", "six_values", "two_planes", "negative_plane",
                                  "infinite_plane"])
@pytest.mark.parametrize("max_n", [1, 30, 1000, 4096])
def test_shared_bits(gpu, kind, max_n):
    g = grid(kind).astype(np.float32)
    assert got(g, max_n, gpu) == ref(g, max_n)


@pytest.mark.parametrize("n", [96, 97, 1025])
def test_many_grids(gpu, n):
    import torch
    rng = np.random.default_rng(n)
    gs = [rng.normal(0, 1, (1 + i % 3, 3 + i % 7, 5 + i % 80)).astype(np.float32) for i in range(n)]
    gs[n - 1] = np.full((1, 100, 100), 2.0, np.float32)
    res = find_local_max([torch.from_numpy(g).to(gpu) for g in gs], 12)
    for g, r in zip(gs, res):
        assert [(int(a["d"]), int(a["x"]), int(a["y"]), float(a["score"])) for a in r] == ref(g, 12)


# 8192 points at most: one workgroup a grid; one more, or one such grid among them: the general kernels
@pytest.mark.parametrize("shapes", [[(2, 64, 64)], [(1, 8192, 1), (8192, 1, 1), (1, 1, 8192)], [(3, 2731, 1)],
                                    [(2, 64, 64), (1, 1, 1), (1, 90, 92)], [(24, 18, 18), (5, 3, 40)]])
@pytest.mark.parametrize("kind", ["noise", "few_values", "equal", "nan"])
@pytest.mark.parametrize("max_n", [1, 25, 4096])
def test_small_grids(gpu, shapes, kind, max_n):
    import torch
    rng = np.random.default_rng(len(shapes) * 10 + max_n)
    gs = [rng.normal(0, 1, s).astype(np.float32) for s in shapes]
    if kind == "few_values":
        gs = [np.round(g) for g in gs]
    elif kind == "equal":
        gs = [np.full_like(g, -1e6) for g in gs]
    elif kind == "nan":  # (one slice: a NaN's place among neighbours in other slices is the comparison's)
        for g in gs:
            g[0].flat[::13] = np.nan
    res = find_local_max([torch.from_numpy(g).to(gpu) for g in gs], max_n)
    for g, r in zip(gs, res):
        if kind == "nan":
            p = np.pad(g, ((1, 1), (1, 1), (1, 1)), constant_values=np.nan)
            n = [p[1, 1 + dy:1 + dy + g.shape[1], 1 + dx:1 + dx + g.shape[2]] for dy in (-1, 0, 1) for dx in (-1, 0, 1)
                 if dy or dx] if g.shape[0] == 1 else None
            if n is None:
                continue
            keep = ~np.any([m > g[0] for m in n], axis=0)
            assert len(r) == min(max_n, int(keep.sum())) and all(keep[a["y"], a["x"]] for a in r)
        else:
            assert [(int(a["d"]), int(a["x"]), int(a["y"]), float(a["score"])) for a in r] == ref(g, max_n)
