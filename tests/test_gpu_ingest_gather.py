"""Score ingestion's gather (each pixel looks for the cell that the reference's
scatter leaves on it) and the scatter it gives way to, against the oracle: the
same LOG_ZERO cells, the same cell behind every other pixel.  The warps sit
where the gather could miss one: half-pixel ties, rotations, shears, boxes on
both sides of its limit, warps without an inverse."""
import math

import numpy as np
import pytest

import oracle
from partapp_amd.api import ingest_scores

pytestmark = pytest.mark.gpu


def rot(a, s, dx, dy):
    c, d = s * math.cos(a), s * math.sin(a)
    return [[c, -d, dx], [d, c, dy], [0, 0, 1]]


WARPS = {
    "identity": [[1, 0, 0], [0, 1, 0], [0, 0, 1]],
    "half_pixel": [[1, 0, 0.5], [0, 1, -0.5], [0, 0, 1]],
    "half_steps": [[0.5, 0, 0.25], [0, 0.5, 0.75], [0, 0, 1]],
    "quarter_turn": [[0, -1, 40], [1, 0, 0], [0, 0, 1]],
    "mirror": [[-1, 0, 50.5], [0, 1, 0], [0, 0, 1]],
    "rot45": rot(math.pi / 4, 1.0, 30.0, -10.0),
    "rot45_two": rot(math.pi / 4, 0.7081, 30.0, -10.0),    # boxes just below and above 2 x 2 cells
    "rot45_three": rot(math.pi / 4, 0.7063, 30.0, -10.0),
    "rot_small": rot(0.13, 1.0, -3.0, 2.5),
    "enlarge": rot(1.1, 3.7, 60.0, -5.0),
    "shrink6": rot(0.4, 1 / 6, 5.0, 3.0),       # boxes of some 100 cells: gather
    "shrink60": rot(0.8, 1 / 60, 20.0, 10.0),   # boxes beyond the limit: scatter
    "shear6": [[1.0, 6.0, -30.0], [0.0, 1.0, 0.0], [0, 0, 1]],
    "shear90": [[1.0, 90.0, -300.0], [0.0, 1.0, 0.0], [0, 0, 1]],  # many cells to test for one that lands: scatter
    "thin": [[1.0, 1.0, 0.0], [1.0, 1.0 + 1e-9, 0.0], [0, 0, 1]],  # inverse entries of 1e9: scatter
    "singular": [[1.0, 2.0, 0.0], [2.0, 4.0, 0.0], [0, 0, 1]],
    "far": [[1.0, 0.0, 1e7], [0.0, 1.0, 0.0], [0, 0, 1]],          # nothing lands on the image
}


def check(sg, T, H, W, gpu):
    import torch
    got = ingest_scores(torch.from_numpy(sg).to(gpu), T, False, H, W).cpu().numpy()
    ref = oracle.ingest_scores(sg, T, False, H, W)
    np.testing.assert_array_equal(got == -1e6, ref == -1e6)
    live = ref != -1e6
    # the same cell: its log to the float log's last bits (two neighbouring cells differ by far more)
    np.testing.assert_allclose(got[live], ref[live], rtol=2e-7, atol=2e-7)


def scores(seed, n, gh, gw):
    rng = np.random.default_rng(seed)
    sg = rng.normal(0.3, 1.0, (n, gh, gw)).astype(np.float32)
    sg[rng.random(sg.shape) < 0.2] = 0.0
    return sg


@pytest.mark.parametrize("dims", [(37, 45, 65, 97), (64, 64, 32, 32), (1, 50, 33, 31), (51, 1, 7, 64)])
@pytest.mark.parametrize("warp", sorted(WARPS))
def test_direct_warps(gpu, warp, dims):
    gh, gw, H, W = dims
    sg = scores(sum(map(ord, warp)) + gh, 2, gh, gw)
    check(sg, np.array([WARPS[warp]] * 2, dtype=np.float64), H, W, gpu)


@pytest.mark.parametrize("n", [80, 81, 1500])
def test_direct_slice_counts(gpu, n):
    # one launch, two, and the table of very many slices; each slice has its own warp
    T = np.array([rot(0.37 * s, 1.0, 8.0 + 0.01 * s, 4.0) for s in range(n)], dtype=np.float64)
    check(scores(n, n, 19, 23), T, 21, 34, gpu)


def test_one_slice_that_needs_the_scatter(gpu):
    T = np.array([WARPS["rot45"], WARPS["singular"], WARPS["identity"]], dtype=np.float64)
    check(scores(5, 3, 37, 45), T, 65, 97, gpu)


def test_scores_of_every_kind(gpu):
    # negative zero and zero are not written, infinities and subnormals are
    sg = scores(6, 1, 40, 40)
    sg.flat[::7] = -0.0
    sg.flat[3::31] = np.inf
    sg.flat[5::37] = -np.inf
    sg.flat[11::41] = 1e-42
    check(sg, np.array([WARPS["rot_small"]], dtype=np.float64), 40, 40, gpu)
