"""Ingestion of many and of small slices: warps in a launch's arguments and in
a table, pixels in square tiles and in rows, for nearest warps that enlarge and
shrink and for bilinear ones; against the oracle, and slice by slice against
calls of one slice."""
import math

import numpy as np
import pytest

import oracle
from partapp_amd.api import ingest_scores

pytestmark = pytest.mark.gpu


def warps(n, s):
    return np.array([[[s * math.cos(0.37 * i), -s * math.sin(0.37 * i), 9.0 + 0.01 * i],
                      [s * math.sin(0.37 * i), s * math.cos(0.37 * i), 5.0], [0, 0, 1]] for i in range(n)])


# tiles of 32 x 32 against rows of 1024: 1 / 1, 2 / 1, 4 / 2, 4 / 4, 4 / 3, 33 / 2, 33 / 33 and 6 / 4 of them
@pytest.mark.parametrize("hw", [(20, 30), (33, 31), (40, 40), (64, 64), (45, 64), (1, 1050), (1050, 32), (50, 70)])
@pytest.mark.parametrize("n", [2, 81])
@pytest.mark.parametrize("scale,interpolate", [(1.0, False), (1 / 6, False), (1.0, True)])
def test_slices(gpu, hw, n, scale, interpolate):
    import torch
    H, W = hw
    rng = np.random.default_rng(H * 1000 + W + n)
    sg = rng.normal(0.3, 1.0, (n, 37, 29)).astype(np.float32)
    sg[rng.random(sg.shape) < 0.2] = 0.0
    T = warps(n, scale)
    got = ingest_scores(torch.from_numpy(sg).to(gpu), T, interpolate, H, W).cpu().numpy()
    ref = oracle.ingest_scores(sg, T, interpolate, H, W)
    np.testing.assert_array_equal(got == -1e6, ref == -1e6)
    live = ref != -1e6
    # one cell or the same four products: its log to the float log's last bits
    np.testing.assert_allclose(got[live], ref[live], rtol=2e-7, atol=2e-7)
    one = ingest_scores(torch.from_numpy(sg[n - 1:]).to(gpu), T[n - 1:], interpolate, H, W).cpu().numpy()
    np.testing.assert_array_equal(got[n - 1], one[0])
