"""Nearest ingestion onto buffers that overlap its input (the same buffer, one
reaching into it from either side) equals the one into a buffer of its own."""
import ctypes
import math

import numpy as np
import pytest

from partapp_amd._lib import check, lib
from partapp_amd.api import ingest_scores

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shift", [0, 1, -1, 2000, -2000])
@pytest.mark.parametrize("angle", [0.0, 0.7])
def test_overlap(gpu, shift, angle):
    import torch
    n, gh, gw, H, W = 5, 70, 90, 90, 70
    c, s = math.cos(angle), math.sin(angle)
    T = np.tile(np.array([[c, -s, 21.0], [s, c, -13.0], [0, 0, 1]]), (n, 1, 1))
    buf = torch.zeros(n * gh * gw + 4000, device=gpu)
    grid = buf[2000:2000 + n * gh * gw]
    grid.copy_(torch.rand(n * gh * gw, device=gpu, generator=torch.Generator("cuda").manual_seed(1)) - 0.1)
    want = ingest_scores(grid.view(n, gh, gw).clone(), T, False, H, W)
    out = buf[2000 + shift:2000 + shift + n * H * W]
    t = np.ascontiguousarray(T.reshape(n, 9))
    check(lib().ps_ingest_scores(grid.data_ptr(), n, gh, gw, t.ctypes.data_as(ctypes.POINTER(ctypes.c_double)), 0, H, W,
                                 out.data_ptr(), None), "ps_ingest_scores")
    assert torch.equal(out.view(n, H, W), want)
