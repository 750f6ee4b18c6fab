"""DPM scores that are slices of the part they are added to: the slices follow
one another, a slice already added to being read as it then is."""
import numpy as np
import pytest

from partapp_amd.api import DPM_LOG, add_dpm_score

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("first,n_dpm", [(0, 1), (7, 1), (13, 1), (0, 7), (3, 7), (7, 7)])
def test_slices_of_the_part(gpu, first, n_dpm):
    import torch
    S, R, H, W, w = 2, 7, 33, 45, np.float32(0.7)
    g = np.random.default_rng(first).normal(-3, 1, (S * R, H, W)).astype(np.float32)
    part = torch.from_numpy(g.copy()).to(gpu)
    add_dpm_score(part.view(S, R, H, W), part[first:first + n_dpm], float(w), DPM_LOG)
    for k in range(S * R):
        g[k] = g[k] + w * g[first + (k % R if n_dpm > 1 else 0)]  # one product, one sum in float32: exact
    np.testing.assert_array_equal(part.cpu().numpy(), g)
