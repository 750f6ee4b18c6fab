"""Leaf maxima of masked grids of few columns, several rows a wave: widths
around the powers of two up to 64 and beyond, masked strips and rotations, more
rows than a block takes; whole sweeps against the oracle at the FP32 path's bar
(marginals 1e-5, MAP identical)."""
import pytest

from partapp_amd.api import ExpParam
from test_gpu_block_keys import star, sweep
from test_gpu_parity import check_parity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W", [1, 2, 3, 4, 5, 8, 9, 16, 17, 31, 32, 33, 63, 64, 65])
@pytest.mark.parametrize("strip,H", [(0.0, 150), (0.2, 37)])
def test_narrow(gpu, W, strip, H):
    model, joints = star(2, ExpParam(-180.0, 180.0, 25, 1.0, 1.0, 1, strip), upright=True)
    u, out = sweep("narrow", model, joints, H, W, seed=W)
    check_parity("%dx%d, strip %g" % (H, W, strip), model, u, joints, out, check_f64=False)
