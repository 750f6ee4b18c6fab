"""The maxima and argmaxima that blocks merge before raising them, and the
root kernel's split over rotations, where they can go wrong: grids around its
tiles of 64 and blocks of 128 pixels, rotation counts that four waves share
unevenly (fewer than four among them), one root child and more than eight,
sources at every alignment, masked strips and rotations; whole sweeps against
the oracle at the FP32 path's bar (marginals 1e-5, MAP identical)."""
import numpy as np
import pytest

from partapp_amd.api import ExpParam, Joint, PartModel
from test_gpu_parity import check_parity, run_plan

pytestmark = pytest.mark.gpu


def star(K, ep, upright=False):
    joints = [Joint(k, 0, (0.5 * k, -1.0), (1.0, 0.3 * k), (3.0 + k, 0, 0, 2.0), 0.1 * k, 0.3) for k in range(1, K + 1)]
    return PartModel([1] * (K + 1), [int(upright)] * (K + 1), [1] + [0] * K, joints, ep), joints


def sweep(name, model, joints, H, W, seed):
    S, R = model.exp_param.num_scale_steps, model.exp_param.num_rotation_steps
    u = np.random.default_rng(seed).normal(-3.0, 1.0, (len(model.is_detect), S, R, H, W)).astype(np.float32)
    return u, run_plan(model, [u], [joints])[0]


@pytest.mark.parametrize("hw", [(1, 1), (1, 63), (4, 16), (5, 13), (7, 18), (8, 16), (3, 43), (11, 23), (13, 21)])
@pytest.mark.parametrize("R", [2, 3, 24, 48, 63, 64])
def test_pixel_and_rotation_tiles(gpu, R, hw):
    model, joints = star(2, ExpParam(-180.0, 180.0, R, 1.0, 1.0, 1, 0.0))
    u, out = sweep("tiles", model, joints, *hw, seed=R * 100 + hw[1])
    check_parity("R %d, %dx%d" % (R, *hw), model, u, joints, out, check_f64=False)


@pytest.mark.parametrize("K", [1, 8, 9, 16])
def test_root_children(gpu, K):
    model, joints = star(K, ExpParam(-180.0, 180.0, 24, 1.0, 1.0, 1, 0.0))
    u, out = sweep("star", model, joints, 9, 29, seed=K)
    check_parity("K %d" % K, model, u, joints, out, check_f64=False)


@pytest.mark.parametrize("strip", [0.0, 0.1, 0.45])
@pytest.mark.parametrize("hw", [(17, 31), (33, 30), (40, 129)])
def test_masks_and_alignment(gpu, strip, hw):
    # scales and parts of an odd number of elements put the sources at every alignment
    ep = ExpParam(-180.0, 180.0, 25, 0.9, 1.1, 2, strip)
    model, joints = star(3, ep, upright=True)
    u, out = sweep("masks", model, joints, *hw, seed=hw[1])
    check_parity("strip %g, %dx%d" % (strip, *hw), model, u, joints, out, check_f64=False)
