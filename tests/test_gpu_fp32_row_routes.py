"""The routes of the FP32 row and column pass around the rules that choose
between them (blocks per CU, columns per thread, narrow and short grids) and
where waves lie past the row: single messages against the float32 oracle, at its
bar for messages."""
import numpy as np
import pytest

import oracle
from partapp_amd.api import ExpParam, Joint, PartModel, compute_rot_joint_marginal

pytestmark = pytest.mark.gpu


# (rotations, H, W, route): a CU takes two blocks of 24 slices and 720 columns on the vector unit, one on the matrix
# cores (half width 36), if the launch has more blocks than CUs
@pytest.mark.parametrize("R,H,W", [
    (24, 5, 512), (24, 5, 513), (24, 5, 577), (24, 5, 1025),      # matrix cores, one column a thread and more
    (24, 260, 690), (24, 260, 730), (24, 250, 730), (24, 260, 810),  # matrix cores, vector, too few blocks, matrix cores
    (48, 5, 512), (48, 5, 513), (48, 5, 640), (48, 5, 1025),      # matrix cores, vector
    (48, 260, 810), (48, 260, 1024), (48, 260, 1030),             # matrix cores, matrix cores, vector
    (24, 40, 16), (24, 40, 17), (24, 12, 100), (24, 13, 100),     # narrow rows, and a column pass of few rows, vector
])
def test_routes(gpu, R, H, W):
    import torch
    child = np.random.default_rng(H * 10000 + W).normal(-3, 1, (R, H, W)).astype(np.float32)
    ep = ExpParam(-180.0, 180.0, R, 1.0, 1.0, 1, 0.0)
    model = PartModel([1, 1], [0, 0], [1, 0], [Joint(1, 0, (0, 0), (0, 0), (4, 0, 0, 4), 0.0, 0.2)], ep)
    args = dict(offset_c=(3.3, -2.7), offset_p=(-1.4, 4.9), C=(144.0, 0, 0, 4.0), rot_mean=0.2, rot_sigma=0.3, scale=1.0)
    ref = oracle.rot_joint_marginal(oracle.exp_param_from(ep), child, **args)
    out = compute_rot_joint_marginal(model, torch.from_numpy(child).to(gpu), args["offset_c"], args["offset_p"], args["C"],
                                     args["rot_mean"], args["rot_sigma"], args["scale"]).cpu().numpy()
    np.testing.assert_array_equal(out <= -9e5, ref <= -9e5)
    live = ref > -9e5
    np.testing.assert_allclose(out[live], ref[live], rtol=1e-5, atol=5e-5)
