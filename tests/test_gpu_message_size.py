"""Messages of very large grids: 2^31 states and more where the kernels index
in 64 bits (any rotation count but 24 and 48, full covariance), refused where
they do not; grids of more than 4 GB."""
import math

import numpy as np
import pytest

from partapp_amd._lib import PsError
from partapp_amd.api import ExpParam, Joint, PartModel, compute_rot_joint_marginal

pytestmark = pytest.mark.gpu


def model(R):
    ep = ExpParam(-180.0, 180.0, R, 1.0, 1.0, 1, 0.0)
    return PartModel([1, 1], [0, 0], [1, 0], [Joint(1, 0, (0, 0), (0, 0), (4, 0, 0, 4), 0.0, 0.2)], ep)


def test_more_than_2_31_states(gpu):
    # a constant grid but for its last state, the maximum: inside, a message is the constant plus the log of the taps' sum
    import torch
    R, H, W = 2, 131080, 8192
    assert R * H * W > 1 << 31
    if torch.cuda.mem_get_info()[0] < 80 << 30:
        pytest.skip("needs 80 GB of device memory")
    C = (4.0, 0.05, 0.05, 9.0)
    child = torch.full((R, H, W), -3.0, device=gpu)
    child[-1, -1, -1] = 1.0
    out = compute_rot_joint_marginal(model(R), child, (0.0, 0.0), (0.0, 0.0), C, 0.0, 0.0, 1.0)
    want = -3.0
    for s2 in np.linalg.eigvalsh(np.array(C).reshape(2, 2)):
        k = math.floor(3 * math.sqrt(s2) + 0.5)
        want += math.log(sum(math.exp(-i * i / (2 * s2)) for i in range(-k, k + 1)))
    for rows in (slice(40, 80), slice(H // 2, H // 2 + 40), slice(H - 80, H - 40)):
        got = out[:, rows, 40:-40]
        # float weights and sums of 13 x 19 taps, exp and log of the hardware (1 ulp each)
        assert (got - want).abs().max().item() < 1e-4
    del child, out
    torch.cuda.empty_cache()


def test_source_beyond_4_gb(gpu):
    # 24 rotations: the last rows of the last slice lie beyond the grid's first 4 GB; each output is the same sum as in
    # a grid of the last rows alone
    import torch
    R, H, W, tail = 24, 32000, 1400, 200
    assert 1 << 30 < R * H * W - 100 * W and R * H * W < 1 << 31
    if torch.cuda.mem_get_info()[0] < 30 << 30:
        pytest.skip("needs 30 GB of device memory")
    args = ((3.3, -2.7), (-1.4, 4.9), (4.0, 0.0, 0.0, 5.5), 0.2, 0.3, 1.0)
    child = torch.full((R, H, W), -3.0, device=gpu)
    child[:, -tail:] = torch.randn((R, tail, W), device=gpu, generator=torch.Generator("cuda").manual_seed(0)) - 3.0
    want = compute_rot_joint_marginal(model(R), child[:, -tail:].contiguous(), *args)
    out = compute_rot_joint_marginal(model(R), child, *args)
    assert torch.equal(out[:, -100:], want[:, -100:])
    del child, out
    torch.cuda.empty_cache()


@pytest.mark.parametrize("R,C", [(24, (4.0, 1.0, 1.0, 9.0)), (48, (4.0, 0.0, 0.0, 9.0)), (2, (4.0, 0.0, 0.0, 9.0))])
def test_refused(gpu, R, C):
    # (one address stands for the grids: the call is refused before it reads them)
    import torch
    import ctypes
    from partapp_amd._lib import check, lib
    m, t = model(R), torch.zeros(64, device=gpu)
    two, four = ctypes.c_double * 2, ctypes.c_double * 4
    H = (1 << 31) // (R * 256) + 1
    with pytest.raises(PsError) as e:
        check(lib().ps_message(m.handle, t.data_ptr(), t.data_ptr(), H, 256, two(0, 0), two(0, 0), four(*C), 0.0, 0.0, 1.0,
                               0, None), "ps_message")
    assert e.value.status == -5
