"""The FP32 filters on the matrix cores where they can go wrong: widths around
the 64-column tiles, heights around the 32-row tiles, every remainder of the
taps by 4, rows and filters too large for their operands in LDS (vector unit),
the fill value overflowing; single messages against the float32 oracle.  The
sums are the sequential dot products, so the bar is that of the messages
elsewhere: exp's and log's last bits."""
import numpy as np
import pytest

import oracle
from partapp_amd.api import ExpParam, Joint, PartModel, compute_rot_joint_marginal

pytestmark = pytest.mark.gpu


def run(gpu, R, H, W, C, child, **kw):
    import torch
    ep = ExpParam(-180.0, 180.0, R, 1.0, 1.0, 1, 0.0)
    model = PartModel([1, 1], [0, 0], [1, 0], [Joint(1, 0, (0, 0), (0, 0), (4, 0, 0, 4), 0.0, 0.2)], ep)
    args = dict(offset_c=(3.3, -2.7), offset_p=(-1.4, 4.9), C=C, rot_mean=0.2, rot_sigma=0.3, scale=1.0)
    args.update(kw)
    out = compute_rot_joint_marginal(model, torch.from_numpy(child).to(gpu), args["offset_c"], args["offset_p"], C,
                                     args["rot_mean"], args["rot_sigma"], args["scale"]).cpu().numpy()
    return out, oracle.rot_joint_marginal(oracle.exp_param_from(ep), child, **args)


def check(out, ref):
    np.testing.assert_array_equal(out <= -9e5, ref <= -9e5)
    live = ref > -9e5
    np.testing.assert_allclose(out[live], ref[live], rtol=1e-5, atol=5e-5)


@pytest.mark.parametrize("R", [24, 48])
@pytest.mark.parametrize("hw", [(1, 1), (5, 63), (31, 64), (32, 65), (33, 128), (64, 129), (65, 40), (97, 193)])
def test_tile_edges(gpu, R, hw):
    child = np.random.default_rng(hw[0] * 1000 + hw[1]).normal(-3, 1, (R, *hw)).astype(np.float32)
    check(*run(gpu, R, hw[0], hw[1], (25.0, 0, 0, 36.0), child))


@pytest.mark.parametrize("k", [1, 2, 3, 4, 5, 12, 13, 14, 15, 35, 43, 60])
def test_filter_lengths(gpu, k):
    # half widths k and k + 1: 2 k + 1 leaves every remainder by 4
    child = np.random.default_rng(k).normal(-3, 1, (24, 70, 90)).astype(np.float32)
    check(*run(gpu, 24, 70, 90, ((k / 3.0) ** 2, 0, 0, ((k + 1) / 3.0) ** 2), child))


@pytest.mark.parametrize("rot_sigma", [0.0, -1.0, 2.0])
def test_rotation_modes(gpu, rot_sigma):
    child = np.random.default_rng(7).normal(-3, 1, (24, 40, 70)).astype(np.float32)
    out, ref = run(gpu, 24, 40, 70, (16.0, 0, 0, 9.0), child, rot_sigma=rot_sigma)
    check(out, ref)


@pytest.mark.parametrize("W", [520, 1500, 1600])
def test_wide_rows(gpu, W):
    # more columns than threads; rows whose padding does not fit LDS beside 24 slices (vector unit)
    child = np.random.default_rng(W).normal(-3, 1, (24, 6, W)).astype(np.float32)
    check(*run(gpu, 24, 6, W, (64.0, 0, 0, 4.0), child))


def test_long_y_filter(gpu):
    # half width 286: its rows fit LDS only without the tap operand (vector unit)
    child = np.random.default_rng(286).normal(-3, 1, (24, 300, 20)).astype(np.float32)
    check(*run(gpu, 24, 300, 20, (4.0, 0, 0, (286 / 3.0) ** 2), child))


@pytest.mark.parametrize("R", [24, 48])
def test_fill_value_overflows(gpu, R):
    # a grid far below LOG_ZERO: exp(LOG_ZERO - M) is infinite at every pixel the warp leaves empty,
    # whose zero taps must not turn the pixels beyond the filter's reach into NaN
    H, W = 120, 160
    child = (np.random.default_rng(R).normal(0, 1, (R, H, W)) - 1.001e6).astype(np.float32)
    out, ref = run(gpu, R, H, W, (4.0, 0, 0, 9.0), child, offset_c=(0.0, 0.0), offset_p=(0.0, 0.0), rot_mean=0.0)
    np.testing.assert_allclose(out, ref, rtol=1e-5)
    out, ref = run(gpu, R, H, W, (4.0, 0, 0, 9.0), child, offset_c=(20.0, 0.0), offset_p=(0.0, 0.0), rot_mean=0.0)
    k = 12  # further than both filters reach, padding included
    far = np.zeros((R, H, W), bool)
    inf = ~np.isfinite(ref)
    assert inf.any() and not inf.all()
    for r, y, x in zip(*np.nonzero(inf)):
        far[:, max(0, y - k):y + k, max(0, x - k):x + k] = True
    far = ~far
    assert far.any()
    np.testing.assert_allclose(out[far], ref[far], rtol=1e-5)


def test_nan_stays_local(gpu):
    # a NaN that does not become the grid's maximum (sign bit set) reaches the outputs of its filters, no others
    R, H, W = 24, 80, 150
    child = np.random.default_rng(3).normal(-3, 1, (R, H, W)).astype(np.float32)
    kw = dict(offset_c=(0.0, 0.0), offset_p=(0.0, 0.0), rot_mean=0.0, rot_sigma=0.0)
    clean, ref = run(gpu, R, H, W, (16.0, 0, 0, 25.0), child, **kw)
    check(clean, ref)
    bad = child.copy()
    bad.view(np.uint32)[5, 40, 75] = 0xFFC00000
    out, _ = run(gpu, R, H, W, (16.0, 0, 0, 25.0), bad, **kw)
    kx, ky, pad = 12, 15, 3
    near = np.zeros((R, H, W), bool)
    near[5, 40 - ky - pad:40 + ky + pad + 1, 75 - kx - pad:75 + kx + pad + 1] = True
    np.testing.assert_array_equal(out[~near], clean[~near])
    assert (out[5, 40 - ky:40 + ky + 1, 75 - kx:75 + kx + 1] < -9e5).all()
