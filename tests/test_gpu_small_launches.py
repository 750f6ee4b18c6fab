"""A launch of few blocks cuts the column passes' strips into parts and takes
fewer rows per block of the BF16 row pass; neither changes a value: one image
alone has the outputs, bit for bit, that it has among twelve, whose launches
are cut otherwise."""
import numpy as np
import pytest

from partapp_amd.api import ExpParam, Plan, decode_maps, person_model, synth_joints

pytestmark = pytest.mark.gpu


def sweep(gpu, model, images, method):
    import torch
    n, hw = len(images), images[0].shape[3:]
    plan = Plan(model, [hw] * n)
    plan.set_method(method)
    un = torch.from_numpy(np.concatenate([u.ravel() for u in images])).to(gpu)
    marg = torch.full_like(un, float("nan"))
    root = torch.full((plan.root_numel,), float("nan"), device=gpu)
    maps = torch.zeros((plan.map_numel * 4,), dtype=torch.int32, device=gpu)
    plan.execute(un, marg, root, maps)
    torch.cuda.synchronize()
    m = decode_maps(maps, plan.n_instances, plan.S, plan.P)
    out = [(plan.instance_view(marg, i).cpu().numpy(), plan.instance_view(root, i, "root").cpu().numpy(), m[i])
           for i in range(n)]
    plan.close()
    return out


# heights at the ends of 32- and 64-row tiles; strips of one and of two 64-column tiles
@pytest.mark.parametrize("hw", [(31, 40), (64, 70), (65, 64), (96, 33), (128, 65), (129, 50), (200, 90)])
@pytest.mark.parametrize("method", ["fp32", "bf16", "bf16mix"])
@pytest.mark.parametrize("R", [24, 48])
def test_alone_as_among_many(gpu, R, method, hw):
    model = person_model(ExpParam(-180.0, 180.0, R, 1.0, 1.0, 1, 0.0), synth_joints(3))
    rng = np.random.default_rng(hw[0] + R)
    images = [rng.normal(-3.0, 0.5, (10, 1, R, *hw)).astype(np.float32) for _ in range(12)]
    many = sweep(gpu, model, images, method)
    for i in (0, 11):
        alone = sweep(gpu, model, [images[i]], method)[0]
        for a, b in zip(alone[:2], many[i][:2]):
            np.testing.assert_array_equal(a.view(np.uint32), b.view(np.uint32))
        assert alone[2].tobytes() == many[i][2].tobytes()
