"""Memory that outlives a call or a plan: results do not depend on what held
the block before, on a plan destroyed while it runs, or on threads and streams
calling at once; the library gives the memory back when asked."""
import threading

import numpy as np
import pytest

from partapp_amd._lib import lib
from partapp_amd.api import (ExpParam, Plan, compute_rot_joint_marginal, find_local_max, person_model, synth_joints)

pytestmark = pytest.mark.gpu

EP = ExpParam(-180.0, 180.0, 24, 1.0, 1.0, 1, 0.0)


def unary(seed, n, gpu):
    import torch
    return torch.empty(n, device=gpu).normal_(-3.0, 0.5, generator=torch.Generator("cuda").manual_seed(seed))


def sweep(size, seed, gpu, method="fp32", keep=None):
    import torch
    plan = Plan(person_model(EP, synth_joints(seed)), [size])
    plan.set_method(method)
    un = unary(seed, plan.unary_numel, gpu)
    marg = torch.full_like(un, float("nan"))
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    plan.execute(un, marg, None, None, stream=s)
    if keep is not None:
        keep.append((un, s))  # the caller's buffers outlive the plan, the plan does not wait
    else:
        s.synchronize()
    plan.close()
    return marg


def test_plan_destroyed_while_it_runs(gpu):
    import torch
    want = sweep((96, 120), 1, gpu)
    keep = []
    got = [sweep((96, 120), 1, gpu, keep=keep) for _ in range(4)]
    sweep((90, 110), 2, gpu, method="bf16mix", keep=keep)  # would reuse the first plan's blocks
    torch.cuda.synchronize()
    assert all(torch.equal(g, want) for g in got)


def test_threads_and_streams(gpu):
    import torch
    model = person_model(EP)
    args = ((7.3, -11.2), (-3.9, 8.8), (30.0, 12.0, 12.0, 50.0), 0.3, 0.25, 1.0)
    sizes = [(41, 57), (64, 40), (33, 90), (50, 50)]
    child = [unary(10 + i, 24 * h * w, gpu).view(24, h, w) for i, (h, w) in enumerate(sizes)]
    want = [compute_rot_joint_marginal(model, c, *args) for c in child]
    peaks = [find_local_max(c, 200) for c in child]
    torch.cuda.synchronize()
    bad = []

    def work(i):
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            for _ in range(20):
                got = compute_rot_joint_marginal(model, child[i], *args, stream=s)
                found = find_local_max(child[i], 200, stream=s)
                if not torch.equal(got, want[i]) or not np.array_equal(found, peaks[i]):
                    bad.append(i)

    t = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    [x.start() for x in t]
    [x.join() for x in t]
    assert not bad


def test_memory_given_back(gpu):
    import torch
    torch.cuda.empty_cache()  # torch keeps memory of its own
    assert lib().ps_release_memory() == 0
    free0 = torch.cuda.mem_get_info()[0]
    sweep((300, 300), 3, gpu)  # 130 MB of scratch
    torch.cuda.empty_cache()
    assert torch.cuda.mem_get_info()[0] <= free0 - (100 << 20)
    assert lib().ps_release_memory() == 0
    assert torch.cuda.mem_get_info()[0] >= free0 - (8 << 20)
