"""The first choice of a BF16 method and the first MAP guard of a plan while a
stream is being captured (on its thread, and on another; a stream that waits for
the default one, and one that does not): both make tables,
none of which belongs in the graph, and the graph's replays equal the eager
sweep."""
import ctypes
import threading

import pytest

from partapp_amd.api import ExpParam, Plan, person_model, synth_joints

pytestmark = pytest.mark.gpu


def setup(gpu):
    import torch
    model = person_model(ExpParam(-180.0, 180.0, 24, 1.0, 1.0, 1, 0.0), synth_joints(3))
    plan = Plan(model, [(60, 70)])
    un = torch.empty(plan.unary_numel, device=gpu).normal_(-3, 0.5, generator=torch.Generator("cuda").manual_seed(1))
    return plan, (un, torch.zeros_like(un), torch.zeros(plan.root_numel, device=gpu),
                  torch.zeros(plan.map_numel * 4, dtype=torch.int32, device=gpu))


def outputs(bufs):
    return [b.clone() for b in bufs[1:]]


@pytest.mark.parametrize("blocking", [False, True])
@pytest.mark.parametrize("what", ["method", "guard", "method in another thread"])
def test_first_use(gpu, what, blocking):
    import torch
    stream = None
    if blocking:  # torch's own streams do not wait for the default one
        made = ctypes.c_void_p()
        assert ctypes.CDLL("libamdhip64.so").hipStreamCreate(ctypes.byref(made)) == 0
        stream = torch.cuda.ExternalStream(made.value)
    ref_plan, ref = setup(gpu)
    ref_plan.set_method("fp32" if what == "guard" else "bf16mix")
    ref_plan.execute(*ref)
    torch.cuda.synchronize()
    plan, bufs = setup(gpu)
    if what == "guard":  # loads the kernels, which is not what this is about
        plan.execute(*bufs)
    torch.cuda.synchronize()

    def first_use():
        if what == "guard":
            plan.set_map_guard(1e-3)
        else:
            plan.set_method("bf16mix")

    x = torch.zeros(8, device=gpu)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=stream):
        x.add_(1)
        if what.endswith("thread"):
            raised = []

            def run():
                try:
                    first_use()
                except Exception as e:
                    raised.append(e)

            t = threading.Thread(target=run)
            t.start()
            t.join()
            assert not raised, raised
        else:
            first_use()
        plan.execute(*bufs)
    for replay in range(3):
        for b in bufs[1:]:
            b.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert x[0].item() == replay + 1
        for a, b in zip(outputs(bufs), ref[1:]):
            assert torch.equal(a, b)
        ref_plan.execute(*ref)  # eager work between the replays
        torch.cuda.synchronize()
    del g
    plan.close()
    ref_plan.close()
