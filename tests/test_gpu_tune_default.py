"""Launch-shape knobs taken back to their defaults, and the autotuner's choice
among them: the outputs stay those of an untouched plan, and the default row
count of the BF16 x pass (by the launch's size) is a candidate."""
import pytest

from partapp_amd._lib import PsError
from partapp_amd.api import ExpParam, Plan, person_model, synth_joints

pytestmark = pytest.mark.gpu


def test_default_after_tuning(gpu):
    import torch
    model = person_model(ExpParam(-180.0, 180.0, 24, 1.0, 1.0, 1, 0.0), synth_joints(5))
    plan = Plan(model, [(90, 100), (60, 150)])
    un = torch.empty(plan.unary_numel, device=gpu).normal_(-3, 0.5, generator=torch.Generator("cuda").manual_seed(2))

    def sweep():
        bufs = (torch.full_like(un, float("nan")), torch.full((plan.root_numel,), float("nan"), device=gpu),
                torch.zeros(plan.map_numel * 4, dtype=torch.int32, device=gpu))
        plan.execute(un, *bufs)
        torch.cuda.synchronize()
        return bufs

    for method, knob, value in (("bf16mix", plan.TUNE_MFMA_ROWS, 16), ("fp32", plan.TUNE_FP32_ROW_THREADS, 64),
                                ("fp32", plan.TUNE_FP32_COL_ROWS, 16)):
        plan.set_method(method)
        want = sweep()
        for cls in (None, 0, len(plan.classes()) - 1):
            plan.tune(knob, value)
            plan.tune(knob, None, cls=cls)
            assert all(torch.equal(a, b) for a, b in zip(sweep(), want))
        plan.tune(knob, None)
    with pytest.raises(PsError):
        plan.tune(plan.TUNE_MFMA_ROWS, None, cls=len(plan.classes()))
    with pytest.raises(PsError):
        plan.tune(9, None)
    plan.set_method("bf16mix")
    want = sweep()
    bufs = sweep()
    tuned = plan.autotune(un, *bufs, max_classes=4)
    assert {"default", "1", "2", "4"} <= set(tuned["knobs"][0]["all"])
    assert all(torch.equal(a, b) for a, b in zip(sweep(), want))
    plan.close()
