"""What a closed plan leaves with the library goes back to the device on
request, from Python."""
import pytest

from partapp_amd.api import ExpParam, Plan, person_model, release_memory, synth_joints

pytestmark = pytest.mark.gpu


def test_release_memory(gpu):
    import torch
    release_memory()
    plan = Plan(person_model(ExpParam(-180.0, 180.0, 24, 1.0, 1.0, 1, 0.0), synth_joints(3)), [(300, 300)])
    scratch = plan.scratch_bytes()
    plan.close()
    kept = torch.cuda.mem_get_info()[0]
    release_memory()
    # the scratch, less the slack of allocation sizes
    assert torch.cuda.mem_get_info()[0] - kept >= scratch - (4 << 20)
    release_memory()  # nothing left: no error
