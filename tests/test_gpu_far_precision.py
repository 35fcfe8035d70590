"""The FP32 sum that tracking launches, clusters included, at the states a tracked beam visits.

The states and the bar of tests/test_gpu_precision.py (FP32 against FP64, 1e-6 at every point), in the blocks that are
tracked together: 512 protons per recorded step, some of them out of the bore and a millimetre from the windings."""
import numpy as np
import pytest
import torch

from tests.test_gpu_precision import RECORD_EVERY, recorded  # noqa: F401 - the fixture

from cctpy_amd import engine  # noqa: E402

pytestmark = pytest.mark.gpu

BEAM = 512


@pytest.mark.parametrize("ppl", [1, 2, 4, -2])
def test_tracked_fp32_field_within_1e6_at_recorded_states(recorded, ppl, monkeypatch):  # noqa: F811
    model, pts, b64, _ = recorded
    # the choice of a track of the whole section, where it has one (2 points per lane, see below)
    if ppl != 2:
        monkeypatch.setattr(engine.DeviceModel, "_far_pays", lambda *a: True)
    plan = model.plan([BEAM], ppl)
    _, partial = model.workspace(plan)
    assert model.far_field(plan, 33, 2510) is not None
    worst, far, same = 0.0, torch.empty((3, BEAM), dtype=torch.float64, device=pts.device), True
    full = torch.empty_like(far)
    for i in range(pts.shape[1] // BEAM):
        p = pts[:, i * BEAM:(i + 1) * BEAM].contiguous()
        want = b64[:, i * BEAM:(i + 1) * BEAM]
        model.tracked_field_tensors(plan, 33, p, partial, far, 2510)
        worst = max(worst, float(((far - want).norm(dim=0) / want.norm(dim=0)).max()))
        if i % 50 == 0:
            model.field_tensors(plan, 33, p, partial, full)
            same = same and bool(torch.equal(far, full))
    print(f"ppl {ppl}: {pts.shape[1]} states every {RECORD_EVERY} steps, worst {worst:.3e}")
    assert not same  # series they were
    assert np.isfinite(worst) and worst <= 1e-6
