"""The tuner times what tracking launches."""
import numpy as np
import pytest
import torch

from tests._helpers import ensure_built, gpu_available

pytestmark = pytest.mark.gpu

ensure_built()

from cctpy_amd import autotune, engine, workloads as W  # noqa: E402
from cctpy_amd.magnets import device_parts  # noqa: E402

if not gpu_available():
    pytest.skip("no GPU visible", allow_module_level=True)


def _case(precision):
    wl = W.single_cct(n_particles=8)
    bl = W.build_beamline(wl.designs[0])
    ps = W.beam_particles(wl.beams[0], bl)
    pts = torch.tensor([p.position.to_list() for p in ps], dtype=torch.float64, device=engine.device()).T.contiguous()
    return engine.DeviceModel([device_parts(bl).spec()], fp32=precision != 64), [len(ps)], pts


@pytest.mark.parametrize("precision,fast", [(64, 4), (64, -4), (33, 2), (33, -2), (32, 4)])
def test_the_shape_with_the_fastest_steps_wins(precision, fast, monkeypatch):
    """One shape's steps cost nothing and the others' a millisecond each."""
    model, npt, pts = _case(precision)
    track = engine.DeviceModel._track

    def slow(self, plan, *a, **k):
        track(self, plan, *a, **k)
        if plan.ppl != fast:
            torch.cuda._sleep(2_000_000)

    monkeypatch.setattr(engine.DeviceModel, "_track", slow)
    best = autotune.tune(model, npt, precision, pts, launches=1, use_cache=False, rounds=1)
    assert best["ppl"] == fast and best["ms"] > 0.0
    assert best["target_items"] % engine.cu_count() == 0


@pytest.mark.parametrize("precision", [64, 33])
def test_the_steps_are_those_of_a_long_track(precision, monkeypatch):
    """With the clusters where a long track takes them, at the points given, which stay as they are."""
    def pays(self, plan, precision, steps):  # 16-point blocks of the FP32 path have no such kernel
        return steps > 1000 and (precision, plan.ppl) != (33, -4)

    monkeypatch.setattr(engine.DeviceModel, "_far_pays", pays)
    model, npt, pts = _case(precision)
    before, used = pts.clone(), []
    track = engine.DeviceModel._track

    def seen(self, plan, precision, state, *a, **k):
        at = state[:3].clone()
        track(self, plan, precision, state, *a, **k)
        used.append((plan.ppl, (precision in plan.far) == pays(self, plan, precision, 2000), bool(torch.equal(at, state[:3])), bool(torch.equal(at, before))))

    monkeypatch.setattr(engine.DeviceModel, "_track", seen)
    autotune.tune(model, npt, precision, [pts, pts], launches=2, use_cache=False, rounds=1)
    assert used and all(u[1:] == (True, True, True) for u in used)
    assert np.array_equal(before.cpu().numpy(), pts.cpu().numpy())
