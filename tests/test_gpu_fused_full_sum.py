"""The fused RK4 stages where every segment is summed.

Sets with segment clusters take two launches per stage whatever CCTAMD_FUSED_STAGES says, so the designs of
tests/test_gpu_fused.py no longer reach the fused kernels by themselves at most shapes; here they do."""
import numpy as np
import pytest

from tests import test_gpu_fused as F

pytestmark = pytest.mark.gpu

engine = F.engine


@pytest.fixture(autouse=True)
def every_segment(monkeypatch):
    monkeypatch.setattr(engine.DeviceModel, "_far_pays", lambda *a: False)

    def no_clusters(*a, **k):
        raise AssertionError("the fused stages have no segment clusters")

    monkeypatch.setattr(engine, "FarField", no_clusters)


@pytest.mark.parametrize("precision", [64, 33, 32])
@pytest.mark.parametrize("ppl", [1, 2, 4])
def test_fused_stages_give_the_two_launch_bits(precision, ppl):
    F.test_fused_stages_give_the_two_launch_bits(precision, ppl)


def test_fused_stages_replay_in_a_graph():
    F.test_fused_stages_replay_in_a_graph()


def test_clusters_take_two_launches(monkeypatch):
    """CCTAMD_FUSED_STAGES=1 changes nothing where a track takes the clusters."""
    monkeypatch.undo()
    monkeypatch.setattr(engine.DeviceModel, "_far_pays", lambda *a: True)
    bls, npt, state, kq, dt, ns = F._case(n_particles=40)
    model = engine.DeviceModel([F.device_parts(bl).spec() for bl in bls], fp32=False)
    with F._fused():
        fused, _ = model.track(state, kq, dt, ns, npt, precision=64, ppl=1)
    assert 64 in model._far
    two, _ = model.track(state, kq, dt, ns, npt, precision=64, ppl=1)
    assert np.array_equal(fused, two)
    monkeypatch.setattr(engine.DeviceModel, "_far_pays", lambda *a: False)
    assert not np.array_equal(model.track(state, kq, dt, ns, npt, precision=64, ppl=1)[0], two)
