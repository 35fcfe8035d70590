"""A model and its segment clusters copied, pickled, and used from several streams and threads."""
import copy
import pickle

import numpy as np
import pytest
import torch

from tests._helpers import ensure_built, gpu_available

pytestmark = pytest.mark.gpu

ensure_built()

from cctpy_amd import engine, workloads as W  # noqa: E402
from cctpy_amd.magnets import device_parts  # noqa: E402

if not gpu_available():
    pytest.skip("no GPU visible", allow_module_level=True)

STEPS = 20


def _case(precision):
    """(model, states (6, P), kq, dt, nsteps, particles per design) of three designs that take the far field."""
    wl = W.population(n_designs=3, n_particles=40, seed=9)
    bls = [W.build_beamline(d) for d in wl.designs]
    ps = [p for bl, beam in zip(bls, wl.beams) for p in W.beam_particles(beam, bl)]
    state = np.array([p.position.to_list() + p.velocity.to_list() for p in ps])
    sd = [engine.rk4_steps(STEPS * 1e-3, 1e-3, p.speed) for p in ps]
    dev = engine.device()
    model = engine.DeviceModel([device_parts(bl).spec() for bl in bls], fp32=precision != 64)
    return (model, torch.from_numpy(np.ascontiguousarray(state.T)).to(dev),
            torch.tensor([p.e / p.relativistic_mass for p in ps], dtype=torch.float64, device=dev),
            torch.tensor([d for _, d in sd], dtype=torch.float64, device=dev),
            torch.tensor([n for n, _ in sd], dtype=torch.int64, device=dev), [40] * 3)


def _track(model, precision, state, kq, dt, ns, npt):
    """Final states on the host, every buffer made on the current stream."""
    plan = model.plan(npt, 1)
    scratch, partial = model.workspace(plan)
    st = state.clone()
    model.track_tensors(plan, precision, st, kq, dt, ns, int(STEPS), scratch, partial)
    return st.cpu().numpy()


@pytest.mark.parametrize("precision", [64, 33])
@pytest.mark.parametrize("tracked", [False, True])
@pytest.mark.parametrize("how", [copy.deepcopy, copy.copy, lambda m: pickle.loads(pickle.dumps(m))])
def test_copies_of_a_model_track_alike(how, tracked, precision, monkeypatch):
    monkeypatch.setattr(engine.DeviceModel, "_far_pays", lambda *a: True)
    model, *rest = _case(precision)
    if tracked:
        _track(model, precision, *rest)
    other = how(model)
    want = _track(model, precision, *rest)
    assert precision in model._far
    assert np.all(np.isfinite(want)) and np.array_equal(_track(other, precision, *rest), want)
