"""Tracking with the far field of segment clusters against the sum over every segment.

Single steps of 0.2 m, so that a relative field error e turns into a velocity error of about
0.2 m / 0.95 m x e: with the cut of the series below 1e-15 and sums of up to 10^5 terms in another
order (1e-14 at the worst of the forms below, which come to within centimetres of the windings) the
states agree to 1e-13 of the velocity and 1e-13 m.  FP32 path: both sums within 1e-6 of the
field, so 2 x 0.21 x 1e-6 of each other."""
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

TOLERANCE = {64: 1e-13, 33: 4.2e-7}


def _specs():
    """Designs of 1, 33 and 17 tiles of raw elements (parts of clusters; one tile, one small cluster and a
    tile, one large cluster and a bit), an empty one, and two with windings."""
    rng = np.random.default_rng(3)
    specs = []
    for n in (5, 17 * 32 - 3, 0, 65 * 32 + 1):
        m = rng.uniform(-0.1, 0.1, (n, 3)) + np.array([0.5, 0.3, 0.0])
        specs.append(engine.DesignSpec(raw_kl=1e-7 * 9000 * rng.normal(0, 1e-3, (n, 3)), raw_m=m))
    wl = W.population(n_designs=2, n_particles=1, seed=5)
    return specs + [device_parts(W.build_beamline(d)).spec() for d in wl.designs]


def _beam(npt):
    """Particles per design: a tight bunch in the bore or outside, one design's spread over a metre, one
    of a single particle."""
    rng = np.random.default_rng(8)
    rows = []
    for d, n in enumerate(npt):
        spread = 0.5 if d == 3 else 3e-3
        p = rng.normal(0, spread, (n, 3)) + np.array([0.3, -0.02, 0.01])
        v = rng.normal(0, 2e-3, (n, 3)) + np.array([1.0, 0.0, 0.0])
        rows.append(np.concatenate([p, 1.8e8 * v / np.linalg.norm(v, axis=1, keepdims=True)], axis=1))
    return np.concatenate(rows)


def _track(model, plan, precision, state, steps, far):
    dev = engine.device()
    P = state.shape[0]
    scratch, partial = model.workspace(plan)
    st = torch.from_numpy(np.ascontiguousarray(state.T)).to(dev)
    kq = torch.full((P,), 7.0e7, dtype=torch.float64, device=dev)
    dt = torch.full((P,), 0.2 / 1.8e8, dtype=torch.float64, device=dev)
    ns = torch.tensor([steps - (i % 2 if steps > 1 else 0) for i in range(P)], dtype=torch.int64, device=dev)
    model._track(plan, precision, st, kq, dt, ns, steps, scratch, partial, None, 1, far_field=far)
    torch.cuda.synchronize()
    return st.cpu().numpy()


@pytest.mark.parametrize("precision,ppl", [(64, 1), (64, 2), (64, 4), (64, -2), (64, -4), (33, 1), (33, 2), (33, 4),
                                           (33, -2)])
@pytest.mark.parametrize("steps", [1, 3])
def test_far_field_matches_the_full_sum(precision, ppl, steps, monkeypatch):
    monkeypatch.setattr(engine.DeviceModel, "_far_pays", lambda *a: True)
    specs = _specs()
    npt = [3, 130, 2, 40, 1, 257]
    model = engine.DeviceModel(specs, fp32=precision != 64)
    state = _beam(npt)
    for target in (None, 40):  # one item per block or a few
        plan = model.plan(npt, ppl, target)
        got = _track(model, plan, precision, state, steps, True)
        assert plan.far[precision].nwork <= plan.nwork
        want = _track(model, plan, precision, state, steps, False)
        assert np.all(np.isfinite(got)) and not np.array_equal(got, state.T)
        tol = TOLERANCE[precision]
        assert np.max(np.abs(got[:3] - want[:3])) <= tol
        assert np.max(np.abs(got[3:] - want[3:])) <= tol * 1.8e8
        # the same bits again
        assert np.array_equal(_track(model, plan, precision, state, steps, True), got)


def test_far_field_keeps_particles_apart(monkeypatch):
    """A particle that is not finite, or far outside, leaves the others of its design as they are."""
    monkeypatch.setattr(engine.DeviceModel, "_far_pays", lambda *a: True)
    specs = _specs()[4:5]
    model = engine.DeviceModel(specs, fp32=False)
    state = _beam([100])
    plan = model.plan([100], 1)
    want = _track(model, plan, 64, state, 1, False)
    state[7, 0], state[70, 1] = np.nan, 1.0e6
    got = _track(model, plan, 64, state, 1, True)
    others = np.delete(np.arange(100), [7, 70])
    assert np.isnan(got[:3, 7]).any()
    assert np.max(np.abs(got[:3, others] - want[:3, others])) <= 1e-13
    assert np.max(np.abs(got[3:, others] - want[3:, others])) <= 1e-13 * 1.8e8


def test_far_field_of_a_map_matches_the_full_sum(monkeypatch):
    """B of one evaluation: relative to its largest value both sums are within 1e-13 (10^5 terms in
    another order, points from 3 mm to metres off the windings)."""
    model = engine.DeviceModel(_specs(), fp32=False)
    npt = [3, 130, 2, 40, 1, 257]
    pts = torch.from_numpy(np.ascontiguousarray(_beam(npt)[:, :3].T)).to(engine.device())
    for ppl in (1, 2, -2):
        plan = model.plan(npt, ppl)
        _, partial = model.workspace(plan)
        out = []
        for far in (True, False):
            monkeypatch.setattr(engine.DeviceModel, "_far_pays", lambda *a: far)
            b = torch.full_like(pts, float("nan"))
            model.field_tensors(plan, 64, pts, partial, b)
            out.append(b.cpu().numpy())
        assert np.all(np.isfinite(out[0]))
        for d, (a, b) in enumerate(zip(*[np.split(o, np.cumsum(npt)[:-1], axis=1) for o in out])):
            assert np.max(np.abs(a - b)) <= 1e-13 * max(np.max(np.abs(b)), 1e-300), (ppl, d)

@pytest.mark.parametrize("precision,ppl", [(64, 1), (64, 2), (64, -2), (64, -4), (33, 1), (33, 2), (33, -2)])
def test_the_number_of_items_does_not_change_the_sum(precision, ppl, monkeypatch):
    """The series' rows and the near segments dealt out to the waves of few items or of many (more waves
    than rows in the designs of few tiles): the same terms, added up in another order.  The FP32 path
    sums whole tiles, so its tile sums are the same too."""
    monkeypatch.setattr(engine.DeviceModel, "_far_pays", lambda *a: True)
    npt = [3, 130, 2, 40, 1, 257]
    model = engine.DeviceModel(_specs(), fp32=precision != 64)
    state = _beam(npt)
    results, items = [], []
    for cus in (1, 3, 100, 1000):  # items per block from one to one per tile
        monkeypatch.setattr(engine, "cu_count", lambda: cus)
        model._plans.clear()
        plan = model.plan(npt, ppl, 8192)
        results.append(_track(model, plan, precision, state, 1, True))
        items.append(plan.far[precision].nwork)
    assert items == sorted(items) and items[-1] > 2 * items[0]
    for r in results[1:]:
        np.testing.assert_allclose(r[:3], results[0][:3], rtol=0, atol=1e-13)
        v = np.linalg.norm(results[0][3:], axis=0)
        assert (np.abs(r[3:] - results[0][3:]) <= 1e-13 * v).all()
