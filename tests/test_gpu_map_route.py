"""Field maps through the segment clusters, and those whose points have no use for them.

An FP64 map of many points lets far clusters act through series (within 1e-13 of the sum of every segment: up to 10^5
terms in another order), unless its blocks reach across the magnet, where every segment is summed (the same bits).
What a call gives depends on its points alone, not on the calls before it."""
import weakref

import numpy as np
import pytest
import torch

from tests._helpers import ensure_built, gpu_available

pytestmark = pytest.mark.gpu

ensure_built()

from cctpy_amd import _native as N, engine, workloads as W  # noqa: E402
from cctpy_amd.magnets import device_parts  # noqa: E402

if not gpu_available():
    pytest.skip("no GPU visible", allow_module_level=True)

POINTS = [700, 0, 3, 450]  # the third design without windings


@pytest.fixture(autouse=True)
def maps_of_any_size(monkeypatch):
    monkeypatch.setattr(engine.DeviceModel, "_far_pays", lambda *a: True)
    monkeypatch.setattr(engine, "_FAR_MAP_PAIRS", 0.0)


def _beamlines():
    designs = W.population(n_designs=3, n_particles=1, seed=5).designs
    return [W.build_beamline(d) for d in designs]


def _model(bls):
    specs = [device_parts(bl).spec() for bl in bls]
    specs.insert(2, engine.DesignSpec(qs=np.zeros((0, 16)), bconst=np.array([0.0, 0.0, 0.5])))
    return engine.DeviceModel(specs, fp32=False)


def _points(bls, order):
    """Along each design's orbit, 20 mm around it, in order or shuffled within the design."""
    rng = np.random.default_rng(4)
    rows = []
    for bl, n in zip(bls[:2] + [bls[0]] + bls[2:], POINTS):
        q = [bl.trajectory.point_at(float(s)) for s in np.linspace(0, bl.get_length(), n + 2)[1:-1]]
        p = np.array([[p.x, p.y, 0.0] for p in q]).reshape(n, 3) + rng.uniform(-0.02, 0.02, (n, 3))
        rows.append(p if order == "ordered" else rng.permutation(p))
    return torch.from_numpy(np.ascontiguousarray(np.concatenate(rows).T)).to(engine.device())


def _field(model, pts, ppl, far=True):
    plan = model.plan(POINTS, ppl)
    _, partial = model.workspace(plan)
    out = torch.full_like(pts, float("nan"))
    if far:
        model.field_tensors(plan, 64, pts, partial, out)
    else:
        soa = [engine._p(t) for t in (pts, partial, out)]
        model._call(N.lib.cctamd_bs_field, "cctamd_bs_field", plan, 64, None, soa[0], plan.npt, soa[1], soa[2])
    return out.cpu().numpy()


@pytest.mark.parametrize("ppl", [1, 2, 4, -2, -4])
def test_ordered_maps_take_the_clusters(ppl):
    bls = _beamlines()
    model, pts = _model(bls), _points(bls, "ordered")
    got = _field(model, pts, ppl)
    want = _field(model, pts, ppl, far=False)
    assert 64 in model._far and not np.array_equal(got, want)
    assert np.max(np.abs(got - want)) <= 1e-13 * np.max(np.abs(want))
    assert np.array_equal(_field(model, pts, ppl), got)


@pytest.mark.parametrize("ppl", [1, 2, 4, -2, -4])
def test_shuffled_maps_sum_every_segment(ppl):
    bls = _beamlines()
    model, pts = _model(bls), _points(bls, "shuffled")
    want = _field(model, pts, ppl, far=False)
    assert np.array_equal(_field(model, pts, ppl), want)
    assert not model._far  # nothing built for them
    # nor do clusters that are there change it
    ordered = _points(bls, "ordered")
    first = _field(model, ordered, ppl)
    assert 64 in model._far
    assert np.array_equal(_field(model, pts, ppl), want)
    assert np.array_equal(_field(model, ordered, ppl), first)
    assert np.array_equal(_field(_model(bls), ordered, ppl), first)


def test_points_that_are_not_finite():
    """They reach everywhere: a map of them sums every segment; one of them leaves the other points as they are."""
    bls = _beamlines()
    model, pts = _model(bls), _points(bls, "ordered")
    want = _field(model, pts, 2, far=False)
    one = pts.clone()
    one[0, 5] = float("nan")
    got = _field(model, one, 2)
    others = np.delete(np.arange(pts.shape[1]), 5)
    assert np.isnan(got[:, 5]).all()
    assert np.max(np.abs(got[:, others] - want[:, others])) <= 1e-13 * np.max(np.abs(want))
    every = torch.full_like(pts, float("inf"))
    assert np.array_equal(_field(model, every, 2), _field(model, every, 2, far=False), equal_nan=True)


def test_a_captured_map_follows_its_points():
    """The choice is the device's: replays with other points in the buffer are the eager calls on them."""
    bls = _beamlines()
    model = _model(bls)
    sets = [_points(bls, "ordered"), _points(bls, "shuffled")]
    want = [_field(model, p, 2) for p in sets]
    plan = model.plan(POINTS, 2)
    _, partial = model.workspace(plan)
    pts, out = sets[0].clone(), torch.empty_like(sets[0])
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        model.field_tensors(plan, 64, pts, partial, out)
    for rep in range(4):
        pts.copy_(sets[rep % 2])
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(out.cpu().numpy(), want[rep % 2]), rep
        assert np.array_equal(_field(model, sets[rep % 2], 2), want[rep % 2]), rep


def test_what_the_device_found_outlives_the_launches(monkeypatch):
    """The call holds the counts of the points until its kernels are on the stream: their memory cannot go to another
    thread's tensors before."""
    bls = _beamlines()
    model, pts = _model(bls), _points(bls, "ordered")
    want = _field(model, pts, 2)
    found, alive = [], []
    empty, call = torch.empty, model._call

    def noted(*a, **k):
        t = empty(*a, **k)
        if k.get("dtype") == torch.int64:
            found.append(weakref.ref(t))
        return t

    def launched(*a, **k):
        alive.append(found[-1]() is not None)
        call(*a, **k)

    monkeypatch.setattr(torch, "empty", noted)
    monkeypatch.setattr(model, "_call", launched)
    assert np.array_equal(_field(model, pts, 2), want)
    assert alive == [True] and found[-1]() is None


@pytest.mark.parametrize("precision,ppl", [(64, 1), (64, -2), (33, 1), (33, -2)])
def test_host_particles_all_along_the_orbit_sum_every_segment(precision, ppl):
    """A bunch takes the clusters, particles at all places of the orbit do not (and nothing is built for them)."""
    bls = _beamlines()[:2]
    model = engine.DeviceModel([device_parts(bl).spec() for bl in bls], fp32=precision != 64)
    rng = np.random.default_rng(6)
    n = 60
    bunch, along = [], []
    for bl in bls:
        for rows, places in ((bunch, rng.normal(0.3, 2e-3, n)), (along, rng.uniform(0.05, 0.95, n) * bl.get_length())):
            for s in places:
                p, d = bl.trajectory.point_at(float(s)), bl.trajectory.direct_at(float(s))
                rows.append([p.x, p.y, 0.0, 1.8e8 * d.x, 1.8e8 * d.y, 0.0])
    args = (np.full(2 * n, 7.0e7), np.full(2 * n, 1e-3 / 1.8e8), np.full(2 * n, 3), [n, n])

    def full(state):
        plan = model.plan([n, n], ppl)
        scratch, partial = model.workspace(plan)
        st, kq, dt, ns = (torch.from_numpy(np.ascontiguousarray(a)).to(engine.device())
                          for a in (np.array(state).T, *args[:3]))
        model._track(plan, precision, st, kq, dt, ns, 3, scratch, partial, None, 1, far_field=False)
        return st.cpu().numpy().T

    assert np.array_equal(model.track(np.array(along), *args, precision=precision, ppl=ppl)[0], full(along))
    assert not model._far
    got, want = model.track(np.array(bunch), *args, precision=precision, ppl=ppl)[0], full(bunch)
    assert precision in model._far and not np.array_equal(got, want)
    np.testing.assert_allclose(got, want, rtol=1e-6 if precision == 33 else 1e-12, atol=1e-9)
    assert np.array_equal(model.track(np.array(along), *args, precision=precision, ppl=ppl)[0], full(along))
