"""A model and its segment clusters copied, pickled, and used from several streams and threads."""
import copy
import gc
import pickle
import threading
import weakref

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


def _stream_of(tensor):
    """The stream whose pool a tensor's memory is from."""
    for seg in torch.cuda.memory_snapshot():
        if seg["address"] <= tensor.data_ptr() < seg["address"] + seg["total_size"]:
            return seg["stream"]
    raise AssertionError("not an allocation of torch")


@pytest.mark.parametrize("precision", [64, 33])
def test_clusters_live_as_long_as_the_segments(precision, monkeypatch):
    """Built by the first call on another stream, used by a third: the memory belongs to the model's stream, like its
    segments', not to the stream that happened to come first."""
    monkeypatch.setattr(engine.DeviceModel, "_far_pays", lambda *a: True)
    model, *rest = _case(precision)
    torch.cuda.synchronize()
    want = None
    for _ in range(2):
        side = torch.cuda.Stream()
        with torch.cuda.stream(side):
            got = _track(model, precision, *rest)
        side.synchronize()
        want = got if want is None else want
        assert np.array_equal(got, want)
    assert np.array_equal(_track(model, precision, *rest), want)
    far, items = model._far[precision], model.plan(rest[-1], 1).far[precision]
    own = _stream_of(model.seg64)
    for t in (far.geo, far.geo_large, far.coef, far.coef_large, far.rows, far.tiles, items.work, items.wbase, items.nchunk):
        assert t is None or _stream_of(t) == own


@pytest.mark.parametrize("precision", [64, 33])
def test_threads_share_the_first_build(precision, monkeypatch):
    """Several threads, a stream each, track a model that has no clusters yet."""
    monkeypatch.setattr(engine.DeviceModel, "_far_pays", lambda *a: True)
    model, *rest = _case(precision)
    want = _track(model, precision, *rest)
    model, *rest = _case(precision)
    torch.cuda.synchronize()
    start, got, failed = threading.Barrier(4), [None] * 4, []

    def work(i):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                start.wait(30)
                got[i] = _track(model, precision, *rest)
        except BaseException as e:  # noqa: BLE001 - shown below
            failed.append(e)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    assert not failed and list(model._far) == [precision]
    for g in got:
        assert np.array_equal(g, want)


@pytest.mark.parametrize("precision", [64, 33])
def test_a_graph_keeps_what_it_reads(precision, monkeypatch):
    monkeypatch.setattr(engine.DeviceModel, "_far_pays", lambda *a: True)
    model, state, kq, dt, ns, npt = _case(precision)
    want = _track(model, precision, state, kq, dt, ns, npt)
    plan = model.plan(npt, 1)
    st = state.clone()
    graph = engine.TrackGraph(model, plan, precision, st, kq, dt, ns, STEPS, *model.workspace(plan))
    alive, items = weakref.ref(model), weakref.ref(plan.far[precision].work)
    del model, plan
    gc.collect()
    assert alive() is not None and items() is not None
    for _ in range(2):
        st.copy_(state)
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(st.cpu().numpy(), want)


@pytest.mark.parametrize("precision", [64, 33])
@pytest.mark.parametrize("where", ["FarField", "_far_plan"])
def test_clusters_that_do_not_fit(where, precision, monkeypatch):
    """The model says so once and sums every segment from then on, also when there is room again: equal calls give
    equal bits."""
    rule = engine.DeviceModel._far_pays
    model, *rest = _case(precision)
    monkeypatch.setattr(engine.DeviceModel, "_far_pays", lambda *a: False)
    full = _track(model, precision, *rest)
    monkeypatch.setattr(engine.DeviceModel, "_far_pays", lambda *a: True)
    tries = []

    def no_room(*a, **k):
        tries.append(1)
        raise torch.OutOfMemoryError("no room")

    with monkeypatch.context() as m:
        m.setattr(engine if where == "FarField" else engine.DeviceModel, where, no_room)
        with pytest.warns(RuntimeWarning, match="segment clusters"):
            assert np.array_equal(_track(model, precision, *rest), full)
        assert np.array_equal(_track(model, precision, *rest), full)
    assert np.array_equal(_track(model, precision, *rest), full)
    assert len(tries) == 1 and not model._far
    monkeypatch.setattr(engine.DeviceModel, "_far_pays", rule)
    assert not model._far_pays(model.plan(rest[-1], 1), precision, 10 ** 6)


@pytest.mark.parametrize("precision", [64, 33])
def test_a_capture_builds_no_clusters(precision, monkeypatch):
    """Captured before anything was tracked, a track sums every segment (the eager call of a model without them); with the
    clusters there, it takes them."""
    monkeypatch.setattr(engine.DeviceModel, "_far_pays", lambda *a: False)
    model, state, kq, dt, ns, npt = _case(precision)
    full = _track(model, precision, state, kq, dt, ns, npt)
    monkeypatch.setattr(engine.DeviceModel, "_far_pays", lambda *a: True)
    plan = model.plan(npt, 1)
    scratch, partial = model.workspace(plan)
    st = state.clone()

    def captured():
        graph = torch.cuda.CUDAGraph()
        torch.cuda.synchronize()
        with torch.cuda.graph(graph):
            model.track_tensors(plan, precision, st, kq, dt, ns, STEPS, scratch, partial)
        return graph

    def replayed(graph):
        st.copy_(state)
        graph.replay()
        torch.cuda.synchronize()
        return st.cpu().numpy()

    before = captured()
    assert not model._far and np.array_equal(replayed(before), full)
    far = _track(model, precision, state, kq, dt, ns, npt)
    assert not np.array_equal(far, full)
    after = captured()
    for _ in range(3):
        assert np.array_equal(replayed(after), far)
        assert np.array_equal(replayed(before), full)
        assert np.array_equal(_track(model, precision, state, kq, dt, ns, npt), far)
