"""The orders of the far field's series at the distances from which they are taken, for the clusters that
need most of them, against extended-precision sums.

Each design is one cluster (512 segments, its ball about the origin) and one point just past one of the
distances of the table, so that the whole field is one series.  Clusters: one strong element on the rim, facing
the point or a few degrees off; a bar; a ring; elements all over the ball."""
import math
import os
import re

import numpy as np
import pytest
import torch

from tests._helpers import ROOT, ensure_built, gpu_available

pytestmark = pytest.mark.gpu

ensure_built()

from cctpy_amd import _native as N, engine  # noqa: E402
from cctpy_amd.engine import _p  # noqa: E402

if not gpu_available():
    pytest.skip("no GPU visible", allow_module_level=True)

EPS = 2.0 ** -52
# FP64: the cut (4e-16 at the worst, tests/test_far_orders.py) below one rounding per order of the series.
# FP32: its series are cut at 2e-9 at the worst and evaluated in FP64.
TOLERANCE = {64: 32 * EPS, 33: 2e-9}


def ratios(precision):
    with open(os.path.join(ROOT, "cctpy_amd", "csrc", "far.hpp")) as f:
        text = f.read()
    body = text.split("struct FarOrders<%s>" % ("true" if precision == 64 else "false"))[1]
    return [float(x) for x in re.search(r"ratio\[n\] = \{([^}]*)\}", body).group(1).split(",")]


def _cluster(shape, u, E, rng):
    """(kl, m) of 512 elements whose bounding box has its middle at the origin and whose radius is E."""
    half = rng.normal(size=(255, 3))
    half *= (0.9 * E * rng.uniform(0, 1, (255, 1)) ** (1 / 3)) / np.linalg.norm(half, axis=1, keepdims=True)
    m = np.concatenate([[E * u, -E * u], half, -half])
    kl = rng.normal(size=(512, 3))
    side = np.cross(u, [0.3, -0.5, 0.8])
    side /= np.linalg.norm(side)
    if shape == "rim":
        kl *= 1e-7
        kl[0] = side
    elif shape == "bar":
        m = np.linspace(-E, E, 512)[:, None] * u
        kl[:] = side
    elif shape == "ring":
        a = 2 * np.pi * np.arange(512) / 512
        w = np.cross(u, side)
        m = E * (np.cos(a)[:, None] * u + np.sin(a)[:, None] * w)
        kl = -np.sin(a)[:, None] * u + np.cos(a)[:, None] * w
    return 1e-7 * kl, m


def _cases(precision):
    rng = np.random.default_rng(17)
    specs, pts, want, size = [], [], [], []
    for ratio in ratios(precision):
        for u in ([1.0, 0.0, 0.0], [0.0, 0.0, 1.0], [0.6, -0.48, 0.64]):
            u = np.array(u)
            v = np.cross(u, [0.3, -0.5, 0.8])
            v /= np.linalg.norm(v)
            for shape, degrees in (("rim", 0), ("rim", 4), ("rim", 10), ("bar", 0), ("ring", 0), ("ball", 0)):
                E = 0.04
                kl, m = _cluster(shape, u, E, rng)
                a = math.radians(degrees)
                radius = max(np.linalg.norm(m - 0.5 * (m.min(0) + m.max(0)), axis=1))
                q = radius * ratio * (1 + 1e-5) * (math.cos(a) * u + math.sin(a) * v)
                r = q.astype(np.longdouble) - m.astype(np.longdouble)
                w = np.sqrt((r * r).sum(1)) ** -3
                terms = np.cross(kl.astype(np.longdouble), r) * w[:, None]
                specs.append(engine.DesignSpec(raw_kl=kl, raw_m=m))
                pts.append(q)
                want.append(terms.sum(0))
                size.append(np.sqrt((terms * terms).sum(1)).sum())
    return specs, np.array(pts), np.array(want), np.array(size, float)


@pytest.mark.parametrize("precision,ppl", [(64, 1), (64, 2), (64, 4), (64, -2), (64, -4), (33, 1), (33, 2), (33, 4),
                                           (33, -2)])
def test_series_at_the_distances_they_are_taken_from(precision, ppl, monkeypatch):
    monkeypatch.setattr(engine.DeviceModel, "_far_pays", lambda *a: True)
    specs, pts, want, size = _cases(precision)
    model = engine.DeviceModel(specs, fp32=precision != 64)
    plan = model.plan([1] * len(specs), ppl)
    far = model.far_field(plan, precision, 0)
    soa = torch.from_numpy(np.ascontiguousarray(pts.T)).to(engine.device())
    _, partial = model.workspace(plan)
    out = torch.empty_like(soa)
    model._call(N.lib.cctamd_bs_field_far, "cctamd_bs_field_far", plan, precision, far, _p(soa), plan.npt, _p(partial),
                _p(out))
    err = np.linalg.norm((out.cpu().numpy().T - want).astype(float), axis=1) / size
    print(f"precision {precision} ppl {ppl}: worst {err.max():.2e} of the cluster's sum of |terms|")
    assert err.max() <= TOLERANCE[precision], err.reshape(len(ratios(precision)), -1).max(1)
    # series they were, not the segments one by one
    full = torch.empty_like(soa)
    model._call(N.lib.cctamd_bs_field, "cctamd_bs_field", plan, precision, None, _p(soa), plan.npt, _p(partial), _p(full))
    assert not np.array_equal(full.cpu().numpy(), out.cpu().numpy())
