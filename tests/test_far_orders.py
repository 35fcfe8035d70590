"""The far field's table of orders (csrc/far.hpp) against the worst cut of a series (no GPU)."""
import math
import os
import re

import pytest

from tests._helpers import ROOT


def _table(fp64):
    with open(os.path.join(ROOT, "cctpy_amd", "csrc", "far.hpp")) as f:
        body = f.read().split("struct FarOrders<%s>" % ("true" if fp64 else "false"))[1]
    return [[float(x) for x in re.search(name + r"\[n\] = \{([^}]*)\}", body).group(1).split(",")]
            for name in ("ratio", "order")]


def _cut(order, ratio):
    """Largest error of the field of one element on the rim of a ball of radius 1, its potential cut before
    degree `order`, at distance `ratio` from the centre, relative to the element's field: gradient of
    sum over n >= order of P_n(cos a) / ratio^(n + 1), over angles a and all directions of the element."""
    worst = 0.0
    for i in range(361):
        c = math.cos(math.pi * i / 360)
        s = math.sqrt(1 - c * c)
        radial = angular = 0.0
        p0, p1, d0, d1 = 1.0, c, 0.0, 1.0
        for n in range(2, order + 80):
            p0, p1 = p1, ((2 * n - 1) * c * p1 - (n - 1) * p0) / n
            d0, d1 = d1, d0 + (2 * n - 1) * p0
            if n >= order:
                radial += (n + 1) * p1 * ratio ** -(n + 2)
                angular += s * d1 * ratio ** -(n + 2)
        worst = max(worst, math.hypot(radial, angular) * (ratio * ratio - 2 * ratio * c + 1))
    return worst


@pytest.mark.parametrize("fp64,bound", [(True, 4e-16), (False, 2e-9)])
def test_every_order_cuts_below_its_bound(fp64, bound):
    """FP64: below the rounding of the terms that a series replaces, also where one element has all the
    current.  FP32: below its terms' rounding (6e-8) and its sums' error (2e-8)."""
    ratios, orders = _table(fp64)
    assert len(ratios) == len(orders) >= 7 and ratios == sorted(ratios) and orders == sorted(orders, reverse=True)
    cuts = {(n, r): _cut(int(n), r) for r, n in zip(ratios, orders)}
    assert max(cuts.values()) <= bound, cuts
