"""Work items of the far-field kernels (host planner, no GPU)."""
import ctypes

import numpy as np
import pytest

from tests._helpers import ensure_built

ensure_built()

from cctpy_amd import _native as N  # noqa: E402


def _far_plan(ntile, npt, ppl, target):
    ntile, npt = np.asarray(ntile, np.int64), np.asarray(npt, np.int64)
    coff = np.concatenate([[0], np.cumsum(4 * -(-ntile // 64))]).astype(np.int64)
    poff = np.concatenate([[0], np.cumsum(npt)]).astype(np.int64)

    def p(a):
        return a.ctypes.data_as(ctypes.c_void_p)

    args = (len(ntile), p(ntile), p(npt), p(coff), p(poff), ppl, target)
    n = N.lib.cctamd_far_plan(*args, None, None, None)
    if n < 0:
        return n
    work, wbase, nch = np.zeros((max(n, 1), 8), np.int32), np.zeros(len(ntile), np.int64), np.zeros(len(ntile), np.int32)
    assert N.lib.cctamd_far_plan(*args, p(work), p(wbase), p(nch)) == n
    return work[:n], wbase, nch, coff, poff


@pytest.mark.parametrize("ppl", [1, 2, 4, -2, -4])
@pytest.mark.parametrize("target", [1, 7, 300, 5000])
def test_items_cover_every_block_once(ppl, target):
    ntile, npt = [37, 0, 5, 1200, 3], [300, 17, 0, 64, 1]
    work, wbase, nch, coff, poff = _far_plan(ntile, npt, ppl, target)
    pb = 64 * ppl if ppl > 0 else 64 // -ppl
    blocks = sum(-(-n // pb) for n in npt)
    assert blocks <= len(work) <= max(target, 1) + blocks
    seen = set()
    for i, (d, ps, pc, cl, ncl, c, nc, b) in enumerate(work.tolist()):
        assert i == wbase[d] + b * nc + c and nc == nch[d] and 0 <= c < nc  # where the partial sums are looked up
        assert ps == poff[d] + b * pb and pc == min(pb, npt[d] - b * pb)
        assert cl == coff[d] and ncl == -(-ntile[d] // 16) and nc <= max(ntile[d], 1)
        seen.add((d, b, c))
    assert len(seen) == len(work)
    assert {(d, b) for d, b, _ in seen} == {(d, b) for d, n in enumerate(npt) for b in range(-(-n // pb))}


@pytest.mark.parametrize("ntile,npt,ppl,target", [([-1], [4], 1, 8), ([4], [-1], 1, 8), ([4], [4], 3, 8),
                                                  ([4], [4], 1, 0)])
def test_bad_arguments_are_refused(ntile, npt, ppl, target):
    assert _far_plan(ntile, npt, ppl, target) == -22


@pytest.mark.parametrize("ppl", [1, 2, 4, -2, -4])
@pytest.mark.parametrize("precision", [33, 64])
def test_items_fill_whole_rounds(precision, ppl):
    """Designs that differ: no items past a full round of what the CUs have under way (two 8-wave items per CU,
    one 4-wave item), unless the next round is nearly full too; never more than the caller's."""
    from cctpy_amd.engine import far_items

    cus = 256
    each = 2 * cus if ppl > 0 else cus
    for clusters in (1, 900, 1275, 2000, 2650, 3030, 4260, 5200, 9600, 100000):
        for most in (7, 255, 300, 530, 986, 1025, 1536, 4096):
            n = far_items(clusters, False, False, precision, ppl, cus, most)
            assert 0 < n <= most and n <= 6 * cus
            over = n % each
            assert n == most and (most < each or over >= 0.7 * each) or over == 0, (clusters, most, n)
    # maps: four per CU, whatever the designs
    assert far_items(28800, True, True, precision, ppl, cus, 5000) == 4 * cus
    assert far_items(28800, False, True, precision, ppl, cus, 900) == 900

def test_bad_arguments_of_a_routed_field_are_refused():
    """On the host, before any launch."""
    some = ctypes.c_void_p(64)
    assert N.lib.cctamd_point_spread(3, some, some, 1, some, 1, some, None) == -22
    assert N.lib.cctamd_point_spread(2, some, some, 1, some, 1, None, None) == -22
    assert N.lib.cctamd_point_spread(2, some, None, 1, some, 1, some, None) == -22
    args = dict(spread=some, geo=some, geo_large=some, coef=some, coef_large=some, rows=some, far_work=some, far_nwork=1,
                far_wbase=some, far_nchunk=some, precision=64, ppl=2)
    rest = [some, None, None, some, 1, some, some, some, 1, some, some, some, some, 1, some, some, None]
    for name, value in (("spread", None), ("geo", None), ("coef_large", None), ("rows", None), ("far_work", None),
                        ("far_nwork", 0), ("far_nwork", 2), ("far_nchunk", None), ("precision", 33), ("ppl", 3)):
        assert N.lib.cctamd_bs_field_routed(*{**args, name: value}.values(), *rest) == -22, name
