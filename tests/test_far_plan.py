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


def _pays(precision, ppl, segments, points, steps, designs=1):
    """DeviceModel._far_pays of designs of so many segments and points each."""
    from cctpy_amd import engine

    model = object.__new__(engine.DeviceModel)
    model.ndesign, model.nseg_padded = designs, designs * segments
    model._far_no_room = set()
    model.cluster_rows = designs * -(-segments // 2048) * 2048
    pb = engine.points_per_block(ppl)
    plan = engine.Plan(ppl=ppl, nwork=0, work=None, wbase=None, nchunk=None, design_pt_off=None, npt=designs * points,
                       pairs=float(designs * -(-points // pb) * pb * segments), large=segments / 2048)
    return model._far_pays(plan, precision, steps)


def test_small_blocks_of_the_fp32_path_keep_the_full_sum():
    """Where a bunch gains nothing and particles all along the orbit lose (gantry of 479,520 segments, 32 of them)."""
    assert not _pays(33, -2, 479520, 32, 1000)
    assert not _pays(33, -2, 959040, 32, 1000)
    assert _pays(33, 1, 368640, 64, 1000)
    assert _pays(33, -2, 204800, 32, 1000, designs=64)


@pytest.mark.parametrize("precision,ppl,points", [(64, 2, 512), (64, 1, 64), (64, -2, 32), (33, 2, 512), (33, 1, 64)])
def test_short_tracks_do_not_pay_for_clusters(precision, ppl, points):
    """What a bunch saves of the full sum's time (0.6 on the FP64 path, 0.25 on the FP32 path) pays for the set-up as it
    is measured (0.96 and 0.64 ms for the section) in one track."""
    segments = 368640
    rate = {(64, True): 1.25e12, (64, False): 0.9e12, (33, True): 2.5e12}[precision, ppl > 0]
    saved, setup = {64: (0.6, 0.96e-3), 33: (0.25, 0.64e-3)}[precision]
    from cctpy_amd.engine import points_per_block

    lanes = -(-points // points_per_block(ppl)) * points_per_block(ppl)
    taken = [n for n in range(1, 400) if _pays(precision, ppl, segments, points, n)]
    assert taken and 4 * taken[0] * lanes * segments / rate * saved >= setup


@pytest.mark.parametrize("ppl,segments,points,designs", [(1, 200, 64, 2000), (1, 1000, 64, 500), (1, 3000, 64, 200),
                                                         (1, 8000, 64, 64), (1, 16000, 64, 24), (-2, 23040, 32, 100)])
def test_many_small_designs_keep_the_full_sum(ppl, segments, points, designs):
    """A design takes at least one large cluster of 2,048 rows, whatever it holds, and a few clusters are close to all of
    its points."""
    assert not _pays(64, ppl, segments, points, 1000, designs)


def test_the_clusters_of_a_model_are_bounded():
    assert _pays(64, 1, 400000, 64, 1000, designs=640)
    assert not _pays(64, 1, 400000, 64, 1000, designs=1000)


def test_maps_pay_for_their_clusters_in_one_call():
    assert _pays(64, 2, 368640, 5003, 0) and not _pays(64, 2, 368640, 2000, 0)
    assert not _pays(64, 2, 46080, 20000, 0)  # a single CCT: few clusters, 0.3 of the time saved


def test_rows_past_31_bits_are_refused():
    """Before any launch: the FP64 kernels count packed rows in 31 bits, 512 per cluster.  The FP32 path counts tiles."""
    some = ctypes.c_void_p(64)

    def build(precision, clusters):
        return N.lib.cctamd_far_build(precision, some, 32 if precision == 33 else 8, some, some, some, 1, some, 1, clusters,
                                      some, some, some, some, some, some, some, some, None)

    assert build(64, 1 << 22) == -34
    assert build(64, 1 << 27) == build(33, 1 << 27) == -34
