"""Device engine: HBM-resident segment sets, work plans and calls into libcctamd.

One *design* is one magnet arrangement (a Beamline, a CCT, a CombinedMagnet);
a ``DeviceModel`` holds D designs at once:

* CCT windings are generated on the GPU (``cctamd_winding_generate``) straight
  into an FP64 AoS segment array in the global frame, each design padded to a
  multiple of 32 segments (one *tile*), and packed once into FP32 tiles
  re-centred on an FP64 tile origin, the mean midpoint of the tile
  (``cctamd_pack_fp32``);
* QS magnets travel as the reference's 16-double records, uniform magnets as a
  per-design constant field.

Field and tracking calls take points/particles per design in SoA FP64 and run
on torch's current HIP stream.  There is no CPU path: without a GPU every
entry point raises.
"""
from __future__ import annotations

import collections
import ctypes
import hashlib
import math
import threading
import warnings
from dataclasses import dataclass, field as dc_field
from typing import Dict, List, Optional, Sequence, Tuple

import numpy
import torch

from . import _native as N

_TARGET_WG_PER_CU = 4
_MIN_TILES_PER_ITEM = 4
_LARGE_TILES = 64   # tiles of a large segment cluster (kParts * kSmallTiles in csrc/far.hpp)
_FAR_CHUNK = 16384  # units that are split together (kChunk in csrc/far.hip)
# Where tracking takes the far field (64-point blocks and larger, smaller blocks): lanes x segments of a launch and
# large clusters per design from which it does, or fewer clusters but more lanes x segments (any_*); the pair terms
# per second of the full sum (the same two block sizes) and the share of their time that a bunch saves at the least;
# the set-up in s and s per segment; and the work items per cluster and block of a single design.
# Measured per RK4 stage in us, full sum / far field, for a bunch and for particles all along the orbit.  FP64: one
# in the gantry at 60 segments per winding (1.3e6 pairs, 39 clusters) 12.9 / 12.1 and 13.0 / 11.9, 64 in the AG-CCT
# section at 60 (2.0e6, 15) 11.5 / 13.7, 32 at 120 (2.0e6, 30) 13.6 / 15.6, 16 at 360 (2.9e6, 90) 17.2 / 15.5 and
# 17.6 / 15.7, 32 in the gantry at 120 (5.1e6, 78) 17.0 / 13.4 and 17.6 / 18.2, 200 in one CCT of 720 tiles (5.9e6,
# 11) 16.2 / 16.7, 300 (8.8e6) 20.4 / 18.4, 64 in the gantry at 720 (6.1e7, 468) 68 / 19 and 72 / 89, 512 in the
# section at 720 (1.9e8, 180) 152 / 52 and 155 / 157.  FP32: 64 in the section at 360 (1.2e7, 90) 16.6 / 16.8, at
# 720 (2.4e7, 180) 23.4 / 18.2 and 23.6 / 29.8, 128 in the gantry at 120 (2.0e7, 78) 24.5 / 18.2 and 38.2 / 31.6;
# 32-point blocks: 32 in the gantry at 360 (1.5e7, 234) 19.5 / 20.0 and 24.9 / 29.8, at 720 (3.1e7, 468) 27.1 / 25.7
# and 31.2 / 42.7, four designs x 32 (4.4e7, 166) 33.9 / 28.2 and 35.7 / 41.0; 4,096 in the gantry at 720 (3.9e9)
# 1,500 / 221 and 1,500 / 1,790; single CCTs stay with the full sum there (300 protons, 1,440 tiles: 1.8e7, 22, 19.7
# / 17.3: their clusters are few and close, and series in the place of FP32 terms so near move a track by the FP32
# sum's own error).  Many designs of few clusters, FP64: 2,000 of 200 segments x 64 198 / 242 and 44 ms of set-up,
# 200 of 3,000 x 64 63 / 87, 64 of 8,000 x 64 46 / 49, 24 of 16,000 x 64 36 / 38, 24 of 23,040 x 100 86 / 65, 8 of
# 30,000 x 100 40 / 31; 100 of 23,040 x 32 91 / 105.  Set-up: FP64 0.51 ms for 23,040 segments, 0.96 for 368,640,
# 1.90 for 959,040; FP32 0.37, 0.64, 0.98.
_FAR = {64: dict(pairs=(1.25e6, 1.25e6), large=36, any_pairs=8.5e6, any_large=(10, 36), rate=(1.25e12, 0.9e12),
                 saved=0.6, setup=(0.47e-3, 1.45e-9), share=24),
        33: dict(pairs=(2.0e7, 4.0e7), large=30, any_pairs=math.inf, any_large=(30, 30), rate=(2.5e12, 1.75e12),
                 saved=0.25, setup=(0.40e-3, 0.66e-9), share=6)}
# of a map's time: single CCTs, of few clusters; the section, a population's design and the gantry
_FAR_MAP_SAVED = (0.3, 0.7)
_FAR_MOST_ROWS = 1 << 28  # rows of the clusters (FP64 161 B each, and 140 B while they are built): 43 GB
_FAR_MAP_PAIRS = 5.0e8  # no single evaluation below pays for its clusters


def device() -> torch.device:
    if not torch.cuda.is_available():
        raise RuntimeError("cctpy_amd runs on an AMD Instinct GPU (gfx950); no GPU is visible")
    return torch.device("cuda", torch.cuda.current_device())


def _p(t: Optional[torch.Tensor]):
    """Device address for a void* argument (an int: a ctypes object for each argument costs a field call 1.2 us)."""
    return t.data_ptr() if t is not None and t.numel() > 0 else None


def _np(a: numpy.ndarray):
    return a.ctypes.data_as(ctypes.c_void_p)


def _stream():
    return torch.cuda.current_stream().cuda_stream


def points_per_block(ppl: int) -> int:
    """Point-block size of a points-per-lane code (1, 2, 4 -> 64 ppl; -2, -4 -> 32, 16)."""
    return 64 * ppl if ppl > 0 else 64 // (-ppl)


def block_shape_for(design_npt: Sequence[int], precision: int) -> int:
    """Points-per-lane code whose blocks waste the fewest lanes for these per-design particle
    counts, for callers that do not tune: the smallest of 16, 32, 64 points per block that
    holds the largest design's particles (16 and 32 only where split-wave kernels exist:
    precisions 33 and 64), else 128 (2 points per lane)."""
    m = int(numpy.max(design_npt)) if len(design_npt) else 0
    if precision != 32 and m <= 16:
        return -4
    if precision != 32 and m <= 32:
        return -2
    return 1 if m <= 64 else 2


def cu_count() -> int:
    return int(torch.cuda.get_device_properties(device()).multi_processor_count)


@dataclass
class DesignSpec:
    """Host description of one design: CCT records, QS records, uniform field."""
    cct_params: numpy.ndarray = dc_field(default_factory=lambda: numpy.zeros((0, N.CCT_PARAMS)))
    cct_counts: numpy.ndarray = dc_field(default_factory=lambda: numpy.zeros((0,), numpy.int64))
    qs: numpy.ndarray = dc_field(default_factory=lambda: numpy.zeros((0, 16)))
    bconst: numpy.ndarray = dc_field(default_factory=lambda: numpy.zeros(3))
    # explicit global-frame current elements (kl, midpoint), placed before the CCT windings
    raw_kl: numpy.ndarray = dc_field(default_factory=lambda: numpy.zeros((0, 3)))
    raw_m: numpy.ndarray = dc_field(default_factory=lambda: numpy.zeros((0, 3)))

    @property
    def nseg(self) -> int:
        return int(self.cct_counts.sum()) + int(self.raw_kl.shape[0])

    def key(self) -> bytes:
        h = hashlib.sha1()
        for a in (self.cct_params, self.cct_counts, self.qs, self.bconst, self.raw_kl, self.raw_m):
            h.update(numpy.ascontiguousarray(a).tobytes())
            h.update(str(a.shape).encode())
        return h.digest()


@dataclass
class FarPlan:
    """Work items of the far-field kernels for a plan's point blocks."""
    nwork: int
    work: torch.Tensor
    wbase: torch.Tensor
    nchunk: torch.Tensor


@dataclass
class Plan:
    ppl: int
    nwork: int
    work: torch.Tensor
    wbase: torch.Tensor
    nchunk: torch.Tensor
    design_pt_off: torch.Tensor
    npt: int
    design_npt: tuple = ()
    pairs: float = 0.0  # lanes x segments of a launch
    large: float = 0.0  # large segment clusters per block, in the mean
    # by precision for tracking, by (precision, 0) for single evaluations
    far: Dict[object, FarPlan] = dc_field(default_factory=dict)


def far_items(clusters: int, alike: bool, single: bool, precision: int, ppl: int, cus: int, most: int) -> int:
    """Work items of a far-field launch: ``clusters`` (of every block together), ``alike`` where the blocks'
    designs have as many tiles, ``single`` for one evaluation (a map) instead of a track's stages; at ``most`` so
    many.

    Tracks through designs alike: one or two per CU, as all their items take the same time and between the two
    some CUs have twice the work of others (512 protons in the AG-CCT section, FP32: 256 items 35.7 us per stage,
    320 42.4, 480 35.3, 512 33.9, 640 42.4, 1,024 44.3; 128 protons: 21.5, 25.1, 24.4, 24.4, 33.2; FP64 8 gantries
    x 80: 256 items 23.4, 448 26.6, 512 26.4, 640 33.2).

    Designs that differ balance over smaller items, but over whole rounds of what a CU has under way (two 8-wave
    items; of the 4-wave ones three or four): the items past a round wait for its slowest.  us per stage of a
    bunch / of particles all along the orbit, FP64: 4 designs x 48 protons 530 items 37 / 119, 510 31 / 96; 8 x 48
    852 items 49 / 157, 507 44 / 146; 5 x 100 606 items 60 / 206, 509 56 / 171; 32 x 64 1,025 items 155 / 641,
    1,006 156 / 492; 4 x 32 530 items 27 / 68, 510 25 / 55; FP32: 4 x 48 44 / 101 and 33 / 67.

    A map's blocks see clusters from next to all around, whatever the designs: four per CU (5,003 points in the
    section: 320 items 549 us, 640 375, 960 357; 20,000: 471 items 1,446, 942 1,213)."""
    if single:
        return min(4 * cus, most)
    if alike:
        return min(cus if clusters <= _FAR[precision]["share"] * cus else 2 * cus, most)
    each = 2 * cus if ppl > 0 else cus
    # 0.3: a round that is nearly full
    whole = int(min(max(clusters // 5, 2 * cus), 6 * cus, most) / each + 0.3) * each
    return whole if 0 < whole <= most else most


class FarField:
    """Segment clusters of a model and their multipole coefficients (csrc/far.hip)."""

    def __init__(self, model: "DeviceModel", precision: int):
        dev = model.seg64.device
        large = -(-model.design_ntile // _LARGE_TILES)
        self.cluster_off = numpy.concatenate([[0], numpy.cumsum(4 * large)]).astype(numpy.int64)
        C = int(self.cluster_off[-1])
        unit = N.TILE
        if precision == 64:  # fine units where the design is small or coarse, so that its splits are too
            unit = 1
            while unit < 8 and int(model.design_ntile.max()) * N.TILE > unit * 2 * _FAR_CHUNK:
                unit *= 2
        unit_off = model.design_tile_off * (N.TILE // unit)
        chunk_off = numpy.concatenate([[0], numpy.cumsum(-(-numpy.diff(unit_off) // _FAR_CHUNK))]).astype(numpy.int64)
        U = int(unit_off[-1])
        uo, co, so = torch.from_numpy(numpy.stack([unit_off, self.cluster_off, chunk_off])).to(dev)  # one copy
        key = torch.empty(U, dtype=torch.int64, device=dev)
        centre = torch.empty((U, 4), dtype=torch.float32, device=dev)
        N.check(N.lib.cctamd_far_keys(_p(model.seg64), unit, _p(uo), model.ndesign, U, _p(key), _p(centre),
                                      _stream()), "cctamd_far_keys")
        perm = torch.sort(key, stable=True).indices
        per = int(N.lib.cctamd_far_coef_doubles(precision))

        def empty(n, dtype=torch.float64):
            return torch.empty(n, dtype=dtype, device=dev)

        self.rows = empty(6 * (C * 512 + 4)) if precision == 64 else None
        self.tiles = empty(C * 16, torch.int32) if precision != 64 else None
        self.geo, self.geo_large = empty(8 * C), empty(2 * C)
        self.coef, self.coef_large = empty(C * per), empty(C // 4 * per)
        mom = empty(2 * C * per // 4 * 3)
        N.check(N.lib.cctamd_far_build(precision, _p(model.seg64), unit, _p(centre), _p(uo), _p(so), int(chunk_off[-1]),
                                       _p(co), model.ndesign, C, _p(perm), _p(self.rows), _p(self.tiles),
                                       _p(self.geo), _p(self.geo_large), _p(mom), _p(self.coef),
                                       _p(self.coef_large), _stream()), "cctamd_far_build")


class DeviceModel:
    """D designs resident in HBM (FP64 segments, FP32 tiles, QS records, uniform fields)."""

    def __init__(self, specs: Sequence[DesignSpec], fp32: bool = True, align_cct: bool = False):
        """``align_cct`` starts every CCT on a tile boundary (needed by the adjoint,
        which attributes each tile to one CCT)."""
        dev = device()
        self.specs = list(specs)
        self.ndesign = D = len(self.specs)
        if D == 0:
            raise ValueError("no design given")
        self.align_cct = align_cct
        if align_cct:
            nseg = numpy.array([-(-int(s.raw_kl.shape[0]) // N.TILE) * N.TILE
                                + sum(-(-int(c) // N.TILE) * N.TILE for c in s.cct_counts)
                                for s in self.specs], numpy.int64)
        else:
            nseg = numpy.array([s.nseg for s in self.specs], numpy.int64)
        self.design_ntile = (nseg + N.TILE - 1) // N.TILE
        self.design_tile_off = numpy.concatenate([[0], numpy.cumsum(self.design_ntile)]).astype(numpy.int64)
        self.design_nseg = nseg
        S = int(self.design_tile_off[-1]) * N.TILE
        self.nseg_padded = S
        self.cluster_rows = int((-(-self.design_ntile // _LARGE_TILES)).sum()) * _LARGE_TILES * N.TILE
        self.nseg = int(nseg.sum())
        # pad segments: kl = 0 and a midpoint far from every field point
        seg64 = torch.zeros((max(S, 1), 8), dtype=torch.float64, device=dev)
        seg64[:, 4:7] = 1.0e3
        params, counts, dst, cct_design = [], [], [], []
        for d, s in enumerate(self.specs):
            row = int(self.design_tile_off[d]) * N.TILE
            nraw = int(s.raw_kl.shape[0])
            if nraw:
                rows = numpy.zeros((nraw, 8))
                rows[:, 0:3] = s.raw_kl
                rows[:, 4:7] = s.raw_m
                seg64[row:row + nraw] = torch.from_numpy(rows).to(dev)
                row += nraw
            for k in range(s.cct_params.shape[0]):
                c = int(s.cct_counts[k])
                if c == 0:
                    continue
                if align_cct:
                    row = -(-row // N.TILE) * N.TILE
                params.append(s.cct_params[k])
                counts.append(c)
                dst.append(row)
                cct_design.append((d, k))
                row += c
        self.ncct = len(params)
        self.cct_design = cct_design          # global CCT index -> (design, CCT index within the design)
        self.cct_dst = numpy.array(dst, numpy.int64)
        self.cct_counts = numpy.array(counts, numpy.int64)
        self.cct_params = numpy.array(params, numpy.float64).reshape(len(params), N.CCT_PARAMS)
        self._gen = None
        if self.ncct:
            prm = torch.from_numpy(numpy.ascontiguousarray(self.cct_params)).to(dev)
            off = torch.from_numpy(numpy.concatenate([[0], numpy.cumsum(counts)]).astype(numpy.int64)).to(dev)
            dsts = torch.from_numpy(self.cct_dst).to(dev)
            self._gen = (prm, off, dsts)
            N.check(N.lib.cctamd_winding_generate(_p(prm), _p(off), _p(dsts), self.ncct, int(sum(counts)),
                                                  _p(seg64), _stream()), "cctamd_winding_generate")
        self.seg64 = seg64
        self.seg32 = self.seg32k = self.tile_org = None
        if fp32:
            self.seg32 = torch.empty((max(S, 1), 8), dtype=torch.float32, device=dev)
            self.seg32k = torch.empty((max(S, 1), 12), dtype=torch.float32, device=dev)
            self.tile_org = torch.empty((max(S // N.TILE, 1), 4), dtype=torch.float64, device=dev)
            N.check(N.lib.cctamd_pack_fp32(_p(seg64), S, _p(self.seg32), _p(self.tile_org), _p(self.seg32k),
                                           _stream()), "cctamd_pack_fp32")
        qs = [s.qs for s in self.specs]
        nq = numpy.array([q.shape[0] for q in qs], numpy.int64)
        self.design_qs_off_host = numpy.concatenate([[0], numpy.cumsum(nq)]).astype(numpy.int64)
        allq = numpy.concatenate(qs).reshape(-1, 16) if nq.sum() else numpy.zeros((1, 16))
        self.qs = torch.from_numpy(numpy.ascontiguousarray(allq, dtype=numpy.float64)).to(dev)
        self.design_qs_off = torch.from_numpy(self.design_qs_off_host).to(dev)
        b = numpy.zeros((D, 4))
        for d, s in enumerate(self.specs):
            b[d, :3] = s.bconst
        self.bconst = torch.from_numpy(b).to(dev)
        self._plans: Dict[tuple, Plan] = {}
        self._far: Dict[int, FarField] = {}
        self._far_no_room: set = set()  # precisions whose clusters did not fit
        self._stream = torch.cuda.current_stream()  # that of the tensors above
        self._far_lock = threading.Lock()

    def __getstate__(self) -> dict:  # copies and pickles: everything but the stream and the lock
        return {k: v for k, v in self.__dict__.items() if k not in ("_stream", "_far_lock")}

    def __setstate__(self, state: dict) -> None:
        self.__dict__.update(state)
        self._stream = torch.cuda.current_stream()
        self._far_lock = threading.Lock()

    # --------------------------------------------------------- adjoint data
    def adjoint_data(self):
        """(seg_tan [T][33][8] f32, tile_cct [T] i32, cct_coef [ncct] f64) for cctamd_track_rk4_adjoint."""
        if not self.align_cct:
            raise ValueError("the adjoint needs a model built with align_cct=True")
        if getattr(self, "_adj", None) is None:
            dev = device()
            S = self.nseg_padded
            nt = max(S // N.TILE, 1)
            tan = torch.zeros((nt, N.TILE + 1, 8), dtype=torch.float32, device=dev)
            if self.ncct:
                prm, off, dsts = self._gen
                N.check(N.lib.cctamd_winding_tangents(_p(prm), _p(off), _p(dsts), self.ncct,
                                                      int(self.cct_counts.sum()), _p(tan), _stream()),
                        "cctamd_winding_tangents")
            tc = numpy.full(nt, -1, numpy.int32)
            for c in range(self.ncct):
                t0 = int(self.cct_dst[c]) // N.TILE
                t1 = -(-(int(self.cct_dst[c]) + int(self.cct_counts[c])) // N.TILE)
                tc[t0:t1] = c
            coef = self.cct_params[:, 19].copy() if self.ncct else numpy.zeros(1)
            self._adj = (tan, torch.from_numpy(tc).to(dev), torch.from_numpy(numpy.ascontiguousarray(coef)).to(dev))
        return self._adj

    # ------------------------------------------------------------- plans
    def plan(self, design_npt: Sequence[int], ppl: int = 2, target_items: Optional[int] = None) -> "Plan":
        npt = numpy.asarray(design_npt, numpy.int64)
        if npt.shape != (self.ndesign,):
            raise ValueError("one point count per design is required")
        if target_items is None:
            target_items = _TARGET_WG_PER_CU * cu_count()
        key = (tuple(npt.tolist()), ppl, target_items)
        if key in self._plans:
            return self._plans[key]
        pt_off = numpy.concatenate([[0], numpy.cumsum(npt)]).astype(numpy.int64)
        nt = numpy.ascontiguousarray(self.design_ntile, numpy.int64)
        toff = numpy.ascontiguousarray(self.design_tile_off[:-1], numpy.int64)
        n = N.lib.cctamd_plan(self.ndesign, _np(nt), _np(npt), _np(toff), _np(pt_off), ppl, target_items,
                              _MIN_TILES_PER_ITEM, None, None, None)
        if n < 0:
            N.check(int(n), "cctamd_plan")
        work = numpy.zeros((max(n, 1), N.WORK_INTS), numpy.int32)
        wbase = numpy.zeros(self.ndesign, numpy.int64)
        nchunk = numpy.zeros(self.ndesign, numpy.int32)
        n2 = N.lib.cctamd_plan(self.ndesign, _np(nt), _np(npt), _np(toff), _np(pt_off), ppl, target_items,
                               _MIN_TILES_PER_ITEM, _np(work), _np(wbase), _np(nchunk))
        if n2 != n:
            raise N.CctamdError(f"cctamd_plan: inconsistent work count {n2} != {n}")
        dev = device()
        p = Plan(ppl=ppl, nwork=int(n), work=torch.from_numpy(work).to(dev), wbase=torch.from_numpy(wbase).to(dev),
                 nchunk=torch.from_numpy(nchunk).to(dev), design_pt_off=torch.from_numpy(pt_off).to(dev),
                 npt=int(pt_off[-1]), design_npt=tuple(npt.tolist()))
        pb = points_per_block(ppl)
        blocks = -(-npt // pb)
        tiles = float((blocks * nt).sum())
        p.pairs, p.large = tiles * pb * N.TILE, tiles / max(float(blocks.sum()), 1.0) / _LARGE_TILES
        self._plans[key] = p
        return p

    # --------------------------------------------------------- far field
    def far_field(self, plan: Plan, precision: int, max_steps: int) -> Optional[Tuple[FarField, FarPlan]]:
        """The segment clusters that tracking ``plan`` for ``max_steps`` steps uses (0: one field
        evaluation) and their work items, kept in ``plan.far``; built on first need; None where every
        segment is summed."""
        if not self._far_pays(plan, precision, max_steps):
            return None
        key = precision if max_steps > 0 else (precision, 0)
        far, items = self._far.get(precision), plan.far.get(key)
        if far is not None and items is not None:
            return far, items
        if torch.cuda.is_current_stream_capturing():
            return None  # a capture cannot build them
        with self._far_lock:
            if precision in self._far_no_room:
                return None
            far, items = self._far.get(precision), plan.far.get(key)
            # On the model's own stream: they live as long as its segments, whichever stream tracks first (memory goes
            # back to the stream that it was taken on, which knows nothing of the others' launches).
            with torch.cuda.stream(self._stream):
                try:
                    if far is None:
                        far = FarField(self, precision)
                    if items is None:
                        items = self._far_plan(far, plan, precision, max_steps == 0)
                except torch.OutOfMemoryError:
                    # FP64 161 bytes per row of the clusters for good and 140 while they are built, FP32 38 and 46,
                    # beside 64 (FP32 144) of the segments.  Not tried again: equal calls give equal bits.
                    self._far_no_room.add(precision)
                    warnings.warn("not enough GPU memory for the segment clusters: this model sums every segment",
                                  RuntimeWarning, stacklevel=4)
                    return None
                self._stream.synchronize()  # ready for every stream that tracks this model
            self._far[precision], plan.far[key] = far, items
            return far, items

    def _far_pays(self, plan: Plan, precision: int, max_steps: int) -> bool:
        """Whether tracking ``plan`` for ``max_steps`` steps (0: one evaluation) is faster with the far
        field, its set-up (once per model) included: a function of the sizes alone, so that equal
        calls give equal bits."""
        rule = _FAR.get(precision)
        if rule is None or precision in self._far_no_room:
            return False
        if self.ndesign > 0x7fff or (precision == 33 and plan.ppl == -4):
            return False  # keys hold 15 bits of design; 16-point blocks of the FP32 path have no far-field kernel
        size = 0 if plan.ppl > 0 else 1
        large = rule["large"] if plan.pairs < rule["any_pairs"] else rule["any_large"][size]
        if plan.pairs < rule["pairs"][size] or plan.large < large or self.cluster_rows > _FAR_MOST_ROWS:
            return False
        saved = rule["saved"] if max_steps > 0 else _FAR_MAP_SAVED[plan.large >= 40]
        base, each = rule["setup"]
        return max(4 * max_steps, 1) * saved * plan.pairs / rule["rate"][size] > base + each * self.cluster_rows

    def _far_plan(self, far: FarField, plan: Plan, precision: int, single: bool) -> FarPlan:
        nt = numpy.ascontiguousarray(self.design_ntile, numpy.int64)
        npt = numpy.asarray(plan.design_npt, numpy.int64)
        pt_off = numpy.concatenate([[0], numpy.cumsum(npt)]).astype(numpy.int64)
        blocks = -(-npt // points_per_block(plan.ppl))
        tiles = blocks * nt
        target = far_items(int((blocks * -(-nt // 16)).sum()), bool(tiles.max() <= 1.05 * tiles.min()), single,
                           precision, plan.ppl, cu_count(), plan.nwork)
        while True:  # the caller's partial sums hold plan.nwork items (every point block has one)
            args = (self.ndesign, _np(nt), _np(npt), _np(far.cluster_off), _np(pt_off), plan.ppl)
            n = int(N.lib.cctamd_far_plan(*args, target, None, None, None))
            if n < 0:
                N.check(n, "cctamd_far_plan")
            if n <= plan.nwork or target == 1:
                break
            target = max(1, target - (n - plan.nwork))
        D = self.ndesign  # one buffer, one copy: offsets (8 bytes each), items, chunk counts
        buf = numpy.zeros(2 * D + N.WORK_INTS * max(n, 1) + D, numpy.int32)
        wbase, work, nchunk = buf[:2 * D], buf[2 * D:-D], buf[-D:]
        n2 = N.lib.cctamd_far_plan(*args, target, _np(work), _np(wbase), _np(nchunk))
        if n2 != n or n > plan.nwork:
            raise N.CctamdError(f"cctamd_far_plan: {n2} work items, {n} expected, {plan.nwork} at most")
        on = torch.from_numpy(buf).to(self.seg64.device)
        return FarPlan(n, on[2 * D:-D], on[:2 * D].view(torch.int64), on[-D:])

    def _track(self, plan: Plan, precision: int, state, kq, dt, nsteps, max_steps: int, scratch, partial, record,
               record_every: int, far_field: bool = True, of_steps: int = 0) -> None:
        """``of_steps``: the length of the track that these steps are the beginning of, for the choice of the sum."""
        far = self.far_field(plan, precision, max(max_steps, of_steps)) if far_field and max_steps > 0 else None
        self._call(N.lib.cctamd_track_rk4 if far is None else N.lib.cctamd_track_rk4_far, "cctamd_track_rk4", plan,
                   precision, far, _p(state), plan.npt, _p(kq), _p(dt), _p(nsteps), int(max_steps), _p(scratch),
                   _p(partial), _p(record), int(record_every))

    def tracked_field_tensors(self, plan: "Plan", precision: int, points: torch.Tensor, partial: torch.Tensor,
                              out: torch.Tensor, steps: int) -> None:
        """B (3, P) at device points (3, P) as the RK4 stages of a track of ``steps`` steps sum it: by the same
        launches, clusters included (``field_tensors`` chooses for one evaluation)."""
        far = self.far_field(plan, precision, steps) if steps > 0 else None
        self._call(N.lib.cctamd_bs_field if far is None else N.lib.cctamd_bs_field_far, "cctamd_bs_field", plan,
                   precision, far, _p(points), plan.npt, _p(partial), _p(out))

    def _map_far(self, plan: Plan, points: torch.Tensor) -> Optional[Tuple[torch.Tensor, FarField, FarPlan]]:
        """What the device found of the points (cctamd_point_spread) and the clusters with their work items for
        cctamd_bs_field_routed; None where every segment is summed.  Points in no order (a shuffled map, a raster
        across the magnet) have blocks that are close to every cluster: they are summed segment by segment, which
        the device finds out for every call, so that equal calls give equal bits; the host asks before it builds
        clusters (one wait, with the build's)."""
        built = 64 in self._far
        if not self._far_pays(plan, 64, 0) or (not built and torch.cuda.is_current_stream_capturing()):
            return None
        spread = self._point_spread(plan, points)
        if not built and self._spread_out(spread):
            return None
        far_field = self.far_field(plan, 64, 0)
        return None if far_field is None else (spread, *far_field)

    def _point_spread(self, plan: Plan, points: torch.Tensor) -> torch.Tensor:
        spread = torch.empty(2, dtype=torch.int64, device=points.device)
        N.check(N.lib.cctamd_point_spread(plan.ppl, _p(self.seg64), _p(plan.work), plan.nwork, _p(points), plan.npt,
                                          _p(spread), _stream()), "cctamd_point_spread")
        return spread

    @staticmethod
    def _spread_out(spread: torch.Tensor) -> bool:
        near, every = spread.tolist()
        return 3 * near > 2 * every  # spread_out in csrc/common.hpp

    def _call(self, function, name: str, plan: Plan, precision: int, far_field: Optional[Tuple[FarField, FarPlan]],
              *args, head: tuple = ()) -> None:
        """A library call on this segment set and plan, with its clusters where ``far_field`` gives them;
        ``head`` goes before."""
        seg, org, near = self._seg(precision)
        w = plan
        if far_field is not None:
            far, w = far_field
            head = (_p(far.geo), _p(far.geo_large), _p(far.coef), _p(far.coef_large), _p(far.tiles))
            seg = seg if far.rows is None else far.rows
        N.check(function(*head, precision, plan.ppl, _p(seg), _p(org), _p(near), _p(w.work), w.nwork, _p(w.wbase),
                         _p(w.nchunk), _p(plan.design_pt_off), self.ndesign, _p(self.qs), _p(self.design_qs_off),
                         _p(self.bconst), *args, _stream()), name)

    def _seg(self, precision: int):
        """(segment rows, tile origins, FP64 rows for near tiles) of a precision."""
        if precision == 64:
            return self.seg64, None, None
        if precision in (32, 33):
            if self.seg32 is None:
                raise ValueError("model was built without FP32 tiles")
            return (self.seg32 if precision == 32 else self.seg32k), self.tile_org, self.seg64
        raise ValueError("precision must be 32, 33 or 64")

    # ------------------------------------------------------------- field
    def field(self, points: numpy.ndarray, design_npt: Sequence[int], precision: int = 64,
              ppl: Optional[int] = None) -> numpy.ndarray:
        """B at points (P, 3) grouped by design (design_npt[d] consecutive rows each); ``ppl``
        defaults to the block shape that fits the largest design's point count."""
        pts = numpy.asarray(points, numpy.float64).reshape(-1, 3)
        if ppl is None:
            ppl = block_shape_for(design_npt, precision)
        plan = self.plan(design_npt, ppl)
        if plan.npt != pts.shape[0]:
            raise ValueError("point count does not match design_npt")
        if plan.npt == 0:
            return numpy.zeros((0, 3))
        dev = device()
        soa = torch.from_numpy(numpy.ascontiguousarray(pts.T)).to(dev)
        out = torch.empty_like(soa)
        partial = torch.empty(max(plan.nwork * 3 * points_per_block(ppl), 1), dtype=torch.float64, device=dev)
        self.field_tensors(plan, precision, soa, partial, out)
        return out.cpu().numpy().T.copy()

    # ---------------------------------------------------------- tracking
    def track(self, state: numpy.ndarray, kq: numpy.ndarray, dt: numpy.ndarray, nsteps: numpy.ndarray,
              design_npt: Sequence[int], precision: int = 64, ppl: Optional[int] = None,
              record: bool = False) -> Tuple[numpy.ndarray, Optional[numpy.ndarray]]:
        """RK4 tracking; state (P, 6) rows [x, y, z, vx, vy, vz] grouped by design.

        Returns the final state (P, 6) and, with ``record``, the state after
        every step as (max_steps+1, P, 6) (rows past a particle's own step
        count repeat nothing meaningful and are masked by the caller).  ``ppl``
        defaults to the block shape that fits the largest design's particle count.
        """
        st = numpy.asarray(state, numpy.float64).reshape(-1, 6)
        if ppl is None:
            ppl = block_shape_for(design_npt, precision)
        plan = self.plan(design_npt, ppl)
        if plan.npt != st.shape[0]:
            raise ValueError("particle count does not match design_npt")
        if plan.npt == 0:
            return st.copy(), None
        dev = device()
        ns = numpy.asarray(nsteps, numpy.int64)
        max_steps = int(ns.max()) if ns.size else 0
        soa = torch.from_numpy(numpy.ascontiguousarray(st.T)).to(dev)
        kq_t = torch.from_numpy(numpy.ascontiguousarray(kq, numpy.float64)).to(dev)
        dt_t = torch.from_numpy(numpy.ascontiguousarray(dt, numpy.float64)).to(dev)
        ns_t = torch.from_numpy(numpy.ascontiguousarray(ns)).to(dev)
        scratch = torch.empty((15, plan.npt), dtype=torch.float64, device=dev)
        partial = torch.empty(max(plan.nwork * 3 * points_per_block(ppl), 1), dtype=torch.float64, device=dev)
        rec = torch.empty((max_steps + 1, 6, plan.npt), dtype=torch.float64, device=dev) if record else None
        # particles all along the orbit have no use for the clusters; this call waits for the device anyway
        far = self._far_pays(plan, precision, max_steps) and not self._spread_out(self._point_spread(plan, soa))
        self._track(plan, precision, soa, kq_t, dt_t, ns_t, max_steps, scratch, partial, rec, 1, far_field=far)
        out = soa.cpu().numpy().T.copy()
        return out, (rec.cpu().numpy().transpose(0, 2, 1).copy() if rec is not None else None)

    # ------------------------------------------- device-resident variants
    def workspace(self, plan: "Plan") -> Tuple[torch.Tensor, torch.Tensor]:
        """(scratch [15][P], partial) device buffers for a plan."""
        dev = device()
        return (torch.empty((15, max(plan.npt, 1)), dtype=torch.float64, device=dev),
                torch.empty(max(plan.nwork * 3 * points_per_block(plan.ppl), 1), dtype=torch.float64, device=dev))

    def track_tensors(self, plan: "Plan", precision: int, state: torch.Tensor, kq: torch.Tensor, dt: torch.Tensor,
                      nsteps: torch.Tensor, max_steps: int, scratch: torch.Tensor, partial: torch.Tensor,
                      record: Optional[torch.Tensor] = None, record_every: int = 1) -> None:
        """In-place RK4 tracking of device-resident SoA state (6, P); nothing crosses PCIe."""
        self._track(plan, precision, state, kq, dt, nsteps, max_steps, scratch, partial, record, record_every)

    def field_tensors(self, plan: "Plan", precision: int, points: torch.Tensor, partial: torch.Tensor,
                      out: torch.Tensor) -> None:
        """B (3, P) at device points (3, P): Biot-Savart pass + fixed-order reduction + QS + uniform."""
        # a map pays for its clusters in one call; on the FP32 path a field keeps the terms of every segment
        routed = self._map_far(plan, points) if precision == 64 and plan.pairs > _FAR_MAP_PAIRS else None
        head: tuple = ()
        if routed is not None:
            spread, far, w = routed
            head = (_p(spread), _p(far.geo), _p(far.geo_large), _p(far.coef), _p(far.coef_large), _p(far.rows),
                    _p(w.work), w.nwork, _p(w.wbase), _p(w.nchunk))
        self._call(N.lib.cctamd_bs_field if routed is None else N.lib.cctamd_bs_field_routed, "cctamd_bs_field", plan,
                   precision, None, _p(points), plan.npt, _p(partial), _p(out), head=head)

    def bs_partial_tensors(self, plan: "Plan", precision: int, points: torch.Tensor, partial: torch.Tensor) -> None:
        """One launch of the split-K Biot-Savart kernel on device points (3, P)."""
        seg, org, near = self._seg(precision)
        N.check(N.lib.cctamd_bs_partial(precision, plan.ppl, _p(seg), _p(org), _p(near), _p(plan.work), plan.nwork,
                                        _p(points), plan.npt, _p(partial), _stream()), "cctamd_bs_partial")

    def segments64(self) -> numpy.ndarray:
        """The FP64 segment rows (S, 8) copied to the host (inspection and tests)."""
        return self.seg64.cpu().numpy()[: self.nseg_padded]


class TrackGraph:
    """One tracking pass (every RK4 step of a plan: 8 launches per step) captured
    once as a HIP graph and replayed.

    The graph binds the device buffers given here: refresh ``state`` in place
    (``state.copy_(initial)``) before each replay.  The captured launches hold
    no memset nodes and no host synchronisation.
    """

    def __init__(self, model: DeviceModel, plan: Plan, precision: int, state: torch.Tensor, kq: torch.Tensor,
                 dt: torch.Tensor, nsteps: torch.Tensor, max_steps: int, scratch: torch.Tensor,
                 partial: torch.Tensor):
        self.buffers = (state, kq, dt, nsteps, scratch, partial)  # kept alive with the graph
        self.model, self.plan = model, plan  # and the segments, clusters and work items that it reads
        model.far_field(plan, precision, max_steps)  # built before the capture, which cannot
        self.graph = torch.cuda.CUDAGraph()
        side = torch.cuda.Stream()  # default priority
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.graph(self.graph, stream=side):
            model.track_tensors(plan, precision, state, kq, dt, nsteps, max_steps, scratch, partial)
        torch.cuda.current_stream().wait_stream(side)

    def replay(self) -> None:
        self.graph.replay()


_CACHE: "collections.OrderedDict[bytes, DeviceModel]" = collections.OrderedDict()
_CACHE_SIZE = 8


def model_for(specs: Sequence[DesignSpec], fp32: bool = True, align_cct: bool = False) -> DeviceModel:
    """DeviceModel for the given designs, reused while the magnet parameters are unchanged."""
    h = hashlib.sha1()
    for s in specs:
        h.update(s.key())
    h.update(b"fp32" if fp32 else b"fp64")
    h.update(b"aligned" if align_cct else b"packed")
    k = h.digest()
    m = _CACHE.get(k)
    if m is not None:
        _CACHE.move_to_end(k)
        return m
    m = DeviceModel(specs, fp32=fp32, align_cct=align_cct)
    _CACHE[k] = m
    while len(_CACHE) > _CACHE_SIZE:
        _CACHE.popitem(last=False)
    return m


def model_from_segments(kl: numpy.ndarray, m: numpy.ndarray, fp32: bool = True) -> DeviceModel:
    """A one-design model from raw global-frame current elements kl (n, 3) and midpoints m (n, 3)."""
    spec = DesignSpec(raw_kl=numpy.ascontiguousarray(kl, numpy.float64).reshape(-1, 3),
                      raw_m=numpy.ascontiguousarray(m, numpy.float64).reshape(-1, 3))
    return model_for([spec], fp32=fp32)


def rk4_steps(length: float, footstep: float, speed: float) -> Tuple[int, float]:
    """Step count and time step of one particle, exactly as the reference computes them
    (final_code/packages/particles.py:585-587 and base_utils.py:284-285)."""
    dt = footstep / speed
    t_end = length / speed
    number = math.ceil((t_end - 0.0) / dt)
    return number, (t_end - 0.0) / float(number)


def winding_points(params: numpy.ndarray, npoints: int) -> numpy.ndarray:
    """Local-frame path points of one CCT (npoints, 3) generated on the GPU."""
    dev = device()
    prm = torch.from_numpy(numpy.ascontiguousarray(params, numpy.float64)).to(dev)
    out = torch.empty((max(npoints, 1), 3), dtype=torch.float64, device=dev)
    N.check(N.lib.cctamd_winding_points(_p(prm), npoints, _p(out), _stream()), "cctamd_winding_points")
    return out.cpu().numpy()[:npoints]
