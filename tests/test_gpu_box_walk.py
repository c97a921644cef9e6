"""The box-classified walks at the sizes where their splits can go wrong.

The timed strict walks cut a wave's targets into segments that fit a box, share
each segment's targets and source slices among the lanes, expand leaves in
batches of 64 sources and evaluate windows of staged records. Each case here is
compared with the counting walk of the same precision (lane by lane over the
whole tree, no boxes, no windows): the same pairs and multipoles in another
order, so the short-range lanes agree to the rounding of the sums (FP32 2e-6,
FP64 1e-12; the bounds of test_gpu_target_mapping.py). Sizes around a wave and
a segment, leaves of one source and of several batches, active sets whose
neighbours in visit order lie far apart (single-target segments), accepted
multipoles, and a cutoff so close to half the box that no box frame exists.
"""
from __future__ import annotations

import numpy as np
import pytest

from helpers import options_struct, rel_l2, to_dev

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover - GPU-only module
    pytest.skip("no HIP device", allow_module_level=True)

from cosmosim import ForceAccumulator, TreePmCoordinator  # noqa: E402
from cosmosim import _lib as L  # noqa: E402
from test_oracle_pins import clustered  # noqa: E402


def short_range(x, y, z, m, o, mesh, active, counted):
    dt = torch.float32 if o.precision == L.PRECISION_MIXED else torch.float64
    dev = to_dev(x, y, z, m)
    na = x.size if active is None else active.size
    acc = tuple(torch.zeros(na, dtype=dt, device="cuda:0") for _ in range(3))
    sr = tuple(torch.zeros(x.size, dtype=dt, device="cuda:0") for _ in range(3))
    act = None if active is None else to_dev(active.astype(np.uint32).view(np.int32))[0]
    torch.cuda.synchronize()
    with TreePmCoordinator(mesh) as coord:
        coord.solve_active_set_with_pm_cadence(*dev, ForceAccumulator(acc, act, None, sr), o, False,
                                               want_diagnostics=counted)
        coord.synchronize()
    return np.stack([s.double().cpu().numpy() for s in sr])


def uniform(n, box, seed):
    p = np.random.default_rng(seed).uniform(0.0, box, (3, n))
    return p[0], p[1], p[2], np.random.default_rng(seed + 1).uniform(0.5, 1.5, n)


CASES = [(f"n{n}_leaf{leaf}", uniform(n, 10.0, n), 10.0, dict(eps=0.02, leaf=leaf), 16, None)
         for n, leaf in ((1, 16), (2, 1), (63, 1), (64, 16), (65, 16), (257, 4), (1000, 300), (4097, 1))]
CASES += [
    # neighbours in visit order far apart: segments of one target, waves of few
    ("sparse_active", uniform(5000, 20.0, 3), 20.0, dict(eps=0.01), 32, 41),
    ("unsoftened", uniform(700, 10.0, 4), 10.0, dict(eps=0.0), 16, None),
    ("multipoles", clustered(9000, 8, 20.0), 20.0, dict(eps=0.005, theta=0.7), 32, 3),
    # r_cut = 0.4999 L: no target has a box frame
    ("cutoff_near_half_box", uniform(600, 10.0, 5), 10.0, dict(eps=0.02, rcut_cells=7.998), 16, None),
]


@pytest.mark.parametrize("precision", [L.PRECISION_FP64, L.PRECISION_MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_box_walk_matches_counting_walk(case, precision):
    _, (x, y, z, m), box, kw, mesh, stride = case
    rcut = kw.pop("rcut_cells", None) if "rcut_cells" in kw else None
    o = options_struct(box, **kw)
    if rcut is not None:
        kw["rcut_cells"] = rcut
        o.rcut_cells = rcut
    o.precision = precision
    o.target_mapping = L.TARGETS_PER_LANE
    o.short_range_only = 1
    active = None if stride is None else np.arange(0, x.size, stride)
    timed = short_range(x, y, z, m, o, mesh, active, False)
    counted = short_range(x, y, z, m, o, mesh, active, True)
    assert np.all(np.isfinite(timed))
    rest = np.ones(x.size, bool)
    rest[slice(None) if active is None else active] = False
    assert np.all(timed[:, rest] == 0.0)
    if np.linalg.norm(counted) == 0.0:
        assert np.all(timed == 0.0)
    else:
        assert rel_l2(timed, counted) < (2e-6 if precision == L.PRECISION_MIXED else 1e-12)


# ---- large boxes: L / r_cut in the hundreds and thousands ----------------------
# Node boxes are tested in FP32 differences of 32-bit fixed point, which round
# by up to 64 units at separations of a quarter box; r_cut is 2^32 / (L / r_cut)
# units. The sources below are a chain along x cut by the root's centre plane
# just inside r_cut of the target, so that the half beyond the plane is one leaf
# whose nearest source is the pair at r_cut, and the positions are drawn until
# rounded_excess, the arithmetic of that test, puts the leaf beyond
# r_cut (1 + 5e-6): a margin that does not cover the rounding loses the pair.
CHAIN = 1200
INSIDE = 1e-6  # the pair lies at r_cut (1 - INSIDE): both precisions count it


def float_up(x):
    f = np.float32(x)
    return np.where(f.astype(np.float64) < x, np.nextafter(f, np.float32(np.inf)), f)


def rounded_excess(target, first, last, L, cubic, half_units):
    """Separation of a leaf [first, last] and a target along x in the kernel's
    FP32 steps, lengths in the separation unit (fixed point, or L / 2^32)."""
    scale = 4294967296.0 / L
    d = np.floor(0.5 * (first + last) * scale).astype(np.int64) - np.floor(target * scale).astype(np.int64)
    half = 0.5 * (last - first)
    unit = np.float32(1.0 if cubic else L / 4294967296.0)
    hx = float_up(half * scale + 2.0) if cubic else float_up(half + 2.0 / scale)
    return (np.abs(d.astype(np.float32) * unit) - hx) - np.float32(half_units) * unit


def boundary_chain(ratio, L, cubic, half_units):
    """x of the chain (its target is particle CHAIN // 2 - 1) and r_cut."""
    rng = np.random.default_rng(int(ratio))
    for _ in range(400):
        rc = L / (ratio * (1.0 + 0.01 * rng.random()))
        lo = 1e-4 * L * rng.random(4096)
        hi = L * (1.0 - 1.6 / CHAIN) + lo * rng.random(4096)
        target = 0.5 * (lo + hi) - rc * rng.uniform(0.45, 0.55, 4096)
        first = target + rc * (1.0 - INSIDE)
        sep = L / 4294967296.0 if cubic else 1.0
        e = rounded_excess(target, first, hi, L, cubic, half_units)
        lost = np.flatnonzero(e.astype(np.float64) * sep > rc * (1.0 + 5.5e-6))
        if lost.size:
            k = lost[0]
            n = CHAIN // 2
            left = np.linspace(lo[k], target[k] - 0.3 * rc, n - 2)
            right = np.linspace(first[k] + 0.3 * rc, hi[k], n - 1)
            # one source before the centre, so that the widest gap is the wrap
            mid = 0.5 * (lo[k] + hi[k]) - 0.01 * rc
            return np.concatenate([left, [mid, target[k], first[k]], right]), rc
    raise AssertionError("no separation where the rounding shows")


@pytest.mark.parametrize("ratio", [500, 2000])
@pytest.mark.parametrize("box", [(1.0, 1.0, 1.0), (1.3, 1.3, 0.8)], ids=["cubic", "slab"])
def test_pairs_just_inside_the_cutoff_of_a_large_box(box, ratio):
    cubic = len(set(box)) == 1
    mesh = 32
    for precision, half_units in ((L.PRECISION_FP64, 4.000004), (L.PRECISION_MIXED, 2.0)):
        x, rc = boundary_chain(ratio, box[0], cubic, half_units)
        y, z = np.full(CHAIN, 0.4 * box[1]), np.full(CHAIN, 0.3 * box[2])
        m = np.random.default_rng(3).uniform(0.5, 1.5, CHAIN)
        o = options_struct(box, eps=0.0, leaf=1024, rcut_cells=rc / (np.cbrt(box[0] * box[1] * box[2]) / mesh))
        o.target_mapping = L.TARGETS_PER_LANE
        o.short_range_only = 1
        target = CHAIN // 2 - 1
        active = np.array([target])
        o.precision = L.PRECISION_FP64
        ref = short_range(x, y, z, m, o, mesh, active, True)[:, target]
        o.precision = precision
        # FP32 pairs and fixed-point positions: 1e-4 of this target's few pairs
        # is far below the lost pair's share
        bound = 1e-12 if precision == L.PRECISION_FP64 else 1e-4
        for counted in (False, True):
            got = short_range(x, y, z, m, o, mesh, active, counted)[:, target]
            assert np.linalg.norm(got - ref) < bound * np.linalg.norm(ref), (precision, counted)


def test_window_fill_lies_beyond_every_target():
    # two targets L / 10 apart share a wave's origin halfway between them; the
    # records that fill a window past its sources must lie beyond r_cut of
    # both, wherever r_cut = L / 1280 puts them: neither has a pair
    box, mesh = 1.0, 32
    rc = box / 1280
    for cells in (60.0, 64.2, 70.0):
        p = np.array([0.5 - cells * rc, 0.5 + cells * rc])
        for eps in (0.0, 0.01 * rc):
            o = options_struct(box, eps=eps, rcut_cells=mesh / 1280)
            o.precision = L.PRECISION_MIXED
            o.target_mapping = L.TARGETS_PER_LANE
            o.short_range_only = 1
            assert np.all(short_range(p, p, p, np.ones(2), o, mesh, None, False) == 0.0), (cells, eps)


# ---- above 2^20 sources: the segment's own origin ------------------------------
@pytest.mark.parametrize("kind", ["uniform", "clustered", "slab"])
@pytest.mark.parametrize("stride", [None, 1001], ids=["all", "sparse"])
def test_mixed_walk_above_2_20_sources_matches_counting_walk(kind, stride):
    # a ragged count, spread masses; clusters give waves whose segments are
    # halved, windows that overflow and last windows that are filled up
    n = (1 << 20) + 4097
    box = (60.0, 90.0, 120.0) if kind == "slab" else (100.0, 100.0, 100.0)
    rng = np.random.default_rng(11)
    p = rng.uniform(0.0, 1.0, (3, n))
    if kind == "clustered":
        c = rng.uniform(0.0, 1.0, (3, 200))
        k = n // 4
        p[:, :k] = np.mod(c[:, rng.integers(0, 200, k)] + rng.normal(0.0, 3e-3, (3, k)), 1.0)
    x, y, z = (np.minimum(p[a] * box[a], np.nextafter(box[a], 0.0)) for a in range(3))
    m = rng.uniform(0.5, 1.5, n)
    mesh = 128
    o = options_struct(box, G=1.0, eps=0.1)  # close pairs soft: their separations round differently
    o.precision = L.PRECISION_MIXED
    o.target_mapping = L.TARGETS_PER_LANE
    o.short_range_only = 1
    active = None if stride is None else np.arange(0, n, stride)
    timed = short_range(x, y, z, m, o, mesh, active, False)
    counted = short_range(x, y, z, m, o, mesh, active, True)
    # The sums' order differs (FP32, the 2e-6 above), and a pair whose
    # separation rounds across r_cut is counted by one walk only, with 1.8e-2
    # of Newton's force: a share 3 d of a target's pairs for a relative rounding
    # d. Offsets of some r_cut round by 2^-24 of themselves in each walk, so d is
    # about 1e-7 (one pair in 7e6 differs at these counts); one in 2.6e6 is allowed.
    rc = 4.5 * 1.25 * np.cbrt(np.prod(box)) / mesh
    targets = n if active is None else active.size
    pairs = targets * n / np.prod(box) * 4.0 / 3.0 * np.pi * rc**3 * (4.0 if kind == "clustered" else 1.0)
    flips = np.sqrt(1.0 + pairs / 2.6e6) * 1.5 * 1.8e-2 / rc**2
    assert np.all(np.isfinite(timed))
    err, norm = np.linalg.norm(timed - counted), np.linalg.norm(counted)
    assert err < 2e-6 * norm + flips
