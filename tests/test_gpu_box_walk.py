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
