"""The octree build at the sizes where its passes can go wrong.

Nodes are found from the digits that sorted keys share, in blocks of 512
particles with a window of max_leaf_size keys around each; leaves are ordered
and summed 16, 32 or 64 lanes to a leaf (larger ones by a whole wave); moments
run in subtrees of at most max(512, n / 1024) particles and then the nodes
above them; a build sorts as many digits as the coordinator's last one needed.
Every tree equals the oracle's bit for bit (no tolerance).
"""
from __future__ import annotations

import time

import numpy as np
import pytest

from helpers import empty_dev, options_struct, to_dev
from oracle import oracle as O
from test_oracle_pins import clustered

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover - GPU-only module
    pytest.skip("no HIP device", allow_module_level=True)

from cosmosim import ForceAccumulator, TreePmCoordinator  # noqa: E402

BOX = 10.0


def uniform(n):
    p = np.random.default_rng(n).uniform(0.0, BOX, (3, n))
    m = np.random.default_rng(n + 1).uniform(0.5, 1.5, n)
    m[::5] = 0.0  # leaves and nodes without mass keep their cell's centre
    m[0] = 1.0
    return p[0], p[1], p[2], m


def tight(n, width):
    x, y, z, m = uniform(n)
    p = np.random.default_rng(7).normal(0.0, width * BOX, (3, 40)) + np.array([[1.2], [3.4], [0.9]])
    x[:40], y[:40], z[:40] = p
    return x, y, z, m


def coincident(n, distinct):
    # points at `distinct` places about 1e-13 apart: one leaf at the smallest cell
    rng = np.random.default_rng(n)
    p = 2.0 + 1e-13 * rng.integers(0, distinct, (3, n)) if distinct > 1 else np.full((3, n), 2.0)
    return p[0].copy(), p[1].copy(), p[2].copy(), rng.uniform(0.5, 1.5, n)


def check_tree(coord, sources, leaf):
    x, y, z, m = sources
    acc = tuple(empty_dev(x.size, torch.float64) for _ in range(3))
    o = options_struct(BOX, eps=0.02, leaf=leaf)
    diag = coord.solve_active_set(*to_dev(x, y, z, m), ForceAccumulator(acc), o, want_diagnostics=True).diagnostics
    torch.cuda.synchronize()
    tree = coord.tree_arrays()
    ref = O.build_tree(*(O.unwrap_axis(c, BOX)[0] for c in (x, y, z)), m, leaf, True, 0.02)
    for name in ("order", "begin", "count", "child_index", "geometry", "moments"):
        assert np.array_equal(tree[name], ref[name]), name
    assert diag["node_count"] == ref["count"].size
    assert diag["leaf_count"] == int(np.all(ref["child_index"] == 0xFFFFFFFF, axis=1).sum())


def check_build_only(coord, sources):
    acc = tuple(empty_dev(1, torch.float64) for _ in range(3))
    active = to_dev(np.zeros(1, np.int32))[0]
    o = options_struct(BOX, eps=0.02, leaf=16)
    o.short_range_only = 1
    coord.solve_active_set_with_pm_cadence(*to_dev(*sources), ForceAccumulator(acc, active), o, False)
    coord.synchronize()


@pytest.mark.parametrize("n,leaf", [(1, 16), (2, 1), (511, 16), (512, 16), (513, 17), (1025, 32), (1200, 33),
                                    (1030, 64), (1500, 65), (2500, 1), (3000, 300), (5000, 1024), (20000, 3)])
def test_tree_matches_oracle(n, leaf):
    with TreePmCoordinator((16, 16, 16)) as coord:
        check_tree(coord, uniform(n), leaf)


def test_rebuilds_of_changing_depth_match_oracle():
    with TreePmCoordinator((16, 16, 16)) as coord:
        for sources in (uniform(700), tight(3000, 2.0**-15), uniform(200), tight(3000, 2.0**-18), uniform(5000),
                        clustered(4000, 3, BOX)):
            check_tree(coord, sources, 16)


@pytest.mark.parametrize("n,distinct", [(65, 1), (70, 3), (2000, 4), (40000, 1)])
def test_leaf_at_the_smallest_cell_matches_oracle(n, distinct):
    with TreePmCoordinator((16, 16, 16)) as coord:
        sources = coincident(n, distinct)
        check_tree(coord, sources, 16)
        # a leaf holds any number of coincident sources; ordering it takes no
        # time that grows with their square (40000 would take seconds)
        start = time.perf_counter()
        check_build_only(coord, sources)
        assert time.perf_counter() - start < 1.0


@pytest.mark.parametrize("n", [(1 << 21) - 3, (1 << 21) + 5])
def test_tree_on_both_sides_of_the_device_frame(n):
    # up to 2^21 sources the build's frame stays on the device, beyond it is read back
    with TreePmCoordinator((96, 96, 96)) as coord:
        check_tree(coord, uniform(n), 16)
