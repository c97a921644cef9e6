"""The group walk's traversal, source window and pair table at their edges.

Listed sources within r_cut of the group box fill a window of 64 that is
evaluated when full; groups clear of the box faces skip the image; the pair
table lies in LDS up to 384 cells (r_cut up to 4.9 a) and in memory beyond; open
nodes are expanded eight at a time, one at a time from 96 on (leaves of one
source and a fine tree open the most). Counters equal the oracle's and forces
agree to 1e-12 (the bounds of test_gpu_group_walk.py).
"""
from __future__ import annotations

import numpy as np
import pytest

from helpers import adaptive_struct, options_struct
from test_gpu_group_walk import check_against_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,leaf,size,ratio", [(1, 16, 0, 4.5), (65, 1, 0, 4.5), (700, 16, 0, 5.5), (700, 16, 32, 4.5),
                                               (2500, 1, 16, 4.5), (2500, 1, 0, 5.5), (3000, 200, 0, 4.5),
                                               (3000, 8, 64, 4.9)])
def test_group_walk_matches_oracle_at_its_edges(n, leaf, size, ratio):
    rng = np.random.default_rng(n + leaf)
    x, y, z = rng.uniform(0.0, 10.0, (3, n))
    m = rng.uniform(0.5, 1.5, n)
    o = options_struct(10.0, eps=0.01, leaf=leaf, rcut_cells=ratio * 1.25)
    o.acceptance_policy = 1
    _, c = check_against_oracle(x, y, z, m, o, adaptive_struct(group_size=size), previous=np.full(n, 3.0))
    assert c["group_walk_grouped_targets"] == n
