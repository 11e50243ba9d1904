"""Positions far outside the box: the periodic wrap ends for every finite value
and the mass of the grid is conserved, in any order and in lattice order."""

import numpy as np
import pytest

from exshalos_amd.lib import set_precision
from exshalos_amd.lib import spectrum as SP

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [4, 8])
@pytest.mark.parametrize("n", [5000, 32**3])
def test_huge_positions_end_in_the_box(prec, n):
    set_precision(prec)
    RT = np.float32 if prec == 4 else np.float64
    L, nd = 100.0, 32
    rng = np.random.default_rng(2)
    pos = rng.uniform(0, L, (n, 3)).astype(RT)
    big = np.finfo(RT).max
    far = [big, -big, big / 3, 1e30, -1e30, 1e20, -3.3e17, 1e12, 7.7e9, -1e9, 5 * L, -4 * L]
    pos[: len(far), 0] = np.array(far, dtype=RT)
    pos[20: 20 + len(far), 2] = np.array(far, dtype=RT)
    w = np.ones(n, dtype=RT)
    g = SP.grid_compute(pos, None, w, 1, None, 1, nd, L, 0.31, 0.0, -1, 2, 4.0, 5.0, 1, 1, 0, 1)
    for s in range(2):
        assert abs(g[0, s].astype(np.float64).sum() - n) < 1e-5 * n
