"""Tracers whose position is not finite before or after the redshift-space
shift are left out of the grid and of its mean, in every deposit kernel: the
grid equals the oracle's of the same catalogue without them."""

import numpy as np
import pytest

from oracle import pipeline as O
from exshalos_amd.lib import set_precision
from exshalos_amd.lib import spectrum as SP

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [4, 8])
@pytest.mark.parametrize("n,nd,window,il,mass", [
    (3000, 16, 2, 1, False),       # global atomics
    (140000, 32, 2, 1, False),     # binned by tiles
    (140000, 32, 5, 0, True),
    (32**3, 32, 2, 1, False),      # windows of a lattice's tiles
    (16**3, 16, 2, 1, False),      # one tile, no room for a window's margin
    (500, 16, 3, 1, False),        # spherical window
])
def test_non_finite_tracers_are_left_out(prec, n, nd, window, il, mass):
    set_precision(prec)
    RT = np.float32 if prec == 4 else np.float64
    rng = np.random.default_rng(n + nd)
    L = 100.0
    pos = rng.uniform(0, L, (n, 3)).astype(RT)
    pos[pos >= L] = 0
    vel = rng.normal(0, 300.0, (n, 3)).astype(RT)
    w = rng.uniform(0.5, 2.0, n).astype(RT) if mass else None
    bad = rng.permutation(n)[:60]
    pos[bad[:10], 2] = np.nan
    pos[bad[10:20], 2] = np.inf
    pos[bad[20:30], 0] = -np.inf
    vel[bad[30:40], 2] = np.nan
    vel[bad[40:50], 2] = np.inf
    vel[bad[50:60], 2] = -np.inf
    good = np.ones(n, bool)
    good[bad] = False
    ref = O.grid_compute(pos[good], nd, L, window=window, interlacing=bool(il),
                         mass=w[good] if mass else None, direction=2, vel=vel[good], Om0=0.31,
                         z=0.5, R=8.0, precision=prec)
    g = SP.grid_compute(pos, vel, w, int(mass), None, 1, nd, L, 0.31, 0.5, 2, window, 8.0, 5.0,
                        il, 1, 0, 1)
    d = np.max(np.abs(g.astype(np.float64) - ref)) / np.max(np.abs(ref))
    assert d < (2e-5 if prec == 4 else 1e-12)
