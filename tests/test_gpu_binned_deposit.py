"""Binned deposit of particles in no order against the oracle: grid sides that
the tiles divide and that they do not, one tile, every window, weights, types,
redshift space, particles on the box's faces, and a clump of more particles
than one workgroup sums (its tile is summed in parts)."""

import numpy as np
import pytest

from oracle import pipeline as O
from exshalos_amd.lib import set_precision
from exshalos_amd.lib import spectrum as SP

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [4, 8])
@pytest.mark.parametrize("nd,window,il,mass,ntype,rsd,clump", [
    (64, 2, 1, False, 1, False, 0),
    (50, 2, 1, True, 1, True, 0),       # tiles of 12 and 13 cells
    (34, 5, 1, False, 2, False, 0),
    (130, 5, 0, True, 1, False, 0),     # 9 tiles an axis
    (9, 2, 1, False, 1, False, 0),      # one tile
    (48, 1, 1, False, 3, True, 0),
    (32, 2, 1, False, 1, False, 60000),
    (40, 5, 1, True, 1, False, 40000),
])
def test_matches_the_oracle(prec, nd, window, il, mass, ntype, rsd, clump):
    set_precision(prec)
    RT = np.float32 if prec == 4 else np.float64
    rng = np.random.default_rng(nd + window)
    n = 600000 if window == 1 else 140000  # past the fewest atomics binned for
    L = 200.0
    pos = rng.uniform(0, L, (n, 3))
    pos[:50] = 0.0
    pos[50:100, 1] = np.nextafter(RT(L), RT(0))
    if clump:
        pos[1000:1000 + clump] = (L / 2, L / 3, 0.2) + rng.normal(0, 0.05, (clump, 3))
    pos = np.mod(pos, L).astype(RT)
    pos[pos >= L] = 0
    w = rng.uniform(0.5, 2.0, n).astype(RT) if mass else None
    t = rng.integers(0, ntype, n).astype(np.int32) if ntype > 1 else None
    vel = rng.normal(0, 300.0, (n, 3)).astype(RT) if rsd else None
    direction = 2 if rsd else -1
    ref = O.grid_compute(pos, nd, L, window=window, interlacing=bool(il), mass=w, types=t,
                         ntype=ntype, direction=direction, vel=vel, Om0=0.31, z=0.5,
                         precision=prec)
    g = SP.grid_compute(pos, vel, w, int(mass), t, ntype, nd, L, 0.31, 0.5, direction, window,
                        4.0, 5.0, il, 1, 0, 1)
    assert g.shape == ref.shape
    d = np.max(np.abs(g.astype(np.float64) - ref)) / np.max(np.abs(ref))
    assert d < (2e-5 if prec == 4 else 1e-12)
