"""Deposit of lattice particles through the tiles' windows against the oracle:
tiles of 8, 16 and 24 cells, windows that nearly fill the box, bulk flows past
the box's edge, particles far from their tile, a collapse onto few tiles, and
one onto a point (fixed-point sums that wrap)."""

import numpy as np
import pytest

from oracle import pipeline as O
from exshalos_amd.lib import set_precision
from exshalos_amd.lib import spectrum as SP

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [4, 8])
@pytest.mark.parametrize("nl,nd,window,il,mass,motion", [
    (32, 32, 2, 1, False, "flow"),      # nd = 2 W: windows of 24 cells in 32
    (32, 16, 2, 1, False, "flow"),      # W = 8
    (48, 72, 5, 1, False, "flow"),      # W = 24
    (48, 48, 5, 0, True, "stray"),
    (48, 48, 1, 1, False, "stray"),
    (80, 80, 2, 1, False, "collapse"),  # 125 windows over the tiles in the middle
    (80, 80, 2, 0, True, "collapse"),
    (32, 32, 2, 1, False, "point"),
])
def test_matches_the_oracle(prec, nl, nd, window, il, mass, motion):
    set_precision(prec)
    RT = np.float32 if prec == 4 else np.float64
    rng = np.random.default_rng(nl + nd)
    L = 100.0
    q = (np.stack(np.meshgrid(*[np.arange(nl) + 0.5] * 3, indexing="ij"), -1) * (L / nl)).reshape(-1, 3)
    x = q + rng.normal(0, 0.7 * L / nl, q.shape)
    if motion == "flow":
        x += (0.37 * L, -0.61 * L, 0.05 * L)
    if motion == "stray":
        k = rng.integers(0, len(x), len(x) // 50)
        x[k] = rng.uniform(0, L, (len(k), 3))
        x[0] = np.nan
    if motion == "collapse":
        x = L / 2 + 0.3 * (x - L / 2)
    if motion == "point":
        x[: len(x) // 2] = (L / 2, L / 3, 0.01)
    x = np.mod(x, L).astype(RT)
    x[x >= L] = 0
    w = rng.uniform(0.5, 2.0, len(x)).astype(RT) if mass else None
    # 16384 particles in one cell: the oracle's own FP32 sum drifts by 1.6e-4
    op = 8 if motion == "point" else prec
    ref = O.grid_compute(x[1:] if motion == "stray" else x, nd, L, window=window,
                         interlacing=bool(il),
                         mass=w[1:] if mass and motion == "stray" else w, types=None, ntype=1,
                         direction=-1, vel=None, Om0=0.31, z=0.5, precision=op)
    g = SP.grid_compute(x, None, w, int(mass), None, 1, nd, L, 0.31, 0.5, -1, window, 4.0, 5.0,
                        il, 1, 0, 1)
    assert g.shape == ref.shape
    d = np.max(np.abs(g.astype(np.float64) - ref)) / np.max(np.abs(ref))
    assert d < (2e-5 if prec == 4 else 1e-12)
