"""Window deposits of more tiles than there are CUs, whose positions are read
again for every filling or kept in registers: two workgroups a CU, one (double
sums, windows of 32 cells, larger tiles), one and two grids, and a point whose
fixed-point sum wraps.  The double sums and the smaller grids are compared with
the oracle; a CIC weight of a float grid may differ from its by an ulp of the
scaled coordinate, so the larger grids (and the point, where such differences
add up) are compared with the double sums of the same weights."""

import numpy as np
import pytest

from oracle import pipeline as O
from exshalos_amd.lib import _native as N
from exshalos_amd.lib import set_precision
from exshalos_amd.lib import spectrum as SP

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,nl,nd,window,il,mass,tile,point", [
    (4, 112, 112, 2, 1, False, 16, True),    # 343 tiles, two workgroups a CU
    (4, 112, 112, 5, 0, False, 16, False),
    (4, 112, 168, 5, 0, False, 16, False),   # windows of 32 cells
    (4, 112, 112, 2, 0, True, 16, False),    # double sums
    (8, 112, 112, 2, 0, False, 16, False),
    (8, 112, 112, 5, 1, False, 16, False),   # kept: two grids
    (4, 128, 128, 2, 1, False, 3216, False),
    (4, 160, 160, 2, 0, False, 3216, False),
    (4, 64, 64, 2, 1, False, 32, False),
    (4, 192, 192, 2, 0, False, 32, True),
    (4, 192, 192, 2, 1, False, 32, False),
])
def test_matches_the_reference(prec, nl, nd, window, il, mass, tile, point):
    set_precision(prec)
    RT = np.float32 if prec == 4 else np.float64
    rng = np.random.default_rng(nl + window)
    L = 100.0
    a = (np.arange(nl) + 0.5) * (L / nl)
    x = np.stack(np.meshgrid(a, a, a, indexing="ij"), -1).reshape(-1, 3)
    x += rng.normal(0, 0.7 * L / nl, x.shape)
    if point:
        x[:3000] = (0.3 * L / nl, 0.2 * L / nl, 5.1 * L / nl)
    x = np.mod(x, L).astype(RT)
    x[x >= L] = 0
    w = rng.uniform(0.5, 2.0, len(x)).astype(RT) if mass else None
    ctx, lib = N.context(), N.load()

    def grid(tile, acc):
        N.check(lib.exh_ctx_set_tunable(ctx, N.TUNE_DEPOSIT_TILE, tile))
        N.check(lib.exh_ctx_set_tunable(ctx, N.TUNE_DEPOSIT_ACC, acc))
        try:
            return SP.grid_compute(x, None, w, int(mass), None, 1, nd, L, 0.31, 0.5, -1, window,
                                   4.0, 5.0, il, 1, 0, 1)
        finally:
            N.check(lib.exh_ctx_set_tunable(ctx, N.TUNE_DEPOSIT_TILE, 0))
            N.check(lib.exh_ctx_set_tunable(ctx, N.TUNE_DEPOSIT_ACC, 0))

    g = grid(tile, 0)
    if point or (window == 2 and nd > 128):
        ref = grid(16, 8).astype(np.float64)
    else:
        ref = O.grid_compute(x, nd, L, window=window, interlacing=bool(il), mass=w, Om0=0.31,
                             z=0.5, precision=prec)
    d = np.max(np.abs(g.astype(np.float64) - ref)) / np.max(np.abs(ref))
    assert d < (2e-5 if prec == 4 else 1e-12)
