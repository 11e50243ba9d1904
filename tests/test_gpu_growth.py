"""Growth rounds against the CPU oracle where their phases meet: halos of
one cell (one thread), of a few shells and of thousands of cells (a row of 16
lanes; shells of more than 64 cells and offsets past the 1024 kept in LDS),
grown below the barrier and shrunk back (ellipsoidal barrier), rejected by
Nmin, across the periodic boundary, and in both workgroup widths."""

import numpy as np
import pytest

from oracle import pipeline as O
from exshalos_amd import synth
from exshalos_amd.lib import exshalos as X
from exshalos_amd.lib import set_precision

pytestmark = pytest.mark.gpu


def _field(bbks, nd, Lc, prec, bumps):
    """Gaussian field with smooth bumps [(centre, height, width), ...]."""
    k, P = bbks
    noise = synth.white_noise(nd, 4, np.float32 if prec == 4 else np.float64)
    d, _, _ = O.field_from_modes(k, P, nd, Lc, noise, precision=prec)
    x = np.arange(nd)
    for (ci, cj, ck), h, w in bumps:
        r2 = sum(((s - c + nd // 2) % nd - nd // 2).astype(np.float64) ** 2
                 for s, c in zip(np.meshgrid(x, x, x, indexing="ij"), (ci, cj, ck)))
        d = d + h * np.exp(-r2 / (2 * w * w))
    return np.ascontiguousarray(d.astype(np.float32 if prec == 4 else np.float64))


@pytest.mark.parametrize("prec", [4, 8])
@pytest.mark.parametrize("nd,Lc,barrier,nmin,bumps", [
    # a halo of thousands of cells around the box's corner
    (64, 4.0, (1.0, 0.0, 0.0), 1, [((0, 0, 0), 8.0, 2.6)]),
    # the same shrunk back below an ellipsoidal barrier, small halos rejected
    (64, 2.0, (0.8, 0.4, 0.6), 8, [((63, 1, 30), 9.0, 5.0), ((20, 40, 12), 6.0, 4.0)]),
    # a high barrier of few cells: most growths shrink to no cell, and their
    # centres must not keep later candidates waiting
    (48, 2.75, (1.2, 0.6, 0.6), 1, [((10, 47, 5), 9.0, 3.5)]),
    # no row in use: isolated cells only
    (32, 4.0, (1.0, 0.0, 0.0), 1, None),
    # more than 131072 candidates: 256 of them a workgroup
    (144, 4.0, (1.0, 0.0, 0.0), 3, [((143, 70, 0), 8.0, 2.4)]),
])
def test_growth_matches_the_oracle(bbks, prec, nd, Lc, barrier, nmin, bumps):
    k, P = bbks
    set_precision(prec)
    if bumps is None:
        delta = np.zeros((nd, nd, nd), dtype=np.float32 if prec == 4 else np.float64)
        rng = np.random.default_rng(3)
        delta[::4, ::4, ::4] = rng.uniform(1.7, 3.0, (nd // 4,) * 3)
    else:
        delta = _field(bbks, nd, Lc, prec, bumps)
    a, beta, alpha = barrier
    ref = O.find_halos(delta, k, P, Lc, Nmin=nmin, a=a, beta=beta, alpha=alpha, seed=12345,
                       precision=prec)
    out = X.find_halos(delta, k, P, Lc, 0.31, 0.0, -1.0, nmin, a, beta, alpha, 1, 0, 0)
    cat = X.halo_catalogue()
    if bumps is not None:
        assert ref["count"].max() > 1024
    np.testing.assert_array_equal(cat["x"], ref["x"])
    np.testing.assert_array_equal(cat["count"], ref["count"])
    np.testing.assert_array_equal(out["flag"].reshape(-1), ref["flag"].reshape(-1))
    np.testing.assert_array_equal(out["Mh"], ref["Mh"])
