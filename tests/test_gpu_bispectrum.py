"""Bispectrum products at the edges of their tiles: one and two shells (jobs
shared by several waves), one more than a column tile (17), more jobs than one
group of workgroups holds, three tracers, and a grid side whose cells leave a
partial last chunk.

Triangles that do not close have a vanishing sum over the indicators, so the
sums are compared (B times the triangle count), relative to the largest: a
field's 32-bit transform is good to about 1e-6 and enters three times."""

import numpy as np
import pytest

from oracle import pipeline as O
from exshalos_amd.lib import set_precision
from exshalos_amd.lib import spectrum as SP

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [4, 8])
@pytest.mark.parametrize("nd,ntype,Nk", [(16, 1, 1), (18, 1, 2), (24, 1, 17), (20, 1, 30),
                                         (18, 3, 6)])
def test_products_match_the_oracle(prec, nd, ntype, Nk):
    set_precision(prec)
    RT = np.float32 if prec == 4 else np.float64
    rng = np.random.default_rng(nd + 100 * Nk + ntype)
    L = 5.0 * nd
    grid = rng.normal(size=(ntype, 1, nd, nd, nd)).astype(RT)
    grid[..., :4] += 1.5
    kmin, kmax = 2 * np.pi / L, np.pi / L * nd
    ref = O.bispectrum(grid, ntype, nd, L, window=2, Nk=Nk, precision=prec)
    out = SP.bi_compute(grid, ntype, nd, L, 2, 0.0, 0, Nk, kmin, kmax, 0, 1)
    tol = 1e-5 if prec == 4 else 1e-11

    def off(a, b):  # shells without modes are 0/0 on both sides
        a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
        np.testing.assert_array_equal(np.isnan(a), np.isnan(b))
        return np.nanmax(np.abs(a - b)) / np.nanmax(np.abs(b))

    np.testing.assert_allclose(out["kP"], ref["kP"], rtol=1e-6 if prec == 4 else 1e-12)
    assert off(out["Ntri"], ref["Ntri"]) < tol
    assert off(out["Nk"], ref["Nk"]) < tol
    assert off(out["Pk"], ref["Pk"]) < tol
    closed = out["Ntri"] != 0
    B = out["Bk"].astype(np.float64) * out["Ntri"] * nd**3 / L**1.5
    assert off(B[:, closed], ref["B64"][:, closed]) < tol
