"""P(k) of one tracer by lines of modes: grid sides whose modes per row leave
every kind of remainder against the 64 lanes of a wave, the multipoles, both
sub-grid options, and few and many bins, against the oracle; and the same bits
on every call."""

import numpy as np
import pytest

from oracle import pipeline as O
from exshalos_amd.lib import set_precision
from exshalos_amd.lib import spectrum as SP

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [4, 8])
@pytest.mark.parametrize("nd,il,lmax,direction,Nk", [
    (6, 1, 0, -1, 3),      # 4 modes a row: 16 rows to a wave
    (30, 0, 4, 0, 7),      # 16
    (64, 1, 2, 1, 40),     # 33: one row to a wave
    (96, 0, 0, -1, 200),   # 49, bins of less than a step
    (126, 1, 4, 2, 16),    # 64: full chunks only
    (128, 1, 0, -1, 33),   # 65: a remainder of one
    (180, 0, 2, 2, 12),    # 91: a remainder of 27, two rows to a wave
])
def test_matches_the_oracle(prec, nd, il, lmax, direction, Nk):
    set_precision(prec)
    R = np.float32 if prec == 4 else np.float64
    L = 4.0 * nd
    grid = np.random.default_rng(nd).normal(size=(1, 1 + il, nd, nd, nd)).astype(R)
    kmin, kmax = 2 * np.pi / L, np.pi / L * nd
    ref = O.power_compute(grid, 1, nd, L, window=2, interlacing=bool(il), Nk=Nk, k_min=kmin,
                          k_max=kmax, l_max=lmax, direction=direction, precision=prec)
    outs = [SP.power_compute(grid, 1, nd, L, 2, 4.0, il, Nk, kmin, kmax, lmax, direction, 0, 1)
            for _ in range(3)]
    np.testing.assert_array_equal(outs[0]["Nk"], ref["Nk"])
    d = np.max(np.abs(outs[0]["Pk"] - ref["Pk64"])) / np.max(np.abs(ref["Pk64"]))
    assert d < (1e-5 if prec == 4 else 1e-10)
    for o in outs[1:]:
        np.testing.assert_array_equal(o["Pk"], outs[0]["Pk"])
        np.testing.assert_array_equal(o["k"], outs[0]["k"])
