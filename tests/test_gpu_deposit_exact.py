"""TSC deposit of an FP64 lattice through the tiles' windows where every value
is exact: particles at the cell centres (and, for the second grid, on the cell
faces) of cells of side 49, whose reciprocal is not exact.  The quotients x / 49
are, the weights are 1/8, 3/4 and 1/2, and every cell sums to one."""

import numpy as np
import pytest

from exshalos_amd.lib import set_precision
from exshalos_amd.lib import spectrum as SP

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [32, 48])
def test_tsc_of_cell_centres_is_uniform(n):
    set_precision(8)
    q = (np.arange(n) + 0.5) * 49.0
    x = np.stack(np.meshgrid(q, q, q, indexing="ij"), -1).reshape(-1, 3)
    g = SP.grid_compute(x, None, None, 0, None, 1, n, n * 49.0, 0.31, 0.0, -1, 5, 4.0, 5.0, 1, 1,
                        0, 1)
    assert g.shape[1] == 2 and np.all(g == 0.0)
