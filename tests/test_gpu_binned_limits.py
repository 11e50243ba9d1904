"""Binned deposit past its limits, which small inputs reach by lowering them:
tiles of up to 20 and 24 cells, more bins than the counters hold, a number of
entries that the host reads, room that does not suffice (before and after the
count, whose particle numbers must not be doubled), room for a count that is
not read beside the halo finder, and positions far outside the box."""

import contextlib

import numpy as np
import pytest

from oracle import pipeline as O
from exshalos_amd import synth
from exshalos_amd.lib import _native as N
from exshalos_amd.lib import set_precision
from exshalos_amd.lib import spectrum as SP
from exshalos_amd.pipeline import BoxPipeline

pytestmark = pytest.mark.gpu

MAX, READ, ROOM, ENTRIES = (N.TUNE_BIN_MAX, N.TUNE_BIN_READ, N.TUNE_BIN_ROOM,
                            N.TUNE_BIN_ENTRIES)
ATOMICS, BINNED = N.DEPOSIT_ATOMICS, N.DEPOSIT_BINNED


@contextlib.contextmanager
def limits(values):
    lib, ctx = N.load(), N.context()
    try:
        for key, v in values.items():
            N.check(lib.exh_ctx_set_tunable(ctx, key, v))
        yield
    finally:
        for key in values:
            N.check(lib.exh_ctx_set_tunable(ctx, key, 0))


def path():
    return N.load().exh_ctx_deposit_path(N.context())


@pytest.mark.parametrize("prec", [4, 8])
@pytest.mark.parametrize("nd,window,il,values,expected", [
    (90, 5, 1, {MAX: 200}, BINNED),            # 5 tiles of 18 cells
    (100, 2, 1, {MAX: 300}, BINNED),           # 5 of 20
    (96, 5, 1, {MAX: 100}, BINNED),            # 4 of 24, 110 KB of sums
    (100, 2, 1, {MAX: 100}, ATOMICS),
    (50, 2, 1, {READ: 1000}, BINNED),          # the number of entries is read
    (50, 2, 1, {ROOM: 1}, ATOMICS),            # no room for 8 a particle
    (50, 2, 1, {READ: 1000, ROOM: 1}, ATOMICS),  # nor for one
    (50, 2, 1, {READ: 1000, ROOM: 4}, ATOMICS),  # but for those counted (FP32)
])
def test_matches_the_oracle(prec, nd, window, il, values, expected):
    set_precision(prec)
    RT = np.float32 if prec == 4 else np.float64
    rng = np.random.default_rng(nd)
    n, L = 140000, 100.0
    pos = rng.uniform(0, L, (n, 3))
    pos[:30000] = (0.5, L / 3, L - 1.0) + rng.normal(0, 3.0, (30000, 3))
    pos = np.mod(pos, L).astype(RT)
    pos[pos >= L] = 0
    ref = O.grid_compute(pos, nd, L, window=window, interlacing=bool(il), precision=prec)
    with limits(values):
        g = SP.grid_compute(pos, None, None, 0, None, 1, nd, L, 0.31, 0.0, -1, window, 4.0, 5.0,
                            il, 1, 0, 1)
        assert path() == expected
    d = np.max(np.abs(g.astype(np.float64) - ref)) / np.max(np.abs(ref))
    assert d < (2e-5 if prec == 4 else 1e-12)


@pytest.mark.parametrize("prec", [4, 8])
@pytest.mark.parametrize("window,values,expected", [
    (2, {}, BINNED),
    (5, {READ: 1000}, BINNED),                  # 2 entries a particle, not read
    (2, {READ: 1000, ENTRIES: 17}, ATOMICS),    # 1.06: the device finds no room
    (5, {READ: 1000, ROOM: 1}, ATOMICS),
])
def test_chain_of_a_side_that_no_tile_divides(bbks, prec, window, values, expected):
    k, P = bbks
    set_precision(prec)
    nd = 70
    pipe = BoxPipeline(k, P, nd=nd, Lc=4.0, precision=prec, Nk=24, window=window)
    pipe.set_modes(synth.white_noise(nd, 9, np.float32 if prec == 4 else np.float64))
    with limits(values):
        for _ in range(2):
            pipe.run(fused=True)
            assert path() == expected
    pos = pipe.pos.cpu().numpy()
    ref = O.grid_compute(pos, nd, pipe.L, window=window, interlacing=True, precision=prec)
    g = pipe.grid.cpu().numpy().astype(np.float64)
    d = np.max(np.abs(g - ref)) / np.max(np.abs(ref))
    assert d < (2e-5 if prec == 4 else 1e-12)


@pytest.mark.parametrize("prec", [4, 8])
def test_huge_positions_end_in_the_box(prec):
    set_precision(prec)
    RT = np.float32 if prec == 4 else np.float64
    n, L, nd = 140000, 100.0, 32
    rng = np.random.default_rng(2)
    pos = rng.uniform(0, L, (n, 3)).astype(RT)
    pos[pos >= L] = 0
    big = np.finfo(RT).max
    far = [big, -big, big / 3, 1e30, -1e30, 1e20, -3.3e17, 1e12, 7.7e9, -1e9, 5 * L, -4 * L]
    pos[: len(far), 0] = np.array(far, dtype=RT)
    pos[20: 20 + len(far), 2] = np.array(far, dtype=RT)
    w = np.ones(n, dtype=RT)
    g = SP.grid_compute(pos, None, w, 1, None, 1, nd, L, 0.31, 0.0, -1, 2, 4.0, 5.0, 1, 1, 0, 1)
    assert path() == BINNED
    for s in range(2):
        assert abs(g[0, s].astype(np.float64).sum() - n) < 1e-5 * n
