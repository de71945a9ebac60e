"""Stores sorted as one tile over the interior (the reference's order): the
particle pass takes them in boxes of cell columns, whose sizes need not
divide the grid, and the inflow tail in chunks; stores that do not fill their
boxes go in chunks altogether."""
import time

import numpy as np
import pytest

import plasmasim_amd as ps
from helpers import rel_l2
from oracle_lib import Oracle

pytestmark = pytest.mark.gpu
FIELDS = ["ex", "ey", "ez", "bx", "by", "bz", "jix", "jiy", "jiz", "jex", "jey", "jez", "ni",
          "ne"]


def state(n, tile, precision, fused=True):
    c = ps.preset(1)
    c.nx, c.ny, c.nz = n
    c.ppc = 5
    c.absorb[2] = 2
    c.ballistic_lo[2], c.ballistic_hi[2] = 6.0, c.nz - 2.0
    c.inflow_every, c.sort_every = 3, 5
    c.precision = precision
    c.deposit = ps.PIC_DEPOSIT_DETERMINISTIC
    for a in range(3):
        c.tile[a] = tile[a]
    s = ps.Simulation(c)
    s.load_particles()
    s.begin()
    s.thrust_ave(True)
    if fused:
        s.step(12)
    else:
        for _ in range(3):
            s.renew_grid()
            for sp in (0, 1):
                s.push_deposit_j(sp)
            for sp in (0, 1):
                s.drift_deposit_n(sp)
            s.fold_current()
            s.particle_boundary()
    return s


# (grid, a tiling of it that runs on tile ranges): the smallest grid, one cell
# over and under the boxes' sizes, sizes that nothing divides, many boxes
@pytest.mark.parametrize("n, tile", [((4, 4, 8), (4, 4, 4)), ((5, 7, 9), (5, 7, 3)),
                                     ((9, 3 * 5, 17 * 2), (3, 5, 2)),
                                     ((31, 27, 45), (1, 3, 15)), ((48, 36, 64), (4, 4, 8))])
@pytest.mark.parametrize("fused", [True, False])
def test_one_tile_equals_tiles(n, tile, fused):
    """FP32 with the fixed summation order: bit for bit the fields of the
    tiled run (sorts, inflows and both kinds of tail between).  FP64: sums in
    another order, 32 contributions of 2^-53 each per node and step."""
    a = state(n, (0, 0, 0), ps.PIC_FP32, fused)
    b = state(n, tile, ps.PIC_FP32, fused)
    for k in FIELDS:
        assert np.array_equal(a.download_field(k), b.download_field(k)), k
    if fused:
        fa, fb = a.thrust_ave_get()[0], b.thrust_ave_get()[0]
        # per-lane fp32 sums of another grouping: 2^-24 of the largest part
        assert np.abs(fa - fb).max() <= 1e-5 * max(np.abs(fb).max(), 1e-30)
    a = state(n, (0, 0, 0), ps.PIC_FP64, fused)
    b = state(n, tile, ps.PIC_FP64, fused)
    for k in FIELDS:
        assert rel_l2(a.download_field(k), b.download_field(k)) <= 1e-12, k


def test_one_tile_resumes_without_cell_starts(tmp_path):
    """A loaded checkpoint carries no cell starts: the pass takes the store
    in chunks until the next sort, with the same result."""
    a = state((20, 12, 24), (0, 0, 0), ps.PIC_FP32)
    f = str(tmp_path / "c.bin")
    a.checkpoint_save(f)
    b = ps.Simulation(a.cfg)
    b.checkpoint_load(f)
    a.thrust_ave(False)
    a.step(3)
    b.step(3)
    for k in FIELDS:
        assert np.array_equal(a.download_field(k), b.download_field(k)), k


def uneven(precision, tile, count, lo, hi):
    """32 x 32 x 40 cells (320 boxes) with `count` particles of each species
    between lo and hi, both sorted, one step."""
    c = ps.preset(1)
    c.nx, c.ny, c.nz = 32, 32, 40
    c.capacity = 65536
    c.inflow_every = c.sort_every = 1000
    c.precision = precision
    c.deposit = ps.PIC_DEPOSIT_DETERMINISTIC
    for a in range(3):
        c.tile[a] = tile[a]
    s = ps.Simulation(c)
    r = np.random.default_rng(count)
    for sp in (0, 1):
        # offsets exact in FP32, so that both forms hold the same particles
        x = np.floor(r.uniform(lo, hi, (count, 3)) * 4096) / 4096
        s.upload_particles(sp, np.concatenate([x, r.normal(0, 0.05, (count, 3))], 1))
        s.sort(sp)
    s.step(1)
    return s


# below and above 32 particles per box (10240); a fullest box of 8 times its
# share or more; one cell, the last cell, the first and last layers, a gap
@pytest.mark.parametrize("count, lo, hi", [
    (3, (2, 2, 2), (34, 34, 42)), (10239, (2, 2, 2), (34, 34, 42)),
    (10240, (2, 2, 2), (34, 34, 42)), (20000, (2, 2, 2), (34, 34, 42)),
    (20000, (2, 2, 2), (18, 18, 22)), (20000, (6, 6, 10), (10, 10, 18)),
    (20000, (20, 20, 20), (21, 21, 21)), (20000, (33, 33, 41), (34, 34, 42)),
    (20000, (2, 2, 2), (34, 34, 14)), (20000, (2, 2, 30), (34, 34, 42))])
def test_uneven_stores(count, lo, hi):
    """FP32, fixed summation order: bit for bit the tiled store's fields;
    FP64: sums in another order."""
    a, b = (uneven(ps.PIC_FP32, t, count, lo, hi) for t in ((0, 0, 0), (4, 4, 8)))
    for k in FIELDS:
        assert np.array_equal(a.download_field(k), b.download_field(k)), k
    a, b = (uneven(ps.PIC_FP64, t, count, lo, hi) for t in ((0, 0, 0), (4, 4, 8)))
    for k in FIELDS:
        assert rel_l2(a.download_field(k), b.download_field(k)) <= 1e-12, k


@pytest.mark.parametrize("precision", [ps.PIC_FP64, ps.PIC_FP32])
def test_sort_of_uneven_stores_takes_no_longer(precision, count=200000, lo=64, hi=68):
    """The sort's cost does not depend on where the empty cells are: 0.15 ms
    for 200000 particles in 4^3 of 128^3 cells; one thread writing the starts
    of a run of empty cells takes 25 ms."""
    c = ps.preset(1)
    c.nx = c.ny = c.nz = 128
    c.capacity = 2 * count
    c.precision = precision
    s = ps.Simulation(c)
    r = np.random.default_rng(5)
    s.upload_particles(0, np.concatenate([r.uniform(lo, hi, (count, 3)),
                                          np.zeros((count, 3))], 1))
    best = 1.0
    for _ in range(4):
        t = time.perf_counter()
        s.sort(0)
        s.sync()
        best = min(best, time.perf_counter() - t)
    assert s.particle_count(0) == count
    assert best <= 5e-3


@pytest.mark.parametrize("dx", [1.0, 0.75])
@pytest.mark.parametrize("tile", [(0, 0, 0), (4, 4, 8)])
def test_fp64_pass_in_other_units(dx, tile):
    """FP64 pass in normalised units and with dx away from 1 (its own
    instantiation) against the oracle, inflow and sort between: 15 steps of
    sums in another order."""
    c = ps.preset(1)
    c.nx, c.ny, c.nz = 16, 12, 24
    c.ppc = 6
    c.dx, c.dt = dx, c.dt * dx
    c.absorb[2] = 3
    c.ballistic_lo[2], c.ballistic_hi[2] = 7.0 * dx, (c.nz - 3.0) * dx
    c.inflow_every, c.sort_every = 4, 6
    for a in range(3):
        c.tile[a] = tile[a]
    g, o = ps.Simulation(c), Oracle(c)
    for s in (g, o):
        s.load_particles()
    for s in (g, o):
        s.begin()
        s.step(15)
    for k in FIELDS:
        assert rel_l2(g.download_field(k), o.download_field(k)) <= 1e-12, k
    for sp in (0, 1):
        assert g.particle_count(sp) == o.particle_count(sp)
