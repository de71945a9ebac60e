"""Tiles whose particles go to several workgroups (few tiles, many particles
each): the same result as with whole tiles."""
import numpy as np
import pytest

import plasmasim_amd as ps
from helpers import rel_l2
from oracle_lib import Oracle, Oracle2D

pytestmark = pytest.mark.gpu
FIELDS = ["ex", "ey", "ez", "bx", "by", "bz", "jix", "jiy", "jiz", "jex", "jey", "jez", "ni",
          "ne"]


def run3(n, tile, ppc, precision, cls=None):
    c = ps.preset(1)
    c.nx, c.ny, c.nz = n
    c.ppc = ppc
    c.absorb[2] = 2
    c.ballistic_lo[2], c.ballistic_hi[2] = 6.0, c.nz - 2.0
    c.inflow_every, c.sort_every = 3, 5
    c.precision = precision
    c.deposit = ps.PIC_DEPOSIT_DETERMINISTIC
    for a in range(3):
        c.tile[a] = tile[a]
    s = (cls or ps.Simulation)(c)
    s.load_particles()
    s.begin()
    s.step(8)
    return s


# particles per tile around the limits of 2, 4 and 8 parts; the tiling with
# small tiles keeps whole ones
@pytest.mark.parametrize("tile, ppc", [((4, 4, 8), 9), ((4, 4, 8), 17), ((4, 4, 8), 33),
                                       ((8, 4, 4), 61)])
def test_3d_parts_equal_whole_tiles(tile, ppc):
    """FP32, fixed summation order: bit for bit.  FP64 against the oracle."""
    a = run3((8, 8, 16), tile, ppc, ps.PIC_FP32)
    b = run3((8, 8, 16), (2, 2, 2), ppc, ps.PIC_FP32)
    for k in FIELDS:
        assert np.array_equal(a.download_field(k), b.download_field(k)), k
    a = run3((8, 8, 16), tile, ppc, ps.PIC_FP64)
    o = run3((8, 8, 16), tile, ppc, ps.PIC_FP64, Oracle)
    for k in FIELDS:
        assert rel_l2(a.download_field(k), o.download_field(k)) <= 1e-12, k


@pytest.mark.parametrize("dx", [1.0, 0.75])
@pytest.mark.parametrize("ppc", [5, 40])
def test_2d_parts_against_the_oracle(ppc, dx):
    """16 x 16 tiles of 1280 and 10240 particles, both instantiations of the
    FP64 pass; 8 steps of sums in another order."""
    c = ps.preset2d(0)
    c.nx, c.nz, c.ppc = 32, 64, ppc
    c.tile[0] = c.tile[1] = 16
    c.inflow_every, c.sort_every = 3, 5
    c.dx, c.dt = dx, c.dt * dx
    c.ballistic_lo[1] *= dx
    c.ballistic_hi[1] *= dx
    c.precision = ps.PIC_FP64
    g, o = ps.Simulation2D(c), Oracle2D(c)
    for s in (g, o):
        s.load_particles()
        s.begin()
        s.step(8)
    for k in FIELDS:
        assert rel_l2(g.download_field(k), o.download_field(k)) <= 1e-12, k
