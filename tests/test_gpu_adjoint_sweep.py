"""The reverse sweep's buffers and units: a context that is asked again, with
other windows and parameters, gives what a new one gives; dx away from 1 (its
own instantiation of the transposed pass) against the oracle's gradient; the
FP32 forward's tape, read in its own form, against the FP64 one."""
import numpy as np
import pytest
import torch

import plasmasim_amd as ps
from oracle_lib import Oracle

pytestmark = pytest.mark.gpu
R, NQ = 3.0, 64


def cfg(precision=ps.PIC_FP64, dx=1.0, sort_every=20):
    c = ps.preset(0)
    c.precision = precision
    c.inflow_every, c.sort_every = 3, sort_every
    c.capacity = 16384
    c.dx, c.dt = dx, c.dt * dx
    c.ballistic_lo[2] *= dx
    c.ballistic_hi[2] *= dx
    return c


def params(c, t=0.1):
    M = c.dipole_m
    return np.array([t * M, 0.9 * M, 0.3 * M, c.vdrift[2]])


def grad(s, p, steps, window):
    loss = s.adj_forward(p, steps, window, R, NQ)
    return loss, s.adj_backward(1.0)


@pytest.mark.parametrize("precision", [ps.PIC_FP64, ps.PIC_FP32])
@pytest.mark.parametrize("sort_every", [2, 20])
def test_repeated_sweeps_equal_fresh_ones(precision, sort_every):
    """Buffers kept between sweeps: more steps, longer and shorter windows,
    sorts inside a window.  FP64 atomics: sums in another order."""
    c = cfg(precision, sort_every=sort_every)
    s = ps.Simulation(c)
    tol = 1e-9 if precision == ps.PIC_FP64 else 1e-5
    for steps, window, t in ((6, 2, 0.1), (7, 5, 0.2), (4, 1, 0.1), (6, 2, 0.1)):
        loss, g = grad(s, params(c, t), steps, window)
        f = ps.Simulation(c)
        lf, gf = grad(f, params(c, t), steps, window)
        f.close()
        assert abs(loss - lf) <= tol * abs(lf)
        assert np.all(np.abs(g - gf) <= tol * np.abs(gf)), (steps, window, g, gf)
    s.close()


def test_kept_buffers_are_those_of_the_last_window():
    """After a sweep over long windows and one over short ones a context holds
    what one that has only seen the short ones holds: a forward gives back
    the tape of 7 steps of 2 x 262144 slots (103 MB)."""
    def used(windows):
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        c = cfg(ps.PIC_FP32)
        c.capacity = 262144
        s = ps.Simulation(c)
        for w in windows:
            grad(s, params(c), 8, w)
        left = torch.cuda.mem_get_info()[0]
        s.close()
        return free - left

    used([1])  # what the process loads and keeps on first use
    one, both = used([1]), used([8, 1])
    assert both - one <= 16 << 20, (one, both)


def test_one_tile_segments_run_in_the_forwards_boxes():
    """A recomputed segment of a one-tile store groups its deposits as its
    forward did: at nodes that the particles of a single box reach the current
    of the first step is the forward's, bit for bit (one fixed-point sum of a
    workgroup, one add to the plane; without the cell starts the contributions
    arrive one by one).  Boxes are 4 x 4 x 8 cells, and no particle crosses
    half a cell: nodes 2 along x and y and 2 to 5 along z of each, without the
    boxes at the z faces, where the inflow's chunks add too."""
    c = ps.preset(1)
    c.nx, c.ny, c.nz, c.ppc = 32, 32, 40, 8
    c.precision = ps.PIC_FP32
    c.inflow_every = c.sort_every = 1000
    s = ps.Simulation(c)
    s.adj_forward(params(c), 1, 1, R, NQ)
    planes = ("jix", "jiy", "jiz", "jex", "jey", "jez")
    a = [s.download_field(k) for k in planes]
    s.adj_backward(1.0)
    node = [np.arange(2, n + 2) for n in (c.nx, c.ny, c.nz)]
    z = np.arange(8, c.nz - 8)
    box = np.ix_(node[0][2::4], node[1][2::4], node[2][z[np.isin(z % 8, (2, 3, 4, 5))]])
    for k, j in zip(planes, a):
        assert np.count_nonzero(j[box]), k
        assert np.array_equal(s.download_field(k)[box], j[box]), k
    s.close()


@pytest.mark.parametrize("dx", [1.0, 0.75])
def test_gradient_in_other_units(dx):
    c = cfg(dx=dx)
    s = ps.Simulation(c)
    loss, g = grad(s, params(c), 6, 2)
    lo, go = Oracle(c, threads=4).adj_gradient(params(c), 6, R, NQ)
    assert abs(loss - lo) <= 1e-10 * abs(lo)
    assert np.all(np.abs(g - go) <= 1e-6 * np.abs(go)), (g, go)
    s.close()


def test_fp32_tape_gradient():
    """The FP32 forward's gradient against the FP64 one: their trajectories
    differ by the FP32 rounding of 6 steps."""
    out = []
    for precision in (ps.PIC_FP32, ps.PIC_FP64):
        c = cfg(precision)
        s = ps.Simulation(c)
        out.append(grad(s, params(c), 6, 3)[1])
        s.close()
    assert np.all(np.abs(out[0] - out[1]) <= 1e-5 * np.abs(out[1])), out
