"""Timing classes of the particle passes: a pass counts once per species, in
the class of what it does, whether a launch takes one species or both."""
import numpy as np
import pytest

import plasmasim_amd as ps

pytestmark = pytest.mark.gpu


def counts(s):
    return {k: s.timing_get(k)[1] for k in ("push", "push_sort", "sort")}


def sorting_step(s, reset):
    """One step that begins with the sort, the ions unsorted (uploaded): the
    radix sort for them, the tile sort's permutation for the electrons."""
    ions = s.download_particles(0)
    s.upload_particles(0, ions)
    reset(s)
    s.timing(True)
    s.timing_reset()
    s.step(1)
    c = counts(s)
    s.timing(False)
    return c


def cadence3(s):
    step, c_add, _ = s.counters()
    s.set_counters(step, 0, s.cfg.sort_every)


@pytest.mark.parametrize("precision", [ps.PIC_FP64, ps.PIC_FP32])
def test_passes_in_their_own_class(precision):
    c = ps.preset(1)
    c.precision = precision
    c.inflow_every = c.sort_every = 50
    c.tile[0] = c.tile[1] = 4
    c.tile[2] = 8
    s = ps.Simulation(c)
    s.load_particles()
    s.begin()
    s.step(2)
    got = sorting_step(s, cadence3)
    f32 = precision == ps.PIC_FP32
    assert got == {"push": 1 if f32 else 2, "push_sort": 1 if f32 else 0, "sort": 2}
    cadence3(s)  # both species by the tile sort
    s.timing(True)
    s.timing_reset()
    s.step(1)
    assert counts(s) == {"push": 0 if f32 else 2, "push_sort": 2 if f32 else 0, "sort": 2}
    s.timing_reset()
    s.step(3)
    assert counts(s) == {"push": 6, "push_sort": 0, "sort": 0}


def test_passes_in_their_own_class_2d():
    c = ps.preset2d(0)
    c.precision = ps.PIC_FP32
    c.nx = c.nz = 64
    c.tile[0] = c.tile[1] = 16
    c.inflow_every, c.sort_every = 50, 2
    s = ps.Simulation2D(c)
    s.load_particles()
    s.begin()
    s.step(2)
    got = sorting_step(s, lambda s: None)
    assert got == {"push": 1, "push_sort": 1, "sort": 2}
