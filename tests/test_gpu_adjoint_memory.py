"""The adjoint where the card is nearly full: a call that finds no room says
so, and the next one, with room again, is the first one's equal; what a
context keeps for its next sweep makes room for its own allocations."""
import contextlib

import numpy as np
import pytest
import torch

import plasmasim_amd as ps

pytestmark = pytest.mark.gpu
MIB = 1 << 20


@contextlib.contextmanager
def card_with(left):
    """All of the card's memory but `left` bytes (to 64 MiB) is taken."""
    torch.cuda.synchronize()
    taken = []
    try:
        for _ in range(8):  # what is reported free grows a little with each
            more = torch.cuda.mem_get_info()[0] - left
            if more < 64 * MIB:
                break
            taken.append(torch.empty(more, dtype=torch.uint8, device="cuda"))
        yield
    finally:
        taken.clear()
        torch.cuda.empty_cache()


def cfg(n, ppc):
    c = ps.preset(4)
    c.nx = c.ny = c.nz = n
    c.ppc = ppc
    c.precision = ps.PIC_FP32
    c.ballistic_hi[2] = n - 4.0
    return c


def params(c):
    M = c.dipole_m
    return np.array([0.1 * M, 0.9 * M, 0.3 * M, c.vdrift[2]])


def test_no_half_built_state():
    """160^3: of 800 MiB free the adjoint's first two allocations take 404 MiB,
    the third, of 606 MiB, finds no room."""
    c = cfg(160, 1)
    s = ps.Simulation(c)
    with card_with(800 * MIB):
        with pytest.raises(ps.PicError):
            s.adj_forward(params(c), 2, 2, 10.0, 64)
    loss = s.adj_forward(params(c), 2, 2, 10.0, 64)
    g = s.adj_backward(1.0)
    s.close()
    f = ps.Simulation(c)
    assert abs(loss - f.adj_forward(params(c), 2, 2, 10.0, 64)) <= 1e-6 * abs(loss)
    # FP32 atomics of two steps
    assert np.all(np.abs(g - f.adj_backward(1.0)) <= 1e-4 * np.abs(g))
    f.close()


def test_kept_buffers_make_room_for_checkpoints():
    """64^3 x 32 ppc: a sweep over 8 steps keeps 6 GiB; a forward of 40 steps in
    windows of 8 takes four more checkpoints of 0.5 GiB with 1 GiB free."""
    c = cfg(64, 32)
    s = ps.Simulation(c)
    s.adj_forward(params(c), 8, 8, 10.0, 64)
    g = s.adj_backward(1.0)
    with card_with(1024 * MIB):
        s.adj_forward(params(c), 40, 8, 10.0, 64)
    s.adj_forward(params(c), 8, 8, 10.0, 64)
    assert np.all(np.abs(s.adj_backward(1.0) - g) <= 1e-4 * np.abs(g))
    s.close()
