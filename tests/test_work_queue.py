"""The cooperative kernels' work queue (queue_for_each, pdq_device.h): every lane of a group gets every
drawn instance once, and every lane takes part in every draw.  A draw behind a branch for one lane may
be compiled into a loop that the other lanes never leave.
"""

import ctypes
import os

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "probdiffeq_amd", "csrc")


@pytest.fixture(scope="module")
def emu():
    from emu import emu as M

    M.build()
    M._lib = None
    return M


@pytest.mark.parametrize("G,n", [(4, 0), (4, 7), (16, 3), (64, 5)])
def test_every_lane_takes_part_in_every_draw(emu, G, n):
    taken = np.zeros((max(n, 1), G), dtype=np.int32)
    atomics = emu.lib().pdqemu_queue(G, n, taken.ctypes.data_as(ctypes.c_void_p))
    assert (taken[:n] == 1).all()
    assert atomics == G * (n + 1)  # one draw per instance and the one that ends the loop


def test_every_kernel_draws_this_way():
    """The queue is read in queue_for_each and in the fixed-shape kernel's loop (all lanes there too)."""
    sites = []
    for name in sorted(os.listdir(CSRC)):
        if not name.endswith((".h", ".hip")) or name == "pdq_hostemu.h":
            continue
        with open(os.path.join(CSRC, name)) as f:
            sites += [line.strip() for line in f if "atomicAdd(" in line]
    assert len(sites) >= 1
    for line in sites:
        assert "l == 0 ? 1 : 0" in line and not line.startswith("if"), line
