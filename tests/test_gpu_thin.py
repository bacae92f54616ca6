"""Thin grids: a few cells across, long in one direction (tubes, sheets)."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


class Device:
    """The solver's SoA planes, written and read through their address (a host
    array of rows would be 2.7 GB here)."""

    def __init__(self, solver, mmf):
        self.L = C.CDLL("libamdhip64.so.7")
        self.L.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
        self.address, self.stride = solver.device_state(mmf.STATE_U)

    def at(self, k, cell):
        return self.address + 8 * (k * self.stride + cell)

    def write(self, k, a):
        assert self.L.hipMemcpy(self.at(k, 0), a.ctypes.data, a.nbytes, 1) == 0

    def read(self, cell, count):
        out = np.empty((5, count))
        for k in range(5):
            assert self.L.hipMemcpy(out[k].ctypes.data, self.at(k, cell), 8 * count, 2) == 0
        return out


LONG = (1 << 26) + 8  # 2^32 threads and more where a brick's 64 columns hold one cell


@pytest.mark.parametrize("order,kind,body", [(1, "AUTO", False), (2, "AUTO", False), (1, "MARCH", True)])
def test_longest_tubes(mmf, order, kind, body):
    """A tube of more than 2^26 cells: every cell advances, at both ends."""
    seen = []
    N = LONG
    windows = [0, N // 2, N - 64]
    energy = np.full(N, 2.5)
    energy[5:9] = energy[N // 2 + 20:N // 2 + 24] = energy[N - 9:N - 5] = 3.5
    for k in (kind, "GATHER"):
        s = mmf.Solver(3, [1, 1, N], [0.0] * 3, 1e-3, [0] * 6, None, order)
        if body:
            fluid = np.ones(N, dtype=np.uint8)
            fluid[12:20] = fluid[N - 30:N - 20] = 0
            s.set_cell_flags(fluid)
        s.set_kernel(getattr(mmf, "KERNEL_" + k))
        d = Device(s, mmf)
        d.write(0, np.ones(N))
        d.write(4, energy)
        s.set_time(0.0, 1e30, 0.4)
        s.advance(1)
        seen.append((s.time()[:3], tuple(s.time()[3]), [d.read(w, 64).tobytes() for w in windows]))
        s.close()
    assert seen[0][0][2] == 1
    assert seen[0] == seen[1]


def test_bricks_are_refused_beyond_a_launch(mmf):
    s = mmf.Solver(3, [1, 1, LONG], [0.0] * 3, 1e-3, [0] * 6, None, 1)
    with pytest.raises(mmf.MMFError) as e:
        s.set_kernel(mmf.KERNEL_BRICK)
    assert e.value.status == mmf.ERR_INVALID
    s.close()
