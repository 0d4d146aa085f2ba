"""Xin-Jin sweeps at the line lengths where their launch changes: whole lines
in a block of 512 or 1024 threads with two or four cells a thread, and the
staged form beyond (X over 4096 cells, Y and Z over 1024; 16, 8 and 4 columns
a block up to 256, 512 and 1024). Lengths that are not
a multiple of a thread's cells leave the last thread with the line's first
cells again; line counts that are not a multiple of a block's leave idle ones.
Tolerance: the fluid step's own (relative L1 1e-12 per variable)."""
import pytest

from gpuimogen_amd import abi, gpuclass as gc
from oracle import pyoracle as po

from .test_gpu_sweep_shapes import G, close, state

pytestmark = pytest.mark.gpu

# (direction, nx, ny, nz)
CASES = [(1, n, 3, 2) for n in (4, 5, 6, 7, 9, 64, 127, 1023, 1024, 1025, 2047, 2049, 4095, 4096, 4097)]
CASES += [(1, 131, 40, 60), (1, 21, 130, 131), (1, 2047, 150, 1), (1, 257, 17, 64)]
CASES += [(2, 17, n, 3) for n in (4, 5, 6, 7, 33, 63, 64, 65, 129, 255, 256, 257, 512, 513, 1024, 1025)]
CASES += [(2, 131, 33, 61), (2, 5, 130, 500), (2, 1, 250, 9), (2, 70, 300, 7), (2, 70, 1100, 2)]
CASES += [(3, 17, 3, n) for n in (4, 5, 6, 7, 33, 63, 64, 65, 129, 255, 256, 257, 512, 513, 1024, 1025)]
CASES += [(3, 61, 131, 34), (3, 250, 33, 131), (3, 3, 3, 250), (3, 70, 7, 300)]


@pytest.mark.parametrize("direction,nx,ny,nz", CASES)
def test_xinjin_lines(direction, nx, ny, nz):
    q = state((nz, ny, nx), nx + 7 * ny + 31 * nz)
    print(f"Xin-Jin sweep {direction} of {nx} x {ny} x {nz}", flush=True)
    f = gc.FluidManager(q, G)
    gm = gc.GeometryManager((nx, ny, nz), (0.01, 0.01, 0.01))
    gc.cudaFluidStep([0.0015, 1, G, 1e-8, abi.METHOD_XINJIN, direction], f, gm)
    po.fluid_update_1d(q, direction, 0.15, G, method=po.XINJIN, rhomin=1e-8)
    close(f.state, q, f"direction {direction}, {nx} x {ny} x {nz}")
    f.free()
