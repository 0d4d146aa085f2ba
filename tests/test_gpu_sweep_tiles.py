"""Y and Z sweeps by tiles, at the column lengths and counts where they change:
columns of up to 64 cells are held whole, several to a wave below 33 cells,
longer ones go in parts through the second array. Single sweeps and steps are
compared with the CPU oracle (the fluid step's own tolerance, relative L1 1e-12
per variable); a periodic step equals its three sweeps in place, which march
where the step goes in parts, bitwise: all schemes run the same arithmetic on
the same cells."""
import numpy as np
import pytest

from gpuimogen_amd import abi, gpuclass as gc
from oracle import pyoracle as po

from .test_gpu_sweep_shapes import G, close, state

pytestmark = pytest.mark.gpu

METHODS = {abi.METHOD_HLLC: po.HLLC, abi.METHOD_HLL: po.HLL}
# (direction, nx, ny, nz): lanes filled or not, last block of columns in part
COLUMNS = [(2, nx, n, 3) for nx, n in ((5, 4), (16, 5), (17, 16), (33, 21), (7, 22), (40, 31), (16, 32), (17, 33),
                                       (1, 63), (35, 64))]
COLUMNS += [(3, 11, 3, n) for n in (4, 9, 32, 33, 63, 64)] + [(3, 129, 127, 64), (3, 129, 128, 64), (2, 70, 65, 3)]


@pytest.mark.parametrize("method", sorted(METHODS))
@pytest.mark.parametrize("direction,nx,ny,nz", COLUMNS)
def test_whole_columns(direction, nx, ny, nz, method):
    q = state((nz, ny, nx), nx + ny + nz)
    print(f"sweep {direction} of {nx} x {ny} x {nz}, method {method}", flush=True)
    f = gc.FluidManager(q, G)
    gm = gc.GeometryManager((nx, ny, nz), (0.01, 0.01, 0.01))
    gc.cudaFluidStep([0.002, 1, G, 1e-8, method, direction], f, gm, limiter=abi.LIMITER_VANLEER)
    po.fluid_update_1d(q, direction, 0.2, G, method=METHODS[method], limiter=po.LIM_VANLEER, rhomin=1e-8)
    close(f.state, q, f"direction {direction}, {nx} x {ny} x {nz}")
    f.free()


# parts of one length and of two, the largest part, the limit of their number,
# Y and Z of which one is whole
STEPS = [(65, 20, 1), (17, 65, 1), (33, 112, 1), (50, 113, 1), (300, 169, 1), (512, 896, 1), (513, 896, 1),
         (66, 40, 30), (20, 70, 64), (12, 13, 115)]


@pytest.mark.parametrize("method", sorted(METHODS))
@pytest.mark.parametrize("sh", STEPS)
def test_steps_equal_their_sweeps_in_place(sh, method):
    nx, ny, nz = sh
    q = state((nz, ny, nx), nx + ny + nz)
    h = (0.01, 0.012, 0.014)
    gm = gc.GeometryManager(sh, h)
    for it, order in ((0, (1, 3, 2)), (3, (2, 3, 1))):  # the reference's sweep orders
        print(f"step {sh} order {order}, method {method}", flush=True)
        f = gc.FluidManager(q, G, bc_modes=(abi.circular,) * 6)
        gc.fluidstep([f], None, None, None, [2e-4, 1, -1, it, method], gm)
        ref = q.copy()
        po.fluidstep(ref, h, 2e-4, -1, it, G, METHODS[method], po.LIM_OSPRE, modes=(po.BC_CIRCULAR,) * 6)
        close(f.state, ref, f"{sh} {order}")
        got = f.state
        f.free()
        g = gc.FluidManager(q, G, bc_modes=(abi.circular,) * 6)
        for d in order:
            if sh[d - 1] > 3:
                gc.cudaFluidStep([2e-4, 1, G, f.MINMASS, method, d], g, gm)
        assert np.array_equal(g.state, got), (sh, order)
        g.free()
