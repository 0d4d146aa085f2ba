"""Ghost cells set by the sweep of their direction: const and mirror faces, and
either beside a periodic one, in every sweep that can set them (X lines whole
and in parts with 1 to 6 cells per lane, tiles whole and in parts, marches in
place and out of place), and at the line lengths 13 and 14 where the boundary
launches give way. Steps against the CPU oracle (relative L1 1e-12 per variable,
as the fluid step); the last swept direction's ghosts are exact images."""
import numpy as np
import pytest

from gpuimogen_amd import abi, gpuclass as gc
from oracle import pyoracle as po

from .test_gpu_sweep_shapes import G, close, state

pytestmark = pytest.mark.gpu

K, M, C = (abi.extrapConstant, po.BC_CONST), (abi.mirror, po.BC_MIRROR), (abi.circular, po.BC_CIRCULAR)
FACES = {"const": (K, K), "mirror": (M, M), "const-mirror": (K, M), "mirror-const": (M, K),
         "const-open": (K, C), "open-mirror": (C, M)}
# X: 13/14; whole lines K = 1..4 and 6; parts of K = 1, 2, 3, 4. Y: tiles whole
# and in parts; 3D: marches; a plane too large for tiles
SHAPES = [(13, 20, 1), (14, 13, 1), (15, 14, 1), (50, 14, 1), (64, 70, 1), (128, 1100, 1), (192, 1100, 1),
          (256, 1100, 1), (384, 20, 1), (90, 20, 1), (600, 14, 1), (520, 800, 1), (500, 800, 1), (30, 130, 20),
          (600, 1100, 1), (100, 110, 90), (1024, 1, 1), (60, 1, 1)]


@pytest.mark.parametrize("faces", sorted(FACES))
@pytest.mark.parametrize("sh", SHAPES)
def test_steps_with_their_ghosts(sh, faces):
    nx, ny, nz = sh
    q = state((nz, ny, nx), nx + ny + nz)
    lo, hi = FACES[faces]
    h = (0.01, 0.012, 0.014)
    gm = gc.GeometryManager(sh, h)
    for method, om in ((abi.METHOD_HLLC, po.HLLC), (abi.METHOD_HLL, po.HLL)):
        f = gc.FluidManager(q, G, bc_modes=(lo[0], hi[0]) * 3)
        ref = q.copy()
        for it, order in ((0, (1, 3, 2)), (4, (3, 1, 2)), (3, (2, 3, 1))):
            print(f"step {sh} {faces} order {order}, method {method}", flush=True)
            gc.fluidstep([f], None, None, None, [2e-4, 1, -1, it, method], gm)
            po.fluidstep(ref, h, 2e-4, -1, it, G, om, po.LIM_OSPRE, modes=(lo[1], hi[1]) * 3)
            got = f.state
            last = [d for d in order if sh[d - 1] > 3][-1] if ny > 1 else 1
            a = np.moveaxis(got, 4 - last, 1)
            n = a.shape[1]
            turn = np.ones((5, 1, 1))
            turn[1 + last] = -1
            if n >= 14:
                for i in range(4):
                    if lo is not C:
                        assert np.array_equal(a[:, i], a[:, 8 - i] * turn if lo is M else a[:, 4])
                    if hi is not C:
                        assert np.array_equal(a[:, n - 1 - i], a[:, n - 9 + i] * turn if hi is M else a[:, n - 5])
        close(got, ref, f"{sh} {faces}")
        f.free()
