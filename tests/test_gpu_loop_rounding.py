"""A sweep that folds the CFL minimum is a kernel instance of its own. Products and
sums are contracted within one expression only, so it rounds as the plain one: the
device loop (folding) and the host loop (not) agree bitwise in every scheme."""
import numpy as np
import pytest

from gpuimogen_amd import abi, gpuclass as gc, imogen

from .test_gpu_second_array_faces import smooth
from .test_gpu_sweep_shapes import G

pytestmark = pytest.mark.gpu

# X whole (K = 1, 2, 4, 6) and in parts (K = 1, 3, 4), tiles whole and in parts, marches
SHAPES = [(1, 40, 60), (20, 20, 256), (9, 130, 128), (2, 300, 384), (1, 70, 300), (1, 600, 700), (1, 700, 420), (90, 110, 100)]


@pytest.mark.parametrize("limiter", [abi.LIMITER_OSPRE, abi.LIMITER_VANLEER, abi.LIMITER_MC])
@pytest.mark.parametrize("method", [abi.METHOD_HLLC, abi.METHOD_HLL])
@pytest.mark.parametrize("sh", SHAPES)
def test_folding_rounds_alike(sh, method, limiter):
    print(f"{sh} method {method} limiter {limiter}", flush=True)
    gm = gc.GeometryManager(sh[::-1], (0.01, 0.012, 0.014))
    fa, fb = (gc.FluidManager(smooth(sh), G, bc_modes=(abi.extrapConstant,) * 6) for _ in range(2))
    sim = imogen.Simulation([fa], [method], gm, limiter=limiter)
    loop = imogen.DeviceLoop([fb], [method], gm, limiter=limiter)
    for _ in range(4):  # every direction last at least once
        sim.step()
    loop.run(4)
    assert loop.time == sim.time
    assert np.array_equal(fa.state, fb.state)
    loop.free()
    fa.free()
    fb.free()
