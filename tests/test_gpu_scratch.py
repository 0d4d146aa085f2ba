"""The scratch block that holds the sweeps' second state array: a device loop goes
on, bitwise as the host loop, when another fluid's step has made the block grow
and after GPU_ctrl_reset has dropped it."""
import numpy as np
import pytest

from gpuimogen_amd import abi, gpuclass as gc, imogen

from .test_gpu_sweep_shapes import G, state

pytestmark = pytest.mark.gpu


def test_loop_outlives_its_scratch_block():
    sh = (30, 70, 64)
    h = (0.01, 0.012, 0.014)
    gm = gc.GeometryManager(sh[::-1], h)
    q = state(sh, 3)
    q[2:] *= 0.1
    fa, fb = (gc.FluidManager(q, G, bc_modes=(abi.extrapConstant,) * 6) for _ in range(2))
    big = gc.FluidManager(state((90, 100, 110), 4), G)
    gb = gc.GeometryManager((110, 100, 90), h)
    sim = imogen.Simulation([fa], [abi.METHOD_HLLC], gm)
    for _ in range(24):
        sim.step()
    abi.call("GPU_ctrl_reset")
    loop = imogen.DeviceLoop([fb], [abi.METHOD_HLLC], gm)
    print("loop, small block", flush=True)
    loop.run(8)
    print("step that makes the block grow", flush=True)
    gc.fluidstep([big], None, None, None, [1e-4, 1, 1, 0, abi.METHOD_HLLC], gb)
    loop.run(8)
    abi.call("GPU_ctrl_reset")
    print("loop, no block", flush=True)
    loop.run(8)
    assert loop.time == sim.time
    assert np.array_equal(fa.state, fb.state)
    loop.free()
    for f in (fa, fb, big):
        f.free()
