"""X lines of 384 cells, whole or in parts by method, limiter and line count: on
either side of the rule's edge (512 lines), against the CPU oracle (relative L1
1e-12 per variable, the fluid step's own), alone and in steps with mirrors, whose
ghosts the whole-line sweep sets and the boundary launch sets after the parts."""
import numpy as np
import pytest

from gpuimogen_amd import abi, gpuclass as gc
from oracle import pyoracle as po

from .test_gpu_sweep_shapes import G, close, state

pytestmark = pytest.mark.gpu

METHODS = {abi.METHOD_HLLC: po.HLLC, abi.METHOD_HLL: po.HLL}
LIMITERS = {abi.LIMITER_OSPRE: po.LIM_OSPRE, abi.LIMITER_VANLEER: po.LIM_VANLEER, abi.LIMITER_MC: po.LIM_MC}


@pytest.mark.parametrize("lines", [511, 512])
@pytest.mark.parametrize("limiter", sorted(LIMITERS))
@pytest.mark.parametrize("method", sorted(METHODS))
def test_sweep_and_steps(method, limiter, lines):
    what = f"{lines} lines of 384, method {method}, limiter {limiter}"
    print(what, flush=True)
    q = state((1, lines, 384), lines)
    h = (0.01, 0.012, 0.014)
    gm = gc.GeometryManager((384, lines, 1), h)
    f = gc.FluidManager(q, G, bc_modes=(abi.mirror,) * 6)
    ref = q.copy()
    gc.cudaFluidStep([0.002, 1, G, 1e-8, method, 1], f, gm, limiter=limiter)
    po.fluid_update_1d(ref, 1, 0.2, G, method=METHODS[method], limiter=LIMITERS[limiter], rhomin=1e-8)
    close(f.state, ref, what)
    f.set_state(q)
    ref = q.copy()
    for it in (0, 3):
        gc.fluidstep([f], None, None, None, [2e-4, 1, 1, it, method], gm, limiter=limiter)
        po.fluidstep(ref, h, 2e-4, 1, it, G, METHODS[method], LIMITERS[limiter], modes=(po.BC_MIRROR,) * 6)
    close(f.state, ref, "steps of " + what)
    f.free()
