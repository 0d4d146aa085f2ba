"""The sweeps' launch shapes at the lengths where they change.

X lines are swept whole, or split into parts of at most 64 K - 8 cells with
K = 1..4 cells per lane, chosen by length and line count; Y and Z columns are
cut into segments, in place or, paired with another sweep of the step, through
a second state array. Each is compared with the CPU oracle at the edges of its
range; the tolerance is the fluid step's own (relative L1 1e-12 per variable).
A step through the second array and one in place run the same arithmetic on
the same cells, so they agree bitwise.
"""
import ctypes

import numpy as np
import pytest

from gpuimogen_amd import abi, gpuclass as gc
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu

G = 5.0 / 3.0
MODES = {"const": (abi.extrapConstant, po.BC_CONST), "circular": (abi.circular, po.BC_CIRCULAR),
         "mirror": (abi.mirror, po.BC_MIRROR)}


def state(sh, seed):
    rng = np.random.default_rng(seed)
    q = np.zeros((5,) + sh)
    q[0] = rng.uniform(0.3, 2.0, sh)
    v = rng.uniform(-1.0, 1.0, (3,) + sh)
    q[1] = rng.uniform(0.2, 2.0, sh) / (G - 1) + 0.5 * q[0] * (v ** 2).sum(0)
    q[2:] = q[0] * v
    return q


def close(got, ref, what):
    rel = np.abs(got - ref).reshape(5, -1).sum(1) / np.abs(ref).reshape(5, -1).sum(1)
    print(what, rel, flush=True)
    assert np.all(rel <= 1e-12), (what, rel)


# (cells per line, lines): K = 1 parts of 56, 2 of 120, 3 of 184, 4 of 248
LINES = [(56, 3), (57, 3), (64, 3), (65, 3), (113, 2), (256, 204), (256, 206), (257, 2), (257, 800), (368, 770),
         (369, 515), (384, 2), (448, 2), (449, 2), (496, 515), (497, 515), (552, 2), (553, 3), (736, 400), (737, 2),
         (920, 320), (921, 2), (961, 2), (1024, 1), (1024, 260)]


@pytest.mark.parametrize("method", [abi.METHOD_HLLC, abi.METHOD_HLL])
@pytest.mark.parametrize("nx,lines", LINES)
def test_x_lines(nx, lines, method):
    q = state((1, lines, nx), nx + lines)
    print(f"X sweep of {lines} lines of {nx}, method {method}", flush=True)
    f = gc.FluidManager(q, G)
    gm = gc.GeometryManager((nx, lines, 1), (0.01, 0.01, 1.0))
    gc.cudaFluidStep([0.002, 1, G, 1e-8, method, 1], f, gm, limiter=abi.LIMITER_VANLEER)
    po.fluid_update_1d(q, 1, 0.2, G, method=method, limiter=po.LIM_VANLEER, rhomin=1e-8)
    close(f.state, q, f"x {nx} {method}")
    f.free()


# 2D (march paired with X), 3D (Y paired with Z), a plane whose X is not swept
# (nothing to pair with), short columns, ragged rows
STEPS = [(1, 5, 70), (1, 67, 33), (1, 9, 1024), (1, 300, 3), (40, 1, 12), (17, 18, 19), (5, 4, 66), (33, 70, 21)]


@pytest.mark.parametrize("bc", sorted(MODES))
@pytest.mark.parametrize("sh", STEPS)
def test_steps_in_every_order(sh, bc):
    nz, ny, nx = sh
    h = (0.01, 0.012, 0.014)
    mode, omode = MODES[bc]
    if bc != "circular" and min(n for n in sh if n > 3) < 12:
        pytest.skip("faces of a mirror or const pair need 12 cells between them to be set in one pass")
    f = gc.FluidManager(state(sh, nx), G, bc_modes=(mode,) * 6)
    ref = state(sh, nx)
    gm = gc.GeometryManager((nx, ny, nz), h)
    for it in range(6):
        for sign in (1, -1):
            print(f"step {sh} {bc} order {it} {sign}", flush=True)
            gc.fluidstep([f], None, None, None, [2e-4, 1, sign, it, abi.METHOD_HLLC], gm)
            po.fluidstep(ref, h, 2e-4, sign, it, G, po.HLLC, po.LIM_OSPRE, modes=(omode,) * 6)
    close(f.state, ref, f"{sh} {bc}")
    f.free()


@pytest.mark.parametrize("method", [abi.METHOD_HLLC, abi.METHOD_HLL])
def test_second_array_equals_in_place(method):
    # 5 slabs of 124 x 120 x 119 are above the allocation-free step's 64 MiB:
    # it works in place where performFluidUpdate_3D goes through a second array
    sh = (119, 120, 124)
    q = state(sh, 7)
    gm = gc.GeometryManager(sh[::-1], (0.01, 0.012, 0.014))
    out = []
    for entry in ("performFluidUpdate_3D", "performFluidUpdate_3D_noalloc"):
        f = gc.FluidManager(q, G, bc_modes=(abi.extrapConstant,) * 6)
        t = abi.ParallelTopology()
        for i in range(3):
            t.nproc[i] = 1
        for it in (0, 4):
            p = gc.step_params(1e-4, 1, it, method, gm, G, f.MINMASS)
            print(entry, it, flush=True)
            abi.call(entry, f.arrays(), ctypes.byref(t), p, *([None] if entry.endswith("3D") else []))
        out.append(f.state)
        f.free()
    assert np.array_equal(out[0], out[1])
