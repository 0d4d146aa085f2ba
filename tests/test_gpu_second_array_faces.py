"""Steps through the second state array beyond periodic, const and mirror faces
with Ospre and van Leer: boundary launches that act on the state where it is between the
paired sweeps (outflow, linear, freebalance, static cells, and const and mirror
faces too close together for the sweeps to set), and the limiters that are
chosen at run time in tiles, parts and out-of-place marches. Against the CPU
oracle (relative L1 1e-12 per variable, the fluid step's own), or bitwise
against the allocation-free step, which works in place above its 64 MiB."""
import ctypes

import numpy as np
import pytest

from gpuimogen_amd import abi, gpuclass as gc
from oracle import pyoracle as po

from .test_gpu_sweep_shapes import G, close, state

pytestmark = pytest.mark.gpu

H = (0.01, 0.012, 0.014)
METHODS = {abi.METHOD_HLLC: po.HLLC, abi.METHOD_HLL: po.HLL}
OUT, CON, MIR = (abi.outflow, po.BC_OUTFLOW), (abi.extrapConstant, po.BC_CONST), (abi.mirror, po.BC_MIRROR)
LIN, CIR = (abi.extrapLinear, po.BC_LINEAR), (abi.circular, po.BC_CIRCULAR)


def smooth(sh):
    """Gentle waves: linear extrapolation and static cells keep them physical."""
    z, y, x = np.meshgrid(*(np.arange(n) / n for n in sh), indexing="ij")
    q = np.zeros((5,) + sh)
    q[0] = 1 + 0.2 * np.sin(2 * np.pi * (x + y + z) + 0.3)
    for k, a in enumerate((x + 2 * y, y - z, z + x)):
        q[2 + k] = q[0] * 0.3 * np.sin(2 * np.pi * a + k + 0.1)
    q[1] = (1 + 0.2 * np.cos(2 * np.pi * (x - y + z) + 0.2)) / (G - 1) + 0.5 * (q[2:] ** 2).sum(0) / q[0]
    return q


def steps(q, faces, method, limiter, olimiter, what):
    nz, ny, nx = q.shape[1:]
    f = gc.FluidManager(q, G, bc_modes=(faces[0][0], faces[1][0]) * 3)
    gm = gc.GeometryManager((nx, ny, nz), H)
    for it in range(3):  # each swept direction last once
        for sign in (1, -1):
            print(f"{what}, order {it} {sign}", flush=True)
            gc.fluidstep([f], None, None, None, [1e-4, 1, sign, it, method], gm, limiter=limiter)
            po.fluidstep(q, H, 1e-4, sign, it, G, METHODS[method], olimiter, modes=(faces[0][1], faces[1][1]) * 3)
    close(f.state, q, what)
    f.free()


# planes (a Y sweep paired with X) and boxes (Y with Z), parts and marches
PAIRED = [(1, 100, 70), (1, 900, 600), (66, 20, 30), (20, 70, 64), (90, 110, 100)]


@pytest.mark.parametrize("method", sorted(METHODS))
@pytest.mark.parametrize("faces", [(OUT, OUT), (OUT, CON), (MIR, OUT), (LIN, CON)])
@pytest.mark.parametrize("sh", PAIRED)
def test_other_faces(sh, faces, method):
    steps(smooth(sh), faces, method, abi.LIMITER_OSPRE, po.LIM_OSPRE, f"{sh} faces {faces[0][0]} {faces[1][0]}, method {method}")


@pytest.mark.parametrize("faces", [CON, MIR])
@pytest.mark.parametrize("sh", [(1, 100, 10), (1, 100, 11), (1, 13, 600), (1, 70, 13), (10, 70, 20), (12, 13, 90), (70, 12, 11)])
def test_faces_set_one_after_the_other(sh, faces):
    steps(smooth(sh), (faces, faces), abi.METHOD_HLLC, abi.LIMITER_VANLEER, po.LIM_VANLEER, f"{sh} face {faces[0]}")


@pytest.mark.parametrize("method", sorted(METHODS))
@pytest.mark.parametrize("limiter", ["MINMOD", "SUPERBEE", "VANALBADA", "MC", "ZERO"])
@pytest.mark.parametrize("sh", [(1, 40, 60), (1, 100, 300), (1, 600, 1024), (64, 20, 30), (90, 110, 100)])
def test_limiters_chosen_at_run_time(sh, limiter, method):
    # (van Albada's slope between equal states is NaN in the reference's formula:
    # a state without any, and no ghosts that are copies)
    q = state(sh, sum(sh))
    q[2:] *= 0.5
    steps(q, (CIR, CIR), method, getattr(abi, "LIMITER_" + limiter),
          getattr(po, "LIM_" + limiter), f"{sh} {limiter}, method {method}")


@pytest.mark.parametrize("method", sorted(METHODS))
@pytest.mark.parametrize("kind", ["outflow", "statics", "freebalance"])
def test_boundary_data_in_the_second_array(kind, method):
    sh = (119, 120, 124)  # 5 slabs are above 64 MiB
    n = 119 * 120 * 124
    q = smooth(sh)
    gm = gc.GeometryManager(sh[::-1], (0.01, 0.012, 0.014))
    rng = np.random.default_rng(2)
    face = {"outflow": abi.outflow, "statics": abi.extrapConstant, "freebalance": abi.freebalance}[kind]
    phi = 0.01 * np.arange(119).reshape(119, 1, 1) + np.zeros(sh)
    idx = rng.choice(n, 500, replace=False).astype(np.float64)
    out = []
    for entry in ("performFluidUpdate_3D", "performFluidUpdate_3D_noalloc"):
        modes = (abi.extrapConstant,) * 4 + (face, abi.extrapConstant)
        if kind == "outflow":
            modes = (face,) * 6
        f = gc.FluidManager(q, G, bc_modes=modes)
        arr = f.arrays()
        pot, tab = gc.GPU_Type(phi), gc.GPU_Type(np.stack([idx, np.full(500, 1.3), np.full(500, 0.5)]))
        pm, tm = pot.mgarray(), tab.mgarray()
        keep = []
        for k in range(5):
            bd = abi.ImogenBoundaryData()
            if kind == "freebalance" and k == 0:
                bd.gravpot = ctypes.pointer(pm)
                bd.gamma = G
            if kind == "statics" and k < 2:
                bd.statics = ctypes.pointer(tm)
                bd.compOffset[0], bd.compOffset[1] = 0.0, 500.0
            keep.append(bd)
            arr[k].boundaryConditions.externalData = ctypes.cast(ctypes.pointer(bd), ctypes.c_void_p)
        topo = abi.ParallelTopology()
        for i in range(3):
            topo.nproc[i] = 1
        for it in range(3):
            for sign in (1, -1):
                p = gc.step_params(1e-4, sign, it, method, gm, G, f.MINMASS)
                print(f"{entry} {kind}, method {method}, order {it} {sign}", flush=True)
                abi.call(entry, arr, ctypes.byref(topo), p, *([None] if entry.endswith("3D") else []))
        out.append(f.state)
        for a in (f, pot, tab):
            a.free()
    assert np.isfinite(out[0]).all()
    assert np.array_equal(out[0], out[1])
