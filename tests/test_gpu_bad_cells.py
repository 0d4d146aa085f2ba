"""A NaN cell in a finite state: a sweep spreads it exactly as far as the
reference's formulas do (a NaN difference gives no slope, so only the cell's own
faces and fluxes are lost), and every other cell stays within the fluid step's
tolerance of the oracle (relative L1 1e-12 per variable)."""
import numpy as np
import pytest

from gpuimogen_amd import abi, gpuclass as gc
from oracle import pyoracle as po

from .test_gpu_sweep_shapes import G, close, state

pytestmark = pytest.mark.gpu

METHODS = {abi.METHOD_HLLC: po.HLLC, abi.METHOD_HLL: po.HLL}
LIMITERS = {abi.LIMITER_OSPRE: po.LIM_OSPRE, abi.LIMITER_VANLEER: po.LIM_VANLEER}
# X lines whole (K = 1, 2, 4, 6) and in parts (K = 1, 3, 4), Y and Z by tiles and marches
SWEEPS = [(1, 60, 3, 1), (1, 128, 1100, 1), (1, 256, 1100, 1), (1, 384, 4500, 1), (1, 100, 3, 1), (1, 300, 700, 1),
          (1, 450, 700, 1), (2, 20, 40, 3), (2, 70, 100, 3), (3, 9, 4, 50), (3, 65, 4, 130)]


def sweep_with_bad_cells(q, direction, method, limiter, bad=True, dt=0.001, rhomin=1e-8):
    """The sweep on the GPU and by the oracle; bad: a cell that is NaN in every
    variable and one whose energy alone is, half a line apart."""
    axis = 4 - direction
    n = q.shape[axis]
    line = [0] * 4
    if bad:
        for at, slabs in ((n // 5, slice(None)), (n // 5 + n // 2, 1)):
            line[axis] = at
            q[(slabs,) + tuple(line[1:])] = np.nan
    f = gc.FluidManager(q, G)
    gm = gc.GeometryManager(q.shape[:0:-1], (0.01, 0.01, 0.01))
    gc.cudaFluidStep([dt, 1, G, rhomin, method, direction], f, gm, limiter=limiter)
    po.fluid_update_1d(q, direction, dt / 0.01, G, method=METHODS[method], limiter=LIMITERS[limiter], rhomin=rhomin)
    got = f.state
    f.free()
    return got, q


def compare(got, ref, what):
    lost = np.isnan(ref)
    print(what, "NaN per variable", lost.reshape(5, -1).sum(1), np.isnan(got).reshape(5, -1).sum(1), flush=True)
    assert np.array_equal(np.isnan(got), lost), what
    close(np.where(lost, 0.0, got), np.where(lost, 0.0, ref), what)


@pytest.mark.parametrize("limiter", sorted(LIMITERS))
@pytest.mark.parametrize("method", sorted(METHODS))
@pytest.mark.parametrize("direction,nx,ny,nz", SWEEPS)
def test_nan_cell_spreads_as_in_the_reference(direction, nx, ny, nz, method, limiter):
    what = f"sweep {direction} of {nx} x {ny} x {nz}, method {method}, limiter {limiter}"
    print(what, flush=True)
    q = state((nz, ny, nx), nx + ny + nz)
    q[2:] *= 0.3  # subsonic: with the energy kept, the pressure only grows
    got, ref = sweep_with_bad_cells(q, direction, method, limiter)
    assert np.isnan(ref).any() and np.isfinite(ref).any()
    compare(got, ref, what)


@pytest.mark.parametrize("flow", [4.0, -4.0])
@pytest.mark.parametrize("limiter", sorted(LIMITERS))
@pytest.mark.parametrize("method", sorted(METHODS))
@pytest.mark.parametrize("direction,nx,ny,nz", SWEEPS)
def test_nan_cell_in_supersonic_flow(direction, nx, ny, nz, method, limiter, flow):
    # where every wave of the good side leaves the bad cell, the interface's flux
    # is that side's own: the bad side must not reach its sound speed
    what = f"flow {flow}, sweep {direction} of {nx} x {ny} x {nz}, method {method}, limiter {limiter}"
    print(what, flush=True)
    q = state((nz, ny, nx), nx + ny + nz)
    ke = 0.5 * (q[2:] ** 2).sum(0) / q[0]
    q[2:] *= 0.3
    q[1 + direction] += flow * q[0]
    q[1] += 0.5 * (q[2:] ** 2).sum(0) / q[0] - ke
    got, ref = sweep_with_bad_cells(q, direction, method, limiter)
    compare(got, ref, what)


@pytest.mark.parametrize("limiter", sorted(LIMITERS))
@pytest.mark.parametrize("method", sorted(METHODS))
@pytest.mark.parametrize("direction,nx,ny,nz", SWEEPS)
def test_densities_whose_product_underflows(direction, nx, ny, nz, method, limiter):
    # products of two densities underflow in these units; momenta and pressures,
    # whose squares the formulas take, stay in the double range
    rho, v = 1e-160, 1e10
    what = f"density {rho}, sweep {direction} of {nx} x {ny} x {nz}, method {method}, limiter {limiter}"
    print(what, flush=True)
    q = state((nz, ny, nx), nx + ny + nz)
    q *= np.array([rho, rho * v * v, rho * v, rho * v, rho * v]).reshape(5, 1, 1, 1)
    got, ref = sweep_with_bad_cells(q, direction, method, limiter, bad=False, dt=0.001 / v, rhomin=1e-8 * rho)
    assert np.isfinite(ref).all()
    compare(got, ref, what)
