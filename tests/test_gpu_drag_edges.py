"""The drag rate's exponentials and logarithms away from ordinary states: flat
viscosity and cross-section laws (T^0), Knudsen numbers below the Cunningham
exponential's underflow and far above 1, cold and hot gas, decays that
underflow, and cells at and around the |dv| cut-off.

Bars: |ln Re| and |ln Kn| stay below 60 here, so a rate is within about
4 x 60 x 1.1e-16 = 3e-14 of the oracle's, and a decay factor e^{-x} within
x e^{-x} <= 0.37 of that: 1e-12 relative L1 per slab, as at ordinary states
(1e-10 for the adaptive integrator, whose steps may differ)."""
import copy

import numpy as np
import pytest

from oracle import pyoracle as po

from .test_gpu_drag import compare_slabs, random_pair
from .test_gpu_hllc import gc
from .test_oracle_drag import gas_dust_thermo

pytestmark = pytest.mark.gpu

STATES = {
    # scale of rho_g, of the specific energy, of the velocities; (muTindex, sigmaTindex)
    "flat laws": (1.0, 1.0, 1.0, (0.0, 0.0)),
    "small Kn": (1e8, 1.0, 1.0, None),
    "large Kn": (1e-8, 1.0, 1.0, None),
    "cold": (1.0, 1e-8, 1e-4, None),
    "hot": (1.0, 1e8, 1e4, None),
}


@pytest.mark.parametrize("method,tol", [(4, 1e-12), (5, 1e-12), (6, 1e-10)])
@pytest.mark.parametrize("state", list(STATES))
def test_drag_rate_over_wide_states(state, method, tol):
    rho, e, v, laws = STATES[state]
    sh = (2, 3, 67)
    g, d = random_pair(sh, seed=40 + method)
    d[2:, 0, 1, :4] = d[0, 0, 1, :4] * g[2:, 0, 1, :4] / g[0, 0, 1, :4]
    d[2, 0, 1, :4] += d[0, 0, 1, :4] * np.array([1e-10, 0.9e-9, 1.1e-9, 1e-8]) / v  # around the cut-off
    for s in (g, d):
        s[0] *= rho
        s[2:] *= rho * v
        s[1] *= rho * e
    tg, td = gas_dust_thermo()
    if laws:
        tg = copy.copy(tg)
        tg.muTindex, tg.sigmaTindex = laws
    P9 = po.drag_params(tg, td)
    dv = np.sqrt(((g[2:] / g[0] - d[2:] / d[0]) ** 2).sum(0))
    u = (g[1] - .5 * (g[2:] ** 2).sum(0) / g[0]) / g[0]
    k = np.median([po.drag_k(P9, *c) for c in zip(g[0].ravel(), d[0].ravel(), dv.ravel(), u.ravel())])
    from gpuimogen_amd import abi as a

    ag, ad = (a.ThermoDetails(*[getattr(t, f) for f, _ in t._fields_]) for t in (tg, td))
    for dt in (0.3 / k, 30.0 / k, 5e3 / k):
        print(f"drag {state} method {method} dt k {dt * k:.0e}", flush=True)
        fg = gc().FluidManager(g, tg.gamma, thermoDetails=ag)
        fd = gc().FluidManager(d, td.gamma, thermoDetails=ad)
        geo = gc().GeometryManager((sh[2], sh[1], sh[0]), (0.1, 0.1, 0.1))
        gc().cudaSource2FluidDrag([fg, fd], geo, [dt, method])
        gg, dd = fg.state, fd.state
        fg.free()
        fd.free()
        rg, rd = g.copy(), d.copy()
        po.drag(rg, rd, tg, td, dt, method)
        assert np.all(np.isfinite(rg)) and np.all(np.isfinite(rd))
        compare_slabs(gg, rg, tol, f"gas {state} m{method}")
        compare_slabs(dd, rd, tol, f"dust {state} m{method}")
