"""The states of test_gpu_drag_edges (flat laws, Knudsen numbers far below and
above 1, cold and hot gas) through the explicit integrators, exponential Euler
and the learned source. The explicit ones take dt k of 1e-3 at the median, where
no stage leaves the positive range; bar as there, 1e-12 relative L1 per slab.
The learned source accepts a cell only within its residual tolerance and leaves
the others to the adaptive integrator: within 1e-6 of that everywhere."""
import copy

import numpy as np
import pytest

from gpuimogen_amd import abi, learned_drag as L
from oracle import pyoracle as po

from .test_gpu_drag import compare_slabs, random_pair
from .test_gpu_drag_edges import STATES
from .test_gpu_hllc import gc
from .test_oracle_drag import gas_dust_thermo

pytestmark = pytest.mark.gpu


def wide_pair(name, seed):
    rho, e, v, laws = STATES[name]
    g, d = random_pair((2, 3, 67), seed=seed)
    d[2:, 0, 0, :3] += 0.1 * d[0, 0, 0, :3]  # every cell moves
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
    return g, d, tg, td, k


def run(g, d, tg, td, dt, method):
    ag, ad = (abi.ThermoDetails(*[getattr(t, f) for f, _ in t._fields_]) for t in (tg, td))
    fg = gc().FluidManager(g, tg.gamma, thermoDetails=ag)
    fd = gc().FluidManager(d, td.gamma, thermoDetails=ad)
    geo = gc().GeometryManager((67, 3, 2), (0.1, 0.1, 0.1))
    gc().cudaSource2FluidDrag([fg, fd], geo, [dt, method])
    out = fg.state, fd.state
    fg.free()
    fd.free()
    return out


@pytest.mark.parametrize("method,dtks", [(0, (1e-3,)), (1, (1e-3,)), (2, (0.3, 30.0, 5e3))])
@pytest.mark.parametrize("name", list(STATES))
def test_explicit_methods(name, method, dtks):
    g, d, tg, td, k = wide_pair(name, 80 + method)
    for dtk in dtks:
        print(f"drag {name} method {method} dt k {dtk}", flush=True)
        gg, dd = run(g, d, tg, td, dtk / k, method)
        rg, rd = g.copy(), d.copy()
        po.drag(rg, rd, tg, td, dtk / k, method)
        assert np.all(np.isfinite(rg)) and np.all(np.isfinite(rd))
        compare_slabs(gg, rg, 1e-12, f"gas {name} m{method}")
        compare_slabs(dd, rd, 1e-12, f"dust {name} m{method}")


@pytest.mark.parametrize("dtk", [1e-3, 0.3, 30.0])
@pytest.mark.parametrize("name", list(STATES))
def test_learned_against_adaptive(name, dtk):
    params, norm, _ = L.load_model()
    L.set_model(params, norm)
    g, d, tg, td, k = wide_pair(name, 90)
    print(f"learned drag {name} dt k {dtk}", flush=True)
    got = run(g, d, tg, td, dtk / k, abi.DRAG_LEARNED)
    ref = run(g, d, tg, td, dtk / k, abi.DRAG_EXACT)
    compare_slabs(got[0], ref[0], 1e-6, f"gas {name}")
    compare_slabs(got[1], ref[1], 1e-6, f"dust {name}")
