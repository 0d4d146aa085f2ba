"""Gas cells without internal energy, and dust moving through them: T = 0, where
the powers of the temperature are 0, 1 or infinite by the laws' exponents. Every
call reports such cells; they are updated as the formula falls (finite, at rest
with the dust, or NaN), and the other cells as without them."""
import copy

import numpy as np
import pytest

from gpuimogen_amd import abi
from oracle import pyoracle as po

from .test_gpu_drag import random_pair
from .test_gpu_hllc import gc
from .test_oracle_drag import gas_dust_thermo

pytestmark = pytest.mark.gpu


# (muTindex, sigmaTindex): viscosity and cross section ~ T^index
@pytest.mark.parametrize("laws", [(0.7, 0.2), (0.0, 0.0), (0.0, 0.2), (0.0, -0.3), (-0.5, 0.2), (-0.5, 0.0), (0.7, -0.3)])
@pytest.mark.parametrize("method", [0, 1, 2, 4, 5])
def test_cells_at_zero_temperature(method, laws):
    if method < 2 and laws == (0.0, -0.3):
        pytest.skip("the explicit integrators leave the finite range in most ordinary cells too")
    sh = (2, 3, 67)
    g, d = random_pair(sh, seed=60)
    g[1:, 1, 2, 10:30] = 0.0  # at rest, so that the internal energy is exactly 0
    tg, td = gas_dust_thermo()
    tg = copy.copy(tg)
    tg.muTindex, tg.sigmaTindex = laws
    ag, ad = (abi.ThermoDetails(*[getattr(t, f) for f, _ in t._fields_]) for t in (tg, td))
    print(f"cold gas, laws {laws}, method {method}", flush=True)
    fg = gc().FluidManager(g, tg.gamma, thermoDetails=ag)
    fd = gc().FluidManager(d, td.gamma, thermoDetails=ad)
    geo = gc().GeometryManager((67, 3, 2), (0.1, 0.1, 0.1))
    with pytest.raises(abi.ImogenError) as e:
        gc().cudaSource2FluidDrag([fg, fd], geo, [1e-4, method])
    assert e.value.code == abi.ERROR_CRASH
    got = np.stack([fg.state, fd.state])
    fg.free()
    fd.free()
    po.drag(g, d, tg, td, 1e-4, method)
    ref = np.stack([g, d])
    lost = np.isnan(ref)
    assert np.array_equal(np.isnan(got), lost), (np.isnan(got).sum(), lost.sum())
    fin = np.isfinite(ref)
    assert np.array_equal(got[~fin & ~lost], ref[~fin & ~lost])
    rel = np.abs(got[fin] - ref[fin]).sum() / np.abs(ref[fin]).sum()
    print(f"{lost.sum()} values NaN, relative L1 of the others {rel:.2e}", flush=True)
    assert rel <= 1e-12
