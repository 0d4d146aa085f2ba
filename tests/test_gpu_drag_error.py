"""The drag source's rounding error. The kernels use their own exponential,
logarithm and quotients; a call is to be no further from the formulas' exact
values than plain FP64 arithmetic with library functions and IEEE divisions is.
Both errors are measured here against the same formulas in 80-bit arithmetic, as
means over 53 thousand cells (a mean of that many roundings is known to about
half a per cent; FMA contraction and the order of products move it by two or
three), and the kernel's may be a tenth above the plain formula's. At dt k of 0.4
a rate with twice the plain formula's error shows as 1.15 or more in the dust."""
import numpy as np
import pytest

from oracle import pyoracle as po

from .test_gpu_drag import random_pair, run_gpu_drag
from .test_oracle_drag import gas_dust_thermo

pytestmark = pytest.mark.gpu

SHAPE = (30, 35, 51)


def rate(P, rg, rd, s, u):
    lT = np.log(P[3] * u)
    Re = P[5] * rg * s * np.exp(P[1] * lT)
    Kn = P[4] * np.exp(P[2] * lT) / rg
    cunningham = 1 + Kn * (1.142 + 0.558 * np.exp(-0.999 / Kn))
    return (3 / Re + .45 * np.exp(-.319 * np.log(Re)) + .0509 * Re / (8710 + Re)) / cunningham * s * (rg + rd) * P[6]


def drag(gas, dust, P, dt, method, T):
    """One call in the number type T: exponential Euler (2), LogTrap2 (4) or LogTrap3 (5)."""
    g, d, P, dt = gas.astype(T), dust.astype(T), P.astype(T), T(dt)
    rg, rd = g[0], d[0]
    dv = g[2:] / rg - d[2:] / rd
    s = np.sqrt(dv[0] * dv[0] + dv[1] * dv[1] + dv[2] * dv[2])
    u = (g[1] - .5 * (g[2] * g[2] + g[3] * g[3] + g[4] * g[4]) / rg) / rg
    mu = rd / (rg + rd)
    k = rate(P, rg, rd, s, u)
    if method != 2:
        def at(a):
            return rate(P, rg, rd, s * np.exp(-dt * a), u - .5 * s * s * mu * np.expm1(-2 * a * dt))
        ksum = k + at(k)
        k = .5 * ksum if method == 4 else ksum / T(6) + T(2) / T(3) * at(.25 * ksum)
    f = np.exp(-dt * k)
    stick = (g[2:] + d[2:]) / (rg + rd)
    old = (d[2:] ** 2).sum(0)
    g[2:] = rg * stick + dv * f * (mu * rg)
    d[2:] = rd * stick - dv * f * (mu * rg)
    g[1] -= .5 * ((d[2:] ** 2).sum(0) - old) / rd
    return g, d


@pytest.mark.parametrize("method", [2, 4, 5])
@pytest.mark.parametrize("dtk", [1e-3, 0.1, 0.4])
def test_error_is_the_plain_formulas(method, dtk):
    gas, dust = random_pair(SHAPE, seed=3 + method)
    dust[2:, 0, 0, :3] += 0.1 * dust[0, 0, 0, :3]  # every cell moves
    P = po.drag_params(*gas_dust_thermo())
    wide = np.longdouble
    assert np.finfo(wide).nmant >= 63
    dv = gas[2:] / gas[0] - dust[2:] / dust[0]
    u = (gas[1] - .5 * (gas[2:] ** 2).sum(0) / gas[0]) / gas[0]
    dt = dtk / float(np.median(rate(P, gas[0], dust[0], np.sqrt((dv ** 2).sum(0)), u)))
    ref = drag(gas, dust, P, dt, method, wide)
    plain = drag(gas, dust, P, dt, method, np.float64)
    got = run_gpu_drag(gas, dust, dt, method, SHAPE)
    for name, x, y, r, slabs in (("gas", got[0], plain[0], ref[0], slice(1, 5)),
                                 ("dust", got[1], plain[1], ref[1], slice(2, 5))):
        scale = np.abs(r[slabs]).sum()
        kernel, formula = (float(np.abs(a[slabs] - r[slabs]).sum() / scale) for a in (x, y))
        print(f"method {method} dt k {dtk} {name}: error {kernel:.3e}, plain formula {formula:.3e}", flush=True)
        assert kernel <= 1.1 * formula
