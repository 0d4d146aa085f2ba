"""Ensembles larger than their second pool (1 GiB) go through it group by group:
every problem must come out bitwise as it does in an ensemble of its own, on
both sides of a group's border, eager and replayed."""
import numpy as np
import pytest

from gpuimogen_amd import ensemble as ens

pytestmark = pytest.mark.gpu


def test_groups_equal_one_group():
    # 104 x 512 x 504 x 5 doubles are 1.07e9 bytes: the last problems, of other
    # sizes, are in a second group
    nx = np.array([512] * 104 + [130, 9])
    ny = np.array([504] * 104 + [70, 300])
    states = {}
    for k, (w, h) in enumerate(((512, 504), (130, 70), (9, 300))):
        rng = np.random.default_rng(k)
        q = np.zeros((5, h, w))
        q[0] = rng.uniform(0.5, 2.0, (h, w))
        q[2], q[3] = q[0] * rng.uniform(-0.5, 0.5, (2, h, w))
        q[1] = rng.uniform(0.5, 2.0, (h, w)) / 0.4 + 0.5 * (q[2] ** 2 + q[3] ** 2) / q[0]
        states[(w, h)] = q
    big = ens.Ensemble(nx, ny, 1.0 / nx, 1.0 / ny)
    small = ens.Ensemble(nx[-3:], ny[-3:], 1.0 / nx[-3:], 1.0 / ny[-3:])
    for e in (big, small):
        for p in range(e.count):
            e.set_state(p, states[(int(e.nx[p]), int(e.ny[p]))])
        print(f"{e.count} problems", flush=True)
        e.run(1, graph=False)
        e.run(2, graph=True)
    for p, k in ((0, 0), (102, 0), (103, 0), (104, 1), (105, 2)):
        assert np.array_equal(big.state(p), small.state(k)), p
    assert np.array_equal(big.times()[[0, 104, 105]], small.times())
    big.free()
    small.free()
