"""An ensemble whose states exceed the second pool's 2 GiB, in two groups: every
problem bitwise as in a small ensemble, on both sides of the groups' border."""
import numpy as np
import pytest

from gpuimogen_amd import ensemble as ens

pytestmark = pytest.mark.gpu


def test_two_groups_equal_one():
    # 208 x 512 x 504 x 5 doubles are 2.147e9 bytes (2 GiB is 2.1475e9): the small
    # problems after them begin a second group
    nx = np.array([512] * 208 + [200, 130, 9])
    ny = np.array([504] * 208 + [120, 70, 300])
    states = {}
    for k, (w, h) in enumerate(((512, 504), (200, 120), (130, 70), (9, 300))):
        rng = np.random.default_rng(k)
        q = np.zeros((5, h, w))
        q[0] = rng.uniform(0.5, 2.0, (h, w))
        q[2], q[3] = q[0] * rng.uniform(-0.5, 0.5, (2, h, w))
        q[1] = rng.uniform(0.5, 2.0, (h, w)) / 0.4 + 0.5 * (q[2] ** 2 + q[3] ** 2) / q[0]
        states[(w, h)] = q
    big = ens.Ensemble(nx, ny, 1.0 / nx, 1.0 / ny)
    small = ens.Ensemble(nx[-4:], ny[-4:], 1.0 / nx[-4:], 1.0 / ny[-4:])
    for e in (big, small):
        for p in range(e.count):
            e.set_state(p, states[(int(e.nx[p]), int(e.ny[p]))])
        print(f"{e.count} problems", flush=True)
        e.run(1, graph=False)
        e.run(2, graph=True)
    for p, k in ((0, 0), (207, 0), (208, 1), (209, 2), (210, 3)):
        assert np.array_equal(big.state(p), small.state(k)), p
    big.free()
    small.free()
