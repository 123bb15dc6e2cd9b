"""Moments of lattices just within and just past the size that keeps its
readback buffer, read repeatedly, between steps and by several threads."""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(128, 128, 64), (128, 128, 65)])
def test_moments_are_those_of_the_populations(device, shape):
    from biblbm_amd.lattice import Lattice
    rng = np.random.default_rng(shape[2])
    L = Lattice(*shape, periodic=(1, 1, 1), omega=1 / 0.8)
    L.init_equilibrium(rng.uniform(0.99, 1.01, shape), rng.uniform(-0.02, 0.02, shape + (3,)))
    for _ in range(2):
        L.collide_and_stream(1)
        want = 1.0 + L.get_populations().sum(-1)
        with ThreadPoolExecutor(4) as pool:
            got = [f.result() for f in [pool.submit(L.moments) for _ in range(4)]]
        for rho, u in got:
            # two orders of a sum of 19 populations of at most 1/3
            assert np.abs(rho - want).max() <= 20 * np.finfo(float).eps
            assert np.array_equal(u, got[0][1])
    L.close()
