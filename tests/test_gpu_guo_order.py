"""The curved-wall pass where its workgroups are dealt in runs over the
XCDs: node counts below one round of runs, past one, and past several, each
with a remainder, after odd and even step counts (both population layouts)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,rounds", [(7, 0), (31, 1), (65, 3)])
def test_guo_wall_over_all_workgroup_runs(device, nx, rounds):
    from biblbm_amd.lattice import Lattice
    from biblbm_amd.walls import Boundary, GuoWall, outside_mask
    from oracle import oracle_py as O
    shape, per = (nx, 29, 29), (1, 0, 0)
    b, ob = Boundary.pipe(14.0, 14.0, 11.6), O.Boundary.pipe(14.0, 14.0, 11.6)
    mask = outside_mask(b, shape, 1.0)
    rng = np.random.default_rng(nx)
    f0 = O.lbm_init_equilibrium(rng.uniform(0.99, 1.01, shape), rng.uniform(-0.02, 0.02, shape + (3,)))
    w = O.guo_wall_nodes(shape, ob)
    n = len(w["cell"])
    assert n // 2048 == rounds and n % 64  # 32 workgroups of 64 nodes are one round
    vel = np.tile([0.01, 0.0, 0.0], (n, 1))
    L = Lattice(*shape, periodic=per, omega=1 / 0.8)
    L.set_mask(mask)
    L.put_populations(f0)
    W = GuoWall(L, b)
    W.set_wall_velocity([0.01, 0.0, 0.0])
    W.insert()
    chk = mask == 0
    chk[np.unravel_index(w["cell"], shape)] = True
    for steps in (1, 2):
        L.collide_and_stream(1)
        ref = O.lbm_run(f0, np.zeros(shape + (3,)), np.zeros(shape), mask, per, 1 / 0.8, 1 / 0.8, steps, guo=(w, vel))
        # the bar of the curved-wall tests: FP64 round-off of a step or two
        assert np.abs(L.get_populations() - ref)[chk].max() <= 1e-12 * np.abs(ref[chk]).max()
    W.close()
    L.close()
