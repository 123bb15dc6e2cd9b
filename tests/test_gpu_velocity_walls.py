"""Velocity walls on every axis against the oracle, with what the wall cells'
finite differences meet on the wall plane: other wall cells across a periodic
face or up to a plain one, bounce-back, no-dynamics and fluid cells."""
import numpy as np
import pytest

from oracle import oracle_py as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage,tol", [("f64", 1e-13), ("f32", 2e-6)])
@pytest.mark.parametrize("plane", ["whole", "framed", "mixed"])
@pytest.mark.parametrize("tangential", [(1, 1), (0, 1), (1, 0), (0, 0)])
@pytest.mark.parametrize("axis", [0, 1, 2])
def test_velocity_walls_match_the_oracle(device, axis, tangential, plane, storage, tol):
    from biblbm_amd.lattice import BOUNCE_BACK, FLUID, Lattice, NO_DYNAMICS, VELOCITY_WALL
    shape = (11, 9, 13)
    t = [d for d in range(3) if d != axis]
    per = [0, 0, 0]
    per[t[0]], per[t[1]] = tangential
    rng = np.random.default_rng(7 * axis + sum(tangential))
    mask = np.zeros(shape, np.uint8)
    at = [slice(None)] * 3
    at[axis] = [0, -1]
    mask[tuple(at)] = VELOCITY_WALL
    if plane == "framed":  # a duct: the side walls bounce back
        side = [slice(None)] * 3
        side[t[1]] = [0, -1]
        mask[tuple(side)] = BOUNCE_BACK
    elif plane == "mixed":
        kinds = rng.choice([FLUID, BOUNCE_BACK, NO_DYNAMICS, VELOCITY_WALL], shape, p=[.2, .1, .1, .6])
        mask[tuple(at)] = kinds[tuple(at)]
    f0 = O.lbm_init_equilibrium(rng.uniform(0.99, 1.01, shape), rng.uniform(-0.02, 0.02, shape + (3,)))
    F = rng.uniform(-1e-4, 1e-4, shape + (3,))
    u_lo, u_hi = rng.uniform(-0.02, 0.02, (2, 3))
    L = Lattice(*shape, periodic=per, storage=storage, omega=1 / 0.9)
    L.set_velocity_walls(axis, u_lo, u_hi)
    L.set_mask(mask)
    L.set_force_field(F)
    L.put_populations(f0)
    wu = np.concatenate([u_lo, u_hi])
    seen = (mask == FLUID) | (mask == VELOCITY_WALL)
    ref = f0
    for _ in range(3):  # both population layouts
        L.collide_and_stream(1)
        ref = O.lbm_run(ref, F, np.zeros(shape), mask, per, 1 / 0.9, 1 / 0.9, 1, axis, wu)
        # round-off of a few steps; FP32's is of the stored deviations, of order 0.02
        assert np.abs(L.get_populations() - ref)[seen].max() <= tol
    L.close()
