"""The launch shapes that untuned lattices and batches take by their size
(collide order, nontemporal hints, z-segments) give bitwise the values of
the plain shape, at the sizes where the rule changes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _state(L, rng):
    u = 0.02 * rng.standard_normal(L.shape + (3,))
    L.init_equilibrium(None, u)


@pytest.mark.parametrize("storage,shape,even,odd", [
    ("f32", (64, 64, 127), (256, 1, 0), (256, 1, 0)),          # in the cache: each XCD keeps its range
    ("f32", (64, 64, 128), (256, 1, 0), (256, 1, 0)),
    ("f64", (128, 111, 124), (256, 1, 0), (256, 1, 0)),
    ("f64", (131, 128, 127), (256, 1, 0), (256, 64, 0)),       # up to 4/3 of it
    ("f16s", (437, 128, 127), (256, 1, 0), (256, 64, 0)),
    ("f64", (128, 128, 128), (256, 1, 0), (256, 1, 0)),        # with equally aligned planes
    ("f32", (224, 128, 128), (256, 1, 0), (256, 1, 0)),
    ("f16s", (432, 128, 128), (256, 1, 0), (256, 1, 0)),
    ("f16s", (580, 128, 127), (256, 64, 0), (256, 64, 0)),     # beyond
    ("f64", (144, 128, 128), (256, 16, 1), (-128, 64, 1)),     # with equally aligned planes, whole z-segments
    ("f32", (288, 128, 128), (256, 16, 1), (256, 64, 0)),
])
def test_untuned_shapes_by_size(device, storage, shape, even, odd):
    from biblbm_amd.lattice import Lattice, BOUNCE_BACK
    out = []
    for fixed in (False, True):
        L = Lattice(*shape, periodic=(1, 0, 1), storage=storage, omega=1.1)
        mask = np.zeros(shape, np.uint8)
        mask[:, [0, -1]] = BOUNCE_BACK
        L.set_mask(mask)
        L.set_body_force([1e-5, 0, 2e-5])
        for p, want in ((0, even), (1, odd)):
            assert tuple(L.launch(p).values()) == want
        if fixed:
            L.set_launch(256, True)
            assert tuple(L.launch(0).values()) == (256, 1, 0)
        _state(L, np.random.default_rng(2))
        L.collide_and_stream(5)
        out.append(L.moments())
        L.close()
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])


@pytest.mark.parametrize("storage,shape,even,odd", [
    ("f32", (128, 111, 124), (256, 1, 0), (256, 1, 0)),        # in the cache, as without
    ("f64", (131, 128, 127), (256, 16, 1), (256, 64, 0)),      # up to 4/3 of it
    ("f64", (128, 128, 128), (256, 16, 1), (256, 64, 0)),
    ("f16s", (437, 128, 127), (256, 1, 0), (256, 64, 0)),
])
def test_untuned_shapes_with_a_force_field(device, storage, shape, even, odd):
    from biblbm_amd.lattice import Lattice
    rng = np.random.default_rng(4)
    F = 1e-5 * rng.standard_normal(shape + (3,))
    out = []
    for fixed in (False, True):
        L = Lattice(*shape, periodic=(1, 1, 1), storage=storage, omega=1.1)
        L.set_force_field(F)
        for p, want in ((0, even), (1, odd)):
            assert tuple(L.launch(p).values()) == want
        if fixed:
            L.set_launch(256, True)
        _state(L, np.random.default_rng(2))
        L.collide_and_stream(3)
        out.append(L.moments())
        L.close()
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])


@pytest.mark.parametrize("storage,n", [("f64", 128), ("f32", 154), ("f16s", 194)])
def test_untuned_shapes_with_staging(device, storage, n):
    """Coupled steps beyond the cache with the velocity staging carried by
    the collision."""
    from biblbm_amd import workloads
    out = []
    for fixed in (False, True):
        w = workloads.taylor_green(storage, n=n, n_caps=2)
        w.ibm.set_fused_staging(1)
        if fixed:
            w.lattice.set_launch(256, True)
        w.ibm.coupled_steps(4, use_graph=False)
        out.append((w.ibm.positions(), w.ibm.velocities(), w.lattice.moments()[1]))
        w.ibm.close()
        w.lattice.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("storage,sides,beyond", [
    ("f64", (32, 48), False), ("f64", (96, 96, 96), True),
    ("f32", (32, 48, 64), False), ("f32", (96,) * 4, True),
    ("f16s", (96,) * 7, False), ("f16s", (96,) * 8, True),
])
def test_untuned_batches_by_size(device, storage, sides, beyond):
    """Batches whose populations fit the 256 MiB cache and whose do not,
    against another order and level of hints than the size gives them."""
    from biblbm_amd import workloads
    from biblbm_amd.ensemble import Ensemble
    size = {"f64": 8, "f32": 4, "f16s": 2}[storage]
    assert (sum(19 * size * s ** 3 for s in sides) > 256 << 20) == beyond
    out = []
    for fixed in (False, True):
        ws = [workloads.shear_box(storage, s, 0.9, 0.3, G=0.004, seed=k, radius=9.0 if s > 32 else 6.0)
              for k, s in enumerate(sides)]
        ens = Ensemble([(w.lattice, w.ibm) for w in ws])
        if fixed:
            for parity in (0, 1):
                ens.set_launch(parity, *((0, 0) if beyond else (16, 1)))
        ens.steps(4)
        assert ens.batched
        out.append([(w.ibm.positions(), w.lattice.moments()[1]) for w in ws])
        ens.close()
        for w in ws:
            w.ibm.close()
            w.lattice.close()
    for a, b in zip(*out):
        assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])
