"""Spreading and interpolation of every kernel against the oracle, over what
changes their path: periodic extents in which a stencil meets itself or wraps
inside one tile, faces that cut it, tiles of few and of many entries, and a
vertex numbering that overflows the binning's table of tiles."""
import numpy as np
import pytest

from oracle import oracle_py as O

pytestmark = pytest.mark.gpu

EPS = {"f64": np.finfo(np.float64).eps, "f32": np.finfo(np.float32).eps}


def _boundary(kernel, storage, shape, periodic, mesh, centres):
    from biblbm_amd.ibm import CAPSULE_SKALAK, ImmersedBoundary
    from biblbm_amd.lattice import Lattice
    rng = np.random.default_rng(5)
    u = rng.uniform(-0.02, 0.02, shape + (3,))
    L = Lattice(*shape, periodic=periodic, storage=storage, omega=1 / 0.9)
    L.put_populations(O.lbm_init_equilibrium(rng.uniform(0.99, 1.01, shape), u))
    v, t = mesh
    ib = ImmersedBoundary(L, kernel)
    sid = ib.add_shape(v, t)
    for c in centres:
        ib.add_particle(sid, CAPSULE_SKALAK, [0.02, 10.0], v * rng.uniform(0.9, 1.1, 3) + c)
    ib.init()
    return L, ib


def _check(L, ib, kernel, storage, shape, periodic):
    """One interpolation and one spreading.  A weight is off by a few units of
    the vertex type (its three factors are at most 3/4), so a cell's force by
    a few units of all vertex forces' sum, and a velocity, 64 products, by a
    few units of the largest cell velocity times the sum of 64."""
    ib.interpolate()
    vel = ib.velocities()
    _, u = L.moments()
    pos = ib.positions()
    ref = O.interpolate(kernel, u, periodic, pos)
    # the reduced storage's moments are its own, formed in its arithmetic
    assert np.abs(vel - ref).max() <= 64 * EPS[storage] * max(np.abs(u).max(), EPS[storage])
    ib.compute_forces()
    ib.spread()
    f = ib.forces()
    assert np.abs(f).max() > 0
    want = O.spread(kernel, shape, periodic, pos, f)
    got = L.force()
    assert np.abs(got - want).max() <= 8 * EPS[storage] * np.abs(f).sum(0).max()
    return got


@pytest.mark.parametrize("storage", ["f64", "f32"])
@pytest.mark.parametrize("kernel", ["tophat", "roma", "peskin"])
@pytest.mark.parametrize("n", [4, 5, 6, 7, 8])
@pytest.mark.parametrize("axis", [0, 1, 2, None])
def test_small_periodic_extents(device, axis, n, kernel, storage):
    from biblbm_amd import meshes
    shape = [13, 14, 15]
    for d in range(3):
        if axis in (d, None):
            shape[d] = n
    shape = tuple(shape)
    rng = np.random.default_rng(n)
    for cells in (1, 3, 10):  # of 42 vertices: tiles of 64 entries or fewer, 128, 420
        centres = rng.uniform(0, 1, (cells, 3)) * shape
        L, ib = _boundary(kernel, storage, shape, (1, 1, 1), meshes.icosphere(1, 1.3), centres)
        pos = ib.positions()
        if cells == 10:  # a stencil starts at every node of the small extents
            for d in range(3):
                if axis in (d, None):
                    assert len(set(O.support_base(kernel, pos[:, d]) % n)) == n
        _check(L, ib, kernel, storage, shape, (1, 1, 1))
        ib.close()
        L.close()


@pytest.mark.parametrize("storage", ["f64", "f32"])
@pytest.mark.parametrize("kernel", ["tophat", "roma", "peskin"])
@pytest.mark.parametrize("periodic", [(0, 0, 0), (1, 0, 1), (0, 1, 0)])
def test_faces_cut_the_stencil(device, periodic, kernel, storage):
    from biblbm_amd import meshes
    shape = (14, 13, 17)
    centres = [(0.2, 6.1, 8.3), (13.1, 12.2, 0.4), (5.5, 0.1, 16.2), (7.0, 7.0, 8.0)]
    L, ib = _boundary(kernel, storage, shape, periodic, meshes.icosphere(2, 2.6), centres)
    _check(L, ib, kernel, storage, shape, periodic)
    ib.close()
    L.close()


@pytest.mark.parametrize("storage", ["f64", "f32"])
@pytest.mark.parametrize("kernel", ["tophat", "peskin"])
@pytest.mark.parametrize("copies", [1, 2])
def test_scattered_numbering_overflows_the_tile_table(device, copies, kernel, storage):
    """One mesh of 40 962 vertices is binned 32 a workgroup, two 256; numbered at random
    256 touch some 2 000 tiles, twice what the workgroup's table holds."""
    from biblbm_amd import meshes
    shape = (96, 92, 94)
    v, t = meshes.icosphere(6, 41.0)
    p = np.random.default_rng(9).permutation(len(v))
    mesh = (v[p], np.argsort(p)[t].astype(np.int32))
    out = []
    for _ in range(2):
        L, ib = _boundary(kernel, storage, shape, (1, 1, 1), mesh, [(48.0, 46.0, 47.0), (48.3, 45.1, 47.9)][:copies])
        assert (len(ib.positions()) >= 65536) == (copies == 2)
        out.append(_check(L, ib, kernel, storage, shape, (1, 1, 1)))
        ib.close()
        L.close()
    assert np.array_equal(out[0], out[1])  # whatever order the atomics gave


@pytest.mark.parametrize("storage", ["f64", "f32"])
@pytest.mark.parametrize("cells", [9, 10])
def test_paired_binning_below_and_above_its_line(device, cells, storage):
    """One vertex a lane group (23 058) and eight (25 620) in the launch that
    the binning shares with the element forces, against the stages one by one."""
    from biblbm_amd import meshes
    shape = (96, 92, 94)
    centres = [(16.0 + 32 * (k % 3), 15.0 + 30 * (k // 3 % 3), 18.0 + 40 * (k // 9)) for k in range(cells)]
    out = []
    for paired in (True, False):
        L, ib = _boundary("peskin", storage, shape, (1, 1, 1), meshes.icosphere(4, 11.0), centres)
        start = ib.positions()
        if paired:
            ib.coupled_steps(6, use_graph=True)
        else:
            for _ in range(6):
                ib.step()
                L.collide_and_stream(1)
        assert np.abs(ib.positions() - start).max() > 0
        out.append((ib.positions(), ib.forces(), L.force()))
        ib.close()
        L.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)  # the same sums in the same order


@pytest.mark.parametrize("storage", ["f64", "f32"])
@pytest.mark.parametrize("kernel", ["roma", "peskin"])
@pytest.mark.parametrize("level", [5, 4])
def test_many_vertices_near_a_wall(device, level, kernel, storage):
    """Three membranes of 10 242 vertices (a lane group takes eight) and of
    2 562 (one), some of them across the blend to the top hat at the plates."""
    from biblbm_amd import meshes
    from biblbm_amd.walls import Boundary
    shape, per, plates = (60, 41, 56), (1, 0, 1), (0.5, 39.5)
    centres = [(15.0, 14.9, 14.0), (44.0, 24.7, 15.0), (30.0, 20.0, 41.0)]
    L, ib = _boundary(kernel, storage, shape, per, meshes.icosphere(level, 13.0), centres)
    ib.set_boundary(Boundary.plates(*plates))
    b = O.Boundary.plates(*plates)
    pos = ib.positions()
    assert pos[:, 1].min() < plates[0] + 1.4 and len(pos) == 3 * (10 * 4 ** level + 2)
    ib.interpolate()
    _, u = L.moments()
    assert np.abs(ib.velocities() - O.interpolate_near(kernel, u, per, pos, b)).max() <= 64 * EPS[storage] * np.abs(u).max()
    ib.compute_forces()
    ib.spread()
    f = ib.forces()
    want = O.spread_near(kernel, shape, per, pos, f, b)
    # as in _check; the blend weight, a distance of up to 20 less the half support, adds 20 units to each factor
    assert np.abs(L.force() - want).max() <= 32 * EPS[storage] * np.abs(f).sum(0).max()
    ib.close()
    L.close()
