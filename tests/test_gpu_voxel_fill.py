"""The voxelised phase against the oracle's sorted column fill, where the
bit-parity fill could differ: hits exactly on nodes, between the last two
nodes, on the last one and beyond it, columns of one word of nodes more or
less, membranes across the periodic faces, a node that keeps its value."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BOX = np.array([[x, y, z] for x in (0, 1) for y in (0, 1) for z in (0, 1)], float)
BOX_TRI = np.array([[0, 1, 3], [0, 3, 2], [4, 6, 7], [4, 7, 5], [0, 4, 5], [0, 5, 1],
                    [2, 3, 7], [2, 7, 6], [0, 2, 6], [0, 6, 4], [1, 5, 7], [1, 7, 3]], np.int32)


@pytest.mark.parametrize("nz", [31, 32, 33, 64, 65])
@pytest.mark.parametrize("per_z", [0, 1])
def test_phase_of_boxes_against_the_sorted_fill(device, nz, per_z):
    from biblbm_amd.ibm import ImmersedBoundary
    from biblbm_amd.lattice import Lattice
    from oracle import oracle_py as O
    shape, per = (17, 14, nz), (1, 0, per_z)
    L = Lattice(*shape, periodic=per, omega=1.0, omega_in=0.7)
    ib = ImmersedBoundary(L, "roma")
    sid = ib.add_shape(BOX * [6.3, 5.1, 7.0], BOX_TRI)
    for _ in range(2):
        ib.add_particle(sid, 0, [1e-12, 1.0], BOX * [6.3, 5.1, 7.0] + [3.25, 4.4, 5.0])
    ib.init()
    want = np.zeros(shape, np.uint8)
    top = nz - 1.0
    # (corner, height) of the two boxes: the second rides above, inside or across the first
    cases = [((3.25, 4.4, 5.0), 7.0, (3.6, 4.6, 5.0), 7.0),                 # faces on the same nodes
             ((3.25, 4.4, 2.0), 4.5, (5.1, 3.3, top - 5.0), 5.0),           # a face exactly on the last node
             ((3.25, 4.4, 2.0), 4.5, (5.1, 3.3, top - 5.0), 4.5),           # between the last two: it keeps its value
             ((13.3, 4.4, 9.0), 3.0, (14.2, 5.2, top - 3.0), 3.3),          # beyond the last node, across the x face
             ((13.3, 4.4, 9.0), 3.0, (5.2, 5.2, top - 3.0), 2.7),
             ((2.2, 4.4, -0.4), 6.0, (8.2, 5.2, 1.0), 0.5),                 # at the bottom, none and one node high
             ((2.2, 4.4, 40.3 % nz), 2.0, (8.2, 5.2, 31.0 % (nz - 4)), 1.0)]
    for a, ha, b, hb in cases:
        pos = [BOX * [6.3, 5.1, ha] + a, BOX * [6.3, 5.1, hb] + b]
        ib.set_positions(np.concatenate(pos))
        ib.move()  # at rest: the centre-of-mass mapping and the voxelisation
        now = ib.positions()
        hits = np.concatenate([O.ray_hits_z(BOX_TRI, now[8 * k:8 * k + 8]) for k in (0, 1)])
        # the oracle starts from the field it fills, as the device does
        fresh = O.voxel_fill(shape, per, hits)
        kept = np.zeros(shape[:2], bool)
        for i in range(shape[0]):
            for j in range(shape[1]):
                z = hits[(hits[:, 0] % shape[0] == i) & (hits[:, 1] == j), 2]
                if per_z:
                    z = z - nz * np.floor((z + 0.5) / nz)
                kept[i, j] = len(z) and nz - 2 < z.max() < nz - 1
        keep = want[..., -1].copy()
        want = fresh
        want[..., -1] = np.where(kept, keep, want[..., -1])
        assert np.array_equal(ib.phase(), want)
    ib.close()
    L.close()
