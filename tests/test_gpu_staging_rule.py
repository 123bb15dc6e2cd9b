"""Velocity staging by the rule on sizes (off the touched-tile list, a thread
per cell, or carried by the collision) against the staging it did not take:
the same trajectory, replayed as a graph and called stage by stage, on
lattices whose sides are no multiples of a tile."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

#   sides, cells of 642 vertices, the other staging
CASES = [((165, 159, 161), 1, 1),   # few tiles of more than 2^22 cells: the list
         ((165, 159, 161), 13, 1),  # an eighth as many vertices as tiles: the list's last, one more: not
         ((165, 159, 161), 14, 1),
         ((131, 83, 101), 1, 1),    # few cells: a thread per cell
         ((101, 66, 103), 18, 0),   # most tiles of more than 96 MiB: the collision
         ((101, 66, 97), 18, 1)]    # the same a little below: a thread per cell


@pytest.mark.parametrize("sides,cells,other", CASES)
def test_staging_rule_keeps_the_trajectory(device, sides, cells, other):
    from biblbm_amd import workloads
    W = [workloads.suspension("f64", *sides, n642=cells, n2562=0, n162=1, cell_radius=9.0) for _ in range(3)]
    start = W[0].ibm.positions()
    W[1].ibm.set_fused_staging(other)
    W[0].ibm.coupled_steps(6, use_graph=True)
    W[1].ibm.coupled_steps(6, use_graph=True)
    for _ in range(6):
        W[2].ibm.step()
        W[2].lattice.collide_and_stream(1)
    moved = np.abs(W[0].ibm.positions() - start).max()
    f = W[0].lattice.get_populations()
    assert moved > 0
    for w in W[1:]:
        # FP64 moments summed in one order or another
        assert np.abs(w.ibm.positions() - W[0].ibm.positions()).max() <= 1e-12
        assert np.abs(w.lattice.get_populations() - f).max() <= 1e-13
    for w in W:
        w.ibm.close()
        w.lattice.close()
