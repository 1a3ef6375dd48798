"""Box moves that only grow the box are scanned for overlaps unless no pair can come closer by them (sides that keep their
directions and grow by one factor; for spheres, any growth of a box with right angles): a side that turns by a part in
1e7, or sides that grow by different factors, can push rods into overlap."""
import numpy as np
import pytest

import oracle_lib
import rampack_amd as ra
from rampack_amd import lattice

pytestmark = pytest.mark.gpu

SC = ra.Shape("spherocylinder", radius=0.5, length=5.0)
HS = ra.Shape("sphere", radius=0.5)


def inclined_rods(gap, along):
    """Two parallel rods inclined by 45 degrees in the x-z plane, `gap` apart and shifted along their axis."""
    axis, across = np.array([1.0, 0.0, 1.0]) / np.sqrt(2), np.array([1.0, 0.0, -1.0]) / np.sqrt(2)
    rot = np.column_stack([across, [0.0, 1.0, 0.0], axis])
    if np.linalg.det(rot) < 0:
        rot[:, 1] *= -1
    d = (1.0 + gap) * across + along * axis
    return np.array([[100.0, 100.0, 100.0], [100.0, 100.0, 100.0] + d]), np.tile(rot.reshape(1, 9), (2, 1))


def scaled(shape, box, new_box, pos, rot):
    """The result of rp_try_scaling and the oracle's overlaps in the scaled packing."""
    length = 5.0 if shape is SC else 0.0
    kind = 1 if shape is SC else 0
    assert oracle_lib.oracle().snapshot_stats(kind, 0.5, length, box, pos, rot)[0] == 0
    pk = ra.GpuPacking(shape, box, pos, rot, seed=1)
    dE = pk.try_scaling(new_box)
    overlaps = oracle_lib.oracle().snapshot_stats(kind, 0.5, length, *pk.download())[0]
    pk.close()
    return dE, overlaps


def test_unequal_growth_of_a_box_of_rods():
    pos, rot = inclined_rods(1e-4, -3.0)
    box = np.diag([200.0, 200.0, 200.0])
    dE, overlaps = scaled(SC, box, box @ np.diag([1.3, 1.001, 1.001]), pos, rot)
    assert overlaps == 1 and dE == np.inf


def test_a_side_that_turns_by_a_part_in_ten_million():
    pos, rot = inclined_rods(1e-9, 0.5)
    box = np.diag([200.0, 200.0, 200.0])
    new_box = box * (1 + 1e-11)
    new_box[0, 2] += 2e-5  # the z side leans towards x by 1e-7
    dE, overlaps = scaled(SC, box, new_box, pos, rot)
    assert overlaps == 1 and dE == np.inf


@pytest.mark.parametrize("shape, factors", [(SC, (1.2, 1.2, 1.2)), (SC, (1 + 1e-13,) * 3), (HS, (1.2, 1.0 + 1e-9, 1.1))])
def test_growth_that_brings_no_pair_closer_is_accepted(shape, factors):
    if shape is SC:
        pos, rot = inclined_rods(1e-9, -3.0)
    else:
        pos, rot = np.array([[100.0, 100.0, 100.0], [100.6, 100.8, 100.0 + 1e-6]]), np.tile(np.eye(3).reshape(1, 9), (2, 1))
    box = np.diag([200.0, 200.0, 200.0])
    dE, overlaps = scaled(shape, box, box @ np.diag(factors), pos, rot)
    assert overlaps == 0 and dE == 0.0


def test_scans_of_growing_boxes():
    """Isotropic moves of rods scan only the boxes that shrink; triclinic moves with steps so short that sides hardly turn
    scan every proposal that passes the Metropolis test."""
    start = lattice.spherocylinder_lattice((14, 14, 3), (1.6, 1.6, 6.6))
    counts = {}
    for kind, step in (("log", 1e-3), ("delta_triclinic", 1e-9)):
        pk = ra.GpuPacking(SC, *start, seed=2)
        pk.set_environment(1.0, 1e-3, 0.1, None, box_move=(kind, step))
        counts[kind] = pk.run_cycles(40)
        pk.close()
    assert counts["log"]["box_scans"] < counts["log"]["box_accepted"]  # (at this pressure most growth is accepted)
    assert counts["delta_triclinic"]["box_scans"] >= counts["delta_triclinic"]["box_accepted"] > 0
