"""The speculative all-pairs sweep (packings without a neighbour grid) where it can go wrong: fewer particles than a
wavefront, word boundaries of the hit rows, chunks of 64 moves that end short or hold many moves of one particle.  Every
decision and the end state against the oracle's replay of the reference's move test."""
import pytest

import rampack_amd as ra
from rampack_amd import lattice
from test_gpu_replay import HS, SC, check_record

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape, n_side, spacing, step, samplers", [
    (SC, (2, 2, 1), (6.5, 6.5, 13.0), 0.8, 4),   # 4 particles, 16 moves: nearly every move is of a moved particle
    (SC, (4, 4, 2), (2.9, 2.9, 6.4), 0.2, 2),    # 32 particles, 64 moves
    (SC, (11, 3, 1), (1.7, 6.0, 12.5), 0.2, 2),  # 33 particles, 66 moves
    (SC, (8, 8, 2), (1.6, 1.6, 6.6), 0.1, 1),    # 128
    (SC, (14, 14, 3), (1.4, 1.4, 6.4), 0.1, 1),  # 588
    (HS, (3, 3, 3), (1.2, 1.2, 1.2), 0.15, 3),   # 27 particles, 81 moves
])
def test_allpairs_sweep_replays(shape, n_side, spacing, step, samplers):
    box, pos, rot = lattice.spherocylinder_lattice(n_side, spacing)
    pk = ra.GpuPacking(shape, box, pos, rot, seed=23)
    pk.set_environment(1.0, 1.0, step, None, box_move=("log", 0.001))
    if samplers > 1:
        pk.set_move_samplers([("rototranslation", (step, step))] * samplers)
    pk.run_cycles(3)
    for _ in range(3):
        rec = pk.record_sweep()
        assert rec["cells"] == [1, 1, 1]
        check_record(shape, rec, rejections=False)
    pk.close()
