"""The speculative sweep (eight wavefronts, every move of a chunk of 32 tested at once) where it can go wrong, every
decision and the end state against the oracle's replay of the reference's move test: chunks that end short and cells
with more than one chunk, few moves per cell, nearly every move accepted (many stale moves and own-pair updates), steps
that leave the cell, cells at the grid's periodic edge."""
import pytest

import rampack_amd as ra
from rampack_amd import lattice
from test_gpu_replay import SC, check_record

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [ra.PREC_FP64, ra.PREC_GUARDED_FP32])
@pytest.mark.parametrize("n_side, spacing, step, moves_per_cell", [
    ((28, 28, 4), (1.2, 1.2, 6.3), 0.1, (33, 64)),     # two chunks, dense
    ((24, 24, 4), (1.36, 1.36, 6.3), 0.02, (32, 64)),  # small steps: most moves are accepted
    ((22, 22, 4), (1.4, 1.4, 6.3), 0.5, (17, 32)),     # one chunk; steps across the cell's faces
    ((7, 7, 4), (3.8, 3.8, 6.3), 0.5, (3, 8)),         # few moves per cell, stencils of little over a hundred
])
def test_speculative_sweep_replays(n_side, spacing, step, moves_per_cell, precision, monkeypatch):
    monkeypatch.setenv("RAMPACK_SWEEP_WAVES", "8")
    box, pos, rot = lattice.spherocylinder_lattice(n_side, spacing)
    pk = ra.GpuPacking(SC, box, pos, rot, seed=77, precision=precision)
    pk.set_environment(1.0, 2.0, step, None, box_move=("log", 0.001))
    pk.run_cycles(5)
    for _ in range(2):
        rec = pk.record_sweep()
        assert moves_per_cell[0] <= rec["moves_per_cell"] <= moves_per_cell[1], rec["moves_per_cell"]
        check_record(SC, rec, rejections=False)
    pk.close()
