"""What the guarded sweep counts as pairs: every candidate of every trial pose that stays in its cell, the moved particle
itself left out, whether a move is accepted or not: the number of tests less one per pose."""
import pytest

import rampack_amd as ra
from rampack_amd import lattice
from test_gpu_replay import SC

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [ra.PREC_GUARDED_FP32, ra.PREC_GUARDED_FP32_VERIFY])
@pytest.mark.parametrize("spacing", [(1.0001, 1.0001, 6.0001), (1.3, 1.3, 6.4)])  # no move accepted; many
def test_pairs_leave_out_the_moved_particle(spacing, precision, monkeypatch):
    monkeypatch.setenv("RAMPACK_SWEEP_WAVES", "8")
    box, pos, rot = lattice.spherocylinder_lattice((28, 28, 4), spacing)
    pk = ra.GpuPacking(SC, box, pos, rot, seed=3, precision=precision)
    pk.set_environment(1.0, 1.0, 0.3, None, box_move=None)
    c = pk.run_cycles(2)
    st = pk.guard_stats()
    assert (c["moves_accepted"] > 0) == (spacing[0] > 1.2)
    assert c["moves_left_cell"] > 0 and c["unstaged_blocks"] == 0
    assert st["pairs"] == c["pair_tests"] - (c["moves_attempted"] - c["moves_left_cell"])
    assert st["mismatches"] == 0
    pk.close()
