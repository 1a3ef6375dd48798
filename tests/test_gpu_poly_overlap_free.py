"""The speculative polysphere sweep against the oracle: beads of their own sizes, one to sixteen per particle, with box
moves; the state has no overlapping beads by the oracle's count, and the device's full and early-exit counts agree."""
import numpy as np
import pytest

import oracle_lib
import rampack_amd as ra
from rampack_amd import lattice
from test_gpu_poly import chain_start

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("waves", ["4", "16"])
@pytest.mark.parametrize("beads, n_side, spacing, step", [
    (1, (9, 9, 9), (1.3, 1.3, 1.3), 0.3),
    (2, (9, 9, 6), (1.3, 1.3, 2.5), 0.3),
    (5, (12, 12, 4), (1.3, 1.3, 5.6), 0.3),
    (11, (14, 14, 3), (1.25, 1.25, 11.6), 0.25),
    (16, (14, 14, 3), (1.25, 1.25, 16.8), 0.2),
])
def test_states_are_overlap_free_by_the_oracle(beads, n_side, spacing, step, waves, monkeypatch):
    monkeypatch.setenv("RAMPACK_SWEEP_WAVES", waves)
    centres, radii = lattice.kinked_chain(beads, 1.0, 30.0) if beads > 1 else (np.zeros((1, 3)), np.array([0.5]))
    centres, radii = np.array(centres), np.array(radii) * np.linspace(1.0, 0.8, beads)
    box, pos, rot = chain_start(n_side, spacing)
    pk = ra.GpuPacking(ra.Shape("polysphere", centres=centres, radii=radii), box, pos, rot, seed=47)
    pk.set_environment(1.0, 3.0, step, None, box_move=("log", 0.003))
    for _ in range(3):
        c = pk.run_cycles(8)
        state = pk.download()
        assert oracle_lib.oracle().snapshot_stats(2, 0.0, 0.0, *state, centres=centres, radii=radii)[0] == 0
        assert pk.count_total_overlaps() == pk.count_total_overlaps(True) == 0
    assert pk.timing()["sweep_waves"] == int(waves)
    assert c["moves_accepted"] > 0 and c["box_scans"] > 0
    pk.close()
