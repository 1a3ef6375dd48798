"""The speculative polysphere sweep where it can go wrong: one bead to sixteen (bead groups of one to four, short groups),
stencils that end within a unit, chunks of 64 moves and more, steps that leave the cell.  The trajectory is that of the
sweep that makes one move at a time (forced by one wavefront), bit for bit, and no bead overlaps by the oracle."""
import numpy as np
import pytest

import rampack_amd as ra
from rampack_amd import lattice
from test_gpu_poly import chain_start

pytestmark = pytest.mark.gpu


def shape(beads):
    centres, radii = lattice.kinked_chain(beads, 1.0, 30.0) if beads > 1 else (np.zeros((1, 3)), np.array([0.5]))
    radii = np.array(radii) * np.linspace(1.0, 0.8, beads)  # every bead of its own size
    return ra.Shape("polysphere", centres=centres, radii=radii)


def run(beads, n_side, spacing, step, samplers, waves, cycles, monkeypatch):
    monkeypatch.setenv("RAMPACK_SWEEP_WAVES", waves)
    box, pos, rot = chain_start(n_side, spacing)
    pk = ra.GpuPacking(shape(beads), box, pos, rot, seed=91)
    pk.set_environment(1.0, 1.0, step, None, box_move=("log", 0.002))
    if samplers > 1:
        pk.set_move_samplers([("rototranslation", (step, step))] * samplers)
    c = pk.run_cycles(cycles)
    out = pk.download()
    pk.close()
    assert c["moves_accepted"] > 0 and c["moves_left_cell"] > 0
    return out, (c["moves_accepted"], c["moves_left_cell"], c["box_accepted"])


@pytest.mark.parametrize("waves", ["4", "8", "16"])
@pytest.mark.parametrize("beads, n_side, spacing, step, samplers", [
    (1, (9, 9, 9), (1.3, 1.3, 1.3), 0.3, 1),
    (2, (9, 9, 6), (1.3, 1.3, 2.5), 0.3, 1),
    (4, (9, 9, 4), (1.3, 1.3, 4.6), 0.3, 1),
    (5, (12, 12, 4), (1.3, 1.3, 5.6), 0.3, 1),
    (11, (28, 28, 3), (1.25, 1.25, 11.6), 0.25, 1),
    (16, (40, 40, 3), (1.25, 1.25, 16.8), 0.2, 4),  # 88 moves per cell: more than one chunk
])
def test_poly_sweep_equals_one_move_at_a_time(beads, n_side, spacing, step, samplers, waves, monkeypatch):
    cycles = 12 if beads < 8 else 4
    ref, counts = run(beads, n_side, spacing, step, samplers, "1", cycles, monkeypatch)
    got, other = run(beads, n_side, spacing, step, samplers, waves, cycles, monkeypatch)
    assert counts == other
    assert all(np.array_equal(a, b) for a, b in zip(ref, got))
