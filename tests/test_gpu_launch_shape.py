"""A launch shape pinned by the autotuner or the environment runs the kernel that it names, with several move samplers as
with one: eight wavefronts with schedule 2 on hard spherocylinders are the speculative sweep (guarded FP32 where asked
for), and its decisions replay through the oracle."""
import numpy as np
import pytest

import rampack_amd as ra
from rampack_amd import lattice
from test_gpu_replay import SC, check_record, rod_start

pytestmark = pytest.mark.gpu


def packing(samplers, precision):
    pk = ra.GpuPacking(SC, *rod_start(), seed=31, precision=precision)
    pk.set_environment(1.0, 2.0, 0.2, None, box_move=("delta_triclinic", 0.002))
    if samplers > 1:
        pk.set_move_samplers([("translation", 0.2), ("rotation", 0.2)])
    return pk


@pytest.mark.parametrize("samplers", [1, 2])
@pytest.mark.parametrize("precision", [ra.PREC_FP64, ra.PREC_GUARDED_FP32])
def test_pinned_eight_wavefronts_stay_speculative(samplers, precision, monkeypatch):
    monkeypatch.setenv("RAMPACK_SWEEP_WAVES", "8")
    monkeypatch.setenv("RAMPACK_SWEEP_PIPELINE", "2")
    pk = packing(samplers, precision)
    pk.run_cycles(3)
    assert pk.timing()["sweep_waves"] == 8
    assert (pk.guard_stats()["pairs"] > 0) == (precision != ra.PREC_FP64)
    check_record(SC, pk.record_sweep(), rejections=False)
    pk.close()


def test_autotuned_guarded_sweep_of_two_samplers_stays_guarded():
    pk = packing(2, ra.PREC_GUARDED_FP32)
    pk.autotune(2)
    before = pk.guard_stats()["pairs"]
    pk.run_cycles(2)
    assert pk.timing()["sweep_waves"] == 8 and pk.guard_stats()["pairs"] > before > 0
    pk.close()


@pytest.mark.parametrize("n_side, spacing, samplers, waves", [
    ((28, 28, 6), (2.2, 2.2, 6.6), 1, 8),    # stencils of 212, 75 workgroups per colour: the chip is not full
    ((60, 60, 10), (2.2, 2.2, 6.6), 1, 2),   # 201, 605 workgroups
    ((60, 60, 10), (2.2, 2.2, 6.6), 2, 2),
    ((60, 60, 10), (2.6, 2.6, 7.0), 1, 1),   # 144, 845 workgroups
    ((60, 60, 10), (1.8, 1.8, 6.6), 2, 8),   # 300, 405 workgroups
    ((86, 86, 24), (2.4, 2.4, 6.4), 1, 2),   # about 160, over 1024 workgroups
])
def test_thin_stencils_of_rods(n_side, spacing, samplers, waves):
    box, pos, rot = lattice.spherocylinder_lattice(n_side, spacing)
    pk = ra.GpuPacking(SC, box, pos, rot, seed=7)
    pk.set_environment(1.0, 0.5, 0.2, None, box_move=("log", 0.001))
    if samplers > 1:
        pk.set_move_samplers([("translation", 0.2), ("rotation", 0.2)])
    pk.run_cycles(3)
    assert pk.timing()["sweep_waves"] == waves
    check_record(SC, pk.record_sweep(), rejections=False)
    pk.close()


def test_stencils_of_over_2048_particles_stay_in_lds(monkeypatch):
    """Layered rods of L/D = 10 in stencils of about 1 850 and up to 2 300 particles (the queue entries of the scan name
    2048): the same cells as on one wavefront read their stencil from memory, and the trajectory is the same."""
    shape = ra.Shape("spherocylinder", radius=0.5, length=10.0)
    start = lattice.spherocylinder_lattice((46, 46, 7), (1.45, 1.45, 11.6))
    runs = []
    for waves in (None, "1"):
        if waves:
            monkeypatch.setenv("RAMPACK_SWEEP_WAVES", waves)
        pk = ra.GpuPacking(shape, *start, seed=19)
        pk.set_environment(1.0, 0.5, 0.05, None, box_move=None)
        c = pk.run_cycles(10)
        assert pk.timing()["sweep_waves"] == int(waves or 8) and pk.timing()["sweep_cap"] > 2048
        runs.append((pk.download(), c["unstaged_blocks"]))
        pk.close()
    (s0, u0), (s1, u1) = runs
    assert u0 == u1 > 0
    assert all(np.array_equal(a, b) for a, b in zip(s0, s1))
