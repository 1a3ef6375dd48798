"""Hard spherocylinders in stencils of about 200 and 300 particles, where the launch rule takes the speculative sweep, with
one sampler and with two, and of about 150, where it keeps one wavefront: every decision against the oracle's replay."""
import pytest

import rampack_amd as ra
from rampack_amd import lattice
from test_gpu_replay import SC, check_record

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("samplers", [1, 2])
@pytest.mark.parametrize("n_side, spacing, waves", [
    ((24, 24, 6), (2.6, 2.6, 7.0), 1),
    ((28, 28, 6), (2.2, 2.2, 6.6), 8),
    ((28, 28, 6), (1.8, 1.8, 6.6), 8),
])
def test_sparse_rods_replay(n_side, spacing, waves, samplers):
    box, pos, rot = lattice.spherocylinder_lattice(n_side, spacing)
    pk = ra.GpuPacking(SC, box, pos, rot, seed=19)
    pk.set_environment(1.0, 0.5, 0.3, None, box_move=("delta_triclinic", 0.005))
    if samplers == 2:
        pk.set_move_samplers([("translation", 0.3), ("rotation", 0.2)])
    pk.run_cycles(20)
    for _ in range(2):
        rec = pk.record_sweep()
        assert pk.timing()["sweep_waves"] == waves
        check_record(SC, rec, rejections=False)
    pk.close()
