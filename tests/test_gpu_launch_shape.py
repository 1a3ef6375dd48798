"""A launch shape pinned by the autotuner or the environment runs the kernel that it names, with several move samplers as
with one: eight wavefronts with schedule 2 on hard spherocylinders are the speculative sweep (guarded FP32 where asked
for), and its decisions replay through the oracle."""
import pytest

import rampack_amd as ra
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
