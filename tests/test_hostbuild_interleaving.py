"""What the order of wavefronts can change, on the CPU build (tests/hostbuild).

* The speculative sweeps under different orders of the wavefronts between barriers: the lowest wavefront always first, the
  highest always first, and drawn orders.  A missing barrier shows as another trajectory than that of one wavefront making
  one move at a time.  Cells have more moves than a chunk holds, so that a chunk's end and the next one's start meet.
* Early-exit overlap counts whose flag another workgroup raises between two wavefronts' reads of it, with LDS as another
  kernel may have left it: no access outside an allocation, and the same count.
"""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(HERE, "hostbuild"))


@pytest.fixture(scope="module")
def host_lib():
    import host_build
    sources = [os.path.join(d, f) for d in (host_build.CSRC, host_build.HERE, os.path.join(host_build.HERE, "include", "hip"))
               for f in os.listdir(d) if f.endswith((".hip", ".cpp", ".h", ".py"))]
    if os.path.exists(host_build.LIB) and \
            os.path.getmtime(host_build.LIB) > max(os.path.getmtime(f) for f in sources):
        return host_build.LIB
    try:
        return host_build.build()
    except RuntimeError as e:
        pytest.fail(str(e))


def run_case(lib, *args, **env):
    import host_build
    env = dict(os.environ, LD_PRELOAD=host_build.asan_runtime(), ASAN_OPTIONS="detect_leaks=0:abort_on_error=1", **env)
    res = subprocess.run([sys.executable, os.path.join(HERE, "hostbuild", "interleaving_case.py"), lib] +
                         [str(a) for a in args], capture_output=True, text=True, timeout=600, env=env)
    print(res.stdout[-3000:])
    assert res.returncode == 0, res.stdout[-2000:] + res.stderr[-4000:]
    assert "case passed" in res.stdout


@pytest.mark.parametrize("order, samplers, precision", [("lowest", 1, 0), ("lowest", 1, 1), ("highest", 1, 0), ("3", 2, 0)])
def test_rods_follow_one_wavefront(host_lib, order, samplers, precision):
    """About 50 moves per cell and sampler: two or four chunks."""
    run_case(host_lib, "rods", "28,28,4", "1.2,1.2,6.3", 0.1, samplers, precision, 2, EMU_SCHED_SEED=order)


@pytest.mark.parametrize("order", ["lowest", "3"])
def test_chains_follow_one_wavefront(host_lib, order):
    run_case(host_lib, "chains", 16, "20,20,2", "1.25,1.25,16.8", 0.2, 4, 1, EMU_SCHED_SEED=order)


@pytest.mark.parametrize("order", ["lowest", "highest", "3"])
def test_packings_without_a_grid_replay(host_lib, order):
    run_case(host_lib, "nogrid", "8,8,2", "1.6,1.6,6.6", 0.1, 1, 2, EMU_SCHED_SEED=order)


@pytest.mark.parametrize("fill", ["1", "165"])
@pytest.mark.parametrize("order", ["highest", "3"])
@pytest.mark.parametrize("kind", ["rods", "spheres", "beads"])
def test_early_exit_flag_raised_between_two_wavefronts(host_lib, kind, order, fill):
    run_case(host_lib, "count", kind, EMU_FLAG_ODDS="9", EMU_LDS_FILL=fill, EMU_SCHED_SEED=order)
