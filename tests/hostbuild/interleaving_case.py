"""One case of tests/test_hostbuild_interleaving.py on the CPU build, in a process of its own (EMU_SCHED_SEED, read once
per process, draws the order in which the wavefronts of a workgroup advance).

    python tests/hostbuild/interleaving_case.py LIB rods N_SIDE SPACING STEP SAMPLERS PRECISION CYCLES
    python tests/hostbuild/interleaving_case.py LIB chains BEADS N_SIDE SPACING STEP SAMPLERS CYCLES
    python tests/hostbuild/interleaving_case.py LIB nogrid N_SIDE SPACING STEP SAMPLERS CYCLES
    python tests/hostbuild/interleaving_case.py LIB count KIND   # early-exit overlap counts; EMU_FLAG_ODDS raises the flag

N_SIDE and SPACING are three numbers joined by commas.
"""
import os
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path[:0] = [os.path.dirname(os.path.dirname(HERE)), os.path.dirname(HERE),
                os.path.join(os.path.dirname(HERE), "golden")]

import numpy as np  # noqa: E402

import rampack_amd as ra  # noqa: E402

ra.load_library(sys.argv[1])

import oracle_lib  # noqa: E402
from rampack_amd import lattice  # noqa: E402

SC = ra.Shape("spherocylinder", radius=0.5, length=5.0)


def numbers(text, of):
    return tuple(of(x) for x in text.split(","))


def end_state(shape, start, step, samplers, waves, cycles, precision=ra.PREC_FP64):
    """The state and the counters after `cycles` cycles with `waves` wavefronts per cell (None: the launch rule's)."""
    os.environ.pop("RAMPACK_SWEEP_WAVES", None)
    if waves:
        os.environ["RAMPACK_SWEEP_WAVES"] = str(waves)
    pk = ra.GpuPacking(shape, *start, seed=77, precision=precision)
    pk.set_environment(1.0, 2.0, step, None, box_move=("log", 0.001))
    if samplers > 1:
        pk.set_move_samplers([("rototranslation", (step, step))] * samplers)
    c = pk.run_cycles(cycles)
    out = pk.download()
    print(f"{waves} wavefronts: moves {c['moves_accepted']}/{c['moves_attempted']}, box {c['box_accepted']}", flush=True)
    pk.close()
    return out, (c["moves_accepted"], c["moves_left_cell"], c["box_accepted"])


def same(a, b):
    assert a[1] == b[1], (a[1], b[1])
    assert all(np.array_equal(x, y) for x, y in zip(a[0], b[0]))


def rods(n_side, spacing, step, samplers, precision, cycles):
    start = lattice.spherocylinder_lattice(numbers(n_side, int), numbers(spacing, float))
    one = end_state(SC, start, float(step), int(samplers), 1, int(cycles))
    eight = end_state(SC, start, float(step), int(samplers), 8, int(cycles), int(precision))
    assert oracle_lib.oracle().snapshot_stats(1, 0.5, 5.0, *eight[0])[0] == 0
    same(one, eight)


def chains(beads, n_side, spacing, step, samplers, cycles):
    from test_gpu_poly import chain_start
    centres, radii = lattice.kinked_chain(int(beads), 1.0, 30.0)
    shape = ra.Shape("polysphere", centres=centres, radii=radii)
    start = chain_start(numbers(n_side, int), numbers(spacing, float))
    one = end_state(shape, start, float(step), int(samplers), 1, int(cycles))
    same(one, end_state(shape, start, float(step), int(samplers), 16, int(cycles)))


def nogrid(n_side, spacing, step, samplers, cycles):
    """The all-pairs sweep: its decisions replay through the oracle."""
    from test_gpu_replay import check_record
    start = lattice.spherocylinder_lattice(numbers(n_side, int), numbers(spacing, float))
    pk = ra.GpuPacking(SC, *start, seed=77)
    pk.set_environment(1.0, 2.0, float(step), None, box_move=("log", 0.001))
    if int(samplers) > 1:
        pk.set_move_samplers([("rototranslation", (float(step), float(step)))] * int(samplers))
    pk.run_cycles(int(cycles))
    rec = pk.record_sweep()
    assert rec["cells"] == [1, 1, 1]
    check_record(SC, rec, rejections=False)
    pk.close()


def count(kind):
    """Layers of particles with a gap between them, so that cells without any alternate with full ones, and one
    overlapping pair: the early-exit count is 1 whichever workgroup finds it and whenever the others learn of it."""
    if kind == "rods":
        shape, (box, pos, rot) = SC, lattice.spherocylinder_lattice((16, 16, 4), (1.3, 1.3, 15.0))
    elif kind == "spheres":
        shape, (box, pos, rot) = ra.Shape("sphere", radius=0.5), lattice.hard_sphere_lattice(10, 0.3)
    else:
        from test_gpu_poly import chain_start
        shape = ra.Shape("polysphere", centres=[[0, 0, -0.5], [0, 0, 0.5]], radii=[0.5, 0.5])
        box, pos, rot = chain_start((9, 9, 6), (1.3, 1.3, 4.5))
    pos[-1] = pos[-2] + [0.3, 0.0, 0.0]
    pk = ra.GpuPacking(shape, box, pos, rot, seed=3)
    for _ in range(40):
        assert pk.count_total_overlaps(True) == 1
    pk.close()


if __name__ == "__main__":
    {"rods": rods, "chains": chains, "nogrid": nogrid, "count": count}[sys.argv[2]](*sys.argv[3:])
    print("case passed", flush=True)
