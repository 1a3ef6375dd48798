"""Performance cases: what users of this framework have it do, through its public entry points.

Most cases are one block of a Monte Carlo run as the casino driver makes it: `cycles` cycles with frozen steps on a
packing resident on the GPU, then the block's observables (and, for soft shapes, its total energy) and the state in the
caller's order, as a snapshot or a trajectory frame takes it.  Two cases are the learned candidate ordering: the
gradient of one training batch and the scores of one set of candidate pairs.

  listed()             the fixed cases
  draw(rng)            one more case of the same ranges (rng: random.Random)
  prepare(case, seed)  what a program holds before the call: an equilibrating packing on the GPU, or network and pairs
  run(state)           one pass; the outputs whole
  work(case)           bytes and operations one pass cannot do without
  exact(case, seed)    what run returns, in 64 bits without this framework (None: no such value)

A Markov chain's end state has no closed form (one flipped decision gives another trajectory of the same ensemble), so
exact() covers the network cases only.
"""
from __future__ import annotations

import math

import numpy as np

import rampack_amd as ra
from rampack_amd import lattice

ROD_V0 = math.pi * 0.25 * 5.0 + 4.0 / 3 * math.pi * 0.125  # L = 5, r = 0.5


# ------------------------------------------------------------------------------------------------------------ cases

def listed():
    return [
        # Hard-sphere equation of state, the smallest runs: 1000 spheres at p* = 5 (log box moves).
        dict(name="spheres_1000", family="spheres", n_side=10, phi=0.30, pressure=5.0, box="log", cycles=100),
        # A liquid of 300 rods: a box too small for a neighbour grid, every pair through the nearest image.
        dict(name="liquid_300", family="rods", n=300, phi=0.30, pressure=1.0, start="sites", box="delta_triclinic",
             precision="fp64", cycles=50),
        # 8000 rods from a packing fraction of 0.25 at p* = 1, guarded FP32 overlap tests.
        dict(name="rods_8000_guarded", family="rods", n=8000, phi=0.25, pressure=1.0, start="sites",
             box="delta_triclinic", precision="guarded", cycles=100),
        # The headline workload: 1e5 rods, an AA-stacked smectic at 0.45, p* = 2, FP64.
        dict(name="rods_100000", family="rods", n=100000, phi=0.45, pressure=2.0, start="smectic",
             box="delta_triclinic", precision="fp64", cycles=100),
        # The large dense system: 1e6 rods, a smectic at 0.50, p* = 2.5.
        dict(name="smectic_1000000", family="rods", n=1000000, phi=0.50, pressure=2.5, start="smectic",
             box="delta_triclinic", precision="fp64", cycles=50),
        # Kinked 11-bead chains at p* = 3, the large multi-centre system.
        dict(name="chains_50653", family="chains", beads=11, kink=30.0, nx=37, nz=37, gap=1.1, z_gap=11.2,
             pressure=3.0, box="delta_triclinic", cycles=8),
        # Hard dumbbells at p* = 1.5, a small multi-centre system.
        dict(name="dimers_1183", family="chains", beads=2, kink=0.0, nx=13, nz=7, gap=1.25, z_gap=2.3, pressure=1.5,
             box="log", cycles=50),
        # Soft (WCA) spheres at constant pressure.
        dict(name="wca_spheres_4913", family="soft_spheres", soft="wca", n_side=17, phi=0.40, pressure=5.0,
             temperature=1.0, box="delta_v", cycles=50),
        # The compound variant: hard rods that also repel by WCA on the segment distance.
        dict(name="compound_rods_100000", family="soft_rods", n=100000, phi=0.45, pressure=2.0, start="smectic",
             box="delta_triclinic", cycles=5),
        # Overlap relaxation of 8000 randomly oriented rods on a lattice: moves accepted by their overlap counts.
        dict(name="relaxation_8000", family="relaxation", n=8000, phi=0.25, pressure=1.0, start="sites",
             box="delta_triclinic", cycles=20),
        # Learned ordering: the gradient of one training batch.
        dict(name="ordering_gradient_4096", family="gradient", batch=4096),
        # Learned ordering: scores of the close candidates of 4000 trial moves (about 298 each).
        dict(name="ordering_scores_1194001", family="scores", pairs=1194001),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    family = rng.choice(["rods", "rods", "rods", "spheres", "chains", "soft_spheres", "soft_rods", "relaxation",
                         "gradient", "scores"])
    if family == "rods":
        n = _log_int(rng, 300, 300000)
        return dict(family="rods", n=n, phi=round(rng.uniform(0.31, 0.42), 3), pressure=round(rng.uniform(1.5, 3.0), 2),
                    start="sites", box=rng.choice(["delta_triclinic", "log", "linear", "none"]),
                    precision=rng.choice(["fp64", "fp64", "guarded"]),
                    cycles=100 if n < 10000 else (50 if n < 100000 else 20))
    if family == "spheres":
        n_side = rng.randint(7, 47)
        return dict(family="spheres", n_side=n_side, phi=round(rng.uniform(0.20, 0.45), 3),
                    pressure=round(rng.uniform(1.0, 9.0), 2), box=rng.choice(["log", "delta_v", "none"]),
                    cycles=100 if n_side < 20 else 40)
    if family == "chains":
        beads = rng.randint(2, 11)
        # at least two total ranges (about 2 beads) across every side
        nx = rng.randint(max(9, int(math.ceil(4.4 * beads / 1.2))), max(20, 4 * beads))
        nz = rng.randint(5, 16)
        return dict(family="chains", beads=beads, kink=rng.choice([0.0, 15.0, 30.0]), nx=nx, nz=nz,
                    gap=round(rng.uniform(1.2, 1.5), 3), z_gap=round(beads + rng.uniform(0.3, 0.6), 3),
                    pressure=round(rng.uniform(0.5, 3.0), 2), box=rng.choice(["delta_triclinic", "log", "none"]),
                    cycles=20 if nx * nx * nz < 5000 else 6)
    if family == "soft_spheres":
        n_side = rng.randint(9, 31)
        return dict(family="soft_spheres", soft=rng.choice(["wca", "lj", "sic"]), n_side=n_side,
                    phi=round(rng.uniform(0.25, 0.42), 3), pressure=round(rng.uniform(1.0, 6.0), 2),
                    temperature=round(rng.uniform(0.8, 2.0), 2), box=rng.choice(["delta_v", "log", "none"]),
                    cycles=50 if n_side < 20 else 20)
    if family == "soft_rods":
        return dict(family="soft_rods", n=_log_int(rng, 2000, 60000), phi=round(rng.uniform(0.31, 0.36), 3),
                    pressure=round(rng.uniform(1.5, 2.5), 2), start="sites",
                    box=rng.choice(["delta_triclinic", "none"]), cycles=6)
    if family == "relaxation":
        return dict(family="relaxation", n=_log_int(rng, 1500, 40000), phi=round(rng.uniform(0.31, 0.36), 3),
                    pressure=round(rng.uniform(1.5, 2.5), 2), start="sites",
                    box=rng.choice(["delta_triclinic", "none"]), cycles=10)
    if family == "gradient":
        return dict(family="gradient", batch=_log_int(rng, 256, 16384))
    return dict(family="scores", pairs=_log_int(rng, 2000, 1190000))


# ---------------------------------------------------------------------------------------------------------- prepare

class _State:
    """What a program holds between calls: a packing (with the cycles of a block), or network and pairs."""

    def __init__(self, family, packing=None, cycles=0, theta=None, x=None, y=None, energy=False):
        self.family, self.packing, self.cycles, self.energy = family, packing, cycles, energy
        self.theta, self.x, self.y = theta, x, y


def _precision(name):
    return {"fp64": ra.PREC_FP64, "guarded": ra.PREC_GUARDED_FP32}[name]


def _box_move(kind, n, v):
    """The box move with a step near the one that step adaptation settles at (acceptance 10 - 20 %): relative steps
    shrink about as 1 / N for triclinic moves of a dense packing."""
    if kind == "none":
        return None
    if kind == "delta_triclinic":
        return ("delta_triclinic", min(0.02, 12.0 / n))
    if kind == "delta_v":
        return ("delta_v", 0.3 * math.sqrt(v * v / n))
    return (kind, (0.3 if kind == "log" else 3.0) / math.sqrt(n) / math.sqrt(max(n, 1000) / 1000.0))


def _rod_start(case):
    if case["start"] == "smectic":
        return lattice.spherocylinder_smectic(case["n"], case["phi"])
    return lattice.rod_replica_start(case["n"], case["phi"])


def _relaxed(shape, start, seed, case, trans, rot, relax, precision=ra.PREC_FP64, temperature=1.0):
    """A packing a short run into its equilibration (`relax` cycles from the lattice), steps frozen from here on."""
    box, pos, orient = start
    pk = ra.GpuPacking(shape, box, pos, orient, seed=1000 + seed, precision=precision)
    n = len(pos)
    pk.set_environment(temperature, case["pressure"], trans, rot,
                       box_move=_box_move(case["box"], n, abs(float(np.linalg.det(box)))))
    if case["family"] == "relaxation":
        pk.set_overlap_counting(True)
    pk.run_cycles(relax)
    return pk


# network of the learned ordering: 12 -> 64 -> 64 -> 64 -> 1, parameters in the order of rp_mlp_get_weights
_LAYERS = ((64, 12), (64, 64), (64, 64), (1, 64))


def _network(seed):
    rng = np.random.Generator(np.random.PCG64(7000 + seed))
    parts = []
    for fan_out, fan_in in _LAYERS:
        a = math.sqrt(6.0 / (fan_in + fan_out))
        parts += [rng.uniform(-a, a, fan_out * fan_in), rng.uniform(-0.05, 0.05, fan_out)]
    parts[-1][:] = -2.0  # the output bias at the log-odds of an overlap fraction of about 0.12
    return np.concatenate(parts).astype(np.float32)


def _rotations(q):
    """Row-major rotation matrices of the quaternions q (n x 4, any length)."""
    w, x, y, z = (q / np.sqrt((q * q).sum(1))[:, None]).T
    return np.stack([1 - 2 * (y * y + z * z), 2 * (x * y - z * w), 2 * (x * z + y * w),
                     2 * (x * y + z * w), 1 - 2 * (x * x + z * z), 2 * (y * z - x * w),
                     2 * (x * z - y * w), 2 * (y * z + x * w), 1 - 2 * (x * x + y * y)], axis=1)


def _pairs(n, seed):
    """Close candidates relative to a trial pose: positions uniform in the ball of the total range, relative rotations
    of a partly aligned packing, labels by a distance rule of about the right overlap fraction."""
    rng = np.random.Generator(np.random.PCG64(9000 + seed))
    d = rng.standard_normal((n, 3))
    d *= (rng.random(n) ** (1.0 / 3) / np.sqrt((d * d).sum(1)))[:, None]
    q = rng.standard_normal((n, 4)) * np.array([0.0, 0.15, 0.15, 1.0]) + np.array([1.0, 0.0, 0.0, 0.0])
    feats = np.ascontiguousarray(np.concatenate([d, _rotations(q)], axis=1), dtype=np.float32)
    side = np.hypot(d[:, 0], d[:, 1])
    label = (side + 0.3 * rng.random(n) < 0.32).astype(np.float32)
    return feats, label


def _random_rotations(n, seed):
    """Uniform random rotations (unit quaternions of four normal deviates), row-major."""
    q = np.random.Generator(np.random.PCG64(5000 + seed)).standard_normal((n, 4))
    return np.ascontiguousarray(_rotations(q))


def prepare(case, seed):
    family = case["family"]
    if family == "gradient":
        x, y = _pairs(case["batch"], seed)
        return _State(family, theta=_network(seed), x=x, y=y)
    if family == "scores":
        x, _ = _pairs(case["pairs"], seed)
        return _State(family, theta=_network(seed), x=x)
    energy, precision, temperature = False, ra.PREC_FP64, 1.0
    if family == "rods":
        shape = ra.Shape("spherocylinder", radius=0.5, length=5.0)
        start, trans, rot = _rod_start(case), 0.12, 0.22
        relax = 300 if case["n"] < 30000 else (150 if case["n"] < 300000 else 20)
        precision = _precision(case["precision"])
    elif family == "relaxation":
        shape = ra.Shape("spherocylinder", radius=0.5, length=5.0)
        box, pos, _ = _rod_start(case)
        start, trans, rot, relax = (box, pos, _random_rotations(len(pos), seed)), 0.5, 0.3, 10
    elif family == "soft_rods":
        shape = ra.Shape("spherocylinder", radius=0.5, length=5.0, soft="wca_segment", hard_core=True)
        start, trans, rot, relax, energy = _rod_start(case), 0.06, 0.03, 10, True
    elif family == "spheres":
        shape = ra.Shape("sphere", radius=0.5)
        start, trans, rot, relax = lattice.hard_sphere_lattice(case["n_side"], case["phi"]), 0.15, 0.1, 200
    elif family == "soft_spheres":
        shape = ra.Shape("sphere", radius=0.5, soft=case["soft"])
        start, trans, rot, relax, energy = lattice.hard_sphere_lattice(case["n_side"], case["phi"]), 0.2, 0.1, 50, True
        temperature = case["temperature"]
    else:
        centres, radii = lattice.kinked_chain(case["beads"], 1.0, case["kink"])
        shape = ra.Shape("polysphere", centres=centres, radii=radii)
        box, pos = lattice.sc_positions((case["nx"], case["nx"], case["nz"]),
                                        (case["gap"], case["gap"], case["z_gap"]))
        start = (box, pos, np.tile(np.eye(3).reshape(1, 9), (len(pos), 1)))
        long = case["beads"] > 4
        trans, rot, relax = (0.1, 0.02, 10) if long else (0.15, 0.2, 50)
    pk = _relaxed(shape, start, seed, case, trans, rot, relax, precision, temperature)
    return _State(family, packing=pk, cycles=case["cycles"], energy=energy)


# -------------------------------------------------------------------------------------------------------------- run

def _block(pk, counters, energy):
    box, pos, rot = pk.download()
    out = {"box": box, "pos": pos, "rot": rot, "packing_fraction": pk.observables()["packing_fraction"]}
    for key in ("moves_attempted", "moves_accepted", "moves_left_cell", "box_attempted", "box_accepted"):
        out[key] = int(counters[key])
    if energy:
        out["energy"] = pk.total_energy()
    return out


def run(state):
    if state.family == "gradient":
        loss, grad = ra.mlp_gradient(state.theta, state.x, state.y)
        return {"loss": float(loss), "grad": grad}
    if state.family == "scores":
        return {"score": ra.mlp_infer(state.theta, state.x)}
    pk = state.packing
    out = _block(pk, pk.run_cycles(state.cycles), state.energy)
    if state.family == "relaxation":
        out["overlaps"] = pk.cached_overlaps()
    return out


# ------------------------------------------------------------------------------------------------------------- work

RECORD = 96  # FP64 position and 3 x 3 orientation


def _particles(case):
    family = case["family"]
    if family in ("spheres", "soft_spheres"):
        return case["n_side"] ** 3
    if family == "chains":
        return case["nx"] * case["nx"] * case["nz"]
    return case["n"]


def work(case):
    """Bytes and operations of one pass.  A cycle reads every particle record once and writes back the moved ones (about
    a sixth).  A move that is accepted meets every particle within its interaction range: a centre distance each
    (8 operations) and the pair's exact test; a rejected one at least the pair that rejects it.  The last read is the
    state itself."""
    family = case["family"]
    if family in ("gradient", "scores"):
        n = case["batch"] if family == "gradient" else case["pairs"]
        params = sum(o * i + o for o, i in _LAYERS)
        macs = sum(o * i for o, i in _LAYERS)
        if family == "gradient":
            return {"bytes": 4.0 * (13 * n + 2 * params), "flops": 6.0 * macs * n}
        return {"bytes": 4.0 * (13 * n + params), "flops": 2.0 * macs * n}
    n, cycles, accepted = _particles(case), case["cycles"], 1.0 / 6
    if family in ("spheres", "soft_spheres"):
        reach = 1.0 if family == "spheres" else {"wca": 2 ** (1 / 6), "lj": 3.0, "sic": 1.0}[case["soft"]]
        near, pair = 4.0 / 3 * math.pi * reach ** 3 * case["phi"] / (math.pi / 6), 8.0 if family == "spheres" else 40.0
    elif family == "chains":
        beads = case["beads"]
        near = 4.0 / 3 * math.pi * beads ** 3 / (case["gap"] ** 2 * case["z_gap"])
        pair = 8.0 + 2.0 * 8.0 * beads
    else:
        near, pair = 4.0 / 3 * math.pi * 6.0 ** 3 * case["phi"] / ROD_V0, 8.0 + 80.0
    if family in ("soft_spheres", "soft_rods", "relaxation"):
        flops = n * cycles * 2.0 * near * pair  # the sums before and after every move
    else:
        flops = n * cycles * (accepted * near * pair + (1 - accepted) * pair)
    return {"bytes": RECORD * n * (cycles * (1 + accepted) + 1.0), "flops": flops}


# ------------------------------------------------------------------------------------------------------------ exact

def _gelu(x):
    """GELU (tanh form) and the tanh it is made of."""
    t = np.tanh(math.sqrt(2 / math.pi) * (x + 0.044715 * x * x * x))
    return 0.5 * x * (1 + t), t


def _gelu_slope(x, t):
    return 0.5 * (1 + t) + 0.5 * x * (1 - t * t) * math.sqrt(2 / math.pi) * (1 + 3 * 0.044715 * x * x)


def _layers(theta):
    out, at = [], 0
    theta = theta.astype(np.float64)
    for fan_out, fan_in in _LAYERS:
        w = theta[at:at + fan_out * fan_in].reshape(fan_out, fan_in)
        at += fan_out * fan_in
        out.append((w, theta[at:at + fan_out]))
        at += fan_out
    return out


def exact(case, seed):
    if case["family"] == "scores":
        x, _ = _pairs(case["pairs"], seed)
        (w1, b1), (w2, b2), (w3, b3), (w4, b4) = _layers(_network(seed))
        score = np.empty(len(x))
        for a in range(0, len(x), 1 << 12):  # blocks that stay in the cache
            h = x[a:a + (1 << 12)].astype(np.float64)
            for w, b in ((w1, b1), (w2, b2), (w3, b3)):
                h = _gelu(h @ w.T + b)[0]
            score[a:a + (1 << 12)] = 1 / (1 + np.exp(-(h @ w4[0] + b4[0])))
        return {"score": score}
    if case["family"] == "gradient":
        x, y = (a.astype(np.float64) for a in _pairs(case["batch"], seed))
        layers = _layers(_network(seed))
        acts, slopes = [x], []
        for w, b in layers[:3]:
            pre = acts[-1] @ w.T + b
            h, t = _gelu(pre)
            acts.append(h)
            slopes.append(_gelu_slope(pre, t))
        z = acts[-1] @ layers[3][0][0] + layers[3][1][0]
        loss = float(np.mean(np.maximum(z, 0) - z * y + np.log1p(np.exp(-np.abs(z)))))
        delta = ((1 / (1 + np.exp(-z)) - y) / len(y))[:, None]
        grads = []
        for i in (3, 2, 1, 0):
            w = layers[i][0]
            grads.append(np.concatenate([(delta.T @ acts[i]).ravel(), delta.sum(0)]))
            if i:
                delta = (delta @ w) * slopes[i - 1]
        return {"loss": loss, "grad": np.concatenate(grads[::-1])}
    return None
