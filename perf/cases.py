"""Performance cases of the sampler, through the public entry points of pimc_hip.Context.

A pass over a sampling case is one block as the host driver runs it: the samples and bins are
cleared, the moves of `passes` passes run with an estimator sample every `every` passes, and the
block's samples, counters and configuration come back (bins and correlation sums too for a single
chain).  Launch shapes are the library's defaults, which is what a program gets that does not tune.

Configurations are made to look like equilibrated paths: atoms on the sites of a compact cluster
(or of a periodic box), every path a confined free-particle ring whose links have the free
particle's spread at the case's temperature, rotor orientations a smooth closed walk.
"""
import ctypes
import functools
import math
import os
import sys

import numpy as np

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "moribs-pimc_amd"))

import pimc_configs as pc  # noqa: E402
import pimc_hip as ph  # noqa: E402
import pimc_tables as pt  # noqa: E402

LAMBDA_AMU = 0.5 * 100.0 * 1.05457266 ** 2 / (1.6605402 * 1.380658)  # hbar^2/2m of 1 amu, Angstrom^2 K


def listed():
    return [
        # the smallest system in use: one chain of the 8-He cluster deck, where launches, barriers
        # and dependent half-sweeps are all the time
        dict(name="cluster_8he", kind="linear", replicas=1, nmin=8, nmax=8, pmin=128, pmax=128, ratio=1, levels=3,
             tmin=0.37, tmax=0.37, fp64=False, passes=4, every=1),
        # one chain of the 64-He cluster at 512 slices: a long chain alone on the device
        dict(name="cluster_64he", kind="linear", replicas=1, nmin=64, nmax=64, pmin=512, pmax=512, ratio=1, levels=3,
             tmin=0.37, tmax=0.37, fp64=False, passes=2, every=1),
        # the driver's many-chain mode: the 8-He deck as 256 independent chains
        dict(name="chains_8he", kind="linear", replicas=256, nmin=8, nmax=8, pmin=128, pmax=128, ratio=1, levels=3,
             tmin=0.37, tmax=0.37, fp64=False, passes=20, every=4),
        # the headline workload: a scan over cluster size, temperature and slices in one context
        dict(name="scan_256", kind="linear", replicas=256, nmin=1, nmax=100, pmin=64, pmax=512, ratio=1, levels=3,
             tmin=0.3, tmax=2.0, fp64=False, passes=6, every=1),
        # a small scan with odd sizes, four bisection levels and half as many rotor slices
        dict(name="scan_ragged", kind="linear", replicas=23, nmin=3, nmax=77, pmin=96, pmax=240, ratio=2, levels=4,
             tmin=0.4, tmax=1.7, fp64=False, passes=3, every=3),
        # FP64 pair terms, the setting of runs that are checked move for move
        dict(name="scan_fp64", kind="linear", replicas=12, nmin=5, nmax=40, pmin=64, pmax=128, ratio=1, levels=3,
             tmin=0.4, tmax=1.5, fp64=True, passes=3, every=1),
        # bulk helium: periodic boxes under the minimum image, no rotor
        dict(name="box_he", kind="box", replicas=16, atoms=64, slices=64, levels=3, temp=1.5, passes=6, every=1),
        # a rotating asymmetric top in 32 para-H2
        dict(name="top_32h2", kind="top", replicas=1, atoms=32, slices=256, levels=3, temp=0.5, da=False, passes=3,
             every=1),
        # the same with the surrogate's delayed acceptance, the framework's learned first stage
        dict(name="top_32h2_da", kind="top", replicas=1, atoms=32, slices=256, levels=3, temp=0.5, da=True, passes=2,
             every=1),
        # pairs of rigid water rotors on long paths, many chains: the largest rotor sweeps
        dict(name="waters_128", kind="waters", replicas=128, slices=2048, levels=3, temp=1.0, passes=1, every=1),
        # batched PotEnergy queries on a committed configuration, as analysis programs ask for them
        dict(name="queries_100k", kind="queries", replicas=8, nmin=20, nmax=60, slices=128, temp=0.7, queries=100003),
        # training the surrogate network on collected rows
        dict(name="train_64k", kind="train", rows=65537, batch=4096, epochs=2),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear"] * 8 + ["box"] * 2 + ["top", "waters"] + ["queries"] * 2 + ["train"])
    if kind == "linear":
        fp64 = rng.random() < 0.15
        replicas = _log(rng, 1, 16 if fp64 else 64)
        n0, n1 = sorted((_log(rng, 1, 50 if fp64 else 100), _log(rng, 1, 50 if fp64 else 100)))
        p0, p1 = sorted(16 * _log(rng, 2, 10 if fp64 else 32) for _ in range(2))
        t0, t1 = sorted(round(rng.uniform(0.3, 2.0), 2) for _ in range(2))
        return dict(kind=kind, replicas=replicas, nmin=n0, nmax=n1, pmin=p0, pmax=p1, ratio=rng.choice([1, 1, 2]),
                    levels=rng.choice([2, 3, 3, 4]), tmin=t0, tmax=t1, fp64=fp64, passes=rng.randint(1, 3), every=1)
    if kind == "box":
        return dict(kind=kind, replicas=_log(rng, 1, 24), atoms=_log(rng, 9, 100), slices=8 * _log(rng, 3, 16), levels=3,
                    temp=round(rng.uniform(0.8, 2.5), 2), passes=rng.randint(1, 4), every=1)
    if kind == "top":
        return dict(kind=kind, replicas=_log(rng, 1, 4), atoms=_log(rng, 5, 40), slices=16 * _log(rng, 4, 16), levels=3,
                    temp=0.5, da=rng.random() < 0.4, passes=rng.randint(1, 2), every=1)
    if kind == "waters":
        return dict(kind=kind, replicas=_log(rng, 3, 64), slices=64 * _log(rng, 2, 16), levels=3, temp=1.0,
                    passes=1, every=1)
    if kind == "queries":
        n0, n1 = sorted((_log(rng, 2, 100), _log(rng, 2, 100)))
        return dict(kind=kind, replicas=_log(rng, 1, 16), nmin=n0, nmax=n1, slices=8 * _log(rng, 4, 32), temp=0.7,
                    queries=_log(rng, 1, 200000))
    return dict(kind=kind, rows=_log(rng, 8192, 65536) | 1, batch=rng.choice([1024, 2048, 4096]), epochs=1)


# ---------------------------------------------------------------------------- inputs
def _rings(rng, n, P, link_var, sigma):
    """n closed Gaussian paths of P points: links of variance link_var, spread about sigma."""
    conf = max(link_var / (4.0 * sigma ** 4), 1e-12)  # per-point confinement that gives this spread
    k = np.arange(P // 2 + 1)
    amp = 1.0 / np.sqrt(4.0 * np.sin(np.pi * k / P) ** 2 / link_var + conf)
    return np.fft.irfft(np.fft.rfft(rng.standard_normal((n, P)), axis=-1) * amp, n=P, axis=-1)


@functools.lru_cache(maxsize=None)
def _sites(n, spacing, rmin):
    """The n sites of an fcc lattice nearest the origin, none closer to it than rmin."""
    m = np.arange(-8, 9)
    g = np.stack(np.meshgrid(m, m, m, indexing="ij"), -1).reshape(-1, 3)
    g = g[g.sum(1) % 2 == 0] * (spacing / math.sqrt(2.0)) + np.array([0.31, 0.17, 0.05])
    r = np.linalg.norm(g, axis=1)
    g, r = g[r >= rmin], r[r >= rmin]
    return g[np.argsort(r, kind="stable")[:n]]


def _paths(rng, centres, masses, P, T, sigma):
    """[3][atoms*P] coordinates of ring paths around the centres."""
    out = np.empty((3, len(centres), P))
    for m in sorted(set(masses)):
        a = [i for i, x in enumerate(masses) if x == m]
        r = _rings(rng, 3 * len(a), P, 2.0 * LAMBDA_AMU / m / (T * P), sigma * min(1.0, math.sqrt(4.0 / m)))
        out[:, a] = r.reshape(3, len(a), P) + np.asarray(centres)[a].T[:, :, None]
    return out.reshape(3, -1)


def _angles(rng, natoms, first, P, Prot, step):
    """[3][natoms*P] (phi, cos theta, chi): smooth closed walks of the molecules from atom `first`."""
    a = np.zeros((3, natoms, P))
    a[1] = 1.0
    for q in range(first, natoms):
        w = _rings(rng, 3, Prot, step * step, 0.4)
        a[0, q, :Prot] = np.mod(rng.uniform(0, 2 * np.pi) + w[0], 2 * np.pi)
        a[1, q, :Prot] = np.cos(np.clip(rng.uniform(0.9, 2.2) + 0.5 * w[1], 0.15, 3.0))
        a[2, q, :Prot] = np.mod(rng.uniform(0, 2 * np.pi) + w[2], 2 * np.pi)
    return a.reshape(3, -1)


@functools.lru_cache(maxsize=None)
def _pair_tables():
    rg, cg, V = pt.morse_legendre_2d()
    return pt.lj_table(), (rg, cg, rg[1] - rg[0], cg[1] - cg[0], V)


@functools.lru_cache(maxsize=None)
def _linden(T, P):
    return pt.linden(T, P, pc.B_ROTOR_CM)


@functools.lru_cache(maxsize=1)
def _asymrho(T, P, maxj):
    gen = ph.Context(1)
    out = gen.asymrho(T, P, *pc.ABC_H2O, maxj)
    gen.close()
    return out


@functools.lru_cache(maxsize=None)
def _pot3d():
    return pt.legendre_3d_table()


def _systems(case):
    """(N, P, T) of every replica of a scan: the case's own, the same for every seed."""
    rng = np.random.default_rng(985456376)
    lo, hi = case["pmin"], case.get("pmax", case["pmin"])
    grid = 1 << max(case["levels"], 1)
    grid *= 2 * case["ratio"] // math.gcd(grid, 2 * case["ratio"])
    out = []
    for _ in range(case["replicas"]):
        n = int(rng.integers(case["nmin"], case["nmax"] + 1))
        p = int(grid * round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / grid))
        t = round(float(rng.uniform(case["tmin"], case["tmax"])), 2)
        out.append((n, max(p, grid * 2), t))
    return out


def _linear(ctx, systems, ratio, levels, rng, rotating=True):
    (r1, v1), two = _pair_tables()
    ctx.add_pot1d(r1, v1)
    ctx.add_pot2d(*two)
    rot = {}
    for _, P, T in systems:
        if (T, P // ratio) not in rot:
            rot[T, P // ratio] = ctx.add_rotdens(*_linden(T, P // ratio))
    for i, (n, P, T) in enumerate(systems):
        ctx.set_replica(i, 2, [n, 1], [0, 1], [levels] * 2, [pc.STEP_HE, pc.STEP_ROTOR], [pc.MASS_HE4, pc.MASS_CO2], P,
                        P // ratio if rotating else 0, T, pc.ROT_STEP, pot1d=[0, -1], pot2d=[-1, 0],
                        rotdens=rot[T, P // ratio])
    ctx.commit()
    coords = []
    for i, (n, P, T) in enumerate(systems):
        c = np.concatenate([_sites(n, 3.7, 3.3) + rng.normal(0, 0.1, (n, 3)), np.zeros((1, 3))])
        xyz = _paths(rng, c, [pc.MASS_HE4] * n + [pc.MASS_CO2], P, T, 0.5)
        ctx.set_state(i, xyz, _angles(rng, n + 1, n, P, P // ratio, 0.1))
        coords.append(xyz)
    return coords


def _network():
    """Surrogate weights: seeded hidden layers, the output layer fitted to the 3D table."""
    rng = np.random.default_rng(7)
    x, v = _rows(rng, 6000)
    norm = np.concatenate([x.mean(0), x.std(0), [v.mean(), v.std()]]).astype(np.float32)
    a = lambda o, i: rng.uniform(-1, 1, (o, i)) * math.sqrt(6.0 / (o + i))  # noqa: E731
    W = [2.0 * a(128, 4), 1.5 * a(128, 128), 1.5 * a(128, 128)]
    b = [rng.normal(0, 0.5, 128) for _ in W]
    h = (x - norm[:4]) / norm[4:8]
    for w, c in zip(W, b):
        z = h @ w.T + c
        h = z / (1.0 + np.exp(-z))
    h = np.concatenate([h, np.ones((len(h), 1))], 1)
    y = (v - norm[8]) / norm[9]
    w4 = np.linalg.solve(h.T @ h + 1e-3 * len(h) * np.eye(129), h.T @ y)
    w4 = np.round(w4 * 4096.0) / 4096.0  # the same bits whatever order the solve sums in
    theta = np.concatenate([W[0].ravel(), b[0], W[1].ravel(), b[1], W[2].ravel(), b[2], w4])
    return theta.astype(np.float32), norm


def _rows(rng, n):
    """Features (R, u) and table energies of atom-rotor pairs around the well."""
    nr, nth, nch, r0, r1, v = _pot3d()
    R = rng.uniform(2.9, 9.0, n)
    u = rng.standard_normal((n, 3))
    u /= np.linalg.norm(u, axis=1)[:, None]
    ir = np.clip((R / 0.529177249 - r0) / (r1 - r0) * (nr - 1), 0, nr - 1).astype(int)
    it = np.degrees(np.arccos(u[:, 2])).astype(int)
    ic = np.clip(np.degrees(np.arctan2(np.abs(u[:, 1]), np.abs(u[:, 0]))), 0, nch - 1).astype(int)
    return (np.concatenate([R[:, None], u], 1).astype(np.float32),
            np.asarray(v)[(ir * nth + it) * nch + ic].astype(np.float32))


@functools.lru_cache(maxsize=1)
def _cached_network():
    return _network()


def prepare(case, seed):
    rng = np.random.default_rng([seed, 11])
    kind = case["kind"]
    if kind == "train":
        ctx = ph.Context(1)
        x, v = _rows(rng, case["rows"])
        return dict(case=case, ctx=ctx, x=x, v=v + rng.normal(0, 0.5, len(v)).astype(np.float32), seed=int(seed) & 0xFFFF)
    R = case["replicas"]
    ctx = ph.Context(R, flags=ph.FLAG_FP64 if case.get("fp64") else 0, seed=int(seed) & 0x7FFFFFFF)
    if kind == "linear":
        systems = _systems(case)
        _linear(ctx, systems, case["ratio"], case["levels"], rng)
    elif kind == "queries":
        P, T = case["slices"], case["temp"]
        systems = _systems(dict(case, pmin=P, ratio=1, levels=3, tmin=T, tmax=T))
        coords = _linear(ctx, systems, 1, 3, rng)
        q = case["queries"]
        rep = rng.integers(0, R, q).astype(np.int32)
        natoms = np.array([s[0] + 1 for s in systems])
        atom = (rng.random(q) * natoms[rep]).astype(np.int32)
        it = rng.integers(0, systems[0][1], q).astype(np.int32)
        pos = np.empty((q, 3))
        for r in range(R):
            s = rep == r
            pos[s] = coords[r][:, atom[s] * systems[r][1] + it[s]].T + rng.normal(0, 0.15, (int(s.sum()), 3))
        return dict(case=case, ctx=ctx, rep=rep, atom=atom, it=it, pos=pos)
    elif kind == "box":
        N, P, T = case["atoms"], case["slices"], case["temp"]
        m = math.ceil(N ** (1.0 / 3.0))
        L = 3.6 * m
        grid = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)[:N] * 3.6 - 0.5 * L
        r1, v1 = pt.lj_table()
        ctx.add_pot1d(r1, v1)
        for i in range(R):
            ctx.set_replica(i, 1, [N], [0], [case["levels"]], [0.6], [pc.MASS_HE4], P, 0, T, 0.0, pot1d=[0], pot2d=[-1])
            ctx.set_minimum_image(i, L)
        ctx.commit()
        for i in range(R):
            ctx.set_state(i, _paths(rng, grid + rng.normal(0, 0.1, (N, 3)), [pc.MASS_HE4] * N, P, T, 0.45))
        systems = [(N - 1, P, T)] * R
    else:
        P, T = case["slices"], case["temp"]
        if kind == "top":
            N = case["atoms"]
            if case["da"]:
                ctx.set_option("delayed_acceptance", 1)
            ctx.add_pot1d(*pt.h2h2_table())
            ctx.add_pot3d(*_pot3d())
            # the density of 256 slices at this temperature for every path length: a table file in hand
            ctx.add_rot3d(*_asymrho(T, 256, 20))
            for i in range(R):
                ctx.set_replica(i, 2, [N, 1], [0, 2], [case["levels"]] * 2, [0.3, 0.1], [pc.MASS_H2, pc.MASS_H2O], P, P,
                                T, 0.4, pot1d=[0, -1], pot2d=[-1, -1], pot3d=0, rot3d=0)
            centres = np.concatenate([_sites(N, 3.8, 3.4), np.zeros((1, 3))])
            masses, first, step, sig = [pc.MASS_H2] * N + [pc.MASS_H2O], N, 0.25, 0.45
        else:
            ctx.add_rot3d(*_asymrho(T, 2048, 44))
            for i in range(R):
                ctx.set_replica(i, 1, [2], [2], [case["levels"]], [0.05], [pc.MASS_H2O], P, P, T, 0.3, pot1d=[-1],
                                pot2d=[-1], pot3d=-1, rot3d=0)
            centres = np.array([[-1.45, 0.0, 0.0], [1.45, 0.0, 0.0]])
            masses, first, step, sig = [pc.MASS_H2O] * 2, 0, 0.1, 0.25
        ctx.commit()
        for i in range(R):
            c = centres + rng.normal(0, 0.05, centres.shape)
            ctx.set_state(i, _paths(rng, c, masses, P, T, sig), _angles(rng, len(c), first, P, P, step))
        if case.get("da"):
            ctx.surrogate_set(*_cached_network())
        systems = [(len(centres) - 1, P, T)] * R
    beads = [(n + 1) * P for n, P, _ in systems]
    return dict(case=case, ctx=ctx, beads=beads, coords=np.empty(3 * sum(beads)), cosines=np.empty(3 * sum(beads)))


# ---------------------------------------------------------------------------- one pass
def run(state):
    case, ctx = state["case"], state["ctx"]
    if case["kind"] == "queries":
        return ctx.pot_energy_slice(state["rep"], state["atom"], state["it"], state["pos"])
    if case["kind"] == "train":
        loss = ctx.surrogate_train(state["x"], state["v"], epochs=case["epochs"], batch=case["batch"], lr=2e-3,
                                   seed=state["seed"])
        theta, norm = ctx.surrogate_get()
        return dict(loss=loss.astype(np.float32), theta=theta, norm=norm)  # the network's outputs are FP32
    ctx.clear_samples()
    ctx.run(case["passes"], case["every"])
    R, n = case["replicas"], case["passes"] // case["every"]
    out = dict(samples=np.stack([ctx.samples(r, n) for r in range(R)]),
               accepted=np.concatenate([ctx.counters(r)[1].reshape(-1) for r in range(R)]),
               coords=state["coords"], cosines=state["cosines"])
    # the configuration of every replica into one array each, [3][atoms*P] per replica
    dp, at = ctypes.POINTER(ctypes.c_double), 0
    for r, b in enumerate(state["beads"]):
        c, s = state["coords"][at:at + 3 * b], state["cosines"][at:at + 3 * b]
        ctx._check(ctx.lib.pimc_get_state(ctx.h, r, c.ctypes.data_as(dp), None, s.ctypes.data_as(dp)))
        at += 3 * b
    if R == 1:
        out["gr"], out["grt"] = ctx.histograms(0)
        if case["kind"] != "box":
            out["rcf"] = ctx.rcf(0)
    return out


# ---------------------------------------------------------------------------- work and exact values
FLOP_1D, FLOP_2D, FLOP_3D, FLOP_DIMER, FLOP_LINK = 28, 36, 90, 330, 120


def work(case):
    """Proposals' pair terms (what a move adds to what the chain already knows) and, in bytes, the
    configuration in and out once and the samples."""
    kind = case["kind"]
    if kind == "train":
        steps = case["epochs"] * (case["rows"] // case["batch"])
        return dict(bytes=case["rows"] * 20.0 * case["epochs"] + 33793 * 28.0 * steps,
                    flops=3.0 * 2 * (4 * 128 + 2 * 128 * 128 + 128) * case["batch"] * steps)
    if kind == "queries":
        s = _systems(dict(case, pmin=case["slices"], ratio=1, levels=3, tmin=1.0, tmax=1.0))
        n = sum(x[0] for x in s) / len(s)
        return dict(bytes=44.0 * case["queries"] + sum(24.0 * (x[0] + 1) * x[1] for x in s),
                    flops=case["queries"] * n * FLOP_1D)
    moved = (1 << case["levels"]) - 1 + 1  # bisection midpoints of a start slice, and the centroid move
    beads = flops = 0.0
    if kind == "linear":
        for n, P, _ in _systems(case):
            beads += (n + 1) * P
            flops += moved * P * (n * (n - 1) * FLOP_1D + 2 * n * FLOP_2D)
            flops += P * (P // case["ratio"]) * (n * case["ratio"] * FLOP_2D + FLOP_LINK)
    else:
        P, R = case["slices"], case["replicas"]
        if kind == "box":
            n = case["atoms"]
            beads, flops = R * n * P, R * moved * P * n * (n - 1) * FLOP_1D
        elif kind == "top":
            n = case["atoms"]
            beads = R * (n + 1) * P
            flops = R * (moved * P * (n * (n - 1) * FLOP_1D + 2 * n * FLOP_3D) + P * P * (n * FLOP_3D + 2 * FLOP_LINK))
        else:
            beads, flops = R * 2 * P, R * (moved * P * 2 * FLOP_DIMER + 2.0 * P * P * (FLOP_DIMER + 2 * FLOP_LINK))
    return dict(bytes=beads * 2 * 48.0, flops=flops * case["passes"])


def _spline2(x, y):
    """Second derivatives of the cubic spline through (x, y), end slopes the first differences."""
    n, h = len(x), np.diff(x)
    s = np.diff(y) / h
    A, b = np.zeros((n, n)), np.zeros(n)
    i = np.arange(1, n - 1)
    A[i, i - 1], A[i, i], A[i, i + 1] = h[:-1] / 6, (h[:-1] + h[1:]) / 3, h[1:] / 6
    b[1:-1] = s[1:] - s[:-1]
    A[0, :2], A[-1, -2:] = (h[0] / 3, h[0] / 6), (h[-1] / 6, h[-1] / 3)
    return np.linalg.solve(A, b)


def exact(case, seed):
    """PotEnergy queries in plain FP64.  The chains' outputs have no value apart from the FP32
    pair terms that decide every move, and the training's none apart from its BF16 products."""
    if case["kind"] != "queries":
        return None
    P, T, R = case["slices"], case["temp"], case["replicas"]
    rng = np.random.default_rng([seed, 11])
    systems = _systems(dict(case, pmin=P, ratio=1, levels=3, tmin=T, tmax=T))
    P = systems[0][1]
    coords, axes = [], []
    for n, _, _ in systems:
        c = np.concatenate([_sites(n, 3.7, 3.3) + rng.normal(0, 0.1, (n, 3)), np.zeros((1, 3))])
        coords.append(_paths(rng, c, [pc.MASS_HE4] * n + [pc.MASS_CO2], P, T, 0.5).reshape(3, n + 1, P))
        a = _angles(rng, n + 1, n, P, P, 0.1).reshape(3, n + 1, P)[:, n]
        st = np.sqrt(1.0 - a[1] ** 2)
        axes.append(np.stack([st * np.cos(a[0]), st * np.sin(a[0]), a[1]]))
    q = case["queries"]
    rep = rng.integers(0, R, q).astype(np.int32)
    natoms = np.array([s[0] + 1 for s in systems])
    atom = (rng.random(q) * natoms[rep]).astype(np.int32)
    it = rng.integers(0, P, q).astype(np.int32)
    (x, y), (rg, cg, dr, dc, V) = _pair_tables()
    y2 = _spline2(x, y)
    alpha = math.log(y[0] / y[1]) / (x[1] - x[0])
    c6 = (y[-1] - y[-2]) / (x[-2] ** -6 - x[-1] ** -6)

    def one(r):
        k = np.clip(np.searchsorted(x, r, side="right") - 1, 0, len(x) - 2)
        h = x[k + 1] - x[k]
        a, b = (x[k + 1] - r) / h, (r - x[k]) / h
        v = a * y[k] + b * y[k + 1] + ((a ** 3 - a) * y2[k] + (b ** 3 - b) * y2[k + 1]) * h * h / 6
        return np.where(r >= x[-1], -c6 * r ** -6.0, np.where(r <= x[0], y[0] * np.exp(alpha * (x[0] - r)), v))

    def two(r, c):
        i = np.clip(np.floor((r - rg[0]) / dr), 0, len(rg) - 2).astype(int)
        j = np.clip(np.floor((c - cg[0]) / dc), 0, len(cg) - 2).astype(int)
        a, b = (r - rg[i]) / (rg[i + 1] - rg[i]), (c - cg[j]) / (cg[j + 1] - cg[j])
        return ((1 - a) * (1 - b) * V[i, j] + a * (1 - b) * V[i + 1, j] + a * b * V[i + 1, j + 1] + (1 - a) * b * V[i, j + 1])

    out = np.empty(q)
    for r, (n, _, _) in enumerate(systems):
        s = np.nonzero(rep == r)[0]
        pos = coords[r][:, atom[s], it[s]].T + rng.normal(0, 0.15, (len(s), 3))
        d = pos[:, :, None] - coords[r][:, :, it[s]].transpose(2, 0, 1)  # mover - partner
        dist = np.sqrt((d ** 2).sum(1))
        own = np.arange(n + 1)[None, :] == atom[s][:, None]
        dist = np.where(own, 1.0, dist)
        cos = np.einsum("qik,iq->qk", d, axes[r][:, it[s]]) / dist
        rotor = atom[s] == n
        v = one(dist)
        v[:, n] = two(dist[:, n], cos[:, n])
        v[rotor] = two(dist[rotor], -cos[rotor])
        out[s] = np.where(own, 0.0, v).sum(1)
    return out
