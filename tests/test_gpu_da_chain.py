"""Delayed-acceptance rotor sweep (MCRot3Dstep, mc_piqmc.cc:938-1199, as three Metropolis factors)
move for move: an FP64 restatement of the three stages on the same draws, with the network's rows
evaluated by pimc_surrogate_eval, and the same chain in short parts (state on chip) and in parts
beyond 256 rotor slices (state in memory).  FP64 pair terms: every decision and stage count equal,
positions and angles within 1e-9 (the bound of the other trajectory tests)."""
import numpy as np
import pytest

import mlp_oracle as M
import oracle as O
import pimc_configs as pc
import pimc_hip as ph
from golden import tables3d
from test_gpu_nonlinear import SEED, nl_workload, rotor_columns

pytestmark = pytest.mark.gpu
TWOPI = 2.0 * np.pi


@pytest.fixture(scope="module")
def rot3d():
    return tables3d.rot3d()


def deck(rot3d, n_h2, nrot, P, ratio=1):
    """n_h2 para-H2 around nrot rotors (two rigid waters when there are no atoms)."""
    wl = nl_workload("h2o_h2" if n_h2 else "water2", rot3d, n_h2=n_h2, P=P, Prot=P // ratio, seed=5)
    rp = wl["replicas"][0]
    if n_h2 > 4:  # two shells
        for a in range(n_h2):
            u = np.random.default_rng(a).standard_normal(3)
            centre = u / np.linalg.norm(u) * (3.5 if a % 2 else 4.6)
            rp["coords"][:, a * P:(a + 1) * P] += (centre - rp["coords"][:, a * P:(a + 1) * P].mean(1))[:, None]
    if n_h2 and nrot == 2:
        rng = np.random.default_rng(6)
        rp["numb"] = [n_h2, 2]
        rp["coords"] = np.concatenate([rp["coords"], np.array([[0.0], [0.2], [2.9]]) + rng.normal(0, 0.12, (3, P))], 1)
        more = np.stack([rng.uniform(0, TWOPI, P), rng.uniform(-1, 1, P), rng.uniform(0, TWOPI, P)])
        rp["angles"] = np.concatenate([rp["angles"], more], 1)
    return wl


def context(wl, copies, net, fp64=True):
    ctx = ph.Context(copies, flags=ph.FLAG_FP64 if fp64 else 0, seed=SEED)
    ctx.set_option("delayed_acceptance", 1)
    pc.load_into_context(ctx, dict(tables=wl["tables"], replicas=wl["replicas"] * copies))
    ctx.surrogate_set(*net)
    return ctx


def network(atoms):
    """A random network whose rows spread over a few Kelvin, as many of them to a move as it has;
    norm leaves the output as it is (ym = 0, ys = 1), so that a row's value is pimc_surrogate_eval's."""
    theta = M.glorot(3) + np.random.default_rng(4).normal(0, 0.02, M.NW)
    o, s = M.OFF["w4"]
    theta[o:o + int(np.prod(s))] *= 20.0 / np.sqrt(max(atoms, 1))
    return theta.astype(np.float32), np.array([4.0, 0, 0, 0, 1.0, 0.6, 0.6, 0.6, 0.0, 1.0], np.float32)


# ------------------------------------------------------------------ the three stages in FP64
def u53(hi, lo):
    return ((hi >> 5) * 67108864.0 + (lo >> 6)) / 9007199254740992.0


def draws(key, pass_, sweep, atom, k, c3):
    """The two uniforms of K_ROT3D's counter word 3 = c3 (words 0, 1 and 2, 3)."""
    w = O.philox([pass_, (4 << 28) | sweep, (atom << 16) | k, c3], [SEED, key])
    return u53(w[0], w[1]), u53(w[2], w[3])


def frames(phi, cth, chi):
    """Columns of the rotation matrix (rotden.f:136-163), rows 0-2, 3-5 and 6-8."""
    cp, sp, ck, sk = np.cos(phi), np.sin(phi), np.cos(chi), np.sin(chi)
    ct, st = np.cos(np.arccos(cth)), np.sin(np.arccos(cth))
    return np.array([cp * ct * ck - sp * sk, sp * ct * ck + cp * sk, -st * ck, -cp * ct * sk - sp * ck,
                     -sp * ct * sk + cp * ck, st * sk, cp * st, sp * st, ct])


class Restated:
    def __init__(self, wl, key, net):
        self.rp, t = wl["replicas"][0], wl["tables"]
        tabs = dict(pot1d=t["pot1d"], pot2d=[], rot=[], pot3d=t["pot3d_list"][0] if t["pot3d_list"] else None,
                    rot3d=t["rot3d_list"][0])
        self.S = O.System(self.rp, tabs, seed=SEED, replica=key)
        self.key, self.rot = key, [np.ascontiguousarray(x) for x in tabs["rot3d"]]
        self.net = ph.Context(1)
        self.net.surrogate_set(*net)
        self.nat = sum(n for n, m in zip(self.rp["numb"], self.rp["molecule"]) if m == 0)
        self.nrot = self.rp["numb"][-1]
        self.da = np.zeros(4)

    def rho(self, e1, e2):
        rel, out, stop = np.zeros(3), np.zeros(3), np.zeros(1, np.int32)
        p = [out[i:].ctypes.data_as(O._dp) for i in range(3)]
        self.S.L.or_rotden(O.P(e1), O.P(e2), rel.ctypes.data_as(O._dp), *p, *[x.ctypes.data_as(O._dp) for x in self.rot],
                           stop.ctypes.data_as(O._ip))
        assert not stop[0]
        return out[0]

    def caleng(self, x1, x2, e1, e2):
        e = np.zeros(1)
        self.S.L.or_caleng(O.P(x1), O.P(x2), e.ctypes.data_as(O._dp), O.P(e1), O.P(e2))
        return e[0]

    def half(self, pass_, sweep, parity, q):
        rp, P, Prot = self.rp, self.rp["P"], self.rp["Prot"]
        RR, tau, nat = P // Prot, 1.0 / (rp["T"] * P), self.nat
        x, a, _ = self.S.state()
        a = a.copy()
        at = lambda p, k: (nat + p) * P + k  # noqa: E731
        eul = lambda p, k: np.array([a[0, at(p, k)], np.arccos(a[1, at(p, k)]), a[2, at(p, k)]])  # noqa: E731
        pos = lambda i, it: x[:, i * P + it]  # noqa: E731

        def link(e0, e1, e2):
            d = self.rho(e0, e1) * self.rho(e1, e2)
            return 0.0 if abs(d) < 1e-10 else abs(d)

        def features(p, k, it, f, fo):
            if nat:
                return [M.pair_features(f, np.linalg.norm(f[6:]), pos(nat + p, it), pos(i, it)) for i in range(nat)]
            return [M.rotor_pair_features(f, fo, pos(nat + p, it), pos(nat + 1 - p, it))]

        moves, rows = [], []
        for k in range(parity, Prot, 2):
            r1, r2 = draws(self.key, pass_, sweep, nat + q, k, 0)
            r3, u1 = draws(self.key, pass_, sweep, nat + q, k, 1)
            u2, u0 = draws(self.key, pass_, sweep, nat + q, k, 2)
            cth = a[1, at(q, k)] + rp["rtstep"] * (r1 - 0.5)
            phi = a[0, at(q, k)] + TWOPI * (rp["rtstep"] * (r2 - 0.5))
            chi = a[2, at(q, k)] + TWOPI * (rp["rtstep"] * (r3 - 0.5))
            phi, chi = [np.fmod(TWOPI + v if v < 0.0 else v, TWOPI) for v in (phi, chi)]
            cth = 2.0 - cth if cth > 1.0 else (-2.0 - cth if cth < -1.0 else cth)
            new, old = np.array([phi, np.arccos(cth), chi]), eul(q, k)
            before, after = eul(q, (k - 1) % Prot), eul(q, (k + 1) % Prot)
            dold, dnew = link(before, old, after), link(before, new, after)
            self.da[0] += 1
            ratio = dnew / dold if dold > 1e-10 else 1.0
            if not (ratio > 1.0 or ratio > u0):
                continue
            its = range(k * RR, (k + 1) * RR)
            other = eul(1 - q, k) if self.nrot == 2 else None
            dpair = sum(self.caleng(pos(nat + q, it), pos(nat + 1 - q, it), e, other) * s
                        for it in its for e, s in ((new, 1.0), (old, -1.0))) if self.nrot == 2 else 0.0
            fn, fo_ = frames(phi, cth, chi), frames(*[a[i, at(q, k)] for i in range(3)])
            fp = frames(*[a[i, at(1 - q, k)] for i in range(3)]) if self.nrot == 2 else None
            n0 = len(rows)
            for it in its:
                rows += features(q, k, it, fn, fp) + features(q, k, it, fo_, fp)
            moves.append((k, (phi, cth, chi), new, old, dpair, u1, u2, n0, len(rows)))
            self.da[3] += RR * nat if nat else 2 * RR
        if not moves:
            return
        out = self.net.surrogate_eval(np.array(rows, np.float32)).astype(np.float64)
        for k, angles, new, old, dpair, u1, u2, n0, n1 in moves:
            o = out[n0:n1].reshape(P // Prot, 2, -1)  # time slice, new or old, partner
            dvs = o[:, 0].sum() - o[:, 1].sum()
            r1 = np.exp(-tau * (dvs + (dpair if nat else 0.0)))
            if not (r1 > 1.0 or r1 > u1):
                continue
            self.da[1] += 1
            dve = dpair
            if nat:  # PotRotE3D less its rotor-rotor term
                e3 = lambda e: sum(self.S.L.or_pot_rot_e3d(self.S.h, nat + q, O.P(e), it)  # noqa: E731
                                   for it in range(k * RR, (k + 1) * RR))
                dve = e3(new) - e3(old) - dpair
            r2 = np.exp(-tau * (dve - dvs))
            if r2 > 1.0 or r2 > u2:
                self.da[2] += 1
                a[:, at(q, k)] = angles
        self.S.set_state(x, a)

    def run(self, npass):
        rp, S = self.rp, 1 << max(self.rp["levels"])
        for pass_ in range(npass):
            for u in range(S):
                for ty in range(rp["ntypes"]):
                    if u == 0:
                        self.S.L.or_molecular_move(self.S.h, ty, pass_)
                    for atom in range(rp["numb"][ty]):
                        for s in range(u, rp["P"], S):
                            self.S.L.or_bisection_atom(self.S.h, ty, atom, s, pass_)
                for s in range(u, rp["P"], S):
                    for parity in (0, 1):
                        for q in range(self.nrot):
                            self.half(pass_, s, parity, q)


@pytest.mark.parametrize("n_h2,nrot,P,ratio", [
    (9, 1, 8, 1),     # one part, its own neighbour; nine rows a move, so a batch of 32 holds pieces of moves
    (10, 1, 32, 1),   # parts that trade; half a wave to a move's exact terms
    (36, 1, 16, 1),   # more rows than a batch, more than 32 exact terms
    (20, 1, 16, 2),   # two time slices a rotor slice
    (3, 2, 16, 1),    # two rotors among atoms: their pair exact in stage 1
    (3, 1, 16, 1),    # three rows a move
    (0, 2, 16, 1),    # the rotor-rotor network
])
def test_every_stage_follows_the_restatement(rot3d, n_h2, nrot, P, ratio):
    wl, net = deck(rot3d, n_h2, nrot, P, ratio), network(n_h2)
    ctx = context(wl, 2, net)
    ctx.run(2)
    R = Restated(wl, 1, net)
    R.run(2)
    assert 0 < R.da[2] < R.da[1] < R.da[0]  # every stage rejects something
    assert np.array_equal(ctx.da_counters(1), R.da), (ctx.da_counters(1), R.da)
    c, a, _ = ctx.get_state(1)
    co, ao, _ = R.S.state()
    cols = np.arange(c.shape[1])[rotor_columns(R.rp)].reshape(-1, P)[:, :P // ratio].reshape(-1)
    assert np.abs(c - co).max() < 1e-9
    assert np.abs(a[:, cols] - ao[:, cols]).max() < 1e-9
    assert np.array_equal(ctx.counters(1)[1][-1][2], R.da[2])
    ctx.close()


@pytest.mark.parametrize("n_h2,nrot,P,fp64", [
    (9, 1, 320, True), (36, 1, 272, True), (3, 2, 160, True), (0, 2, 192, True), (9, 1, 320, False), (0, 2, 192, False)])
def test_long_parts_follow_short_ones(rot3d, n_h2, nrot, P, fp64):
    """300 chains leave whole chains to a workgroup, whose parts of more than 256 rotor slices keep
    their state in memory; two chains are split into short parts.  Same draws, same chain."""
    wl, net = deck(rot3d, n_h2, nrot, P), network(n_h2)
    out = []
    for copies in (2, 300):
        ctx = context(wl, copies, net, fp64)
        ctx.run(1)
        out.append([(ctx.da_counters(r), ctx.counters(r), ctx.get_state(r)) for r in (0, 1)])
        ctx.close()
    for short, long in zip(*out):
        assert np.array_equal(short[0], long[0]), (short[0], long[0])
        assert 0 < short[0][2] < short[0][1] < short[0][0]
        assert np.array_equal(short[1], long[1])
        assert max(np.abs(s - g).max() for s, g in zip(short[2], long[2])) < 1e-9
