"""Systems near the LDS limits of a launch: pimc_commit accepts what each replica's own layout fits,
and the chains are those of the same replicas elsewhere."""
import numpy as np
import pytest

import oracle as O
import pimc_configs as pc
import pimc_hip as ph
import pimc_tables as pt

pytestmark = pytest.mark.gpu
SEED = 985456376


def lattice(n, P, seed):
    m = int(np.ceil(n ** (1.0 / 3.0)))
    g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n] * 3.6
    return (g.T[:, :, None] + np.random.default_rng(seed).normal(0.0, 0.1, (3, n, P))).reshape(3, -1)


def test_a_large_window_beside_a_long_table():
    """A bisection block holds one replica's segments and knots: 1000 atoms with a short table (87 KB)
    and 70 atoms with a table of 10000 knots (86 KB) share a size class, though the larger window and
    the longer table together would not fit."""
    P, levels = 16, 3

    def run(which):
        ctx = ph.Context(len(which), seed=SEED)
        tabs = [ctx.add_pot1d(*pt.lj_table(n=10000)), ctx.add_pot1d(*pt.lj_table(n=500))]
        for i, (n, t) in enumerate(which):
            ctx.set_replica(i, 1, [n], [0], [levels], [0.3], [pc.MASS_HE4], P, 0, 2.0, 0.0, pot1d=[tabs[t]], pot2d=[-1])
        ctx.commit()
        for i, (n, _) in enumerate(which):
            ctx.set_state(i, lattice(n, P, i))
        ctx.run(2)
        out = ctx.get_state(0)[0], ctx.counters(0)[1]
        assert ctx.counters(len(which) - 1)[1][0][:2].min() > 0
        ctx.close()
        return out

    alone, beside = run([(70, 0)]), run([(70, 0), (1000, 1)])
    assert np.array_equal(alone[1], beside[1])
    assert np.abs(alone[0] - beside[0]).max() < 1e-9


def test_the_longest_table_of_a_centroid_part():
    """10200 FP32 knots are 163200 of a workgroup's 163840 bytes; the rest holds the move's sums."""
    P, n = 16, 12
    ctx = ph.Context(1, seed=SEED)
    t = ctx.add_pot1d(*pt.lj_table(n=10200))
    ctx.set_replica(0, 1, [n], [0], [2], [0.3], [pc.MASS_HE4], P, 0, 2.0, 0.0, pot1d=[t], pot2d=[-1])
    ctx.commit()
    ctx.set_state(0, lattice(n, P, 0))
    ctx.run(3)
    total, accepted = ctx.counters(0)
    assert total[0][0] == 3 * n and 0 < accepted[0][0] <= 3 * n
    ctx.close()


@pytest.mark.parametrize("n_he,P,Prot,bytes_", [
    (1238, 16, 8, 158688),   # parts of two slices, two time slices each: 158688 bytes of a workgroup's 163840
    (1238, 68, 68, 79456),   # 34 parts of two slices, two to a CU: with 9 KB more each, an XCD holds 32
])
def test_rotor_parts_that_fill_a_workgroups_lds(n_he, P, Prot, bytes_):
    """Partner geometry of up to all of a workgroup's LDS, as the plan admits it; one pass in FP64
    follows the oracle (acceptances equal, axes and positions to rounding, 1e-9)."""
    rp = pc.replica(0, P, 0.9, SEED, Prot=Prot)
    x = lattice(n_he + 1, P, 3).reshape(3, n_he + 1, P)
    x -= x[:, n_he // 2:n_he // 2 + 1].mean(2, keepdims=True)  # the rotor takes the place of one in the middle
    x = np.concatenate([np.delete(x, n_he // 2, 1), np.zeros((3, 1, P))], 1)
    angles = np.zeros((3, n_he + 1, P))
    angles[1] = 1.0
    angles[1, -1, :Prot] = np.cos(0.1 * np.sin(np.arange(Prot)))
    angles[0, -1, :Prot] = 0.3 * np.arange(Prot)
    rp.update(numb=[n_he, 1], levels=[1, 1], mcstep=[0.02, 0.05], rotdens=0, pot1d=[0, -1], pot2d=[-1, 0],
              coords=x.reshape(3, -1), angles=angles.reshape(3, -1))
    wl = dict(pc.workload("tiny"), replicas=[rp])
    wl["tables"]["rot"] = [pc.rot_table(0.9, Prot)]
    ctx = pc.load_into_context(ph.Context(1, flags=ph.FLAG_FP64, seed=SEED), wl)
    if hasattr(ctx, "launch_shape"):
        assert ctx.launch_shape("rotor_lds_bytes") == bytes_
    ctx.run(1)
    S = O.System(rp, wl["tables"], seed=SEED, replica=0)
    S.run(0, 1, order=O.ORDER_SEGMENTS)
    got, ref = ctx.get_state(0), S.state()
    assert np.array_equal(ctx.counters(0)[1], S.counters()[1])
    assert 0 < ctx.counters(0)[1][1][2] < P * Prot
    assert np.abs(got[0] - ref[0]).max() < 1e-9
    assert np.abs(got[2] - ref[2]).max() < 1e-9
    ctx.close()
