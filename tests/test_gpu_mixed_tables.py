"""Replicas on uniform tables beside replicas on others in one FP32 context.  A chain's pair terms
follow its own tables, so it is the same chain whoever shares the context, and in parts beyond 256
rotor slices: equal counters, positions and orientations (proposals depend on draws and end points
alone, so equal decisions give equal bits).  FP32 pair terms formed in another order of rounding
change about one decision in ten to a hundred million; these runs make 20 to 200 million."""
import numpy as np
import pytest

import pimc_configs as pc
import pimc_hip as ph

pytestmark = pytest.mark.gpu
SEED = 985456376


def stretched_tables():
    """The workload's pair tables on grids that are finer at small r and near the ends of cos theta."""
    r = 1.0 + 29.0 * np.linspace(0.0, 1.0, 500) ** 1.3
    sr6 = (2.556 / r) ** 6
    rg = 1.5 + 20.0 * np.linspace(0.0, 1.0, 1001) ** 1.1
    cg = -np.cos(np.linspace(0.0, np.pi, 201))
    P2, P4 = 0.5 * (3 * cg ** 2 - 1), 0.125 * (35 * cg ** 4 - 30 * cg ** 2 + 3)
    morse = ((1.0 - np.exp(-1.2 * (rg - 3.5))) ** 2 - 1.0)[:, None]
    V = morse * (30.0 + 8.0 * P2 + 2.0 * P4)[None, :]
    return (r, 4.0 * 10.22 * (sr6 * sr6 - sr6)), (rg, cg, rg[1] - rg[0], cg[1] - cg[0], V)


def chains(n_he, P, copies, others, npass, keep=False, **options):
    """State and counters of `copies` replicas on the workload's uniform tables, beside replicas whose
    1D table, 2D table or both (others: pairs of 0 or 1) are the stretched ones."""
    wl = pc.workload("tiny")
    t1, t2 = stretched_tables()
    wl["tables"].update(rot=[pc.rot_table(0.8, P)], pot1d=wl["tables"]["pot1d"] + [t1], pot2d=wl["tables"]["pot2d"] + [t2])
    base = dict(pc.replica(n_he, P, 0.8, SEED), rotdens=0, pot1d=[0, -1], pot2d=[-1, 0])
    wl["replicas"] = [base] * copies + [dict(base, pot1d=[a, -1], pot2d=[-1, b]) for a, b in others]
    ctx = ph.Context(len(wl["replicas"]), seed=SEED)
    for k, v in options.items():
        ctx.set_option(k, v)
    pc.load_into_context(ctx, wl)
    if keep:
        return ctx
    ctx.run(npass)
    out = [(*ctx.get_state(r), *ctx.counters(r)) for r in range(copies)]
    ctx.close()
    return out


def lanes(n_he, P, copies, others, **options):
    """Lanes per segment of the launch on uniform tables and of the others' (one size class)."""
    ctx = chains(n_he, P, copies, others, 0, keep=True, **options)
    name = "bisect_lanes_" + ("small" if n_he < 24 else "medium" if n_he < 64 else "large")
    out = ctx.launch_shape(name), ctx.launch_shape(name + "_general")
    ctx.close()
    return out


def same(a, b):
    for r, (x, y) in enumerate(zip(a, b)):
        assert all(np.array_equal(u, v) for u, v in zip(x, y)), r


@pytest.mark.parametrize("n_he,P,copies,npass", [(8, 64, 64, 600), (40, 64, 48, 60)])
def test_other_tables_beside_do_not_change_a_chain(n_he, P, copies, npass):
    alone = chains(n_he, P, copies, [], npass)
    same(alone, chains(n_he, P, copies, [(1, 1)], npass))
    same(alone, chains(n_he, P, copies, [(1, 0), (0, 1)], npass))


def test_long_parts_keep_the_arithmetic():
    alone = chains(20, 320, 32, [], 60)
    same(alone, chains(20, 320, 32, [], 60, rotor_part_slices=320, rotor_lds_kb=140))


@pytest.mark.parametrize("n_he", [40, 100])
def test_each_launch_has_the_lanes_of_its_own_load(n_he):
    """P = 128 at eight slices a segment: 16 segments a chain, 2048 of 128 chains.  Lanes measured on
    uniform tables made a pass over stretched ones up to 1.4 times as long."""
    full, few = ph.plan_bisect_lanes(n_he + 1, 2048)[0], ph.plan_bisect_lanes(n_he + 1, 16, stretched_1d=True)[0]
    assert lanes(n_he, 128, 128, []) == (full, 64)
    assert lanes(n_he, 128, 128, [(1, 0)]) == (full, few) == (64, 256)
    assert lanes(n_he, 128, 0, [(1, 1)] * 128) == (64, ph.plan_bisect_lanes(n_he + 1, 2048, stretched_1d=True)[0]) == (64, 128)
    assert lanes(n_he, 128, 0, [(0, 1)] * 128) == (64, 64)
