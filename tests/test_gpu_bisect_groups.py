"""Bisection groups (MCBisectionMove, mc_piqmc.cc:194-294): every number of lanes a segment can get,
levels from one to seven (chunks of one to three levels, moves of more midpoints than a group has
lanes), odd numbers of segments, against the oracle's chain on the same draws.  FP64: the moves are
the oracle's, so acceptances are equal and positions agree to rounding (1e-9 Angstrom, as in the
other trajectory tests)."""
import numpy as np
import pytest

import oracle as O
import pimc_configs as pc
import pimc_hip as ph

pytestmark = pytest.mark.gpu
SEED = 985456376


def deck(n_he, P, levels, n_replicas, T=0.9):
    wl = pc.workload("tiny")
    wl["tables"]["rot"] = [pc.rot_table(T, P)]
    reps = []
    for r in range(n_replicas):
        rp = pc.replica(n_he, P, T, SEED + r)
        rp.update(levels=[levels, max(1, levels - 1)], rotdens=0, pot1d=[0, -1], pot2d=[-1, 0])
        reps.append(rp)
    wl["replicas"] = reps
    return wl


def check(wl, which, lanes=0, npass=2):
    ctx = ph.Context(len(wl["replicas"]), flags=ph.FLAG_FP64, seed=SEED)
    for k in ("small", "medium", "large"):
        if lanes:
            ctx.set_option("bisect_lanes_" + k, lanes)
    pc.load_into_context(ctx, wl)
    ctx.run(npass)
    for r in which:
        S = O.System(wl["replicas"][r], wl["tables"], seed=SEED, replica=r)
        S.run(0, npass, order=O.ORDER_SEGMENTS)
        assert np.array_equal(ctx.counters(r)[1], S.counters()[1]), r
        assert np.abs(ctx.get_state(r)[0] - S.state()[0]).max() < 1e-9, r
    ctx.close()


@pytest.mark.parametrize("lanes", [64, 128, 256])
@pytest.mark.parametrize("levels,n_he,P", [(1, 5, 16), (2, 1, 12), (3, 33, 24), (4, 18, 48), (5, 9, 96), (7, 2, 256)])
def test_levels_and_lanes(lanes, levels, n_he, P):
    check(deck(n_he, P, levels, 1), [0], lanes)


@pytest.mark.parametrize("n_he,levels,P", [(2, 3, 24), (17, 2, 12)])
def test_two_segments_share_a_wave(n_he, levels, P):
    """More than 4096 segments of few atoms, three per chain: groups of 32 lanes, some without one."""
    n = 4096 // (P >> levels) + 40
    check(deck(n_he, P, levels, 1), [0])
    check(deck(n_he, P, levels, n), [0, 1, n - 1])


@pytest.mark.parametrize("n_he,fp64", [(40, False), (40, True)])
def test_lanes_by_load_keep_the_chain(n_he, fp64):
    """The default lanes change with the number of segments, the chain does not: replica 0 alone and
    among 48 makes the same moves (its key and draws are the same, sums over pairs are FP64)."""
    out = []
    for n in (1, 48):
        wl = deck(n_he, 128, 3, n)
        ctx = ph.Context(n, flags=ph.FLAG_FP64 if fp64 else 0, seed=SEED)
        pc.load_into_context(ctx, wl)
        ctx.run(2)
        out.append((ctx.get_state(0)[0], ctx.counters(0)[1]))
        ctx.close()
    assert np.array_equal(out[0][1], out[1][1])
    assert np.abs(out[0][0] - out[1][0]).max() < 1e-9
