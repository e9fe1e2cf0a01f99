"""Linear-rotor sweep (MCRotLinStep, mc_piqmc.cc:781-936): every split of the work inside a part --
one and two chain waves, one to many energy lanes per move, parts of two slices, parts beyond 256
slices, chains that are their own neighbour, no partners -- and links outside the staged knots,
against the oracle's chain on the same draws.  FP64: acceptances equal, axes and positions to
rounding (1e-9, as in the other trajectory tests)."""
import numpy as np
import pytest

import oracle as O
import pimc_configs as pc
import pimc_hip as ph

pytestmark = pytest.mark.gpu
SEED = 985456376


def run_both(n_he, P, Prot, T, options, angles=None, fp64=True, npass=2, levels=2, tables=None):
    wl = pc.workload("tiny")
    wl["tables"]["rot"] = [tables or pc.rot_table(T, Prot)]
    rp = pc.replica(n_he, P, T, SEED, Prot=Prot)
    rp.update(levels=[levels, levels], rotdens=0, pot1d=[0, -1], pot2d=[-1, 0])
    if n_he == 0:  # a lone rotor
        for k in ("type_names", "numb", "molecule", "levels", "mcstep", "mass", "pot1d", "pot2d"):
            rp[k] = rp[k][1:]
        rp["ntypes"] = 1
    if angles is not None:
        rp["angles"] = angles(rp)
    wl["replicas"] = [rp]
    ctx = ph.Context(1, flags=ph.FLAG_FP64 if fp64 else 0, seed=SEED)
    for k, v in options.items():
        ctx.set_option(k, v)
    pc.load_into_context(ctx, wl)
    ctx.run(npass)
    S = O.System(rp, wl["tables"], seed=SEED, replica=0)
    S.run(0, npass, order=O.ORDER_SEGMENTS)
    got, ref = ctx.get_state(0), S.state()
    acc = ctx.counters(0)[1], S.counters()[1]
    ctx.close()
    return got, ref, acc


@pytest.mark.parametrize("n_he,P,Prot,options", [
    (3, 16, 16, {}),                                    # one part, its own neighbour, 24 lanes a move
    (1, 16, 4, {}),                                     # two moves a half
    (2, 8, 2, {}),                                      # one move a half: both neighbours are one slice
    (0, 24, 24, {}),                                    # no partners
    (5, 64, 64, dict(rotor_part_slices=2)),             # 32 parts of one move a half
    (7, 96, 48, dict(rotor_part_slices=14)),            # parts of 14 slices, the last shorter, two time slices each
    (40, 64, 64, dict(rotor_part_slices=34)),           # 17 moves: quads of energy lanes, a shorter last part
    (2, 132, 132, {}),                                  # 66 moves: two chain waves, one energy lane a move
    (2, 256, 256, {}),                                  # 128 moves: both chain waves full
    (1, 320, 320, dict(rotor_part_slices=320, rotor_lds_kb=78)),  # beyond 256 slices: chain lanes in turn
    (1, 640, 640, dict(rotor_part_slices=320, rotor_lds_kb=78)),  # the same with a neighbour
])
def test_parts_follow_the_oracle(n_he, P, Prot, options):
    got, ref, acc = run_both(n_he, P, Prot, 0.7, options, npass=1 if P > 256 else 2)
    assert np.array_equal(*acc), acc
    assert np.abs(got[0] - ref[0]).max() < 1e-9
    assert np.abs(got[2] - ref[2]).max() < 1e-9


@pytest.mark.parametrize("npt", [40, 2001])
def test_links_outside_the_staged_knots(npt):
    """A path that crosses itself: links of up to half a turn, far below the knots near
    cos(gamma) = 1 that a part keeps on chip, and a table of fewer knots than it could keep."""
    def folded(rp):
        a = rp["angles"].reshape(3, -1, rp["P"]).copy()
        k = np.arange(rp["P"])
        a[1, -1] = np.where(k % 3 == 0, -0.6, np.where(k % 3 == 1, 0.9, 0.1))
        a[0, -1] = 1.3 * k
        return a.reshape(3, -1)

    T, P = 0.3, 16  # long times: a density that reaches all angles (a 40-knot spline stays positive)
    got, ref, acc = run_both(4, P, P, T, {}, angles=folded, tables=pc.rot_table(T, P, npt=npt))
    assert np.array_equal(*acc), acc
    assert np.abs(got[2] - ref[2]).max() < 1e-9
