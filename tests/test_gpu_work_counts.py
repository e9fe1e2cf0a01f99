"""Pair evaluations as pimc_family_evals counts them: the terms that a bisection move's tests needed
(MCBisectionMove stops at the level it rejects, mc_piqmc.cc:246-275), however many were formed."""
import numpy as np
import pytest

import pimc_configs as pc
import pimc_hip as ph
from golden import tables3d
from test_gpu_nonlinear import nl_workload

pytestmark = pytest.mark.gpu
SEED = 985456376


def flat():
    r = np.linspace(1.0, 30.0, 500)
    return r, np.zeros(500) + 1e-300


def stiff():
    """Every displacement from a distance of 3 raises the energy by far more than kT."""
    r = np.linspace(1.0, 30.0, 500)
    return r, 1e9 * (r - 3.0) ** 2 + 1.0


@pytest.mark.parametrize("lanes", [32, 64, 128, 256])
@pytest.mark.parametrize("levels", [1, 2, 3, 5])
@pytest.mark.parametrize("table,accepts", [(flat, True), (stiff, False)])
def test_bisection_counts_the_levels_it_tested(table, accepts, levels, lanes):
    P, n = 64, 3
    ctx = ph.Context(1, seed=SEED)
    ctx.set_option("bisect_lanes_small", lanes)
    t = ctx.add_pot1d(*table())
    ctx.set_replica(0, 1, [n], [0], [levels], [0.3], [pc.MASS_HE4], P, 0, 1.0, 0.0, pot1d=[t], pot2d=[-1])
    ctx.commit()
    corners = 3.0 / np.sqrt(2.0) * np.array([[0, 0, 0], [1, 1, 0], [1, 0, 1]])  # all distances 3
    ctx.set_state(0, np.repeat(corners.T[:, :, None], P, 2).reshape(3, -1))
    ctx.run(2)
    total, accepted = ctx.counters(0)
    assert accepted[0][1] == (total[0][1] if accepts else 0)
    assert ctx.family_evals("bisect") == total[0][1] * 2 * (n - 1) * ((1 << levels) - 1 if accepts else 1)
    ctx.close()


@pytest.mark.parametrize("levels", [2, 3, 4])
def test_bisection_beside_a_rotor_counts_the_levels_it_tested(levels):
    """Para-H2 held by the stiff table around a non-linear rotor, whose own moves have one level."""
    P, n = 32, 3
    wl = nl_workload("h2o_h2", tables3d.rot3d(), n_h2=n, P=P, Prot=P)
    rp = wl["replicas"][0]
    rp["levels"], wl["tables"]["pot1d"] = [levels, 1], [stiff()]
    corners = 3.0 / np.sqrt(2.0) * np.array([[0, 0, 0], [1, 1, 0], [1, 0, 1]]) + np.array([4.0, 0.0, 0.0])
    rp["coords"][:, :n * P] = np.repeat(corners.T[:, :, None], P, 2).reshape(3, -1)
    ctx = pc.load_into_context(ph.Context(1, seed=SEED), wl)
    ctx.run(2)
    total, accepted = ctx.counters(0)
    assert accepted[0][1] == 0
    assert ctx.family_evals("bisect") == 2 * n * (total[0][1] + total[1][1])
    ctx.close()


def test_two_rotors_count_one_pair_term_a_move():
    """Short parts form the pair's energy for every outcome of the first rotor's move ahead of it."""
    P = 16
    ctx = pc.load_into_context(ph.Context(1, seed=SEED), nl_workload("water2", tables3d.rot3d(), P=P, Prot=P))
    ctx.run(1)
    launches = 4  # start slices
    assert ctx.family_evals("rotor") == 2 * P * P + launches * P
    ctx.close()
