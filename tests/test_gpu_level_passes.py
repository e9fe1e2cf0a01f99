"""Stretched 1D tables under many atoms: on 256 lanes a segment the bisection tests its first three levels
one by one, on fewer lanes in one pass.  Proposals depend on draws and end points alone and the terms are
the same, only added in another order, so the chains, their counters and the midpoints that the tests
needed are the same.  A sum of 10^2 FP64 terms of size 10^2 K rounds by about 10^-12 K, so that one of
the 10^4 to 10^5 tests here meets a draw closer than that about once in 10^7 runs."""
import numpy as np
import pytest

import pimc_configs as pc
import pimc_hip as ph
from test_gpu_mixed_tables import stretched_tables

pytestmark = pytest.mark.gpu
SEED = 985456376


def run(n_he, P, levels, lanes, flags, rotor):
    wl = pc.workload("tiny")
    t1, t2 = stretched_tables()
    wl["tables"].update(rot=[pc.rot_table(0.8, P)], pot1d=[t1], pot2d=[t2])
    rep = dict(pc.replica(n_he, P, 0.8, SEED), rotdens=0, pot1d=[0, -1], pot2d=[-1, 0], levels=[levels, levels])
    if not rotor:  # atoms alone
        n = n_he * P
        rep.update(ntypes=1, type_names=rep["type_names"][:1], Prot=0, coords=np.ascontiguousarray(rep["coords"][:, :n]),
                   angles=np.ascontiguousarray(rep["angles"][:, :n]),
                   **{k: rep[k][:1] for k in ("numb", "molecule", "levels", "mcstep", "mass", "pot1d", "pot2d")})
    wl["replicas"] = [rep]
    ctx = ph.Context(1, seed=SEED, flags=flags)
    ctx.set_option("bisect_lanes_medium", lanes)
    ctx.set_option("bisect_lanes_large", lanes)
    pc.load_into_context(ctx, wl)
    ctx.run(5)
    out = (*ctx.get_state(0), *ctx.counters(0), ctx.family_evals("bisect"))
    ctx.close()
    return out


@pytest.mark.parametrize("flags", [0, ph.FLAG_FP64])
@pytest.mark.parametrize("n_he,P,levels,rotor", [
    (97, 32, 3, True), (98, 32, 3, True), (99, 32, 3, False), (130, 32, 2, True), (130, 32, 1, True),
    (64, 32, 4, True), (65, 32, 4, True), (66, 32, 4, False), (70, 64, 5, True), (100, 64, 4, True)])
def test_passes_per_level_make_the_same_chain(n_he, P, levels, rotor, flags):
    a, b = (run(n_he, P, levels, lanes, flags, rotor) for lanes in (256, 64))
    assert 0 < a[4][0][1] < a[3][0][1]
    for x, y in zip(a, b):
        assert np.array_equal(x, y)
