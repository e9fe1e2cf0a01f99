"""The non-linear rotor sweep in every form a chain's part can take: one part that is its own
neighbour, parts of unequal length, state in LDS with a lane per move, state in memory; enough copies
of the chain fill the device that the split leaves parts that long."""
import numpy as np
import pytest

import oracle as O
import pimc_configs as pc
import pimc_hip as ph
from golden import tables3d
from test_gpu_nonlinear import SEED, nl_workload, rotor_columns

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rot3d():
    return tables3d.rot3d()


@pytest.mark.parametrize("kind,P,ratio,copies", [
    ("water2", 24, 1, 1),     # one part
    ("h2o_h2", 16, 2, 1),     # one part of eight slices
    ("h2o_h2", 92, 2, 1),     # parts of 24 and 22 slices
    ("water2", 512, 1, 200),  # 256 slices of two rotors: a lane per move, in LDS
    ("h2o_h2", 640, 1, 200),  # 320 slices of one rotor among atoms
    ("water2", 1200, 1, 140),  # 600 slices of two rotors: state in memory
])
def test_trajectory_follows_the_oracle(rot3d, kind, P, ratio, copies):
    """FP64 pair terms: one pass, every decision the oracle's and the state within 1e-9 of it (the
    bound of the other trajectory tests: rounding of single operations over a pass)."""
    wl = nl_workload(kind, rot3d, n_h2=3, P=P, Prot=P // ratio, seed=11)
    rp = wl["replicas"][0]
    wl["replicas"] = [rp] * copies
    ctx = pc.load_into_context(ph.Context(copies, flags=ph.FLAG_FP64, seed=SEED), wl)
    ctx.run(1)
    t = wl["tables"]
    tabs = dict(pot1d=t["pot1d"], pot2d=[], rot=[], pot3d=t["pot3d_list"][0] if t["pot3d_list"] else None,
                rot3d=t["rot3d_list"][0])
    for r in {0, copies - 1}:
        S = O.System(rp, tabs, seed=SEED, replica=r)
        S.run(0, 1, order=O.ORDER_SEGMENTS)
        cg, ag, _ = ctx.get_state(r)
        co, ao, _ = S.state()
        tg, acg = ctx.counters(r)
        to, aco = S.counters()
        assert np.array_equal(tg, to) and np.array_equal(acg, aco), (r, acg, aco)
        assert np.abs(cg - co).max() < 1e-9
        rot = np.arange(sum(rp["numb"]) * P)[rotor_columns(rp)].reshape(-1, P)
        cols = rot[:, :rp["Prot"]].reshape(-1)  # the slices that rotate
        assert np.abs(ag[:, cols] - ao[:, cols]).max() < 1e-9
    ctx.close()
