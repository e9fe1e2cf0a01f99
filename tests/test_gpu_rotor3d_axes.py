"""The stored axes of non-linear rotors are the same bits in every form of the sweep: a chain split
into short parts, in parts beyond 256 rotor slices (on chip and in memory), whole in one workgroup, and
with delayed acceptance.  FP64 pair terms: the same decisions, so the same angles."""
import numpy as np
import pytest

import pimc_configs as pc
import pimc_hip as ph
import test_gpu_da_chain as da
from golden import tables3d
from test_gpu_nonlinear import SEED, nl_workload

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rot3d():
    return tables3d.rot3d()


def same(states):
    first = states[0]
    for s in states[1:]:
        assert np.array_equal(s[1], first[1])  # angles
        assert np.array_equal(s[2], first[2])  # axes


@pytest.mark.parametrize("kind,P,copies", [
    ("water2", 512, (1, 200, 600)),  # parts of at most 128 slices; 256, on chip; whole chains
    ("water2", 1200, (1, 140)),      # the last 600 slices, in memory
    ("h2o_h2", 640, (1, 200)),
    ("water2", 24, (1, 2)),          # one part
])
def test_every_form_stores_the_same_axes(rot3d, kind, P, copies):
    wl = nl_workload(kind, rot3d, n_h2=3, P=P, Prot=P, seed=11)
    out = []
    for n in copies:
        ctx = pc.load_into_context(ph.Context(n, flags=ph.FLAG_FP64, seed=SEED),
                                   dict(tables=wl["tables"], replicas=wl["replicas"] * n))
        ctx.run(1)
        out.append(ctx.get_state(0))
        ctx.close()
    same(out)


@pytest.mark.parametrize("n_h2,nrot,P", [(9, 1, 320), (3, 2, 160), (0, 2, 192)])
def test_delayed_acceptance_stores_the_same_axes(rot3d, n_h2, nrot, P):
    wl, net = da.deck(rot3d, n_h2, nrot, P), da.network(n_h2)
    out = []
    for n in (2, 300):
        ctx = da.context(wl, n, net)
        ctx.run(1)
        out.append(ctx.get_state(0))
        ctx.close()
    same(out)
