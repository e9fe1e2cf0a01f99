"""What queries and getters return: a batch of queries at the edges of its blocks, the getters as the host's copy of counters and samples goes out of date, grows past its
room, and as a replica's state outgrows the packed read-back."""
import numpy as np
import pytest

import pimc_configs as pc
import pimc_hip as ph
import pimc_tables as pt

pytestmark = pytest.mark.gpu


def box(replicas, atoms, P, seed=5):
    ctx = ph.Context(replicas, seed=seed)
    ctx.add_pot1d(*pt.lj_table())
    for r in range(replicas):
        ctx.set_replica(r, 1, [atoms], [0], [2], [0.3], [pc.MASS_HE4], P, 0, 1.5, 0.0, pot1d=[0], pot2d=[-1])
    ctx.commit()
    rng = np.random.default_rng(seed)
    m = int(np.ceil(atoms ** (1.0 / 3.0)))
    sites = 3.6 * np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)[:atoms]
    states = []
    for r in range(replicas):
        c = np.repeat(sites.T[:, :, None], P, 2).reshape(3, -1) + rng.normal(0, 0.1, (3, atoms * P))
        ctx.set_state(r, c)
        states.append(c)
    return ctx, states


@pytest.mark.parametrize("taken", [1, 16, 17])
def test_samples_up_to_and_past_the_read_back(taken):
    """256 replicas keep 16 samples each in the read-back; one more is read from the device."""
    ctx, _ = box(256, 2, 8)
    ctx.run(taken, 1)
    first = [ctx.samples(r, 64) for r in (0, 255)]
    assert all(s.shape == (taken, 8) for s in first)
    t0 = ctx.counters(255)[0].sum()
    ctx.run(1, 1)  # the copies are of the run before
    second = [ctx.samples(r, 64) for r in (0, 255)]
    assert all(s.shape == (taken + 1, 8) and np.array_equal(s[:taken], f) for s, f in zip(second, first))
    assert ctx.counters(255)[0].sum() > t0 and ctx.pass_counter(255) == taken + 1
    ctx.clear_samples()
    assert ctx.samples(0, 64).shape == (0, 8)
    c, a, cs = ctx.get_state(255)
    ctx.restore_state(255, c, a, cs, 40)
    assert ctx.pass_counter(255) == 40 and ctx.pass_counter(0) == taken + 1
    ctx.close()


@pytest.mark.parametrize("atoms,P", [(3, 8), (64, 2728), (64, 2736)])
def test_state_round_trip(atoms, P):
    """64 * 2730.67 beads fill the packed read-back's 4 MB."""
    ctx, states = box(1, atoms, P)
    c, a, cs = ctx.get_state(0)
    assert np.array_equal(c, states[0])
    n = atoms * P
    assert np.array_equal(a, np.repeat([[0.0], [1.0], [0.0]], n, 1)) and np.array_equal(cs, np.repeat([[0.0], [0.0], [1.0]], n, 1))
    ctx.close()


@pytest.mark.parametrize("nq", [1, 31, 32, 33, 1000])
def test_a_batch_of_queries_is_its_queries(nq):
    """Whatever shares a query's block; the energies themselves are checked against the oracle with the
    estimators.  One query's sum runs over the same lanes in any batch, so it is the same bits."""
    ctx, states = box(3, 11, 16)
    rng = np.random.default_rng(nq)
    rep, atom, it = rng.integers(0, 3, nq), rng.integers(0, 11, nq), rng.integers(0, 16, nq)
    pos = np.array([states[r][:, a * 16 + i] for r, a, i in zip(rep, atom, it)]) + rng.normal(0, 0.1, (nq, 3))
    rep, atom, it = (x.astype(np.int32) for x in (rep, atom, it))
    got = ctx.pot_energy_slice(rep, atom, it, pos)
    for q in {0, nq // 2, nq - 1}:
        one = ctx.pot_energy_slice(rep[q:q + 1], atom[q:q + 1], it[q:q + 1], pos[q:q + 1])
        assert one[0] == got[q] and np.isfinite(got[q]) and got[q] != 0.0
    ctx.close()
