"""Launch shapes of a tuned context: the plan's own are candidates, what is reported is what runs, and
it can be asked for again."""
import numpy as np
import pytest

import pimc_configs as pc
import pimc_hip as ph
from golden import tables3d
from test_gpu_nonlinear import nl_workload

pytestmark = pytest.mark.gpu
SEED = 985456376


def chains(n_he, P, copies, **options):
    wl = pc.workload("tiny")
    wl["tables"]["rot"] = [pc.rot_table(0.8, P)]
    wl["replicas"] = [dict(pc.replica(n_he, P, 0.8, SEED), rotdens=0, pot1d=[0, -1], pot2d=[-1, 0])] * copies
    ctx = ph.Context(copies, seed=SEED)
    for k, v in options.items():
        ctx.set_option(k, v)
    return pc.load_into_context(ctx, wl)


def test_lanes_where_two_segments_share_a_wave():
    """4096 segments of 9 atoms: the plan's 32 lanes are timed like the others, and the tuned shapes
    given as options make the same chains."""
    tuned, plain = chains(8, 64, 512), chains(8, 64, 512)
    shapes = tuned.autotune(passes=2)
    assert shapes["bisect_lanes_small"] in ph.plan_bisect_lanes(9, 4096) and 32 in ph.plan_bisect_lanes(9, 4096)
    asked = chains(8, 64, 512, **{k: v for k, v in shapes.items()})
    small = chains(8, 64, 512, bisect_lanes_small=32)
    for c in (tuned, plain, asked, small):
        c.run(2)
    for r in (0, 511):
        for c in (tuned, asked, small):
            assert np.array_equal(c.counters(r)[1], plain.counters(r)[1])
            assert all(np.array_equal(a, b) for a, b in zip(c.get_state(r), plain.get_state(r)))


def test_other_classes_keep_whole_waves():
    ctx = ph.Context(1, seed=SEED)
    for k in ("bisect_lanes_medium", "bisect_lanes_large"):
        with pytest.raises(ph.PimcError, match="64, 128 or 256"):
            ctx.set_option(k, 32)
    ctx.close()


def test_proposals_follow_the_tuned_parts():
    """Chains committed with few large rotor parts leave CUs free for the next proposals; the budgets
    that the tuner times make more parts than that, and the proposals then run between the launches."""
    ctx = chains(100, 512, 16, rotor_lds_kb=150)
    cu = ctx.launch_shape("compute_units")
    assert ctx.launch_shape("rotor_blocks") <= cu // 2 and ctx.launch_shape("proposals_beside") == 1
    assert ctx.autotune(passes=1)["rotor_lds_kb"] < 150
    assert ctx.launch_shape("rotor_blocks") > cu // 2 and ctx.launch_shape("proposals_beside") == 0
    ctx.close()


@pytest.mark.parametrize("kb,state_kb", [(8, 8), (16, 8), (17, 8), (52, 43), (150, 141)])
def test_rotor_budget_of_a_part(kb, state_kb):
    """The budget holds the kernel's own 9 KB, and a part's slices get 8 KB at least."""
    ctx = chains(40, 128, 1, rotor_lds_kb=kb)
    want = ph.plan_rotor_parts([128], [1], [41], lds_kb=state_kb)[2]
    assert ctx.launch_shape("rotor_lds_bytes") == want
    ctx.close()


@pytest.mark.parametrize("n_h2,copies,flags,lanes", [
    (9, 129, 0, 64), (10, 128, 0, 128), (10, 129, 0, 64), (18, 129, 0, 64), (10, 129, ph.FLAG_FP64, 128), (19, 64, 0, 256),
    (19, 65, 0, 128), (19, 65, ph.FLAG_FP64, 128), (32, 65, ph.FLAG_FP64, 256), (32, 129, ph.FLAG_FP64, 128)])
def test_lanes_of_a_segment_beside_a_non_linear_rotor(n_h2, copies, flags, lanes):
    """32 slices at four a segment: eight segments a chain, 1024 of 128 chains."""
    wl = nl_workload("h2o_h2", tables3d.rot3d(), n_h2=n_h2, P=32, Prot=32)
    ctx = ph.Context(copies, seed=SEED, flags=flags)
    pc.load_into_context(ctx, dict(tables=wl["tables"], replicas=wl["replicas"] * copies))
    assert ctx.launch_shape("bisect_lanes_non_linear") == lanes
    ctx.run(1)
    assert ctx.counters(0)[1][0][1] > 0
    ctx.close()
