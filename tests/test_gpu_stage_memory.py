"""Memory of the batched contraction stage: a solve takes the same path (and so
gives the same bits) whether it is served, under a budget that holds its buffers,
or alone, whatever scratch is pooled; its buffers give way to what else the
context has to hold; and a reduced phase that cannot use them holds none.

Which path ran is read from the timing classes of the kernels."""

import numpy as np
import pytest

import aquarius_amd as aq

pytestmark = pytest.mark.gpu


def history(o, v, order):
    """Bytes of a whole DIIS history, each tensor rounded up to 1 MiB."""
    return 2 * order * (8 * (o * o * v * v + o * v) + (2 << 20))


def footprint(o, v, order, **over):
    """(bytes beside integrals and solver, bytes of the stage's buffers, energies) of three
    iterations with no budget to speak of."""
    with aq.Context(hbm_budget=64 << 30) as ctx:
        ints = aq.Integrals.synthetic(ctx, 3, o, v)
        cc = aq.RHFCCSD(ctx, ints, diis_order=order, **over)
        ctx.trim()
        held = ctx.memory()[0]
        energies = [cc.iterate()[0]]
        ctx.trim()   # scratch and operand copies; the stage's buffers stay
        stage = ctx.memory()[0] - held
        slot = history(o, v, 1)
        energies += [cc.iterate()[0] for _ in range(2)]
        cc.close()
        ints.free()
    return held, stage - min(stage, slot), energies


def classes(ctx):
    return {k.split("_")[0] + "_" + k.split("_")[1] for k in ctx.timing()}


@pytest.mark.parametrize("o,v", [(13, 75), (18, 90), (30, 30)])
def test_served_takes_the_path_it_takes_alone(o, v):
    print(f"case: served o={o} v={v}", flush=True)
    cfg = lambda: aq.default_config(diis_order=8, max_iterations=6, convergence=0.0)
    with aq.Context() as ctx:
        ints = aq.Integrals.synthetic(ctx, 3, o, v)
        ctx.sync()
        cc = aq.RHFCCSD(ctx, ints, config=cfg())
        alone = cc.run()
        cc.close()
        with aq.Server(slots=2, hbm_budget=24 << 30) as s:
            for jobs in ({"inputs": ints}, {}):     # the caller's integrals, and the job's own
                r = s.wait(s.submit(3, o, v, config=cfg(), **jobs))
                assert r["status"] == aq.JOB_DONE, r["error"]
                # conv is one element of a residual: a sum in another order shows
                assert (r["energy"], r["conv"]) == (alone["energy"], alone["conv"])
        ints.free()


@pytest.mark.parametrize("pooled", [False, True])
def test_pooled_scratch_does_not_change_the_path(pooled):
    o, v, order = 8, 40, 4
    print(f"case: pooled scratch {pooled}", flush=True)
    held, stage, want = footprint(o, v, order)
    assert stage > 0
    with aq.Context(hbm_budget=held + history(o, v, order) + 3 * stage // 2) as ctx:
        ints = aq.Integrals.synthetic(ctx, 3, o, v)
        cc = aq.RHFCCSD(ctx, ints, diis_order=order)
        ctx.trim()
        if pooled:   # an aliased sum's snapshot stays in the pool
            x = ctx.tensor((stage // 4 // 24, 3))
            ctx.sum(1.0, x, "ab", 1.0, x, "ab")
            y = ctx.tensor((max(int((stage // 4 // 8) ** 0.5), 2),) * 2)
            ctx.sum(1.0, y, "aa", 0.5, y, "ab")
            x.free()
            y.free()
        ctx.enable_timing(True)
        got = [cc.iterate()[0] for _ in range(3)]
        assert "stage_contract" in classes(ctx)
        assert got == want
        cc.close()
        ints.free()


def test_buffers_give_way():
    """A tensor that fits beside the solver, but not beside the stage's buffers too: it is
    allocated, and the solve goes on along the general path."""
    o, v, order = 30, 30, 4
    print("case: buffers give way", flush=True)
    held, stage, _ = footprint(o, v, order)
    with aq.Context() as ctx:
        ints = aq.Integrals.synthetic(ctx, 3, o, v)
        cc = aq.RHFCCSD(ctx, ints, diis_order=order)
        want = [cc.iterate()[0] for _ in range(6)]
        cc.close()
        ints.free()
    with aq.Context(hbm_budget=held + history(o, v, order) + 4 * stage) as ctx:
        ints = aq.Integrals.synthetic(ctx, 3, o, v)
        cc = aq.RHFCCSD(ctx, ints, diis_order=order)
        ctx.enable_timing(True)
        got = [cc.iterate()[0] for _ in range(2)]
        assert "stage_contract" in classes(ctx)
        extra = ctx.tensor((int(3.6 * stage) // 8,), zero=False)
        ctx.timing_reset()
        got += [cc.iterate()[0] for _ in range(2)]
        assert "stage_contract" not in classes(ctx)
        cc.hbar(with_wabej=True)
        extra.free()
        got += [cc.iterate()[0] for _ in range(2)]
        np.testing.assert_allclose(got, want, rtol=1e-9, atol=0)
        cc.close()
        ints.free()


def test_reduced_phase_holds_no_buffers():
    o, v, order = 30, 30, 4
    print("case: reduced phase", flush=True)
    _, stage, _ = footprint(o, v, order)
    over = dict(precision="bf16x3", refine_below=0.0)
    _, reduced, _ = footprint(o, v, order, min_reduced_flops=1e5, **over)
    _, every, _ = footprint(o, v, order, min_reduced_flops=1e18, **over)   # every product in FP64 arithmetic
    assert stage > 50 << 20 and every == stage
    assert reduced < 8 << 20
