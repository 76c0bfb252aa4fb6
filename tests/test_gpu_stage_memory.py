"""Memory of the batched contraction stage: a reduced phase that cannot use its
buffers holds none."""

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


def test_reduced_phase_holds_no_buffers():
    o, v, order = 30, 30, 4
    print("case: reduced phase", flush=True)
    _, stage, _ = footprint(o, v, order)
    over = dict(precision="bf16x3", refine_below=0.0)
    _, reduced, _ = footprint(o, v, order, min_reduced_flops=1e5, **over)
    _, every, _ = footprint(o, v, order, min_reduced_flops=1e18, **over)   # every product in FP64 arithmetic
    assert stage > 50 << 20 and every == stage
    assert reduced < 8 << 20
