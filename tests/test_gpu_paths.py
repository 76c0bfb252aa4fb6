"""The kernels that a call is meant for are the ones that run (read from the timing
classes): aliased sums under a permutation that is its own inverse, and the batched
stage up to the sizes where it is used, in both arithmetics."""

import numpy as np
import pytest

import aquarius_amd as aq

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("src,dst,in_place", [
    ("baji", "abij", True), ("abji", "abij", True), ("abij", "abij", False), ("jbai", "abij", False), ("ijab", "abij", True)])
def test_aliased_sums_in_place(src, dst, in_place):
    print(f"case: sum {src} -> {dst}", flush=True)
    n = 9
    x = np.random.default_rng(1).standard_normal((n,) * 4)
    with aq.Context() as ctx:
        t = ctx.from_numpy(x)
        ctx.enable_timing(True)
        ctx.sum(-0.5, t, src, 2.0, t, dst)
        ran = ctx.timing()
        want = 2.0 * x - 0.5 * np.einsum(f"{src}->{dst}", x)
        np.testing.assert_allclose(t.numpy(), want, rtol=0, atol=4 * 2.0 ** -53 * 2.5 * abs(x).max())
    assert ("sum_pairs" in ran) == in_place, sorted(ran)


@pytest.mark.parametrize("o,v,precision,batched", [
    (19, 98, "fp64", True), (20, 94, "fp64", False), (10, 109, "bf16x3", True), (10, 110, "bf16x3", False)])
def test_batched_stage_up_to_its_limit(o, v, precision, batched):
    print(f"case: stage o={o} v={v} {precision}", flush=True)
    with aq.Context() as ctx:
        ints = aq.Integrals.synthetic(ctx, 5, o, v)
        cc = aq.RHFCCSD(ctx, ints, precision=precision, min_reduced_flops=1e18)
        ctx.enable_timing(True)
        cc.iterate()
        assert ("stage_contract" in ctx.timing()) == batched
        cc.close()
        ints.free()
