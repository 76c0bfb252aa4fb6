"""Sums of a tensor into itself under a permutation of its indices: in place
where the permutation is its own inverse (tiles exchanged, or whole rows),
through a snapshot otherwise.  Bit-exact against the oracle, at lengths around
the 32 x 32 tile."""

import numpy as np
import pytest

import aquarius_amd as aq
from oracle import ctf_ops as ops

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    with aq.Context(0) as c:
        yield c


@pytest.mark.parametrize("src,dst,shape", [
    ("baji", "abij", (1, 1, 4, 4)), ("baji", "abij", (33, 33, 3, 3)), ("baij", "abij", (31, 31, 2, 5)),
    ("ba", "ab", (65, 65)), ("nmji", "mnij", (7, 7, 7, 7)), ("abji", "abij", (5, 3, 6, 6)), ("acb", "abc", (32, 9, 9)),
    ("bjai", "aibj", (4, 6, 4, 6)), ("cba", "abc", (17, 2, 17)),
    ("bca", "abc", (8, 8, 8)), ("bcad", "abcd", (4, 4, 4, 3))])   # the last two are no involutions
def test_aliased_permuted_sum(ctx, src, dst, shape):
    rng = np.random.default_rng(len(src) + sum(shape))
    X = rng.standard_normal(shape)
    print(f"case: {src}->{dst} {shape}", flush=True)
    for alpha, beta in ((1.0, 1.0), (-0.5, 2.0), (0.75, 0.0)):
        ref = X.copy()
        ops.tsum(alpha, ref.copy(), src, beta, ref, dst)
        t = ctx.from_numpy(X)
        ctx.sum(alpha, t, src, beta, t, dst)
        assert np.array_equal(t.numpy(), ref), (src, dst, alpha, beta)
        t.free()
