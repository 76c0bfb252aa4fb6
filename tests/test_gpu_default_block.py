"""The block a BF16x3 or FP32 GEMM takes without a tuner never changes its
result: default against the 128 x 128 block, bit for bit, on both sides of the
rule (rounds of resident blocks), at ragged edges, with and without split
partials, batches and inner extents that are no multiple of the k step; and
the split sums against FP64 within the format's bound."""

import numpy as np
import pytest

import aquarius_amd as aq

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    with aq.Context(0) as c:
        yield c


@pytest.mark.parametrize("prec,tol", [("bf16x3", 5e-5), ("fp32", 2e-6)])
@pytest.mark.parametrize("m,n,k,b", [(255, 4000, 40, 1), (256, 256, 33, 1), (2945, 2817, 40, 1), (2945, 2817, 41, 1),
                                     (1300, 700, 700, 1), (300, 260, 4097, 1), (70, 50, 9000, 1), (17, 300, 600, 3),
                                     (600, 700, 96, 17)])
def test_default_equals_small_block(ctx, prec, tol, m, n, k, b):
    print(f"case: {prec} {m} {n} {k} {b}", flush=True)
    rng = np.random.default_rng(m + n + k)
    A, B = ctx.from_numpy(rng.standard_normal((m, k, b))), ctx.from_numpy(rng.standard_normal((k, n, b)))
    C0 = rng.standard_normal((m, n, b))
    outs = []
    ctx.set_precision(prec, 0.0)
    try:
        for variant in (-1, 0):
            ctx.set_gemm_variant(prec, variant)
            C = ctx.from_numpy(C0)
            ctx.contract(0.3, A, "mkb", B, "knb", -0.7, C, "mnb")
            outs.append(C.numpy())
            C.free()
    finally:
        ctx.set_precision("fp64")
        ctx.set_gemm_variant(prec, -1)
    assert np.array_equal(outs[0], outs[1])
    ref = 0.3 * np.einsum("mkb,knb->mnb", A.numpy(), B.numpy(), optimize=True) - 0.7 * C0
    assert np.linalg.norm(outs[0] - ref) <= tol * np.linalg.norm(ref)
    A.free()
    B.free()
