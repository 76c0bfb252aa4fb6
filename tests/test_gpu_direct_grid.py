"""Products over one long batch label, a block for each of its values: up to the
largest grid of 256-thread blocks (fewer than 2^32 threads) they run; beyond it
they are refused as any batch too large for the GEMM kernels is, not by a failing
launch."""

import numpy as np
import pytest

import aquarius_amd as aq

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [65535, 65536, (1 << 24) - 1, 1 << 24])
def test_scaled_columns(n):
    print(f"case: {n} columns", flush=True)
    rng = np.random.default_rng(n)
    a, b = np.asfortranarray(rng.standard_normal((2, n))), rng.standard_normal(n)
    with aq.Context() as ctx:
        ta, tb, tc = ctx.from_numpy(a), ctx.from_numpy(b), ctx.tensor((2, n))
        if n < 1 << 24:
            ctx.contract(2.0, ta, "mi", tb, "i", 0.0, tc, "mi")
            np.testing.assert_array_equal(tc.numpy(), 2.0 * (a * b))   # one rounding each
        else:
            with pytest.raises(aq.AqError, match="batch too large"):
                ctx.contract(2.0, ta, "mi", tb, "i", 0.0, tc, "mi")
