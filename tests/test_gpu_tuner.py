"""The GEMM tuner tries the variants that need no large scratch memory: the four-wave
256 x 256 tile of the BF16x3 arithmetic is left out, and runs when it is asked for."""

import numpy as np
import pytest

import aquarius_amd as aq

pytestmark = pytest.mark.gpu


def test_spilling_variant_is_not_tried():
    n, k = 2100, 256
    print(f"case: tuner at {n} x {n} x {k}", flush=True)
    rng = np.random.default_rng(3)
    a, b = rng.standard_normal((n, k)), rng.standard_normal((k, n))
    with aq.Context() as ctx:
        ctx.set_precision("bf16x3", 0.0)
        ta, tb = ctx.from_numpy(a), ctx.from_numpy(b)
        out = []
        for tune, variant in ((True, -1), (False, 4)):
            ctx.set_autotune(tune)
            ctx.set_gemm_variant("bf16x3", variant)
            tc = ctx.tensor((n, n))
            ctx.contract(1.0, ta, "mk", tb, "kn", 0.0, tc, "mn")
            out.append(tc.numpy())
    np.testing.assert_array_equal(out[0], out[1])
    tried = [e for e in aq.autotune_table() if e["precision"] == aq.PRECISIONS["bf16x3"]]
    assert tried and all(e["ms"][4] < 0 and e["variant"] != 4 for e in tried)
    assert any(e["ms"][0] >= 0 and e["ms"][3] >= 0 for e in tried)
