"""The device DIIS over several tensors per call: more tensors and history
slots than one launch holds, sizes around the block size, and the same tensor
given as x and as dx (its extrapolation must come from the stored copies, as
if x were a tensor of its own), against the oracle."""

import numpy as np
import pytest

import aquarius_amd as aq
from oracle import rhfccsd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order,nx,ndx,shared", [(2, 1, 5, False), (9, 6, 3, False), (17, 2, 2, False), (4, 2, 2, True)])
def test_many_tensors_equal_oracle(order, nx, ndx, shared):
    rng = np.random.default_rng(100 * order + nx)
    sizes = [1, 255, 257, 1024, 4097, 33]
    ref = rhfccsd.DIIS({"order": order, "start": 1, "damping": 0.0}, nx, ndx)
    with aq.Context(0) as ctx:
        d = aq.DIIS(ctx, order, 1, 0.0, nx, ndx)
        for it in range(order + 2):
            dx = [rng.standard_normal(sizes[j]) * 0.7 ** it for j in range(ndx)]
            x = [a.copy() for a in dx] if shared else [rng.standard_normal(sizes[j]) for j in range(nx)]
            tdx = [ctx.from_numpy(a) for a in dx]
            tx = tdx if shared else [ctx.from_numpy(a) for a in x]
            d.extrapolate(tx, tdx)
            ref.extrapolate(x, dx)
            for t, a in list(zip(tx, x)) + list(zip(tdx, dx)):
                np.testing.assert_allclose(t.numpy(), a, rtol=1e-9, atol=1e-11 * np.abs(a).max(), err_msg=f"it {it}")
            for t in tdx + ([] if shared else tx):
                t.free()
        d.close()
