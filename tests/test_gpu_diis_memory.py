"""A DIIS history slot that does not fit the budget: the call fails, leaves no slot
half filled, and the extrapolation goes on, from the later calls, once there is room;
in between the tensors are the caller's own."""

import numpy as np
import pytest

import aquarius_amd as aq
from oracle import rhfccsd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fits", [0, 1, 2, 3])   # tensors of the slot (x0, x1, dx0, dx1) that do
def test_half_a_slot(fits):
    print(f"case: {fits} of 4 tensors fit", flush=True)
    order, n, mib = 3, 1 << 17, 1 << 20
    rng = np.random.default_rng(fits)
    new = lambda: [rng.standard_normal(n) for _ in range(2)]
    with aq.Context(hbm_budget=64 * mib) as ctx:
        d = aq.DIIS(ctx, order, 1, 0.0, 2, 2)
        x, dx = new(), new()
        tx, tdx = ([ctx.from_numpy(a) for a in v] for v in (x, dx))
        in_use, budget = ctx.memory()
        fill = ctx.tensor(((budget - in_use - fits * mib) // 8 // (mib // 8) * (mib // 8),), zero=False)
        with pytest.raises(aq.AqError):
            d.extrapolate(tx, tdx)
        for t, a in zip(tx + tdx, x + dx):
            np.testing.assert_array_equal(t.numpy(), a)
        fill.free()
        ref = rhfccsd.DIIS({"order": order, "start": 1, "damping": 0.0}, 2, 2)
        for it in range(order + 2):
            x, dx = new(), new()
            for t, a in zip(tx + tdx, x + dx):
                t.write_all(a)
            d.extrapolate(tx, tdx)
            ref.extrapolate(x, dx)
            for t, a in zip(tx + tdx, x + dx):
                np.testing.assert_allclose(t.numpy(), a, rtol=1e-9, atol=1e-11 * np.abs(a).max(), err_msg=f"it {it}")
        d.close()
