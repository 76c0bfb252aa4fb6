"""Which kernels a contraction takes at both sides of the lines between the direct
kernels and the GEMM, and of those between the direct tile shapes (read from the
timing classes), and its values there against numpy: sums of K rounded products in
any order, (K + 8) 2^-53 sum |a||b|."""

import numpy as np
import pytest

import aquarius_amd as aq

pytestmark = pytest.mark.gpu

CASES = [
    # the batch index contiguous in the operands, and outermost
    ("bmk,bkn,bmn", dict(b=40, m=30, k=50, n=3), "gemm_f64"),
    ("bmk,bkn,bmn", dict(b=300, m=8, k=20, n=8), "direct_f64"),
    ("mkb,knb,mnb", dict(b=40, m=30, k=50, n=3), "direct_f64"),
    ("mkb,knb,mnb", dict(b=70, m=100, k=16, n=4), "gemm_f64"),
    ("mkb,knb,mnb", dict(b=70, m=100, k=17, n=4), "direct_f64"),
    ("mkb,knb,mnb", dict(b=700, m=5, k=3, n=7), "direct_f64_16x16"),
    # matrices as they lie: few columns, short sums, both contiguous along k
    ("mk,kn,mn", dict(m=16000, k=40, n=12), "direct_f64"),
    ("mk,kn,mn", dict(m=16700, k=40, n=12), "gemm_f64"),
    ("mk,kn,mn", dict(m=16000, k=64, n=34), "direct_f64"),
    ("mk,kn,mn", dict(m=16400, k=64, n=34), "gemm_f64"),
    ("mk,kn,mn", dict(m=16400, k=65, n=34), "direct_f64"),
    ("km,kn,mn", dict(m=16400, k=65, n=34), "gemm_f64"),
    ("mk,kn,mn", dict(m=1500, k=33, n=1500), "direct_f64"),
    ("mk,kn,mn", dict(m=1501, k=33, n=1499), "gemm_f64"),
    # shapes: a ring whose 64 x 64 tiles need a split, a long operand with few columns
    ("amie,ebmj,abij", dict(a=74, b=74, e=74, i=15, j=15, m=15), "direct_f64_64x64"),
    ("abej,ei,abij", dict(a=60, b=60, e=60, i=14, j=14), "direct_f64_256x16"),
]


@pytest.mark.parametrize("form,dim,want", CASES)
def test_route(form, dim, want):
    print(f"case: route {form} {dim}", flush=True)
    ia, ib, ic = form.split(",")
    rng = np.random.default_rng(sum(dim.values()))
    A, B = (rng.standard_normal([dim[c] for c in lab]) for lab in (ia, ib))
    spec = f"{ia},{ib}->{ic}"
    ref, mag = np.einsum(spec, A, B, optimize=True), np.einsum(spec, abs(A), abs(B), optimize=True)
    with aq.Context() as ctx:
        tA, tB, tC = ctx.from_numpy(A), ctx.from_numpy(B), ctx.tensor([dim[c] for c in ic])
        ctx.enable_timing(True)
        ctx.contract(1.0, tA, ia, tB, ib, 0.0, tC, ic)
        ran = [k for k in ctx.timing() if k.startswith(("gemm", "direct_f64"))]
        assert len(ran) == 1 and ran[0].startswith(want), ran
        K = int(np.prod([dim[c] for c in set(ia) & set(ib) - set(ic)]))
        assert (abs(tC.numpy() - ref) <= (K + 8) * 2.0 ** -53 * mag).all()
