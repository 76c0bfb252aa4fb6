"""FP64 contractions on operands in any label order: random label groups,
orders and lengths (units and odd lengths among them, merged and unmerged
digits, k contiguous in neither, one or both operands, a batch label), and
sizes around the kernels' edges: tiles of 16, 32, 64 and 256, chunks of 16 k,
tables of 1024 k, split inner extents.  Reference: numpy einsum.  Each element
is within the bound of a sum of K rounded products in any order,
(K + 8) 2^-53 (|alpha| sum |a||b| + |beta c|)."""

import numpy as np
import pytest

import aquarius_amd as aq

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    with aq.Context(0) as c:
        yield c


def check(ctx, ia, ib, ic, dim, alpha, beta, seed):
    rng = np.random.default_rng(seed)
    A = rng.standard_normal([dim[c] for c in ia])
    B = rng.standard_normal([dim[c] for c in ib])
    Cm = rng.standard_normal([dim[c] for c in ic]) if beta else np.full([dim[c] for c in ic], np.nan)
    spec = f"{ia},{ib}->{ic}"
    ref = alpha * np.einsum(spec, A, B, optimize=True)
    mag = abs(alpha) * np.einsum(spec, abs(A), abs(B), optimize=True)
    if beta:
        ref, mag = ref + beta * Cm, mag + abs(beta * Cm)
    K = int(np.prod([dim[c] for c in set(ia) & set(ib) - set(ic)] or [1]))
    tA, tB, tC = ctx.from_numpy(A), ctx.from_numpy(B), ctx.from_numpy(Cm)
    ctx.contract(alpha, tA, ia, tB, ib, beta, tC, ic)
    got = tC.numpy()
    for t in (tA, tB, tC):
        t.free()
    bad = ~(abs(got - ref) <= (K + 8) * 2.0 ** -53 * mag)
    assert not bad.any(), (spec, dim, alpha, beta, int(bad.sum()), np.argwhere(bad)[:3])


@pytest.mark.parametrize("seed", range(48))
def test_random_forms(ctx, seed):
    rng = np.random.default_rng(1000 + seed)
    names = list("abcdefghijkl")
    take = lambda n: [names.pop(0) for _ in range(n)]
    M, N, K, Bt = (take(int(rng.integers(lo, hi))) for lo, hi in ((0, 4), (0, 4), (0, 4), (0, 2)))
    dim = {c: int(rng.choice([1, 2, 3, 4, 5, 7, 8, 12, 16, 17])) for c in M + N + K + Bt}
    mix = lambda labs: "".join(rng.permutation(labs)) if labs else ""
    print(f"case: random form {seed}", flush=True)
    check(ctx, mix(M + K + Bt), mix(K + N + Bt), mix(M + N + Bt), dim, float(rng.choice([1.0, -0.5, 2.0])),
          float(rng.choice([0.0, 1.0, -0.25])), seed)


EDGES = [(1, 1, 1), (16, 16, 16), (17, 15, 15), (31, 33, 17), (64, 64, 64), (65, 63, 1), (257, 5, 19), (5, 257, 33),
         (33, 33, 1023), (20, 20, 1024), (3, 18, 1025), (13, 13, 40000), (75, 13, 9001), (300, 17, 3000), (400, 400, 48)]


@pytest.mark.parametrize("form", ["mk,kn,mn", "km,kn,mn", "mk,nk,mn", "km,nk,nm", "mk,kn,nm"])
@pytest.mark.parametrize("size", EDGES)
def test_edges(ctx, form, size):
    print(f"case: edges {form} {size}", flush=True)
    check(ctx, *form.split(","), dict(zip("mnk", size)), 0.5, 1.0, sum(size))


def test_infinities_stay_in_their_rows(ctx):
    """An inner extent that is no multiple of the chunk: elements past it are
    zeroed in both operands, so an infinity in the last k gives infinities (not
    NaN) in its own row and column only."""
    m, n, k = 37, 21, 19
    A, B = np.ones((m, k)), np.ones((k, n))
    A[3, k - 1], B[k - 1, 5] = np.inf, -np.inf
    tA, tB, tC = ctx.from_numpy(A), ctx.from_numpy(B), ctx.tensor((m, n))
    ctx.contract(1.0, tA, "mk", tB, "kn", 0.0, tC, "mn")
    got = tC.numpy()
    with np.errstate(invalid="ignore"):
        ref = A @ B
    np.testing.assert_array_equal(got, ref)
    for t in (tA, tB, tC):
        t.free()
