"""FP64 contractions large enough for the tiles staged through LDS (64 x 64 and
128 x 128) and for the 256 x 32 tiles of a few columns, straight from labelled layouts: each operand contiguous along its
rows or along k, digits that do not merge, partial tiles, partial chunks of 16
k, several tables of 512 k, split inner extents, a batch label.  Reference:
numpy.  Each element is within the bound of a sum of K rounded products in any
order, (K + 8) 2^-53 (|alpha| sum |a||b| + |beta c|)."""

import numpy as np
import pytest

import aquarius_amd as aq

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    with aq.Context(0) as c:
        yield c


def check(ctx, form, dim, alpha, beta):
    ia, ib, ic = form.split(",")
    rng = np.random.default_rng(sum(map(ord, form)) + sum(dim.values()))
    A = rng.standard_normal([dim[c] for c in ia])
    B = rng.standard_normal([dim[c] for c in ib])
    C = rng.standard_normal([dim[c] for c in ic])
    spec = f"{ia},{ib}->{ic}"
    ref = alpha * np.einsum(spec, A, B, optimize=True) + beta * C
    mag = abs(alpha) * np.einsum(spec, abs(A), abs(B), optimize=True) + abs(beta * C)
    K = int(np.prod([dim[c] for c in set(ia) & set(ib) - set(ic)]))
    tA, tB, tC = ctx.from_numpy(A), ctx.from_numpy(B), ctx.from_numpy(C)
    ctx.contract(alpha, tA, ia, tB, ib, beta, tC, ic)
    got = tC.numpy()
    for t in (tA, tB, tC):
        t.free()
    bad = ~(abs(got - ref) <= (K + 8) * 2.0 ** -53 * mag)
    assert not bad.any(), (form, dim, int(bad.sum()), np.argwhere(bad)[:3])


# unit stride (the first label): rows and rows, rows and k, k and rows
FORMS = ["efmn,afin,amie", "amie,ebmj,abij", "eabm,afim,befi", "emai,bmej,abij", "amie,mebj,jbia"]


@pytest.mark.parametrize("beta", [0.0, 1.0])
@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("o,v", [(3, 70), (7, 93), (12, 121), (20, 140), (19, 149)])
def test_rings(ctx, form, o, v, beta):
    if form == FORMS[2]:
        v = min(v, 60)   # three virtual labels in one operand
    print(f"case: staged {form} o={o} v={v} beta={beta}", flush=True)
    check(ctx, form, {c: v if c < "i" else o for c in form if c != ","}, 0.5, beta)


@pytest.mark.parametrize("M,N,K", [(65, 129, 513), (200, 210, 1023), (640, 96, 2048), (90, 80, 20011), (1021, 515, 517)])
@pytest.mark.parametrize("form", ["xmk,nyk,xnmy", "kxm,kny,nmyx", "xmkz,nyzk,xnmy"])
def test_around_the_edges(ctx, form, M, N, K):
    print(f"case: staged edges {form} {M} {N} {K}", flush=True)
    check(ctx, form, {"m": M // 3 + 1, "x": 3, "n": N // 2 + 1, "y": 2, "k": K, "z": 2}, -1.0, 0.25)


@pytest.mark.parametrize("beta", [0.0, 1.0])
@pytest.mark.parametrize("o,v", [(17, 130), (20, 97), (27, 61), (31, 90), (32, 64), (33, 70)])
@pytest.mark.parametrize("form", ["abej,ei,abij", "abej,ie,abij"])
def test_few_columns(ctx, form, o, v, beta):
    print(f"case: few columns {form} o={o} v={v} beta={beta}", flush=True)
    check(ctx, form, {c: v if c < "i" else o for c in form if c != ","}, 1.0, beta)


def test_batch_label(ctx):
    check(ctx, "mkb,bkn,nmb", {"m": 260, "n": 131, "k": 700, "b": 3}, 1.0, 1.0)
