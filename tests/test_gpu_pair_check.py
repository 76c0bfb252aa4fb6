"""The packed ladder's symmetry check at the edges of its 32 x 32 tiles: a solver
takes the packed ladder on symmetric integrals, and the full one when a single
element of a mirrored pair is off."""

import pytest

import aquarius_amd as aq

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    with aq.Context(0) as c:
        yield c


@pytest.mark.parametrize("v", [31, 32, 33])
@pytest.mark.parametrize("at", [None, (0, 0, 0, 1), (1, 0, 0, 0), (-1, -2, -1, -1), (5, 7, 2, 9)])
def test_pair_symmetry_check_sees_every_element(ctx, v, at):
    ints = aq.Integrals.synthetic(ctx, 3, 2, v, 20)
    if at is not None:
        key = [k % v for k in at]
        flat = sum(k * v ** n for n, k in enumerate(key))
        old = ints.t["VABCD"].read([flat])
        ints.t["VABCD"].write([flat], old + 1e-9)
    cc = aq.RHFCCSD(ctx, ints)
    mirrored = at is None or (at[0] == at[1] and at[2] == at[3])
    assert cc.packed_ladder == mirrored
    cc.close()
    ints.free()
