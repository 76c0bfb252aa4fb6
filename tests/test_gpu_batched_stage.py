"""The contraction stage of a small closed-shell iteration as batched launches:
every tensor that it forms against the oracle, at sizes on the edges of its
tiles (16, 32, 64), with long contractions that are split, with a ladder that
is not packed, and just below and just above the size where it is used.

Both sides are FP64 sums of at most n = o v^2 + 12 products (the longest
contraction and the terms of an output), so an element is off by at most
n 2^-53 of the sum of magnitudes; that sum stays below 16 here, and two
iterations feed the error back a few times."""

import numpy as np
import pytest

import aquarius_amd as aq
from oracle import rhfccsd, synth

pytestmark = pytest.mark.gpu

NAMES = ("FAE", "FMI", "FME", "WMNIJ", "WMNEJ", "WAMIJ", "WAMEI", "WAMIE", "T1", "T2")


@pytest.mark.parametrize("precision", ["fp64", "bf16x3"])   # bf16x3: every product is below min_reduced_flops
@pytest.mark.parametrize("o,v,symmetric", [
    (1, 1, True), (1, 2, True), (2, 1, True), (1, 17, True), (3, 16, True), (4, 17, False), (5, 19, True),
    (7, 33, True), (8, 32, False), (15, 31, True), (16, 16, True), (3, 65, True), (17, 64, True), (19, 98, True), (20, 94, True)])
def test_stage_matches_oracle(o, v, symmetric, precision):
    seed, nQ = 100 * o + v, o + v + 3
    print(f"case: stage o={o} v={v} symmetric={symmetric} {precision}", flush=True)
    eps, B = aq.synth_host(seed, o, v, nQ)
    f, V = synth.fock(eps[:o], eps[o:]), synth.blocks_from_B(B, o)
    if not symmetric:
        V["VABCD"][0, 1, 1, 2] += 0.05
    ref = rhfccsd.RHFCCSD(f, V, rhfccsd.default_config())
    tol = 16 * 16 * (o * v * v + 12) * 2.0 ** -53
    with aq.Context() as ctx:
        ints = aq.Integrals.from_numpy(ctx, f, V)
        cc = aq.RHFCCSD(ctx, ints, precision=precision, min_reduced_flops=1e18)
        for it in range(2):
            e, _ = cc.iterate()
            ref.iterate()
            assert abs(e - ref.energy) <= tol * max(1.0, abs(ref.energy)), (it, e, ref.energy)
            for name in NAMES:
                want = getattr(ref, name)
                np.testing.assert_allclose(cc.tensor(name).numpy(), want, rtol=0,
                                           atol=tol * max(1.0, np.abs(want).max()), err_msg=f"{name} {it}")
        cc.close()
        ints.free()


@pytest.mark.parametrize("spare", [16, 32, 256])
def test_tight_budget(spare):
    """`spare` doubles tensors beyond the solver and its DIIS history: too few
    for the batched stage's buffers (the first two) the iteration runs with
    evictable operand copies, to the same energy."""
    o, v, order = 6, 30, 4
    print(f"case: stage budget {spare}", flush=True)
    eps, B = aq.synth_host(9, o, v, 40)
    f, V = synth.fock(eps[:o], eps[o:]), synth.blocks_from_B(B, o)
    cfg = rhfccsd.default_config()
    cfg["diis"]["order"] = order
    ref = rhfccsd.RHFCCSD(f, V, cfg)
    held = 0
    for bounded in (False, True):
        with aq.Context(hbm_budget=held + (2 * order + spare) * 8 * (o * v) ** 2 if bounded else 0) as ctx:
            ints = aq.Integrals.from_numpy(ctx, f, V)
            cc = aq.RHFCCSD(ctx, ints, diis_order=order)
            if not bounded:
                held = ctx.memory()[0]
            else:
                for _ in range(6):
                    e, _ = cc.iterate()
                    ref.iterate()
                assert abs(e - ref.energy) <= 1e-9 * abs(ref.energy)
            cc.close()
            ints.free()
