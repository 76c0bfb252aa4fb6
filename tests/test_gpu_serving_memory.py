"""Memory that a server keeps between jobs: jobs of very different sizes, in an
order that reuses, outgrows and splits what was kept, give the energies of the
direct solver bit for bit on every slot count; and the device has its memory
back when the server is gone."""

import numpy as np
import pytest
import torch

import aquarius_amd as aq

pytestmark = pytest.mark.gpu

SIZES = [(3, 12), (8, 48), (4, 30), (8, 48), (2, 9), (7, 52), (3, 12), (5, 41)]


@pytest.mark.parametrize("slots", [1, 3])
@pytest.mark.parametrize("prec", ["fp64", "bf16x3"])
def test_reused_blocks_do_not_change_results(slots, prec):
    cfg = lambda: aq.default_config(diis_order=6, max_iterations=60, precision=prec, min_reduced_flops=1e6)
    alone = {}
    with aq.Context() as ctx:
        for k, (o, v) in enumerate(SIZES):
            ints = aq.Integrals.synthetic(ctx, 50 + k, o, v)
            cc = aq.RHFCCSD(ctx, ints, config=cfg())
            alone[k] = cc.run()["energy"]
            cc.close()
            ints.free()
        ctx.trim()
    torch.cuda.synchronize()
    free0 = torch.cuda.mem_get_info()[0]
    with aq.Server(slots=slots) as s:
        for _ in range(2):
            ids = [s.submit(50 + k, o, v, config=cfg()) for k, (o, v) in enumerate(SIZES)]
            for k, i in enumerate(ids):
                r = s.wait(i)
                assert r["status"] == aq.JOB_DONE, r["error"]
                assert r["energy"] == alone[k], (k, SIZES[k], r["energy"], alone[k])
                assert r["bytes_peak"] <= r["bytes_reserved"]
    torch.cuda.synchronize()
    assert torch.cuda.mem_get_info()[0] >= free0 - (256 << 20)
