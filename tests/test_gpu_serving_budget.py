"""What a live server holds of the device between jobs: never more than its
budget.  256 MiB on top: the slots' contexts, queues and streams, and the code
objects and kernel scratch that the first jobs load (free memory is taken after
a warm-up job in the same process, so that most of that is there already)."""

import pytest
import torch

import aquarius_amd as aq

pytestmark = pytest.mark.gpu

OVERHEAD = 256 << 20
SIZES = [(10, 60), (12, 70), (9, 80), (14, 66), (11, 76), (13, 58), (8, 84), (15, 62)]


def free():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def serve(s, sizes):
    cfg = aq.default_config(diis_order=4, max_iterations=4, convergence=0.0)
    for i in [s.submit(7 + k, o, v, config=cfg) for k, (o, v) in enumerate(sizes)]:
        r = s.wait(i)
        assert r["status"] == aq.JOB_DONE, r["error"]


@pytest.fixture(scope="module")
def before():
    with aq.Server(slots=2) as s:
        serve(s, [SIZES[0]] * 2)
    return free()


@pytest.mark.parametrize("slots", [1, 2])
def test_idle_server_holds_at_most_its_budget(before, slots):
    """Jobs of different sizes, one after another: the blocks that each leaves
    fit few of the next one's."""
    cfg = lambda o, v: aq.job_bytes_estimate(o, v, diis_order=4)
    budget = max(cfg(o, v) for o, v in SIZES) * 5 // 4
    print(f"case: budget {budget} slots {slots}", flush=True)
    with aq.Server(slots=slots, hbm_budget=budget) as s:
        for _ in range(2):
            serve(s, SIZES)
            s.drain()
            assert before - free() <= budget + OVERHEAD
    assert before - free() <= OVERHEAD


def test_server_returns_what_earlier_contexts_freed(before):
    """Memory that a context left in the device pool (which keeps no more than
    is in use beside it) goes back to the driver when a server starts: it is not
    missing beside the budget."""
    print("case: pool memory at server start", flush=True)
    with aq.Context() as ctx:
        kept = ctx.tensor((3 << 27,), zero=False)   # 3 GiB
        gone = ctx.tensor((1 << 28,), zero=False)   # 2 GiB
        gone.free()
        ctx.sync()
        assert before - free() > 5 * 10 ** 9        # in the pool
        with aq.Server(slots=1, hbm_budget=1 << 30) as s:
            assert before - free() <= (3 << 30) + OVERHEAD
            s.drain()
        kept.free()


def test_trim_of_another_context_takes_back_what_a_server_keeps(before):
    """At least the largest four-virtual block is kept after the jobs; a context created
    then counts it as free in its default budget (nine tenths), and trim gives it back."""
    print("case: trim beside an idle server", flush=True)
    largest = 8 * max(v for _, v in SIZES) ** 4
    with aq.Context() as ctx, aq.Server(slots=2, hbm_budget=24 << 30) as s:
        serve(s, SIZES)
        s.drain()
        kept = free()
        with aq.Context() as other:
            budget = other.memory()[1]
        ctx.trim()
        trimmed = free()
        assert trimmed - kept >= largest
        assert budget >= 0.9 * (trimmed - OVERHEAD)
        assert before - trimmed <= OVERHEAD
        serve(s, SIZES[:3])                      # and the server goes on
