"""Many short served jobs with graphs on: slots capture while others start and
end jobs, which take over and give back memory between the slots.  No job's
capture may be disturbed by that: every job ends well and has the energy of the
same job without graphs."""

import pytest

import aquarius_amd as aq

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["fp64", "bf16x3"])
def test_captures_beside_starting_and_ending_jobs(prec):
    print(f"case: 48 jobs, 4 slots, graphs, {prec}", flush=True)
    jobs = [(60 + k, 3 + k % 4, 12 + 3 * (k % 5)) for k in range(48)]

    def cfg(graph):
        return aq.default_config(diis_order=6, max_iterations=60, precision=prec, min_reduced_flops=0.0, graph=graph)

    with aq.Server(slots=1) as s:
        alone = [s.wait(i) for i in [s.submit(*j, config=cfg(0)) for j in jobs]]
    with aq.Server(slots=4) as s:
        mix = [s.wait(i) for i in [s.submit(*j, config=cfg(1)) for j in jobs]]
    for a, m, job in zip(alone, mix, jobs):
        assert (a["status"], m["status"]) == (aq.JOB_DONE, aq.JOB_DONE), (job, a["error"], m["error"])
        assert (a["energy"], a["iterations"]) == (m["energy"], m["iterations"]), job
