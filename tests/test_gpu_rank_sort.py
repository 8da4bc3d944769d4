"""Unitig heads and branch points on both sides of the line between sorting by
counting and by radix (8,192), one job and two of a batch, one and two words."""
import pytest

import bruno_amd
from gpu_common import compare_all, run_oracle
from helpers import pack, random_reads, thresholds_L
from test_gpu_batch import pack_jobs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [15, 31, 45])
@pytest.mark.parametrize("n,sides", [(500, "below"), (6000, "above")])
def test_unthresholded_reads(k, n, sides):
    _, reads = random_reads(k, 20 * n, n, 120, 0.02)
    b, off = pack(reads)
    g, _ = compare_all(k, None, b, off, stages=False)
    st = g["stats"]
    assert (st["n_unitigs"] > 8192) == (sides == "above")


@pytest.mark.parametrize("k", [31, 45])
@pytest.mark.parametrize("n", [200, 3000])
def test_two_jobs_of_a_batch(k, n):
    jobs = [random_reads(s, 20 * n, n, 120, 0.02)[1] for s in (1, 2)]
    th = thresholds_L(1)
    bt = bruno_amd.GraphBatch(k, th, [2 * n * 120] * 2)
    bt.parse_count(*pack_jobs(jobs))
    bt.run(1)
    for i, job in enumerate(jobs):
        o = run_oracle(k, th, *pack(job))
        assert bt.job(i).unitigs() == o.chain_fasta()
        assert bt.job(i).branch_fasta() == o.branch_fasta()
    bt.close()
