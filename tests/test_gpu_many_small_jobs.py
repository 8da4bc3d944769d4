"""Batches of very many small jobs keep probe windows and the atomic count
(a job costs the region count 32 buckets and a workgroup whatever it holds),
and one very small job among larger ones must not blow up their buffers."""
import numpy as np
import pytest

import bruno_amd
from gpu_common import node_table, oracle_node_table, run_oracle
from helpers import pack, random_reads
from test_gpu_batch import pack_jobs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [31, 63])
def test_many_small_jobs(k):
    n, cap = 2400, 300  # 2^19 slots and more in all
    _, reads = random_reads(k, 3000, n, 90, 0.0)
    jobs = [[reads[i], reads[i]] for i in range(n)]
    bt = bruno_amd.GraphBatch(k, None, [cap] * n)
    bt.parse_count(*pack_jobs(jobs))
    st = bt.stats()
    assert st["count_by_regions"] == 0
    # the slots asked for, a sixteenth more for the side table, and what a batch holds per job
    slot = 32 if k <= 31 else 64
    assert st["device_bytes"] <= n * cap * (slot + 4) + (2 << 20)
    for i in range(0, n, 97):
        want = run_oracle(k, None, *pack(jobs[i]))
        assert node_table(bt.job(i).counts()) == oracle_node_table(want.unfiltered()), i
    bt.close()


@pytest.mark.parametrize("k", [31, 63])
def test_one_small_job_beside_others(k):
    """The buffers of eight jobs counted by regions grow by what a ninth, of 64
    slots, needs, and not by a larger chunk for every bucket."""
    rng = np.random.default_rng(k)
    g = "".join(rng.choice(list("ACGT"), 60_000))
    jobs = [[g[i:i + 150] for i in rng.integers(0, len(g) - 150, 20_000)] for _ in range(8)]
    tiny = [g[:k + 10]]
    peak = []
    for js in (jobs, jobs + [tiny]):
        bt = bruno_amd.GraphBatch(k, None, [1 << 19] * 8 + [64] * (len(js) - 8))
        bt.parse_count(*pack_jobs(js))
        st = bt.stats()
        assert st["count_by_regions"] == 1
        peak.append(st["peak_device_bytes"])
        for i in (0, len(js) - 1):
            want = run_oracle(k, None, *pack(js[i]))
            assert node_table(bt.job(i).counts()) == oracle_node_table(want.unfiltered()), i
        bt.close()
    assert peak[1] < 1.05 * peak[0]


def test_more_jobs_than_workgroups():
    """300 jobs, one of them with most of the reads: it gets more than one
    workgroup of the record parser, and every job its own counts."""
    k, n = 31, 300
    rng = np.random.default_rng(8)
    g = "".join(rng.choice(list("ACGT"), 30_000))

    def reads(m):
        return [g[i:i + 150] for i in rng.integers(0, len(g) - 150, m)]

    jobs = [reads(int(m)) for m in rng.integers(0, 60, n)]
    jobs[170] = reads(60_000)
    bt = bruno_amd.GraphBatch(k, None, [45_000] * n)
    bt.parse_count(*pack_jobs(jobs))
    assert bt.stats()["count_by_regions"] == 1
    for i in list(range(0, n, 23)) + [170]:
        want = run_oracle(k, None, *pack(jobs[i]))
        assert node_table(bt.job(i).counts()) == oracle_node_table(want.unfiltered()), i
        assert bt.job(i).stats()["n_reads"] == len(jobs[i])
    bt.close()
