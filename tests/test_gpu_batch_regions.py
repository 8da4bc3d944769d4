"""Batches counted by region: every job's buckets and regions go through the
same launches, so jobs of any size (a job of 32 regions beside one of
thousands), empty jobs and several calls must give each job what it has
alone; a job that puts one k-mer into a large share of a pass's records sends
that pass to the atomic count.  Also the widest splits: 512 buckets, and 12
region bits per bucket."""
import numpy as np
import pytest

import bruno_amd
from bruno_amd.autotune import get_tuning, set_tuning
from gpu_common import compare_results, node_table, oracle_node_table, run_oracle
from helpers import pack, random_reads, thresholds_L
from test_gpu_batch import mixed_jobs, pack_jobs

pytestmark = pytest.mark.gpu

BIG = 1 << 22


@pytest.fixture(autouse=True)
def regions_on():
    old = get_tuning()
    set_tuning(count_regions=2)
    yield
    set_tuning(**old)


def caps_of(jobs, k, big):
    """Tight tables, but for one job that brings the batch to BIG slots."""
    c = [max(64, sum(max(0, len(r) - k + 1) for r in j) + 64) for j in jobs]
    c[big] = BIG
    return c


def result(bt, i):
    v = bt.job(i)
    st = v.stats()
    st["n_conflicts"] = 0
    return {"nodes": v.nodes(), "fasta": v.unitigs(), "branch_fasta": v.branch_fasta(),
            "chain_nodes": v.chain_nodes(), "branches": v.branches(), "stats": st, "rounds": st["iterations"]}


@pytest.mark.parametrize("k", [31, 15, 63])
@pytest.mark.parametrize("calls", [1, 3])
@pytest.mark.parametrize("big", [0, 4])
def test_jobs_of_any_size(k, calls, big):
    jobs = mixed_jobs(60 + k)
    th = thresholds_L(2)
    bt = bruno_amd.GraphBatch(k, th, caps_of(jobs, k, big))
    for part in range(calls):
        bt.parse_count(*pack_jobs([j[len(j) * part // calls:len(j) * (part + 1) // calls] for j in jobs]))
    assert bt.stats()["count_by_regions"] == 1
    want = [run_oracle(k, th, *pack(j)) for j in jobs]
    for i in range(len(jobs)):
        assert node_table(bt.job(i).counts()) == oracle_node_table(want[i].unfiltered()), i
    bt.filter()
    bt.build_chains()
    bt.list_rank(1)
    bt.compact()
    for i in range(len(jobs)):
        compare_results(k, result(bt, i), want[i], 1, stages=False)
        assert bt.job(i).stats()["n_reads"] == len(jobs[i])
    bt.close()


@pytest.mark.parametrize("first", ["even", "skewed"])
def test_one_kmer_in_most_records(first):
    """The fallback, in a first count and in one that adds to regions."""
    k = 31
    jobs = mixed_jobs(9)[:4]
    poly = ["A" * 131] * 3000  # 303,000 instances of one k-mer
    skew = [jobs[0], jobs[1] + poly, jobs[2], jobs[3]]
    order = [jobs, skew] if first == "even" else [skew, jobs]
    bt = bruno_amd.GraphBatch(k, None, caps_of(jobs, k, 2))
    for js in order:
        bt.parse_count(*pack_jobs(js))
    for i in range(4):
        o = run_oracle(k, None, *pack(order[0][i] + order[1][i]))
        assert node_table(bt.job(i).counts()) == oracle_node_table(o.unfiltered()), i
    bt.close()


@pytest.mark.parametrize("k,cap", [(31, 700_000_000), (31, 1_400_000_000), (63, 350_000_000)])
def test_widest_splits(k, cap):
    """2^20 regions (256 buckets, 12 region bits) and 2^21 (512 buckets)."""
    set_tuning(region_slots=1280)
    b, off = pack(random_reads(5, 20000, 2000, (80, 200), 0.01)[1])
    job = bruno_amd.GraphJob(k, None, capacity=cap)
    job.parse_count(b, off)
    assert job.stats()["count_by_regions"] == 1
    want = oracle_node_table(run_oracle(k, None, b, off).unfiltered())
    assert node_table(job.counts()) == want
    job.parse_count(b, off)
    assert {q: c[-1] for q, c in node_table(job.counts()).items()} == {q: 2 * c[-1] for q, c in want.items()}
    job.close()


@pytest.mark.parametrize("k", [31, 24, 63])
@pytest.mark.parametrize("sizes", [(100, 20000, 100), (20000, 100, 20000)])
def test_calls_of_few_and_many_instances(k, sizes):
    """count_regions 1 in a table of about 2^19 slots filled to the last one:
    calls below and above the line between atomics and regions, in either
    order, give what the oracle gives."""
    set_tuning(count_regions=1)
    rng = np.random.default_rng(k)
    g = "".join(rng.choice(list("ACGT"), 530_000))
    parts = [[g[i:i + 180] for i in rng.integers(0, len(g) - 180, n)] for n in sizes]
    b, off = pack([r for p in parts for r in p])
    want = oracle_node_table(run_oracle(k, None, b, off).unfiltered())
    job = bruno_amd.GraphJob(k, None, capacity=max(len(want), 1 << 19))
    for p in parts:
        job.parse_count(*pack(p))
        assert job.stats()["count_by_regions"] == (len(p) > 100)
    assert node_table(job.counts()) == want
    job.close()


def test_small_table_takes_batches_after_a_fused_count():
    """Asked to fuse the filter, a table of fewer than 2^22 slots counted by
    regions still takes a further batch (its count is not fused)."""
    _, reads = random_reads(4, 60000, 6000, 150, 0.01)
    b, off = pack(reads)
    job = bruno_amd.GraphJob(31, thresholds_L(2), capacity=1 << 21)
    job.set_fused_filter(True)
    for part in (reads[:4000], reads[4000:]):
        job.parse_count(*pack(part))
        assert job.stats()["count_by_regions"] == 1 and job.stats()["filter_fused"] == 0
    want = run_oracle(31, thresholds_L(2), b, off)
    assert node_table(job.counts()) == oracle_node_table(want.unfiltered())
    job.run()
    assert job.unitigs() == want.chain_fasta()
    job.close()
