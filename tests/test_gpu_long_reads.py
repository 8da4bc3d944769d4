"""Reads that the others of a round would wait for are taken by all lanes of a
parser workgroup, a piece of the instances each: every instance once, with the
edges across the pieces and none at the read's ends, whatever the read's length
and alignment, and none of a read with a byte that is no base anywhere."""
import numpy as np
import pytest

import bruno_amd
from bruno_amd.autotune import get_tuning, set_tuning
from gpu_common import node_table, oracle_node_table, run_oracle
from test_gpu_batch import pack_jobs
from test_gpu_crowded_reads import check, in_order

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def every_call_by_regions():
    old = get_tuning()
    set_tuning(count_regions=2)
    yield
    set_tuning(**old)


def reads_of(seed, lens, genome=40_000):
    rng = np.random.default_rng(seed)
    g = rng.choice(np.frombuffer(b"ACGT", np.uint8), genome)
    off = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint64)
    read = np.repeat(np.arange(len(lens)), lens)
    at = np.arange(int(off[-1])) - off[:-1].astype(np.int64)[read] + rng.integers(0, genome, len(lens))[read]
    return g[at % genome], off


def mixed(seed, n, long_lens):
    """n reads of 60 to 250 bases with longer ones spread among them."""
    rng = np.random.default_rng(seed)
    lens = rng.integers(60, 250, n)
    lens[rng.permutation(n)[:len(long_lens)]] = long_lens
    return lens


# lengths about the lines 2^8, 2^9 ..., one instance more or less than lanes
LINES = [256, 257, 512, 513, 1023, 1024, 1025, 1054, 1055, 1086, 2049, 4096, 16_385, 65_537]


@pytest.mark.parametrize("k", [31, 21, 32, 63])
@pytest.mark.parametrize("what", ["one", "few", "lines", "all", "alone"])
def test_long_reads(k, what):
    rng = np.random.default_rng(k)
    lens = {"one": mixed(1, 3000, [200_003]), "few": mixed(2, 70_000, rng.integers(3000, 30_000, 40)),
            "lines": mixed(3, 900, LINES), "all": rng.integers(5000, 15_000, 300), "alone": [700_001]}[what]
    check(k, *reads_of(k, lens))


def test_long_reads_of_512_buckets():
    set_tuning(region_slots=1280)
    check(31, *reads_of(4, mixed(4, 3000, [100_000, 7000])), capacity=1_400_000_000)


@pytest.mark.parametrize("k", [31, 63])
def test_byte_that_is_no_base(k):
    """In the first and last base, in every alignment of a block, across pieces."""
    length, n = 20_000, 60
    b, off = reads_of(k, mixed(5, 2000, [length] * n))
    b = b.copy()
    longs = np.flatnonzero(np.diff(off.astype(np.int64)) == length)
    at = [0, length - 1, 1, length - 2, k, length - k] + list(range(9000, 9040))
    for i, p in zip(longs, at):
        b[int(off[i]) + p] = ord("N")
    job = bruno_amd.GraphJob(k, None, capacity=1 << 20)
    job.parse_count(b, off)
    assert job.stats()["count_by_regions"] == 1
    assert job.stats()["n_reads_dropped"] == len(at)
    o = run_oracle(k, None, b, off)
    assert job.stats()["n_instances"] == o.stat("n_instances")
    km, e, c = job.k2()
    hi = km[:, 1] if km.shape[1] > 1 else np.zeros(len(km), np.uint64)
    assert in_order(km[:, 0], hi, e, c) == in_order(*o.k2())
    job.close()


def test_long_read_in_a_batch():
    k = 31
    parts = [reads_of(20, mixed(6, 5000, [])), reads_of(21, [150_000]), reads_of(22, mixed(7, 100, [40_000, 300]))]
    jobs = [[b[int(o[i]):int(o[i + 1])].tobytes().decode() for i in range(len(o) - 1)] for b, o in parts]
    bt = bruno_amd.GraphBatch(k, None, [1 << 19] * 3)
    bt.parse_count(*pack_jobs(jobs))
    assert bt.stats()["count_by_regions"] == 1
    for i, (b, o) in enumerate(parts):
        assert node_table(bt.job(i).counts()) == oracle_node_table(run_oracle(k, None, b, o).unfiltered()), i
    bt.close()
