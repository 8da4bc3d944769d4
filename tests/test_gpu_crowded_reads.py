"""Reads that put many records into one bucket at once (a share of them
poly-A, spread evenly, as low-complexity and duplicate reads lie in real
input): the record parser's stage for that bucket overflows at every append
while the share of all records stays small, and every count must still be
exact."""
import numpy as np
import pytest

import bruno_amd
from bruno_amd.autotune import get_tuning, set_tuning
from gpu_common import node_table, oracle_node_table, run_oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def every_call_by_regions():
    old = get_tuning()
    set_tuning(count_regions=2)
    yield
    set_tuning(**old)


def reads_with(seed, n, length, poly, poly_length, locus=None):
    """n reads of a 20,000-base genome without errors, of which those numbered
    in poly are poly-A of poly_length bases, and those in locus all begin at
    the same base."""
    rng = np.random.default_rng(seed)
    g = rng.choice(np.frombuffer(b"ACGT", np.uint8), 20_000)
    is_poly = np.zeros(n, bool)
    is_poly[poly] = True
    lens = np.where(is_poly, poly_length, length)
    off = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint64)
    read = np.repeat(np.arange(n), lens)
    at = np.arange(int(off[-1])) - off[:-1].astype(np.int64)[read]
    start = rng.integers(0, len(g) - length, n)
    if locus is not None:
        start[locus] = 7777
    b = np.where(is_poly[read], ord("A"), g[start[read] + at])
    return b.astype(np.uint8), off


def reads_with_poly(seed, n, length, every, poly_length):
    return reads_with(seed, n, length, slice(0, n, every), poly_length)


def in_order(lo, hi, edge, count):
    at = np.lexsort((edge, lo, hi))
    return [np.asarray(v)[at].tolist() for v in (hi, lo, edge, count)]


def check(k, b, off, capacity=1 << 20):
    job = bruno_amd.GraphJob(k, None, capacity=capacity)
    job.parse_count(b, off)
    assert job.stats()["count_by_regions"] == 1
    o = run_oracle(k, None, b, off)
    assert job.stats()["n_instances"] == o.stat("n_instances")
    assert node_table(job.counts()) == oracle_node_table(o.unfiltered())
    # (k-mer, biedge) counts, which do not saturate
    km, e, c = job.k2()
    hi = km[:, 1] if km.shape[1] > 1 else np.zeros(len(km), np.uint64)
    assert in_order(km[:, 0], hi, e, c) == in_order(*o.k2())
    job.close()


# Reads of one wave per workgroup (64 of them) and of several; about 200 records
# of the poly-A k-mer beyond its stage at every append.
@pytest.mark.parametrize("k,n,length,every,poly", [
    (31, 4000, 150, 4, 50), (31, 120_000, 150, 27, 60), (63, 120_000, 150, 8, 75), (25, 300_000, 101, 36, 60),
])
def test_crowded_stage(k, n, length, every, poly):
    check(k, *reads_with_poly(n + k, n, length, every, poly))


# Whole intervals of a workgroup's records in one bucket: more than the stage
# and the park hold, and more than a chunk, from one wave and from many.
@pytest.mark.parametrize("k,n,length,run,poly", [
    (31, 6000, 150, 300, 60), (31, 120_000, 150, 468, 60), (63, 120_000, 150, 468, 90), (25, 600_000, 101, 2000, 40),
])
@pytest.mark.parametrize("what", ["poly", "locus"])
def test_crowded_run(k, n, length, run, poly, what):
    at = slice(n // 3, n // 3 + run)
    if what == "poly":
        check(k, *reads_with(n + k, n, length, at, poly))
    else:
        check(k, *reads_with(n + k, n, length, slice(0, 0), 1, at))


def test_one_bucket_of_all_records_falls_back():
    """A tenth of all records in one bucket would be one workgroup's split: the
    call is counted with atomics, alone and after one counted by regions."""
    k, n = 31, 60_000
    skew = reads_with(3, n, 150, slice(0, n, 4), 100)
    even = reads_with(3, n, 150, slice(0, 0), 1)
    for calls in ((skew,), (even, skew)):
        job = bruno_amd.GraphJob(k, None, capacity=1 << 20)
        for b, off in calls:
            job.parse_count(b, off)
        assert job.stats()["count_by_regions"] == 0
        want = run_oracle(k, None, np.concatenate([b for b, _ in calls]),
                          np.concatenate([calls[0][1]] + [o[1:] + calls[0][1][-1] for _, o in calls[1:]]))
        assert node_table(job.counts()) == oracle_node_table(want.unfiltered())
        job.close()


def test_crowded_run_of_512_buckets():
    set_tuning(region_slots=1280)
    check(31, *reads_with(5, 300_000, 150, slice(100_000, 101_200), 60), capacity=1_400_000_000)


def test_crowded_job_beside_others():
    """A crowded job of a batch leaves the count of the others by regions."""
    k = 31
    parts = [reads_with(70, 20_000, 150, slice(0, 0), 1), reads_with(71, 20_000, 150, slice(5000, 5300), 60),
             reads_with(72, 3000, 100, slice(0, 0), 1)]
    off, first = [np.zeros(1, np.uint64)], np.cumsum([0] + [len(o) - 1 for _, o in parts]).astype(np.uint64)
    for _, o in parts:
        off.append(o[1:] + off[-1][-1])
    bt = bruno_amd.GraphBatch(k, None, [1 << 19] * 3)
    bt.parse_count(np.concatenate([b for b, _ in parts]), np.concatenate(off), first)
    assert bt.stats()["count_by_regions"] == 1
    for i, (b, o) in enumerate(parts):
        assert node_table(bt.job(i).counts()) == oracle_node_table(run_oracle(k, None, b, o).unfiltered()), i
    bt.close()
