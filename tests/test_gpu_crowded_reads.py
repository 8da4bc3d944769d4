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


def reads_with_poly(seed, n, length, every, poly_length):
    """n reads of a 20,000-base genome without errors; each `every`-th one is
    poly-A of poly_length bases."""
    rng = np.random.default_rng(seed)
    g = rng.choice(np.frombuffer(b"ACGT", np.uint8), 20_000)
    poly = np.arange(n) % every < 1
    lens = np.where(poly, poly_length, length)
    off = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint64)
    read = np.repeat(np.arange(n), lens)
    at = np.arange(int(off[-1])) - off[:-1].astype(np.int64)[read]
    start = rng.integers(0, len(g) - length, n)
    b = np.where(poly[read], ord("A"), g[start[read] + at])
    return b.astype(np.uint8), off


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
