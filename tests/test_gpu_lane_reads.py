"""Reads walked by one lane each (record parser, sketch of many reads): every
byte value, alignment and length against the wave-per-read kernels and the
oracle."""
import numpy as np
import pytest

import bruno_amd
from bruno_amd.autotune import get_tuning, set_tuning
from bruno_amd.device import DeviceBuffer
from bruno_amd.pipeline import estimate_distinct
from gpu_common import node_table, oracle_node_table, run_oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def every_call_by_regions():
    old = get_tuning()
    set_tuning(count_regions=2)
    yield
    set_tuning(**old)


def ragged_reads(rng, n, k, long_reads):
    """Reads of k - 1 up to 300 bases, some of either case, some with one byte
    of any value anywhere; long_reads: one longer than a lane takes per 4096."""
    g = rng.choice(np.frombuffer(b"ACGT", np.uint8), 60_000)
    out = []
    for i in range(n):
        L = int(rng.integers(k - 1, 300))
        if long_reads and i % 4096 == 77:
            L = int(rng.integers(2040, 9000))
        p = int(rng.integers(0, len(g) - L))
        r = g[p:p + L].copy()
        if i % 3 == 0:
            r |= rng.choice(np.array([0, 32], np.uint8), L)
        if i % 5 == 0:
            r[int(rng.integers(0, L))] = i // 5 % 256
        out.append(r.tobytes())
    return out


def device(reads):
    b = np.frombuffer(b"".join(reads), np.uint8)
    o = np.zeros(len(reads) + 1, np.uint64)
    o[1:] = np.cumsum([len(r) for r in reads])
    return b, o


@pytest.mark.parametrize("k", [21, 31, 32, 63])
def test_sketch_by_lanes_and_by_waves(k):
    """20,000 reads (a wave each) and the same reads four times (a lane each) have
    the same k-mers, so the same registers and the same estimate."""
    reads = ragged_reads(np.random.default_rng(k), 20_000, k, True)
    ests = []
    for rs in (reads, 2 * (reads + reads[::-1])):
        b, o = device(rs)
        db, do = DeviceBuffer.from_numpy(b), DeviceBuffer.from_numpy(o)
        ests.append(estimate_distinct(k, db.ptr, do.ptr, len(rs))[0])
        db.free()
        do.free()
    assert ests[0] == ests[1] > 0


@pytest.mark.parametrize("k", [21, 31, 47])
def test_any_byte_in_a_read(k):
    reads = ragged_reads(np.random.default_rng(100 + k), 6000, k, False)
    b, o = device(reads)
    job = bruno_amd.GraphJob(k, None, capacity=1 << 20)
    job.parse_count(b, o)
    st = job.stats()
    assert st["count_by_regions"] == 1
    assert st["n_reads_dropped"] == sum(any(c not in b"ACGTacgt" for c in r) for r in reads)
    want = oracle_node_table(run_oracle(k, None, b, o).unfiltered())
    assert node_table(job.counts()) == want
    job.close()
