"""Keys of the region build: during the adds a slot is known by its hash
word, so two-word k-mers whose 64-bit hashes agree must still be told apart,
in a first count and in one that adds to written regions."""
import numpy as np
import pytest

import bruno_amd
from bruno_amd.autotune import get_tuning, set_tuning
from tests.gpu_common import node_table, oracle_node_table, run_oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def every_call_by_regions():
    old = get_tuning()
    set_tuning(count_regions=2)
    yield
    set_tuning(**old)


M = (1 << 64) - 1
MUL, ADD = 0xD6E8FEB86659FD93, 0x9E3779B97F4A7C15


def kmix(x):
    x ^= x >> 32
    x = x * MUL & M
    return x ^ (x >> 32)


def kmer_hash(v):
    return kmix((v & M) ^ kmix((v >> 64) + ADD & M))


def rc(v, k):
    r = 0
    for _ in range(k):
        r = r << 2 | (3 - (v & 3))
        v >>= 2
    return r


def text(v, k):
    return "".join("ACGT"[v >> 2 * (k - 1 - i) & 3] for i in range(k))


def colliding(rng, k, n):
    """n canonical k-mers (40 <= k <= 63) with one hash."""
    bits = 2 * k - 64
    want, out = None, []
    while len(out) < n:
        hi = int(rng.integers(0, 1 << 62)) & ((1 << bits) - 1)
        lo = int(rng.integers(0, 1 << 63)) * 2 + int(rng.integers(0, 2))
        if want is not None:
            # the low word that gives the hash with this high word
            lo = want ^ kmix(hi + ADD & M)
        v = hi << 64 | lo
        if v < rc(v, k) and v not in out:
            want = lo ^ kmix(hi + ADD & M)
            out.append(v)
    assert len({kmer_hash(v) for v in out}) == 1
    return out


@pytest.mark.parametrize("k", [40, 47, 63])
@pytest.mark.parametrize("batches", [1, 2])
def test_equal_hash_words(k, batches):
    rng = np.random.default_rng(k)
    kms = colliding(rng, k, 6)
    reads = []
    for i, v in enumerate(kms):
        for _ in range(i + 1):
            reads.append(text(v, k) + "".join("ACGT"[c] for c in rng.integers(0, 4, 3)))
    order = rng.permutation(len(reads))
    reads = [reads[i] for i in order]
    b = np.frombuffer("".join(reads).encode(), np.uint8)
    L = k + 3
    o = np.arange(len(reads) + 1, dtype=np.uint64) * L
    job = bruno_amd.GraphJob(k, None, capacity=1 << 22)
    cut = len(reads) // 2 if batches == 2 else len(reads)
    job.parse_count(b[:cut * L], o[:cut + 1])
    if batches == 2:
        job.parse_count(b[cut * L:], o[:len(reads) - cut + 1])
    assert job.stats()["count_by_regions"] == 1
    assert node_table(job.counts()) == oracle_node_table(run_oracle(k, None, b, o).unfiltered())
    job.close()
