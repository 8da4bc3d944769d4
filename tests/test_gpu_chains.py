"""List ranking by ruler contraction and the placing of its result: paths
and cycles of lengths around the ruler period, the 64-node bitmap words and
the FASTA tile, against the oracle."""
import numpy as np
import pytest

import bruno_amd
from tests.gpu_common import compare_all

pytestmark = pytest.mark.gpu

PATHS = [3, 4, 7, 8, 9, 15, 16, 17, 31, 33, 63, 64, 65, 127, 129, 255, 513, 2047, 2048, 2049]
CYCLES = [3, 5, 7, 8, 16, 40, 63, 64, 65, 200, 1000, 4099]


def reads_of(seqs):
    b = np.frombuffer("".join(seqs).encode(), np.uint8)
    o = np.concatenate([[0], np.cumsum([len(s) for s in seqs])]).astype(np.uint64)
    return b, o


def random_seq(rng, n):
    return "".join("ACGT"[c] for c in rng.integers(0, 4, n))


def path_and_cycle_reads(rng, k, paths, cycles):
    """One read per path (n nodes: n + k - 1 bases) and per cycle (period p,
    read once round and through its start again)."""
    out = [random_seq(rng, n + k - 1) for n in paths]
    for p in cycles:
        s = random_seq(rng, p)
        out.append((s * ((p + k + 1) // p + 1))[:p + k + 1])
    return [out[i] for i in rng.permutation(len(out))]


@pytest.mark.parametrize("k", [21, 31, 47])
@pytest.mark.parametrize("paths,cycles", [(PATHS, CYCLES), (PATHS, []), ([], CYCLES), ([5], []), ([], [3])])
def test_paths_and_cycles(k, paths, cycles):
    rng = np.random.default_rng(k * 100 + len(paths) + 7 * len(cycles))
    b, o = reads_of(path_and_cycle_reads(rng, k, paths, cycles))
    compare_all(k, None, b, o)


@pytest.mark.parametrize("period", [8, 4096])
def test_ruler_period(period):
    """Dense rulers, and walks as long as the paths (only their ends are
    rulers; cycles without any)."""
    from bruno_amd.autotune import get_tuning, set_tuning
    knobs = get_tuning()
    rng = np.random.default_rng(period)
    b, o = reads_of(path_and_cycle_reads(rng, 31, PATHS * 3, CYCLES * 3))
    try:
        set_tuning(ruler_sample=period)
        compare_all(31, None, b, o)
    finally:
        set_tuning(**knobs)


def test_batch_of_paths_and_cycles():
    """Per-job rounds, cycles and slices when the jobs' paths are placed
    together; jobs of cycles only and of one path only among them."""
    k = 27
    rng = np.random.default_rng(5)
    jobs = [reads_of(path_and_cycle_reads(rng, k, p, c))
            for p, c in ((PATHS, CYCLES), ([], CYCLES), ([9], []), (PATHS, []), ([3, 3, 3], [64]))]
    bases = np.concatenate([b for b, _ in jobs])
    offs, first = [0], [0]
    for b, o in jobs:
        offs += [offs[-1] + int(x) for x in o[1:]]
        first.append(first[-1] + len(o) - 1)
    bt = bruno_amd.GraphBatch(k, None, [4 * len(b) + 64 for b, _ in jobs])
    bt.parse_count(bases, np.array(offs, np.uint64), first)
    bt.run(1)
    for i, (b, o) in enumerate(jobs):
        one = bruno_amd.GraphJob(k, None)
        one.parse_count(b, o)
        one.run(1)
        v, st, s1 = bt.job(i), bt.job(i).stats(), one.stats()
        assert v.unitigs() == one.unitigs()
        assert np.array_equal(v.chain_nodes(), one.chain_nodes())
        assert np.array_equal(v.chain_edges(), one.chain_edges())
        for f in ("iterations", "n_cycle_nodes", "n_isolated", "n_unitigs", "n_unitig_nodes", "n_chain_nodes"):
            assert st[f] == s1[f], (i, f)
        one.close()
    bt.close()
