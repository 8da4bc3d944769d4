"""Results copied to the host in pinned pieces: lengths around the line above
which several threads copy (2 MB) and around a piece (8 MB)."""
import threading

import numpy as np
import pytest

import bruno_amd
from gpu_common import run_oracle
from helpers import pack

pytestmark = pytest.mark.gpu

K = 31


def genome_reads(seed, n):
    """One unitig of n nodes: n + 2 K + 1 bytes of text."""
    g = np.random.default_rng(seed).choice(np.frombuffer(b"ACGT", np.uint8), n + K - 1).tobytes().decode()
    return [g[a:a + 10_000 + K - 1] for a in range(0, n, 10_000)]


@pytest.mark.parametrize("n", [3, 1000, 52428, 52429, 209715, 209716, 250_000])
def test_results_of_length(n):
    """40 n bytes of chain nodes, n + 62 of text from an odd address."""
    b, off = pack(genome_reads(n, n))
    o = run_oracle(K, None, b, off)
    job = bruno_amd.GraphJob(K, None)
    job.parse_count(b, off)
    job.run()
    on, gn = o.chain_nodes(), job.chain_nodes()
    assert gn.nbytes == 40 * n
    assert np.array_equal(gn["k"][:, 0], on["k_lo"]) and np.array_equal(gn["dist"], on["dist"])
    assert np.array_equal(gn["rep"][:, 0], on["rep_lo"])
    assert job.unitigs() == o.chain_fasta()
    assert job.branch_fasta() == o.branch_fasta()
    job.close()


def test_many_threads():
    """Each thread's job has rings and buffers of its own."""
    want, got = {}, {}
    for s in range(6):
        want[s] = run_oracle(K, None, *pack(genome_reads(s, 20_000))).chain_fasta()

    def one(s):
        job = bruno_amd.GraphJob(K, None)
        job.parse_count(*pack(genome_reads(s, 20_000)))
        job.run()
        got[s] = [job.unitigs() for _ in range(3)]
        job.close()

    ts = [threading.Thread(target=one, args=(s,)) for s in range(6)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert got == {s: [want[s]] * 3 for s in want}
