"""Results of more pieces than the pinned ring holds (a slot is filled again),
text from an odd address with helper threads, and several jobs at it at once."""
import ctypes
import threading

import numpy as np
import pytest

import bruno_amd
from gpu_common import run_oracle
from helpers import pack, rc
from test_gpu_copy_out import K, genome_reads

pytestmark = pytest.mark.gpu


def compacted(reads):
    job = bruno_amd.GraphJob(K, None)
    job.parse_count(*pack(reads))
    job.run()
    return job


@pytest.mark.parametrize("n", [629_146, 700_001])
def test_four_pieces(n):
    """40 n bytes of chain nodes: three pieces and a little, four with a part."""
    reads = genome_reads(n, n)
    on = run_oracle(K, None, *pack(reads)).chain_nodes()
    job = compacted(reads)
    for _ in range(2):
        gn = job.chain_nodes()
        assert len(gn) == len(on) >= n - 1  # (a last read of one k-mer gives nothing)
        assert np.array_equal(gn["k"][:, 0], on["k_lo"]) and np.array_equal(gn["dist"], on["dist"])
        assert np.array_equal(gn["rep"][:, 0], on["rep_lo"])
    job.close()


@pytest.mark.parametrize("n", [9_000_003, 26_000_000])
def test_long_text(n):
    """Reads of a random genome that share no k+1-mer are a unitig each: the
    text is known without an oracle."""
    reads = genome_reads(n, n)
    seqs = sorted((min(r, rc(r), key=lambda s: s[:K]) for r in reads if len(r) >= K + 2), key=lambda s: s[:K])
    want = "\n".join(">" + min(s[:K], rc(s[:K])) + "\n" + s for s in seqs).encode()
    job = compacted(reads)
    for _ in range(2):
        assert job.unitigs() == want
    job.close()


def test_jobs_at_once():
    """4 MB of chain nodes each, fetched by a thread per job."""
    want, got = {}, {}
    for s in range(4):
        want[s] = run_oracle(K, None, *pack(genome_reads(s, 100_000))).chain_nodes()["dist"].tolist()

    def one(s):
        job = compacted(genome_reads(s, 100_000))
        got[s] = [job.chain_nodes()["dist"].tolist() for _ in range(5)]
        job.close()

    ts = [threading.Thread(target=one, args=(s,)) for s in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert got == {s: [want[s]] * 5 for s in want}


def test_another_device_current():
    """Results fetched by a thread whose current device is not the job's."""
    hip, n = bruno_amd.lib(), ctypes.c_int()  # (the library's own HIP runtime)
    assert hip.hipGetDeviceCount(ctypes.byref(n)) == 0
    if n.value < 2:
        pytest.skip("needs two devices")
    job = compacted(genome_reads(1, 60_000))
    want, got = job.unitigs(), []

    def fetch():
        hip.hipSetDevice(1)
        got.append(job.unitigs())

    t = threading.Thread(target=fetch)
    t.start()
    t.join()
    assert got == [want]
    job.close()
