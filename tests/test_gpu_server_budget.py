"""The memory that the server's batches hold at once stays within its budget,
the record buffers of their counts and the regions' room in their tables
included; where the budget leaves too little of it, a batch counts with atomics
and its results are the same."""
import threading

import numpy as np
import pytest

import bruno_amd
from bruno_amd.device import pool_stats, pool_trim
from bruno_amd.server import Server
from gpu_common import run_oracle
from helpers import thresholds_L

pytestmark = pytest.mark.gpu


def requests(k, n):
    """Many instances of few k-mers: the records outweigh the table."""
    out = []
    for i in range(n):
        rng = np.random.default_rng(100 * k + i)
        g = rng.choice(np.frombuffer(b"ACGT", np.uint8), 30_000)
        at = rng.integers(0, 30_000 - 150, 60_000)
        out.append((g[at[:, None] + np.arange(150)[None, :]].reshape(-1), np.arange(60_001, dtype=np.uint64) * 150))
    return out


@pytest.mark.parametrize("k", [31, 63])
@pytest.mark.parametrize("budget", [260 << 20, 1 << 30, 8 << 30])
def test_batches_stay_within_the_budget(k, budget):
    th = thresholds_L(2)
    reqs = requests(k, 6)
    want = [run_oracle(k, th, b, o).chain_fasta() for b, o in reqs]
    pool_trim()
    base, peak, stop = pool_stats()["in_use"], [0], threading.Event()

    def watch():
        while not stop.is_set():
            peak[0] = max(peak[0], pool_stats()["in_use"] - base)

    w = threading.Thread(target=watch)
    w.start()
    try:
        with Server(hbm_budget=budget, n_workers=2, max_batch_jobs=2, reserve_pool=False) as srv:
            tickets = [srv.submit_reads(k, th, b, o, capacity=1 << 19) for b, o in reqs]
            for t, fasta in zip(tickets, want):
                assert srv.wait(t)["status"] == 0
                assert srv.unitigs(t) == fasta
            st = srv.stats()
    finally:
        stop.set()
        w.join()
    assert st["jobs_done"] == len(reqs) and st["jobs_failed"] == 0 and st["retries"] == 0
    assert st["peak_reserved"] <= budget
    assert peak[0] <= budget


def test_planner_counts_the_regions_room():
    from bruno_amd.planner import region_slots
    k, caps = 31, [1 << 19, 60_000, 300_000]
    bt = bruno_amd.GraphBatch(k, None, caps)
    assert bt.stats()["capacity"] == sum(region_slots(c, k) for c in caps)
    bt.close()
