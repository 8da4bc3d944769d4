"""Self counts summed 64 nodes a wave (.chain.edges): unitigs that start and
end anywhere in a wave's nodes, many short ones in one, one over many waves."""
import numpy as np
import pytest

from gpu_common import run_oracle
from helpers import pack
from test_gpu_edges_out import gpu_edges

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [24, 31, 63])
@pytest.mark.parametrize("nodes", [[64] * 12, [3] * 200, [3, 61, 63, 65, 66, 127, 128, 129, 5000, 4, 3, 191, 20000, 7]])
def test_unitigs_of_these_lengths(k, nodes):
    rng = np.random.default_rng(k)
    reads = []
    for n in nodes:
        s = "".join(rng.choice(list("ACGT"), n + k - 1))
        reads.append(s)
        for _ in range(3):  # uneven counts along it
            a = int(rng.integers(0, n))
            reads.append(s[a:a + int(rng.integers(k + 2, k + 400))])
    b, off = pack(reads)
    be, ce, st = gpu_edges(k, None, b, off)
    o = run_oracle(k, None, b, off)
    assert be == o.branch_edges() and ce == o.chain_edges()
    assert st["n_unitigs"] >= len(nodes)
