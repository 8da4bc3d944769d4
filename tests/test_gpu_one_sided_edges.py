"""Edges that thresholds on (k-mer, biedge) counts leave on one side only: a
branch keeps its edge to a chain node whose own only edge on that side leads
to another chain node, which points back at it.  The chain nodes are then no
disjoint paths, so list ranking has to follow the rounds, and the outputs are
the oracle's."""
import numpy as np
import pytest

from gpu_common import compare_all, oracle_node_table, run_oracle
from helpers import DEFAULT_T, pack, rc

K2_THREE = [0, DEFAULT_T, 0, DEFAULT_T, 3, DEFAULT_T]  # a biedge is kept from three instances
K = 21


def canon(s):
    return min(s, rc(s))


def as_int(s):
    v = 0
    for ch in s:
        v = v << 2 | "ACGT".index(ch)
    return v


def gadgets(seed, n, flank=40):
    """n times: branch B = y + core[:-1] (two predecessors) and chain node
    D = x + core[:-1] before C = core.  B's biedges into C count three each and
    are kept; C's from B are spread over three successors, two each, and are
    dropped; C's from D count five.  Returns reads and (x, y, core) of each."""
    rng = np.random.default_rng(seed)

    def rand(m):
        return "".join(rng.choice(list("ACGT"), m))

    reads, made = [], []
    for _ in range(n):
        core = rand(K)
        x, y, _, _ = rng.permutation(list("ACGT"))
        o = rng.permutation(list("ACGT"))[:3]
        right = [rand(flank) for _ in range(3)]
        reads += [rand(flank) + x + core + o[0] + right[0]] * 5
        a = rng.permutation(list("ACGT"))[:2]
        for left in (rand(flank) + a[0], rand(flank) + a[1]):
            reads += [left + y + core + o[q] + right[q] for q in range(3)]
        made.append((x, y, core))
    at = rng.permutation(len(reads))
    return [rc(reads[i]) if i % 2 else reads[i] for i in at], made


def one_sided(nodes, x, y, core):
    """B's edge into C is there, C's edge back to B is not, C's to D is."""

    def edges(s, side):  # counts of the out (0) or in (1) edges of s as it reads here
        c = nodes[as_int(canon(s))]
        return list(c[4:8] if side else c[:4]) if canon(s) == s else list((c[:4] if side else c[4:8])[::-1])

    last, b_in = "ACGT".index(core[-1]), edges(core, 1)
    return (edges(y + core[:-1], 0)[last] > 0 and b_in["ACGT".index(y)] == 0 and b_in["ACGT".index(x)] > 0
            and sum(v > 0 for v in edges(y + core[:-1], 1)) == 2)


def test_the_graph_is_one_sided():
    reads, made = gadgets(3, 60)
    b, off = pack(reads)
    nodes = oracle_node_table(run_oracle(K, K2_THREE, b, off).nodes())
    assert sum(one_sided(nodes, *m) for m in made) >= 55


@pytest.mark.gpu
@pytest.mark.parametrize("variant", [1, 0])
@pytest.mark.parametrize("n", [1, 60])
def test_one_sided_edges(n, variant):
    reads, _ = gadgets(3, n)
    compare_all(K, K2_THREE, *pack(reads), variant=variant)
