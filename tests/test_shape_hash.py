"""The shape hash against its definition: every round of the leaf-anchored colour refinement
computed from the texts, on trees and admixture graphs from 2 to 30 leaves (colour counts on
both sides of ten, where the order of the ranks' texts leaves the ranks' order)."""
import numpy as np
import pytest

from steppe_amd import qpgraph


def _hash(edges):
    """2 V + 4 rounds of "own colour|<parents>|<children>" texts, ranked; FNV-1a of the result."""
    nodes = {x for e in edges for x in e}
    parents = {a for a, _ in edges}
    leaf = {n: i for i, n in enumerate(sorted(nodes - parents))}
    up = {n: [a for a, b in edges if b == n] for n in nodes}
    down = {n: [b for a, b in edges if a == n] for n in nodes}
    col = {n: f"L{leaf[n]}" if n in leaf else f"I{len(up[n])}_{len(down[n])}" for n in nodes}
    for _ in range(2 * len(nodes) + 4):
        sig = {n: col[n] + "|<" + "".join(c + "," for c in sorted(col[w] for w in up[n])) + ">|<"
               + "".join(c + "," for c in sorted(col[w] for w in down[n])) + ">" for n in nodes}
        rank = {s: str(i) for i, s in enumerate(sorted(set(sig.values())))}
        col = {n: rank[sig[n]] for n in nodes}
    text = ("N:" + "".join(c + ";" for c in sorted(col.values())) + "E:"
            + "".join(e + ";" for e in sorted(f"{col[a]}>{col[b]}" for a, b in edges)))
    h = 1469598103934665603
    for ch in text.encode():
        h = (h ^ ch) * 1099511628211 % (1 << 64)
    return h


def _graph(rng, n_leaf, n_admix):
    """A random tree, then admixture edges from a split of one edge to a split of a later one."""
    edges = [("r", "x0"), ("r", "x1")]
    tips, k = ["x0", "x1"], 2
    while len(tips) < n_leaf:
        t = tips.pop(int(rng.integers(len(tips))))
        edges += [(t, f"x{k}"), (t, f"x{k + 1}")]
        tips += [f"x{k}", f"x{k + 1}"]
        k += 2
    for m in range(n_admix):
        i, j = sorted(int(x) for x in rng.choice(len(edges), 2, replace=False))
        (a, b), (c, d) = edges[i], edges[j]
        edges[i], edges[j] = (a, f"s{m}"), (c, f"t{m}")
        edges += [(f"s{m}", b), (f"t{m}", d), (f"s{m}", f"t{m}")]
    return edges


@pytest.mark.parametrize("n_leaf", [2, 3, 4, 5, 6, 7, 9, 12, 30])
@pytest.mark.parametrize("n_admix", [0, 1, 3])
def test_hash_is_the_refinements(n_leaf, n_admix):
    rng = np.random.default_rng(100 * n_leaf + n_admix)
    for _ in range(4):
        edges = _graph(rng, n_leaf, min(n_admix, n_leaf - 2))
        assert qpgraph.graph_hash(edges) == _hash(edges), edges
