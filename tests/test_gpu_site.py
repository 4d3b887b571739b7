"""The site kernel (message updates on the matrix cores, every bond <= 16, the site
tensor in LDS) at the edges of its tiles, pairings and launch classes, against the
CPU oracle: one star per case, whose centre has the given bonds, and one sweep
from random messages.

Tolerances, relative to each (normalised) message: FP64 1e-12, sums of at most
2e4 terms of rounding 1e-16 each; FP32 arithmetic 2e-6, at most five products
with 16-term FP32 sums (16 * 6e-8 each at worst) around an FP64 Gram.
"""
import numpy as np
import pytest

import itnbp
from helpers import oracle_graph, oracle_psi, to_index
from oracle import bp_oracle as O

pytestmark = pytest.mark.gpu

BONDS = [(1,), (7,), (16,), (15, 1), (2, 3), (16, 5), (16, 16, 16), (9, 2, 11), (1, 1, 1, 1), (8, 8, 8, 8),
         (5, 7, 3, 2), (4, 4, 4, 4), (10, 10, 10, 10), (3, 3, 3, 3, 3), (2, 3, 2, 4, 2, 3), (12, 3, 13, 2, 1)]


def star(bonds, rng, eltype, d=2):
    """A centre with the given bonds, every leaf with one more site behind it."""
    k = len(bonds)
    g = itnbp.NamedGraph(list(range(2 * k + 1)), [(0, i + 1) for i in range(k)] + [(i + 1, k + i + 1) for i in range(k)])
    link = [0] * g.ne
    for i in range(k):
        link[g.edge_id(0, i + 1)] = bonds[i]
        link[g.edge_id(i + 1, k + i + 1)] = 3
    return g, itnbp.random_tensornetwork(rng, eltype, g, link_space=link, phys_dim=d)


def random_messages(rng, g, psi, symmetric):
    out = {}
    for m in range(2 * g.ne):
        a, b = g.message_edge(m)
        chi = psi.bond_dim(a, b)
        M = rng.standard_normal((chi, chi)).astype(np.float32).astype(np.float64)
        out[(a, b)] = M + M.T if symmetric else M
    return out


@pytest.mark.parametrize("bonds", BONDS, ids=lambda b: "x".join(map(str, b)))
@pytest.mark.parametrize("mode", ["parallel", "parallel-f32", "nonsymmetric", "sequential"])
def test_one_sweep_matches_oracle(bonds, mode):
    f32 = mode == "parallel-f32"
    rng = np.random.default_rng(71)
    g, psi = star(bonds, rng, np.float32 if f32 else np.float64, d=3 if len(bonds) == 2 else 2)
    msgs = random_messages(rng, g, psi, symmetric=mode != "nonsymmetric")
    bpc = itnbp.initialize_cache(psi, messages=msgs)
    schedule = "sequential" if mode == "sequential" else "parallel"
    itnbp.update_(bpc, maxiter=1, edge_sequence=None if schedule == "sequential" else "parallel",
                  precision="f32" if f32 else "f64")
    assert ("[vertex" in bpc.last_update["path"]) == (mode in ("parallel", "parallel-f32"))
    og, opsi = oracle_graph(g), oracle_psi(psi)
    ref, _, md, _ = O.bp_update(og, opsi, to_index(g, msgs), maxiter=1, tol=0.0, schedule=schedule)
    got = to_index(g, bpc.messages())
    tol = 2e-6 if f32 else 1e-12
    for e in ref:
        assert np.linalg.norm(got[e] - ref[e]) <= tol * np.linalg.norm(ref[e]), (bonds, e)
    assert bpc.last_update["mean_diff"] == pytest.approx(md, rel=1e-4 if f32 else 1e-10, abs=1e-6 if f32 else 1e-12)
