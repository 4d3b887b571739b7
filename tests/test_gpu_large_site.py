"""Sites with every bond <= 16 whose tensor does not fit in LDS (passes over pairs of
bonds, k_vertex.hip): every degree, odd ones with their overlapping last pair, chunks
that end inside a run or span several, ragged tiles, all in FP64 and FP32 against the
CPU oracle: one star per case, one sweep from random symmetric messages, then a
second one (the eigenvectors of the first as seeds).

Tolerances, relative to each (normalised) message: FP64 1e-11, eigenvectors and
weighted sums at n eps ~ 1e-14 amplified by the cancellation of indefinite messages
(eigenvalues of either sign; at most ~1e3); FP32 arithmetic 2e-5 by the same factors.
"""
import numpy as np
import pytest

import itnbp
from helpers import oracle_graph, oracle_psi, to_index
from oracle import bp_oracle as O
from test_gpu_site import star

pytestmark = pytest.mark.gpu

# centre's bonds, physical dimension; more than 20480 (FP64) or 40960 (FP32) entries
CASES = [((16, 16, 16), 8), ((13, 15, 16), 8), ((16, 16, 16, 16), 2), ((13, 14, 15, 16), 2), ((16, 15, 9, 11), 3),
         ((1, 16, 16, 16), 8), ((16, 16, 1, 14), 8), ((8, 9, 10, 11, 7), 2), ((16, 3, 16, 2, 16), 4),
         ((7, 5, 6, 7, 6, 5), 2), ((2, 3, 16, 16, 16, 2), 2), ((12, 12, 12, 13), 2)]


def positive_messages(rng, g, psi):
    out = {}
    for m in range(2 * g.ne):
        a, b = g.message_edge(m)
        chi = psi.bond_dim(a, b)
        M = rng.standard_normal((chi, chi + 2)).astype(np.float32).astype(np.float64)
        out[(a, b)] = M @ M.T / chi
    return out


@pytest.mark.parametrize("bonds,d", CASES, ids=lambda b: "x".join(map(str, b)) if isinstance(b, tuple) else str(b))
@pytest.mark.parametrize("precision", ["f64", "f32"])
def test_two_sweeps_match_oracle(bonds, d, precision):
    f32 = precision == "f32"
    rng = np.random.default_rng(81)
    g, psi = star(bonds, rng, np.float32 if f32 else np.float64, d=2)
    t = rng.standard_normal((d,) + bonds) / np.sqrt(np.prod(bonds))
    psi = itnbp.ITensorNetwork(g, {v: t.astype(psi[1].dtype) if v == 0 else psi[v] for v in g.vertices})
    msgs = positive_messages(rng, g, psi)
    # an indefinite message: eigenvalues of either sign
    M = msgs[(1, 0)]
    msgs[(1, 0)] = M - 0.3 * np.trace(M) / len(M) * np.eye(len(M))
    bpc = itnbp.initialize_cache(psi, messages=msgs)
    og, opsi, cur = oracle_graph(g), oracle_psi(psi), to_index(g, msgs)
    for _ in range(2):
        itnbp.update_(bpc, maxiter=2, edge_sequence="parallel", precision=precision)
        assert "[vertex" in bpc.last_update["path"], bpc.last_update["path"]
        cur, _, _, _ = O.bp_update(og, opsi, cur, maxiter=2, tol=0.0, schedule="parallel")
        got = to_index(g, bpc.messages())
        for e in cur:
            err = np.linalg.norm(got[e] - cur[e]) / np.linalg.norm(cur[e])
            assert err <= (2e-5 if f32 else 1e-11), (e, err)
