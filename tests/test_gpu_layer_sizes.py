"""The two-layer message kernel on both sides of its LDS limit (2 D + one open pair
of elements within 160 KB) and at the smallest sites, one Jacobi sweep against the
two-layer oracle from random messages, and a partial sequence, whose other messages
keep their values.

Tolerance, relative to each normalised message: 1e-12, sums of at most 5e4 terms of
rounding 1e-16.
"""
import numpy as np
import pytest

import itnbp
from helpers import oracle_graph, to_index
from oracle import layer_oracle as LO
from test_gpu_layer import as_list

pytestmark = pytest.mark.gpu


# bonds of the star's centre in the ket and the bra, complex: D = d prod(max) elements
CASES = [((1,), (1,), False), ((1, 2), (3, 1), True), ((5, 5, 5, 5), (5, 5, 5, 5), True), ((7, 6, 8, 9), (6, 8, 7, 9), False),
         ((7, 7, 7, 7), (7, 7, 7, 7), True), ((9, 9, 9, 9), (9, 9, 9, 9), False), ((11, 12, 11, 12), (12, 11, 12, 11), True)]


def star_state(rng, g, dims, cplx):
    t = {}
    for v in g.vertices:
        shape = (2,) + (tuple(dims) if v == 0 else (dims[v - 1],))
        a = rng.standard_normal(shape)
        t[v] = 0.5 * (a + 1j * rng.standard_normal(shape) if cplx else a)
    return itnbp.ITensorNetwork(g, t)


@pytest.mark.parametrize("kd,bd,cplx", CASES, ids=lambda x: "x".join(map(str, x)) if isinstance(x, tuple) else str(x))
def test_one_sweep_and_a_partial_sequence(kd, bd, cplx):
    rng = np.random.default_rng(91)
    g = itnbp.NamedGraph(list(range(len(kd) + 1)), [(0, i + 1) for i in range(len(kd))])
    ket, bra = star_state(rng, g, kd, cplx), star_state(rng, g, bd, cplx)
    msgs = {}
    for m in range(2 * g.ne):
        e = g.message_edge(m)
        i = max(e) - 1
        M = rng.standard_normal((kd[i], bd[i]))
        msgs[e] = M + 1j * rng.standard_normal(M.shape) if cplx else M
    c = itnbp.inner_network_cache(bra, ket, messages=msgs)
    before = c.messages()
    seq = [(0, 1)]
    c.update_(maxiter=2, edge_sequence=seq)
    part = c.messages()
    for e in before:
        if e not in seq:
            np.testing.assert_array_equal(part[e], before[e])
    og = oracle_graph(g)
    cur = {k: v for k, v in to_index(g, part).items()}
    ref, _, _ = LO.bp_update2(og, as_list(ket), as_list(bra), cur, maxiter=1, schedule="parallel")
    c.update_(maxiter=1, edge_sequence="parallel")
    got = to_index(g, c.messages())
    for e in ref:
        err = np.linalg.norm(got[e] - ref[e]) / np.linalg.norm(ref[e])
        assert err <= 1e-12, (e, err)


def test_a_non_finite_message_is_an_error():
    """Also one that leaves the tree before the last sweep of a fixed number."""
    rng = np.random.default_rng(92)
    g = itnbp.path_graph(4)
    t = {v: rng.standard_normal((2,) + (3,) * g.degree(v)) for v in g.vertices}
    psi = itnbp.ITensorNetwork(g, t)
    c = itnbp.inner_network_cache(psi, psi, messages="identity")
    c.set_message_((2, 3), np.full((3, 3), np.nan))
    with pytest.raises(itnbp.ITNBPError):
        c.update_(maxiter=6, edge_sequence="parallel")
