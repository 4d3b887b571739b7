"""The split gate pipeline (bonds past the LDS kernel's limits) where its kernels
branch, against the CPU oracle: ragged bonds (chunks of rows, 16-column tiles and
fibre groups with remainders), sides at the tall/wide boundary and of every
degree, environments whose truncation drops eigenvalues (the projector pass),
graded sides (the eigendecomposition instead of the Cholesky factor), bonds that
grow, odd singular-value problems, and a non-finite gate among good ones.

Tolerances: FP64 results to 1e-10 relative, the bar of the other gate tests.
Graded sides (columns down to 1e-6 of the largest): the factors reproduce X to
~eps ||X||, so a singular value s_k carries eps s_0 / s_k <= 1e-16 * 1e6 * n,
about 1e-8, and the rebuilt columns, weighted by sqrt(s_k), stay below 1e-9.
"""
import numpy as np
import pytest

import itnbp
from helpers import oracle_graph, oracle_psi, to_index
from oracle import bp_oracle as O

pytestmark = pytest.mark.gpu


def run_and_compare(g, psi, msgs, bonds, gates, maxdim, tol=1e-10, stol=1e-10, cutoff=None):
    bpc = itnbp.initialize_cache(psi, messages=msgs)
    og, opsi = oracle_graph(g), oracle_psi(psi)
    omsgs = to_index(g, msgs)
    svals = []
    errs = itnbp.apply_gates_(bpc, [itnbp.Gate(G, b) for G, b in zip(gates, bonds)], maxdim=maxdim, cutoff=cutoff,
                              normalize=True,
                              callback=lambda singular_values, truncation_error: svals.append(singular_values))
    new = bpc.tensornetwork()
    for i, ((u, v), G) in enumerate(zip(bonds, gates)):
        ref, s_ref, err_ref = O.apply_gate(G, og, opsi, omsgs, g.index[u], g.index[v], maxdim=maxdim, cutoff=cutoff,
                                           normalize=True)
        assert new.bond_dim(u, v) == len(s_ref), (u, v)
        np.testing.assert_allclose(svals[i], s_ref, rtol=stol, atol=1e-13 * s_ref[0])
        for x in (u, v):
            r = ref[g.index[x]]
            assert new[x].shape == r.shape
            rel = np.linalg.norm(new[x] - r) / np.linalg.norm(r)
            assert rel <= tol, (u, v, x, rel)
        assert errs[i] == pytest.approx(err_ref, rel=1e-8, abs=1e-15)


def random_gates(rng, bonds, d=2, t=0.3):
    out = []
    for _ in bonds:
        H = rng.standard_normal((d * d, d * d))
        out.append(O.expm_sym(0.5 * (H + H.T), -t))
    return out


def positive_messages(rng, psi, rank=None):
    """Random positive messages, well conditioned, of full or given rank."""
    g = psi.graph
    out = {}
    for m in range(2 * g.ne):
        a, b = g.message_edge(m)
        chi = psi.bond_dim(a, b)
        Q = np.linalg.qr(rng.standard_normal((chi, chi)))[0]
        w = rng.uniform(0.3, 1.0, chi)
        if rank is not None:
            w[max(1, int(rank * chi)):] = 0.0
        M = (Q * w) @ Q.T
        out[(a, b)] = 0.5 * (M + M.T) / np.linalg.norm(M)
    return out


# (lattice, bond dimensions, physical dimension): E, n and the tiles at their edges
SHAPES = {
    "ragged": ((3, 3), (9, 14), 2),
    "boundary": ((3, 2), (16, 16), 2),   # corners E = 16 < n = 32, the others E = 256
    "chi17": ((3, 2), (17, 17), 2),      # one past a tile, n = 34, an odd count of row chunks
    "chi31": ((2, 2), (31, 31), 2),      # E = 31 <= n on every site
    "qutrit": ((3, 2), (9, 11), 3),      # Theta up to 99 x 99
    "chain": ((5, 1), (10, 20), 2),      # degrees 1 and 2, E = 1 at the ends
}


@pytest.mark.parametrize("name", sorted(SHAPES))
def test_ragged_sides_match_oracle(name):
    dims, (lo, hi), d = SHAPES[name]
    rng = np.random.default_rng(61)
    g = itnbp.path_graph(dims[0]) if name == "chain" else itnbp.named_grid(dims)
    link = [int(c) for c in rng.integers(lo, hi + 1, g.ne)]
    psi = itnbp.random_tensornetwork(rng, np.float64, g, link_space=link, phys_dim=d)
    msgs = positive_messages(rng, psi)
    for cls in itnbp.edge_coloring(g):
        run_and_compare(g, psi, msgs, cls, random_gates(rng, cls, d), maxdim=min(link) - 1)


def test_projector_and_growth_match_oracle():
    """Environments of rank 8 of 9 (P != 1 on every external bond), bonds growing
    from 9 to 13 (at most the corner's rank of Theta, 16: kept zeros would be noise
    on both sides)."""
    rng = np.random.default_rng(62)
    g = itnbp.named_grid((3, 3))
    psi = itnbp.random_tensornetwork(rng, np.float64, g, link_space=9)
    msgs = positive_messages(rng, psi, rank=0.9)
    bonds = [((2, 2), (2, 3)), ((1, 1), (2, 1))]
    run_and_compare(g, psi, msgs, bonds, random_gates(rng, bonds), maxdim=13)


def test_graded_sides_match_oracle():
    rng = np.random.default_rng(63)
    g = itnbp.named_grid((3, 3))
    psi = itnbp.random_tensornetwork(rng, np.float64, g, link_space=12)
    bond = ((2, 2), (2, 3))
    t = psi[(2, 2)]
    shape = [1] * t.ndim
    shape[g.axis(*bond)] = 12
    psi[(2, 2)] = t * np.logspace(0, -6, 12).reshape(shape)
    run_and_compare(g, psi, positive_messages(rng, psi), [bond], random_gates(rng, [bond]), maxdim=12, tol=1e-9,
                    stol=1e-7)


def test_cutoff_and_a_non_finite_gate():
    """A cutoff cuts the bond; a NaN in one pair leaves its tensors alone and the
    other gate of the call is applied."""
    rng = np.random.default_rng(64)
    g = itnbp.named_grid((4, 2))
    psi = itnbp.random_tensornetwork(rng, np.float64, g, link_space=10)
    msgs = positive_messages(rng, psi)
    bonds = [((1, 1), (1, 2)), ((3, 1), (3, 2))]
    gates = random_gates(rng, bonds)
    run_and_compare(g, psi, msgs, bonds, gates, maxdim=None, cutoff=5e-2)
    bad = psi.copy()
    bad[(3, 1)].flat[7] = np.nan
    bpc = itnbp.initialize_cache(bad, messages=msgs)
    with pytest.raises(itnbp.ITNBPError) as e:
        itnbp.apply_gates_(bpc, [itnbp.Gate(G, b) for G, b in zip(gates, bonds)], maxdim=10, normalize=True)
    assert e.value.code == itnbp._lib.ERR_NONFINITE
    new = bpc.tensornetwork()
    for x in bonds[1]:
        np.testing.assert_array_equal(new[x], bad[x])
    ref, _, _ = O.apply_gate(gates[0], oracle_graph(g), oracle_psi(psi), to_index(g, msgs), g.index[bonds[0][0]],
                             g.index[bonds[0][1]], maxdim=10, normalize=True)
    for x in bonds[0]:
        np.testing.assert_allclose(new[x], ref[g.index[x]], atol=1e-10)


@pytest.mark.parametrize("chi", [15, 16, 17, 31])  # Theta 30, 32 (one kernel), 34 and 62 (the next)
def test_powers_of_two_change_no_bits(chi):
    """Theta is scaled to order 1 by a power of two before its SVD: a site tensor
    times 2^+-300 gives the same gauged tensors bit for bit, singular values and
    all (the norms divide it out again, every step before is homogeneous)."""
    rng = np.random.default_rng(65)
    g = itnbp.path_graph(3)
    psi = itnbp.random_tensornetwork(rng, np.float64, g, link_space=chi)
    msgs = positive_messages(rng, psi)
    bond = (2, 3)
    gate = random_gates(rng, [bond])[0]
    runs = []
    for p in (0, 300, -300):
        q = psi.copy()
        q[2] = np.ldexp(psi[2], p)
        bpc = itnbp.initialize_cache(q, messages=msgs)
        sv = []
        errs = itnbp.apply_gates_(bpc, [itnbp.Gate(gate, bond)], maxdim=chi, normalize=True,
                                  callback=lambda singular_values, truncation_error: sv.append(singular_values))
        new = bpc.tensornetwork()
        runs.append((np.ldexp(sv[0], -p), new[2], new[3], errs[0]))
    for r in runs[1:]:
        for x, y in zip(r, runs[0]):
            np.testing.assert_array_equal(x, y)


@pytest.mark.parametrize("chie,chib,rank,gate", [(32, 16, 5, "full"), (24, 16, 5, "full"), (32, 10, 5, "full"),
                                                  (32, 16, None, "projector"), (32, 10, None, "projector")])
def test_rank_deficient_pairs_keep_the_state(chie, chib, rank, gate):
    """Without truncation the gauged pair contracts to the gate times the old one,
    also where Theta has fewer non-zero singular values than the bond may keep: a
    side of low rank (wide: E <= n, tall: E = 32 > n = 20), whose kept rank is the
    rank's bound, or a gate that halves Theta's rank, whose bond keeps noise
    values.  Bound: products of n x n factors and E-row sums, ~sqrt(n) eps each,
    and rotations to eps sqrt(N): 1e-13 is a few times their sum."""
    rng = np.random.default_rng(66)
    g, n = itnbp.path_graph(4), 2 * chib
    psi = itnbp.random_tensornetwork(rng, np.float64, g, link_space=[chie, chib, chie])
    if rank is not None:
        for v in (2, 3):
            t = (rng.standard_normal((chie, rank)) @ rng.standard_normal((rank, n))).reshape(chie, 2, chib)
            psi[v] = np.asfortranarray(t.transpose(1, 0, 2) if v == 2 else t.transpose(1, 2, 0))
    msgs = positive_messages(rng, psi)
    Q = np.linalg.qr(rng.standard_normal((4, 4)))[0]
    G = Q if gate == "full" else np.diag([1.0, 0.0, 0.0, 0.0])
    bpc = itnbp.initialize_cache(psi, messages=msgs)
    sv = []
    itnbp.apply_gates_(bpc, [itnbp.Gate(G, (2, 3))], maxdim=2 * n, normalize=False,
                       callback=lambda singular_values, truncation_error: sv.append(singular_values))
    new = bpc.tensornetwork()
    exact = np.einsum("xyst,seb,tbf->xeyf", G.reshape((2,) * 4, order="F"), psi[2], psi[3])
    got = np.einsum("xek,ykf->xeyf", new[2], new[3])
    assert np.linalg.norm(got - exact) <= 1e-13 * np.linalg.norm(exact)
    if rank is not None:
        assert len(sv[0]) == 2 * rank
