"""Gates within the LDS limits (external bonds <= 8, Theta <= 32 x 32) where their
two kernels branch, against the CPU oracle: column counts at the 16-column tile,
sides at the tall/wide boundary and of every degree, rows past a multiple of the
16-row tile, dropped environment eigenvalues, bonds that grow; ill-conditioned and
rank-deficient sides against the state itself.

Tolerances: FP64 results to 1e-10 relative, the bar of the other gate tests; the
state to 1e-13 (products of n x n factors and E-row sums, ~sqrt(n) eps each, through
roots of messages of condition 3.4, rotations to eps sqrt(N); a few times their sum).
"""
import numpy as np
import pytest

import itnbp
from test_gpu_apply_split import positive_messages, random_gates, run_and_compare

pytestmark = pytest.mark.gpu

# (lattice, bond dimensions, physical dimension)
SHAPES = {
    "chi1": ((2, 2), (1, 1), 2),       # E = 1, n = 2
    "ragged": ((3, 3), (2, 8), 2),
    "chi8": ((3, 3), (8, 8), 2),       # the largest: E = 512, n = 16
    "boundary": ((3, 2), (4, 4), 2),   # corners E = 4 < n = 8, the others 16 > 8
    "wide": ((2, 1), (5, 5), 2),       # E = 1
    "scalar": ((3, 3), (3, 7), 1),     # d = 1: n = chi
    "qutrit": ((3, 2), (2, 3), 3),
    "ququart": ((3, 3), (2, 2), 4),
    "chain": ((5, 1), (6, 8), 2),      # E = 1 and 6 .. 8
}


@pytest.mark.parametrize("name", sorted(SHAPES))
def test_sides_match_oracle(name):
    dims, (lo, hi), d = SHAPES[name]
    rng = np.random.default_rng(71)
    g = itnbp.path_graph(dims[0]) if dims[1] == 1 else itnbp.named_grid(dims)
    link = [int(c) for c in rng.integers(lo, hi + 1, g.ne)]
    psi = itnbp.random_tensornetwork(rng, np.float64, g, link_space=link, phys_dim=d)
    msgs = positive_messages(rng, psi)
    for cls in itnbp.edge_coloring(g):
        run_and_compare(g, psi, msgs, cls, random_gates(rng, cls, d), maxdim=max(1, min(link) - 1))


def test_tall_scalar_bond_of_two_tiles_matches_oracle():
    """d = 1 with 20 columns: two 16-column tiles, E = 64 rows."""
    rng = np.random.default_rng(72)
    g = itnbp.named_grid((2, 3))
    link = [8] * g.ne
    bond = ((1, 2), (2, 2))
    link[[g.message_edge(2 * e) for e in range(g.ne)].index(bond)] = 20
    psi = itnbp.random_tensornetwork(rng, np.float64, g, link_space=link, phys_dim=1)
    msgs = positive_messages(rng, psi)
    run_and_compare(g, psi, msgs, [bond], [np.array([[1.3]])], maxdim=17)


def test_projector_and_growth_match_oracle():
    """Environments of rank 6 of 7 (P != 1 on every external bond); a bond grows
    from 5 to 9."""
    rng = np.random.default_rng(73)
    g = itnbp.named_grid((3, 3))
    bonds = [((2, 2), (2, 3)), ((1, 1), (2, 1))]
    edges = [g.message_edge(2 * e) for e in range(g.ne)]
    link = [5 if e in bonds else 7 for e in edges]
    psi = itnbp.random_tensornetwork(rng, np.float64, g, link_space=link)
    msgs = positive_messages(rng, psi, rank=0.9)
    run_and_compare(g, psi, msgs, bonds, random_gates(rng, bonds), maxdim=9)


@pytest.mark.parametrize("grade,rank", [(-4.5, None), (-8, None), (-12, None), (-16, None), (0, 3), (-9, 3)])
@pytest.mark.parametrize("chib", [3, 4, 8])  # E = 8 > n = 6 (the QR's further passes), E = n, E < n
def test_ill_conditioned_sides_keep_the_state(chib, grade, rank):
    """Singular values of a side down to 10^grade, mixed over its columns, or only
    `rank` of them: without truncation the gauged pair contracts to the gate times
    the old one."""
    rng = np.random.default_rng(74)
    g, chie, n = itnbp.path_graph(4), 8, 2 * chib
    psi = itnbp.random_tensornetwork(rng, np.float64, g, link_space=[chie, chib, chie])
    for v in (2, 3):
        k = min(n, chie)
        s = np.logspace(0, grade, k)
        if rank is not None:
            s[rank:] = 0.0
        A, B = (np.linalg.qr(rng.standard_normal((m, k)))[0] for m in (chie, n))
        t = ((A * s) @ B.T).reshape(chie, 2, chib)
        psi[v] = np.asfortranarray(t.transpose(1, 0, 2) if v == 2 else t.transpose(1, 2, 0))
    msgs = positive_messages(rng, psi)
    G = np.linalg.qr(rng.standard_normal((4, 4)))[0]
    bpc = itnbp.initialize_cache(psi, messages=msgs)
    itnbp.apply_gates_(bpc, [itnbp.Gate(G, (2, 3))], maxdim=4 * chib, normalize=False)
    new = bpc.tensornetwork()
    exact = np.einsum("xyst,seb,tbf->xeyf", G.reshape((2,) * 4, order="F"), psi[2], psi[3])
    got = np.einsum("xek,ykf->xeyf", new[2], new[3])
    assert np.linalg.norm(got - exact) <= 1e-13 * np.linalg.norm(exact)


def test_non_finite_gate_leaves_its_bond_alone():
    rng = np.random.default_rng(75)
    g = itnbp.path_graph(4)
    psi = itnbp.random_tensornetwork(rng, np.float64, g, link_space=4)
    psi[2] = psi[2].copy()
    psi[2][0, 0, 0] = np.nan
    bpc = itnbp.initialize_cache(psi, messages=positive_messages(rng, psi))
    with pytest.raises(itnbp.ITNBPError):
        itnbp.apply_gates_(bpc, [itnbp.Gate(np.eye(4), (1, 2)), itnbp.Gate(2 * np.eye(4), (3, 4))], maxdim=4)
    new = bpc.tensornetwork()
    for v in (1, 2):
        np.testing.assert_array_equal(new[v], psi[v])
    pair = lambda t: np.einsum("seb,tb->set", t[3], t[4])
    ref = 2 * pair(psi)
    got = pair(new)
    assert np.linalg.norm(got * (np.linalg.norm(ref) / np.linalg.norm(got)) - ref) <= 1e-12 * np.linalg.norm(ref)
