"""Accuracy of Theta's SVD, in each of its kernels: a pair of sites whose environments
are identities, so that the new second site is V sqrt(S) of Theta, its columns
orthogonal as far as the SVD makes them so.  Inner products that the Jacobi sweeps leave
behind turn the kept singular vectors towards each other, amplified by the gaps of the
singular values in the gauged tensors.

Bound: eps sqrt(N), the threshold of a rotation, and as much again for the product
that rebuilds the site (measured: 0.3 of it at most).  With a threshold of 8 eps
sqrt(N) they come to 7 to 8 eps sqrt(N)."""
import numpy as np
import pytest

import itnbp
from test_gpu_apply_split import random_gates

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps
# gate bond before the call, other bonds of each side, maxdim; N = 2 min(E, 2 chi_b)
PAIRS = {
    "lds16": (4, (4, 4), 8), "lds32": (8, (8, 8), 16),
    "split32": (8, (30,), 16), "split64": (16, (32,), 32), "split64tall": (16, (16, 16, 16), 16),
    "split128": (32, (9, 16), 32), "split128all": (32, (9, 16), 64),
}


@pytest.mark.parametrize("name", sorted(PAIRS))
def test_kept_singular_vectors_are_orthogonal(name):
    chib, ext, maxdim = PAIRS[name]
    edges = [(0, 1)] + [(v, 2 + v * len(ext) + i) for v in (0, 1) for i in range(len(ext))]
    g = itnbp.NamedGraph(range(2 + 2 * len(ext)), edges)
    bound = 2 * EPS * np.sqrt(2 * min(int(np.prod(ext)), 2 * chib))
    for seed in range(4):
        rng = np.random.default_rng(seed)
        psi = itnbp.random_tensornetwork(rng, np.float64, g, link_space=[chib] + 2 * list(ext))
        msgs = {g.message_edge(m): np.eye(psi.bond_dim(*g.message_edge(m))) for m in range(2 * g.ne)}
        bpc = itnbp.initialize_cache(psi, messages=msgs)
        itnbp.apply_gates_(bpc, [itnbp.Gate(random_gates(rng, [(0, 1)], 2, 0.1)[0], (0, 1))], maxdim=maxdim,
                           normalize=False)
        t = np.moveaxis(bpc.tensornetwork()[1], g.axis(1, 0), -1)
        t = t.reshape(-1, maxdim).astype(np.longdouble)
        t /= np.sqrt((t * t).sum(0))
        assert np.abs(t.T @ t - np.eye(maxdim)).max() <= bound, seed
