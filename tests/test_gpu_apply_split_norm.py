"""normalize = True on bonds that grow in the split gate pipeline past one pass of its
rebuild (64 // d bond values, so 63 or 60 columns at d = 3, 5, 6 and 7), both sides
tall, against the CPU oracle.  maxdim puts the last kept bond value before, at and
behind the end of a pass.

Tolerance: FP64 results to 1e-10 relative, the bar of the other gate tests; a column
counted twice in the norm is off by about half its weight, 1e-3 and more here."""
import numpy as np
import pytest

import itnbp
from helpers import oracle_graph, oracle_psi, to_index
from oracle import bp_oracle as O
from test_gpu_apply_split import positive_messages, random_gates

pytestmark = pytest.mark.gpu

# d, external bond, gate bond before the call, maxdim
GROWN = [
    (2, 20, 9, 32), (2, 20, 9, 36),  # 64 columns a pass, none left over
    (3, 30, 8, 21), (3, 30, 8, 22), (3, 30, 8, 32), (3, 30, 8, 43),
    (5, 32, 5, 12), (5, 32, 5, 13), (5, 32, 5, 25),
    (6, 20, 3, 10), (6, 20, 3, 11), (6, 20, 3, 18),
    (7, 20, 2, 9), (7, 20, 2, 10), (7, 20, 2, 14),
]


@pytest.mark.parametrize("d,ext,chib,maxdim", GROWN)
def test_grown_bond_is_normalised(d, ext, chib, maxdim):
    rng = np.random.default_rng(67)
    g = itnbp.path_graph(4)
    psi = itnbp.random_tensornetwork(rng, np.float64, g, link_space=[ext, chib, ext], phys_dim=d)
    msgs = positive_messages(rng, psi)
    gate = random_gates(rng, [(2, 3)], d)[0]
    bpc = itnbp.initialize_cache(psi, messages=msgs)
    itnbp.apply_gates_(bpc, [itnbp.Gate(gate, (2, 3))], maxdim=maxdim, normalize=True)
    new = bpc.tensornetwork()
    ref, s, _ = O.apply_gate(gate, oracle_graph(g), oracle_psi(psi), to_index(g, msgs), g.index[2], g.index[3],
                             maxdim=maxdim, normalize=True)
    assert len(s) == maxdim
    for x in (2, 3):
        assert np.linalg.norm(new[x]) == pytest.approx(1.0, rel=1e-12)
        assert np.linalg.norm(new[x] - ref[g.index[x]]) <= 1e-10
