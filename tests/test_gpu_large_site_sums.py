"""FP32 messages out of sites too large for LDS: the Gram sums over a site carry at
most 64 fibres in FP32 before they go to FP64, however the site is cut into chunks.

512 equal sites with six bonds of 11, 1, 2, 3, 16 and 16: the second pair of bonds is
cut into 512 chunks, of 32 and of 1 of the 33 entries before it in turn, and every
fourth chunk is one workgroup's, so half the workgroups get short chunks alone.  The
site has its weight there, as one fibre of size 1 with 255 small ones behind it, whose
squares are 0.9 of half an ulp of 1: a sum of them in FP32 that starts at 1 leaves every
one out, 127 of them in a workgroup, and the elements (1/2 after the division by the
norm) are off by 3/8 * 127 * 0.9 * 2^-24 = 2.5e-6.

Bound: the products are exact or round the small squares alone, a group of 64 fibres
(four entries here) that starts at 1 loses three small squares, 6e-8, and the output
rounds to 2^-25: 5e-7 is three times their sum."""
import numpy as np
import pytest

import itnbp

pytestmark = pytest.mark.gpu

NSITE, DIMS = 512, (11, 1, 2, 3, 16, 16)


def centre():
    c = np.zeros((3,) + DIMS, dtype=np.float32, order="F")
    small = np.sqrt(0.9 * 2.0**-24)
    for i in range(256):
        c[2, 10, 0, 0, 0, i % 16, i // 16] = 1.0 if i == 0 else small
    c[2, 10, 0, 1, 0, 0, 0] = 1.0   # the other element of the message on that bond
    return c


def test_fp32_sums_are_bounded():
    """Stars of such a site and six leaves, every message the identity before the sweep."""
    c = centre()
    k = len(DIMS)
    vertices = [(s, j) for s in range(NSITE) for j in range(k + 1)]
    edges = [((s, 0), (s, j)) for s in range(NSITE) for j in range(1, k + 1)]
    g = itnbp.NamedGraph(vertices, edges)
    assert [g.axis((0, 0), (0, j)) for j in range(1, k + 1)] == list(range(1, k + 1))
    tensors, msgs = {}, {}
    for s in range(NSITE):
        tensors[(s, 0)] = c
        for j in range(1, k + 1):
            n = DIMS[j - 1]
            tensors[(s, j)] = np.ones((1, n), dtype=np.float32, order="F")
            msgs[((s, 0), (s, j))] = np.eye(n)
            msgs[((s, j), (s, 0))] = np.eye(n)
    psi = itnbp.ITensorNetwork(g, tensors)
    bpc = itnbp.initialize_cache(psi, messages=msgs)
    itnbp.update_(bpc, maxiter=1, edge_sequence="parallel", precision="f32")
    got = bpc.messages()[((0, 0), (0, 3))]
    x = c.astype(np.float64)
    ref = np.einsum("sabpqef,sabrqef->pr", x, x)
    ref /= np.linalg.norm(ref)
    assert np.abs(got - ref).max() <= 5e-7
