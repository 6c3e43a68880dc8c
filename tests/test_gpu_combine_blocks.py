"""The assembled right-hand side at widths of the field that take each width of a block, with
remainders, and on large fields of few points a direction, where it takes two launches with
many terms: the bits of the pass and the gather-scatter."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def se():
    import semhip
    return semhip


@pytest.mark.parametrize("nr,ns,Ex,Ey,nterms", [
    (4, 4, 2, 50, 3), (3, 4, 3, 41, 3), (5, 3, 5, 30, 4), (8, 8, 4, 41, 5), (11, 11, 3, 17, 8),
    (9, 9, 15, 5, 3), (8, 8, 19, 31, 5), (8, 8, 150, 3, 8), (7, 5, 61, 7, 3),
    (2, 2, 300, 301, 7), (2, 2, 300, 301, 6), (3, 3, 201, 200, 8), (2, 2, 200, 200, 8)])
def test_same_bits(se, nr, ns, Ex, Ey, nterms):
    import torch
    print(f"combine {nr}x{ns} {Ex}x{Ey} {nterms}", flush=True)
    m = se.Mesh(nr, ns, Ex, Ey, (True, False), se.deform_sinsin(0.1))
    M = se.generateMask("NNDN", m)
    rng = np.random.default_rng(nr * Ex + Ey)
    terms = [(float(rng.standard_normal()), se.to_device(rng.standard_normal((nr * Ex, ns * Ey))),
              q % 2 == 0) for q in range(nterms)]
    y = se.combine(m, terms, M=M, assemble=True)
    assert torch.equal(se.gatherScatter(se.combine(m, terms, M=M), m), y)
    # the terms one after the other, on the host
    B = se.to_host(m.B)
    ref = sum(c * (B * se.to_host(x) if w else se.to_host(x)) for c, x, w in terms)
    got = se.to_host(se.combine(m, terms))
    scale = sum(abs(c) * np.abs(se.to_host(x)).max() for c, x, _ in terms)
    assert np.abs(got - ref).max() <= 16 * 2.3e-16 * scale   # (two roundings a term)
