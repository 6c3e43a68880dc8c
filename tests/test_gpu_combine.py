"""The assembled right-hand side in one launch against the pass and the gather-scatter
that an output among the terms takes: the same bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def se():
    import os
    import sys
    sys.path.insert(0, os.path.join(os.path.dirname(__file__), "..", "spectralelements.jl_amd"))
    import semhip
    return semhip


# one element, rows of one block and of several with a remainder, two points (every node
# on an edge), orders that differ, periodic directions of one element and of many
@pytest.mark.parametrize("nr,ns,Ex,Ey,per,bc", [
    (2, 2, 1, 1, (False, False), "DDDD"), (2, 3, 70, 5, (True, True), "DNDD"),
    (8, 8, 1, 9, (True, False), "NNDN"), (8, 8, 32, 32, (False, False), "DDDD"),
    (10, 10, 13, 1, (False, True), "DDNN"), (17, 5, 16, 11, (True, False), None),
    (4, 20, 33, 7, (False, True), "NDND")])
@pytest.mark.parametrize("nterms", [1, 8])
def test_one_launch_same_bits(se, nr, ns, Ex, Ey, per, bc, nterms):
    import torch
    print(f"[gpu] combine {nr}x{ns} {Ex}x{Ey} {per} {bc} {nterms}", flush=True)
    m = se.Mesh(nr, ns, Ex, Ey, per, se.deform_sinsin(0.1))
    M = se.generateMask(bc, m) if bc else None
    rng = np.random.default_rng(11)
    xs = [se.to_device(rng.standard_normal((nr * Ex, ns * Ey))) for _ in range(nterms)]
    terms = [(float(rng.standard_normal()), x, q % 2 == 0) for q, x in enumerate(xs)]
    y = se.combine(m, terms, M=M, assemble=True)
    assert torch.equal(se.gatherScatter(se.combine(m, terms, M=M), m), y)
    last = xs[-1].clone()
    out = se.combine(m, terms, M=M, assemble=True, out=xs[-1])
    assert out.data_ptr() == xs[-1].data_ptr() and not torch.equal(out, last)
    assert torch.equal(out, y)
