"""The element operator on rows held in registers (nr != ns or more than 16 points,
rows of at most 16, the longer ones only with many elements) against the oracle: the
shortest and longest rows, the first that take the other kernel, many and few rows per
element, remainders of a workgroup."""
import numpy as np
import pytest

from oracle import sem_oracle as o

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def se():
    import semhip
    return semhip


CASES = [(3, 2, 11, 9), (2, 3, 13, 11), (2, 18, 7, 5), (18, 2, 5, 6), (17, 17, 3, 2), (18, 18, 2, 2),
         (4, 19, 3, 2), (19, 4, 3, 2), (5, 17, 1, 1), (60, 3, 2, 3), (64, 8, 1, 1), (64, 17, 1, 2), (7, 12, 37, 1),
         (9, 16, 1, 29), (12, 9, 7, 3), (6, 5, 43, 2), (16, 15, 4, 5), (11, 10, 23, 2),
         (13, 14, 64, 57), (3, 16, 65, 64), (4, 15, 61, 63), (3, 12, 55, 56),
         (2, 9, 48, 49), (5, 11, 53, 54), (3, 13, 58, 58), (4, 10, 51, 51), (13, 14, 5, 4), (8, 6, 32, 1), (10, 13, 6, 5), (8, 11, 4, 9), (9, 4, 29, 1), (8, 7, 8, 5)]


@pytest.mark.parametrize("nr,ns,Ex,Ey", CASES)
def test_operator(se, nr, ns, Ex, Ey):
    print(f"rows {nr}x{ns} {Ex}x{Ey}", flush=True)
    m = se.Mesh(nr, ns, Ex, Ey, (True, False), se.deform_sinsin(0.1))
    mo = o.Mesh(nr, ns, Ex, Ey, (True, False), o.deform_sinsin(0.1), dense_gs=False)
    rng = np.random.default_rng(nr * 100 + ns)
    u = rng.standard_normal(mo.x.shape)
    nu, k = 1.0 + rng.random(mo.x.shape), 0.5 + rng.random(mo.x.shape)
    # the mesh's own factors, so that only the operator is compared: sums of nr + ns
    # products twice, entries of D up to its row count squared / 4: below 1e-12 of
    # the largest value
    for name in ("G11", "G12", "G22", "B"):
        setattr(mo, name, se.to_host(m.field(name)))
    ud = se.to_device(u)
    for a, b in ((0.8, 1.3), (1.0, 0.0), (nu, 0.7), (nu, k), (1.1, k)):
        ref = o.hlmz(u, a, b, mo)
        assert np.abs(se.to_host(se.hlmz(ud, a, b, m)) - ref).max() <= 1e-12 * np.abs(ref).max()
    v = ud.clone()
    se.hlmz(v, nu, 0.7, m, out=v)          # in place
    import torch
    assert torch.equal(v, se.hlmz(ud, nu, 0.7, m))
