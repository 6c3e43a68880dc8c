"""The dealiased convective term (advect.jl:45-64) and its transpose at the edges
of the kernel's work split: element counts around a workgroup's share, fewer and
more dealiasing nodes than nodes, the smallest and largest orders."""
import numpy as np
import pytest

from oracle import sem_oracle as o

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def se():
    import semhip

    return semhip


# p, pd, Ex, Ey: a workgroup takes 128/max(p, pd) elements at most
CASES = [
    (2, 2, 1, 1), (2, 3, 9, 5), (2, 24, 3, 4), (3, 5, 25, 1), (4, 6, 1, 22),
    (5, 8, 16, 1), (6, 9, 15, 1), (7, 4, 6, 3), (8, 12, 10, 2), (8, 12, 5, 7),
    (9, 14, 9, 1), (10, 15, 3, 3), (11, 17, 5, 3), (12, 18, 7, 2), (13, 20, 4, 3),
    (14, 21, 1, 1), (15, 23, 3, 2), (16, 16, 8, 3), (16, 24, 3, 3), (16, 24, 1, 1),
]


@pytest.mark.parametrize("p,pd,Ex,Ey", CASES)
def test_advect_and_transpose(se, p, pd, Ex, Ey):
    print(f"advect p={p} pd={pd} {Ex}x{Ey}", flush=True)
    # a deformed mesh: every metric term is nonzero
    mV, moV = (c.Mesh(p, p, Ex, Ey, (False, False), c.deform_sinsin(0.1)) for c in (se, o))
    mD, moD = (c.Mesh(pd, pd, Ex, Ey, (False, False), c.deform_sinsin(0.1)) for c in (se, o))
    rng = np.random.default_rng(p * 100 + pd)
    T, vx, vy = (rng.standard_normal(moV.x.shape) for _ in range(3))
    for ref, tr in ((o.advect(T, vx, vy, moV, moD), False),
                    (o.advect_transpose(T, vx, vy, moV, moD), True)):
        got = se.advect(T, vx, vy, mV, mD, transpose=tr)
        # sums of at most 4*16 + 2*24 terms a value, growth by D below p^2: 1e-12
        # of the largest value, the bound of the library's other element operators
        assert np.max(np.abs(got - ref)) <= 1e-12 * np.max(np.abs(ref))
