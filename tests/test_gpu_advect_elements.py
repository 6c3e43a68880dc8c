"""The dealiased convective term on both sides of the line in the elements between its two
kernels (an element a workgroup up to it, several beyond), for every order: the largest mesh
before it and ones beyond it whose last workgroup is not full; and the largest and
smallest counts of nodes a phase takes."""
import numpy as np
import pytest

from oracle import sem_oracle as o

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def se():
    import semhip

    return semhip


CASES = [(7, 7, 1280, 1), (7, 7, 1, 1281), (8, 12, 40, 32), (8, 12, 61, 21), (9, 13, 32, 40),
         (9, 13, 1283, 1), (10, 15, 40, 32), (10, 15, 3, 428), (11, 16, 32, 32), (11, 16, 25, 41),
         (12, 18, 32, 32), (12, 18, 1027, 1), (13, 19, 1, 1024), (13, 19, 25, 41), (14, 21, 32, 32),
         (14, 21, 79, 13), (15, 22, 24, 32), (15, 22, 17, 47), (16, 16, 16, 32), (16, 16, 27, 19),
         (16, 16, 25, 41), (16, 24, 16, 32), (16, 24, 27, 19), (2, 24, 32, 32), (2, 24, 25, 41),
         (6, 8, 1, 1), (3, 16, 3, 1), (13, 23, 1, 2), (4, 24, 41, 25)]


@pytest.mark.parametrize("p,pd,Ex,Ey", CASES)
@pytest.mark.parametrize("per", [(False, False), (True, False)])
def test_advect_at_the_line(se, p, pd, Ex, Ey, per):
    print(f"advect p={p} pd={pd} {Ex}x{Ey}", flush=True)
    mV, moV = se.Mesh(p, p, Ex, Ey, per, se.deform_sinsin(0.1)), o.Mesh(
        p, p, Ex, Ey, per, o.deform_sinsin(0.1), dense_gs=False)
    mD, moD = se.Mesh(pd, pd, Ex, Ey, per, se.deform_sinsin(0.1)), o.Mesh(
        pd, pd, Ex, Ey, per, o.deform_sinsin(0.1), dense_gs=False)
    # the reference on the library's own metric terms: those of thin elements (a mesh of
    # 1283x1) hold 12 digits only, as differences of coordinates
    for f in ("rx", "ry", "sx", "sy"):
        setattr(moV, f, se.to_host(getattr(mV, f)))
    moD.B = se.to_host(mD.B)
    rng = np.random.default_rng(p * 100 + pd)
    T, vx, vy = (rng.standard_normal(moV.x.shape) for _ in range(3))
    for ref, tr in ((o.advect(T, vx, vy, moV, moD), False),
                    (o.advect_transpose(T, vx, vy, moV, moD), True)):
        got = se.advect(T, vx, vy, mV, mD, transpose=tr)
        # (the other advect tests' bound; in 1e4 to 3e5 values)
        assert np.max(np.abs(got - ref)) <= 1e-12 * np.max(np.abs(ref))
