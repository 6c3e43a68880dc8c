"""The V-cycle's bilinear levels (tiles with halos, and the levels one workgroup
cycles) against the oracle's V-cycle, oracle/sem_mg.py: level sizes around the
tiles' and the workgroup's limits, periodic and Neumann sides, odd element counts
(a large last level), degrees whose applies need several launches."""
import numpy as np
import pytest

from oracle import sem_mg as omg
from oracle import sem_oracle as o

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def se():
    import semhip
    return semhip


# points, elements, periodic, boundary, nu, k, degree, degree_coarse
CASES = [
    (3, 4, 4, (False, False), "DDDD", 1.0, 1.0, 3, 8),
    (3, 33, 33, (False, False), "DDDD", 1.0, 0.0, 3, 8),      # one workgroup, full
    (3, 34, 33, (False, False), "DDDD", 1.0, 1.0, 3, 8),      # one tile row too many
    (3, 64, 64, (False, False), "DNDD", 0.7, 1.0, 3, 8),
    (3, 96, 40, (True, False), "NNDD", 1.0, 0.5, 3, 8),
    (3, 40, 64, (True, True), "NNNN", 1.0, 1.0, 3, 8),
    (2, 68, 36, (False, True), "DDDD", 1.0, 1.0, 2, 5),       # bilinear finest level
    (4, 47, 71, (False, False), "DDND", 1.0, 1.0, 3, 8),      # large last level
    (3, 53, 61, (False, True), "DDDD", 1.0, 0.0, 3, 20),      # its steps in three launches
    (3, 72, 72, (False, False), "DDDD", 1.0, 1.0, 9, 8),      # smoothing in several launches
    (3, 48, 48, (False, False), "DDDD", 1.0, 1.0, 7, 18),     # no one-workgroup levels
    (3, 80, 48, (False, False), "DDDD", 1.0, 1.0, 1, 1),
    (3, 700, 2, (False, False), "DDDD", 1.0, 1.0, 3, 8),      # long and thin
    (3, 1, 3, (True, False), "DDDD", 1.0, 1.0, 3, 8),
    (3, 2, 40, (True, True), "NNNN", 1.0, 1.0, 3, 8),
]


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("n,Ex,Ey,per,bc,nu,k,deg,degc", CASES)
def test_vcycle(se, n, Ex, Ey, per, bc, nu, k, deg, degc, prec):
    print(f"vcycle n={n} {Ex}x{Ey} {per} {bc} deg={deg},{degc} {prec}", flush=True)
    m = se.Mesh(n, n, Ex, Ey, per, se.deform_sinsin(0.1))
    mo = o.Mesh(n, n, Ex, Ey, per, o.deform_sinsin(0.1), dense_gs=False)
    op = se.SEMOperator(nu, k, m, se.generateMask(bc, m))
    P = se.MG(op, degree=deg, degree_coarse=degc, precision=prec)
    lm = [v[3] for v in P.levels()]
    Po = omg.MG(mo, nu, k, bc, omg.MGParams(degree=deg, degree_coarse=degc), lmax=lm)
    assert [v[:3] for v in P.levels()] == [(L.msh.nr, L.msh.Ex, L.msh.Ey) for L in Po.levels]
    rng = np.random.default_rng(n * 1000 + Ex)
    r = Po.levels[0].M * mo.gs(rng.standard_normal(mo.x.shape))
    z, zo = se.to_host(P(se.to_device(r))), Po(r)
    # FP64: the cycle's bound of the other multigrid tests. FP32: some 50 steps of a
    # few roundings (6e-8) each, taken ten times for the cancellation in residuals
    tol = 1e-10 if prec == "f64" else 1e-4
    assert np.abs(z - zo).max() <= tol * np.abs(zo).max()
