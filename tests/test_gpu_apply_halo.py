"""The apply whose workgroups compute their neighbours' elements (small meshes, one
launch) and the two-row apply with strips of odd width: against the oracle at the
smallest meshes, and bit by bit against strips of one element row with a seam pass
(the SEM_AX_ROWS hook), the form before, up to past the switch between them."""
import numpy as np
import pytest

from oracle import sem_oracle as o

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def se():
    import semhip
    return semhip


# a workgroup writes two rows of 256 // (4 P) - 2 elements, or six
SMALL = [(P, Ex, Ey, per)
         for P in (2, 3, 5, 8, 11, 13, 14, 15, 16)
         for Ex, Ey, per in ((1, 1, (False, False)), (1, 2, (True, True)),
                             (2, 1, (True, True)), (5, 3, (True, False)),
                             (7, 4, (False, True)), (13, 9, (False, False)))]
LARGE = [(9, 20, 73, (False, False)), (9, 26, 130, (True, True)), (16, 32, 32, (True, False)),
          (16, 33, 32, (False, False)), (11, 47, 58, (True, False)), (5, 103, 77, (False, True)),
          (8, 64, 70, (True, True)), (15, 36, 33, (False, False)),
          (4, 113, 101, (True, True)), (6, 81, 85, (False, True)), (8, 80, 79, (False, False)),
          (7, 99, 102, (True, False)), (10, 62, 66, (False, False)), (12, 57, 61, (True, True))]


def _coefficients(rng, shape):
    return (0.7, 1.3), (1.0, 0.0), (1.0 + rng.random(shape), 0.5)


@pytest.mark.parametrize("P,Ex,Ey,per", SMALL)
def test_apply_matches_oracle(se, P, Ex, Ey, per):
    import torch
    print(f"apply P={P} {Ex}x{Ey} {per}", flush=True)
    m = se.Mesh(P, P, Ex, Ey, per, se.deform_sinsin(0.1))
    mo = o.Mesh(P, P, Ex, Ey, per, o.deform_sinsin(0.1), dense_gs=False)
    bc = "DNDD"
    M, Mo = se.generateMask(bc, m), o.generateMask(bc, mo)
    rng = np.random.default_rng(P * 10000 + Ex * 100 + Ey)
    u = rng.standard_normal(mo.x.shape)          # copies need not agree
    for nuv, k in _coefficients(rng, u.shape):
        ref = o.opLHS(u, nuv, k, mo, Mo)
        scale = np.abs(ref).max()
        got = se.to_host(se.SEMOperator(nuv, k, m, M)(se.to_device(u)))
        # the element operators' bound of the parity tests
        assert np.abs(got - ref).max() <= 1e-12 * scale
        op32 = se.SEMOperator(nuv, k, m, M, precision="f32")
        g32 = op32(se.to_device(u.astype(np.float32), dtype=torch.float32))
        assert np.abs(se.to_host(g32) - ref).max() <= 2e-5 * scale


@pytest.mark.parametrize("P,Ex,Ey,per", SMALL + LARGE)
def test_apply_same_bits_as_strips(se, monkeypatch, P, Ex, Ey, per):
    import torch
    print(f"apply bits P={P} {Ex}x{Ey} {per}", flush=True)
    m = se.Mesh(P, P, Ex, Ey, per, se.deform_sinsin(0.1))
    M = se.generateMask("DNDD", m)
    rng = np.random.default_rng(P * 10000 + Ex * 100 + Ey)
    u = rng.standard_normal((P * Ex, P * Ey))
    for nuv, k in _coefficients(rng, u.shape):
        for prec, dt in (("f64", torch.float64), ("f32", torch.float32)):
            ud = se.to_device(u).to(dt)
            op = se.SEMOperator(nuv, k, m, M, precision=prec)
            with monkeypatch.context() as c:
                c.setenv("SEM_AX_ROWS", "1")
                strips = se.SEMOperator(nuv, k, m, M, precision=prec)
            assert torch.equal(op(ud), strips(ud))
