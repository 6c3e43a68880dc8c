"""The resident PCG's forms of exchange: all workgroups on one XCD (up to 32), sums by
XCD first (more than 120), flat in between, and each of the first two told that its
workgroups are not where it expects them (SEM_PCG_RESIDENT=3 at creation), which has
to fall back to the flat one. Four iterations against the launches (=0) from the same
operator: the sums' order is all that differs, 1e-12 (FP32: 1e-5), the bounds of the
other resident tests; on one XCD the fallback adds in the same order, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def se():
    import semhip
    return semhip


# nr, ns, Ex, Ey, periodic; workgroups: a few, 32 and a few more, 121 to 256
CASES = [(8, 8, 4, 13, (False, False)), (8, 8, 32, 31, (True, True)), (5, 5, 40, 33, (True, False)),
         (10, 10, 25, 24, (False, False)), (8, 8, 45, 45, (False, True)), (16, 16, 14, 22, (False, False)),
         (6, 6, 66, 64, (True, True)), (10, 10, 63, 65, (False, True)), (5, 5, 101, 99, (False, False)),
         (12, 12, 51, 50, (False, False)), (8, 8, 127, 128, (True, True)), (16, 16, 60, 62, (False, False)),
         (12, 9, 8, 6, (True, False)), (7, 12, 30, 50, (False, False)), (9, 5, 3, 4, (True, True))]


# (FP32 operators need nr == ns)
@pytest.mark.parametrize("nr,ns,Ex,Ey,per,prec", [(*c, prec) for c in CASES for prec in ("f64", "f32")
                                                  if prec == "f64" or c[0] == c[1]])
def test_forms_agree(se, monkeypatch, nr, ns, Ex, Ey, per, prec):
    import torch
    import warnings
    print(f"exchange {nr}x{ns} {Ex}x{Ey} {per} {prec}", flush=True)
    m = se.Mesh(nr, ns, Ex, Ey, per, se.deform_sinsin(0.1))
    M = se.generateMask("DDDD", m)
    dt = torch.float64 if prec == "f64" else torch.float32
    f = np.random.default_rng(nr * Ex + Ey).standard_normal(m.shape)
    b = se.gatherScatter(se.mask(se.mass(se.to_device(f), m), M), m)
    d = se.Diagonal(se.SEMOperator(1.0, 1.0, m, M).jacobi().to(dt), local=False)
    x = {}
    for mode in ("0", "1", "3"):
        monkeypatch.setenv("SEM_PCG_RESIDENT", mode)
        op = se.SEMOperator(1.0, 1.0, m, M, precision=prec)
        with warnings.catch_warnings():
            warnings.simplefilter("ignore")
            x[mode] = se.pcg(b.to(dt), op, opM=d, mult=m.mult, tol=0.0, maxiter=4)
    scale = float(x["0"].abs().max())
    for mode in ("1", "3"):
        assert float((x[mode] - x["0"]).abs().max()) <= (1e-12 if prec == "f64" else 1e-5) * scale
    if Ex * Ey <= 300:   # at most 32 workgroups
        assert torch.equal(x["1"], x["3"])
