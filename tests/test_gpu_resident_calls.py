"""Calls around the resident PCG (a solve in one launch): its mail in the fixed array of
sem_pcg_noalloc."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def se():
    import semhip
    return semhip


def _problem(se, nr, ns, Ex, Ey, seed=1):
    m = se.Mesh(nr, ns, Ex, Ey, (False, False), se.deform_sinsin(0.1))
    M = se.generateMask("DDDD", m)
    return m, M, se.workloads.helmholtz_rhs(se, m, M, seed=seed)


def _solve(se, ctx, op, b, d=None, tol=0.0, maxiter=4, entry="sem_pcg"):
    """x of a solve through the C ABI, in the given context; and its info"""
    import torch
    from semhip import _lib as L
    x = torch.zeros_like(b)
    info = L.sem_pcg_info()
    L.call(entry, ctx, op.h, L.SEM_PRECOND_IDENTITY if d is None else L.SEM_PRECOND_DIAG,
           None if d is None else C.c_void_p(d.data_ptr()), C.c_void_p(b.data_ptr()),
           C.c_void_p(x.data_ptr()), float(tol), int(maxiter), C.byref(info))
    torch.cuda.synchronize()
    return x, info


# two whose workspace ends 64 bytes past a 128-byte line (254 and 250 parts of 32 bytes),
# with sums by XCD, and one near the array's end, whose mail takes w's place
@pytest.mark.parametrize("n,Ex,Ey,prec", [(9, 80, 80, "f64"), (9, 80, 79, "f32"),
                                          (8, 125, 128, "f64")])
def test_noalloc_mail_on_whole_lines(se, n, Ex, Ey, prec):
    import torch
    print(f"noalloc n={n} {Ex}x{Ey} {prec}", flush=True)
    m, M, b = _problem(se, n, n, Ex, Ey)
    dt = torch.float64 if prec == "f64" else torch.float32
    d = se.SEMOperator(1.0, 1.0, m, M).jacobi().to(dt)
    op = se.SEMOperator(1.0, 1.0, m, M, precision=prec)
    x0, i0 = _solve(se, se.ctx(), op, b.to(dt), d, maxiter=40)
    x1, i1 = _solve(se, se.ctx(), op, b.to(dt), d, maxiter=40, entry="sem_pcg_noalloc")
    assert i0.iters == i1.iters == 40 and i0.res == i1.res
    assert torch.equal(x0, x1)
