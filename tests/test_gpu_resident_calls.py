"""Calls around the resident PCG (a solve in one launch): its mail in the fixed array of
sem_pcg_noalloc, solves of several contexts at a time, what follows a launch that other
work called off, which inner products a mixed solve reports, the tags of its words over their range."""
import ctypes as C
import threading
import time

import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def se():
    import semhip
    return semhip


@pytest.fixture
def contexts(se):
    """two contexts of the library, each on a stream of its own"""
    import torch
    from semhip import _lib as L
    st = [torch.cuda.Stream() for _ in range(2)]
    h = []
    for s in st:
        c = C.c_void_p()
        L.call("sem_ctx_create", torch.cuda.current_device(), C.c_void_p(s.cuda_stream), C.byref(c))
        h.append(c)
    yield list(zip(h, st))
    torch.cuda.synchronize()
    for c in h:
        L.call("sem_ctx_destroy", c)


def _problem(se, nr, ns, Ex, Ey, seed=1):
    m = se.Mesh(nr, ns, Ex, Ey, (False, False), se.deform_sinsin(0.1))
    M = se.generateMask("DDDD", m)
    return m, M, se.workloads.helmholtz_rhs(se, m, M, seed=seed)


def _solve(se, ctx, op, b, d=None, tol=0.0, maxiter=4, entry="sem_pcg", x=None):
    """x of a solve through the C ABI, in the given context; and its info"""
    import torch
    from semhip import _lib as L
    if x is None:
        x = torch.zeros_like(b)
        torch.cuda.current_stream().synchronize()   # (x, b and d are ready for any stream)
    info = L.sem_pcg_info()
    L.call(entry, ctx, op.h, L.SEM_PRECOND_IDENTITY if d is None else L.SEM_PRECOND_DIAG,
           None if d is None else C.c_void_p(d.data_ptr()), C.c_void_p(b.data_ptr()),
           C.c_void_p(x.data_ptr()), float(tol), int(maxiter), C.byref(info))
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


# one workgroup, 8 and 16 on one XCD, blocks of any size: the second context's solve does
# not wait for the first's, whose stream has other work (bounded, one lane) ahead of it.
# (Streams may come to share a hardware queue and then run in order: several are tried.)
@pytest.mark.parametrize("nr,ns,Ex,Ey", [(9, 9, 4, 4), (8, 8, 16, 12), (8, 8, 24, 20),
                                         (12, 9, 4, 3)])
def test_solves_of_two_contexts_side_by_side(se, contexts, nr, ns, Ex, Ey):
    import torch
    from semhip import _lib as L
    print(f"two contexts {nr}x{ns} {Ex}x{Ey}", flush=True)
    (c0, s0), (c1, _) = contexts
    m, M, b = _problem(se, nr, ns, Ex, Ey)
    op = se.SEMOperator(1.0, 1.0, m, M)
    ref, _ = _solve(se, c0, op, b, maxiter=50)
    _solve(se, c1, op, b, maxiter=50)
    x0, x1 = torch.zeros_like(b), torch.zeros_like(b)
    e = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
    with torch.cuda.stream(s0):   # the cycles of a third of a second
        torch.cuda._sleep(1)
        e[0].record()
        torch.cuda._sleep(1000000)
        e[1].record()
    torch.cuda.synchronize()
    cycles = int(1000000 * 333.0 / e[0].elapsed_time(e[1]))

    def first():
        with torch.cuda.stream(s0):
            torch.cuda._sleep(cycles)
        _solve(se, c0, op, b, maxiter=50, x=x0)

    waits = False
    for _ in range(8):
        s1 = torch.cuda.Stream()
        L.call("sem_ctx_set_stream", c1, C.c_void_p(s1.cuda_stream))
        t = threading.Thread(target=first)
        t.start()
        time.sleep(0.1)
        _solve(se, c1, op, b, maxiter=50, x=x1)
        waits = t.is_alive()
        t.join()
        torch.cuda.synchronize()
        assert torch.equal(x1, ref) and torch.equal(x0, ref)
        if waits:
            break
    assert waits


def test_solves_of_two_contexts_that_fill_the_chip(se, contexts):
    import torch
    print("two contexts 128x128", flush=True)
    m, M, b = _problem(se, 8, 8, 128, 128)
    op = se.SEMOperator(1.0, 1.0, m, M)
    ref, _ = _solve(se, contexts[0][0], op, b, maxiter=300)
    out = [torch.zeros_like(b) for _ in range(2)]
    torch.cuda.synchronize()

    def run(i):
        for _ in range(3):
            _solve(se, contexts[i][0], op, b, maxiter=300, x=out[i])

    t = [threading.Thread(target=run, args=(i,)) for i in range(2)]
    for q in t:
        q.start()
    for q in t:
        q.join()
    torch.cuda.synchronize()
    assert torch.equal(out[0], ref) and torch.equal(out[1], ref)


# SEM_PCG_RESIDENT = 4: a launch is called off as if by other work. Its solve and the next
# ones of the context take launches (the bits of = 0), after a rest one launch again.
@pytest.mark.parametrize("nr,ns,Ex,Ey", [(8, 8, 13, 9), (12, 9, 8, 6)])
def test_called_off_is_remembered(se, contexts, monkeypatch, nr, ns, Ex, Ey):
    import torch
    print(f"called off {nr}x{ns} {Ex}x{Ey}", flush=True)
    m, M, b = _problem(se, nr, ns, Ex, Ey)
    op = {}
    for mode in ("0", "1", "4"):
        monkeypatch.setenv("SEM_PCG_RESIDENT", mode)
        op[mode] = se.SEMOperator(1.0, 1.0, m, M)
    (c0, _), (c1, _) = contexts
    launches, _ = _solve(se, c0, op["0"], b, maxiter=60)
    resident, _ = _solve(se, c0, op["1"], b, maxiter=60)
    torch.cuda.synchronize()
    assert not torch.equal(launches, resident)   # (else the solves could not be told apart)
    x = [_solve(se, c1, op[mode], b, maxiter=60)[0] for mode in ("1", "4", "1", "1")]
    other = _solve(se, c0, op["1"], b, maxiter=60)[0]   # another context's: as before
    torch.cuda.synchronize()
    same = [(torch.equal(v, launches), torch.equal(v, resident)) for v in x]
    assert same == [(False, True)] + 3 * [(True, False)]
    assert torch.equal(other, resident)
    time.sleep(0.5)
    again, _ = _solve(se, c1, op["1"], b, maxiter=60)
    torch.cuda.synchronize()
    assert torch.equal(again, resident)


def test_called_off_later_goes_on_from_there(se, monkeypatch):
    # blocks of any size, more iterations than one launch takes (4096), the second launch
    # called off (SEM_PCG_RESIDENT = 5): the same solve by steps takes several times as long,
    # and one that started over longer still
    print("called off later 12x9 64x60", flush=True)
    m, M, b = _problem(se, 12, 9, 64, 60)
    info = {}
    x = {}
    for mode in ("0", "5"):
        monkeypatch.setenv("SEM_PCG_RESIDENT", mode)
        op = se.SEMOperator(1.0, 0.0, m, M)
        d = se.Diagonal(op.jacobi())
        i = info[mode] = se.PCGInfo()
        x[mode] = se.pcg(b, op, opM=d, mult=m.mult, tol=-1e-12, info=i)
        assert i.converged and i.res <= 1e-12 * float(b.abs().max())
    assert info["5"].iters > 4096
    assert abs(info["5"].iters - info["0"].iters) <= info["0"].iters // 100
    assert float((x["5"] - x["0"]).abs().max()) < 1e-9 * float(x["0"].abs().max())
    assert info["5"].elapsed_ms < 0.6 * info["0"].elapsed_ms


@pytest.mark.parametrize("prec", ["f32", "f16x3", "bf16x3", "f16"])
@pytest.mark.parametrize("mode", ["0", "1", "2"])
def test_mixed_solve_says_which_products(se, monkeypatch, capfd, prec, mode):
    print(f"mixed {prec} mode {mode}", flush=True)
    m, M, b = _problem(se, 16, 16, 12, 12)
    tol = 1e-10 * float(b.abs().max())
    op64 = se.SEMOperator(1.0, 1.0, m, M)
    monkeypatch.setenv("SEM_PCG_RESIDENT", mode)
    op = se.SEMOperator(1.0, 1.0, m, M, precision=prec)
    monkeypatch.setenv("SEM_DEBUG_MIXED", "1")
    info = se.PCGInfo()
    x = se.pcg_mixed(b, op64, op, d=op64.jacobi(), tol=tol, inner_tol=1e-2, info=info)
    lines = [v for v in capfd.readouterr().err.splitlines() if v.startswith("[mixed] cycle")]
    assert info.converged and float((b - op64(x)).abs().max()) <= 1.01 * tol
    one = mode == "1" and prec != "f16"
    assert len(lines) == info.outer
    assert all(("FP32 products in one launch" in v) == one for v in lines)
    assert all(("op_lo's products by launches" in v) != one for v in lines)


# each launch uses 4098 tags: the exchanged lines' 16 bits start over every 16 launches,
# the counter (SEM_PCG_TAG at the context's creation) after some million; here on the fourth
@pytest.mark.parametrize("nr,ns,Ex,Ey", [(8, 8, 13, 9), (10, 10, 17, 25), (8, 8, 64, 64),
                                         (12, 9, 20, 14)])
def test_tags_start_over(se, monkeypatch, nr, ns, Ex, Ey):
    import torch
    from semhip import _lib as L
    print(f"tags {nr}x{ns} {Ex}x{Ey}", flush=True)
    m, M, b = _problem(se, nr, ns, Ex, Ey)
    op = se.SEMOperator(1.0, 1.0, m, M)
    ref = None
    for start in (0, 2**32 - 1 - 3 * 4098 - 17):
        monkeypatch.setenv("SEM_PCG_TAG", str(start))
        c = C.c_void_p()
        L.call("sem_ctx_create", torch.cuda.current_device(), None, C.byref(c))
        try:
            for _ in range(36):
                x, _ = _solve(se, c, op, b, maxiter=12)
                torch.cuda.synchronize()
                ref = x if ref is None else ref
                assert torch.equal(x, ref)
        finally:
            L.call("sem_ctx_destroy", c)
