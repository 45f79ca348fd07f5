"""PCG where an iteration breaks off, and preconditioners of the caller's own.

The step length is formed on the device; an iteration that hypre's pcg.c leaves
at it must leave x alone, whoever owns the preconditioner.
"""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PRECOND = ctypes.CFUNCTYPE(ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p)


def set_precond(hx, pcg, solve):
    """A preconditioner of the caller's own; keeps the callbacks alive."""
    pcg.callbacks = PRECOND(solve), PRECOND(lambda *_: 0)
    hx.call("HYPRE_ParCSRPCGSetPrecond", pcg.h, *(ctypes.cast(c, ctypes.c_void_p) for c in pcg.callbacks), None)


def diagonal(hx, d):
    n = len(d)
    return hx.ParCSRMatrix.from_csr(np.arange(n + 1), np.arange(n), np.asarray(d, np.float64))


def test_a_preconditioner_that_runs_pcg(hx, oracle):
    """Diagonal scaling, with and without a PCG solve beside it that ends on
    <s, p> = 0: the outer iteration is the same, bit for bit."""
    A = hx.ParCSRMatrix.laplacian7(13, 12, 11)
    n, _ = A.dims()
    zero, c, y = diagonal(hx, np.zeros(50)), hx.ParVector(50, np.ones(50)), hx.ParVector(50)
    inner = hx.PCG(None)
    inner.setup(zero, c, y)

    def solve(inside):
        b, x = hx.ParVector(n, 2 * oracle.rand_stream(3, n) - 1), hx.ParVector(n)
        pcg = hx.PCG(None, tol=1e-8)
        hx.call("HYPRE_ParCSRPCGSetRelChange", pcg.h, 1)

        def apply(_, a, r, z):
            hx.call("HYPRE_ParCSRDiagScale", None, *map(ctypes.c_void_p, (a, r, z)))
            if inside:
                inner.solve(zero, c, y)
            return 0
        set_precond(hx, pcg, apply)
        pcg.setup(A, b, x)
        pcg.solve(A, b, x)
        return pcg.num_iterations(), np.array(pcg.history()), x.get()
    plain, nested = solve(False), solve(True)
    assert plain[0] == nested[0] > 10
    assert np.array_equal(plain[1], nested[1]) and np.array_equal(plain[2], nested[2])


@pytest.mark.parametrize("how", ["refused", "no_cycle"])
def test_a_cycle_that_does_not_run_gives_zeros(hx, oracle, how):
    """A BoomerAMG preconditioner that refuses its sweeps, or whose tolerance
    lets no cycle run, gives zeros: the vectors of an earlier solve do not
    show, <s, p> is zero and x stays."""
    A = hx.ParCSRMatrix.laplacian27(20, 21, 22)
    n, _ = A.dims()
    b, x = hx.ParVector(n, 2 * oracle.rand_stream(3, n) - 1), hx.ParVector(n)
    amg = hx.BoomerAMG()
    pcg = hx.PCG(amg, tol=1e-8)
    pcg.setup(A, b, x)
    pcg.solve(A, b, x)
    assert pcg.num_iterations() > 3
    start = oracle.rand_stream(5, n)
    x.set(start)
    if how == "refused":
        amg.set(relax_type=14)              # no reversed rows
        with pytest.raises(hx.HypreError) as e:
            pcg.solve(A, b, x)
        assert e.value.code & hx.ERROR_GENERIC and e.value.code & hx.ERROR_CONV
    else:
        amg.set(tol=float("nan"))
        assert pcg.solve(A, b, x) == hx.ERROR_CONV
    assert pcg.num_iterations() == 1
    assert np.array_equal(x.get(), start)


def test_no_cycle_is_printed_for_an_iteration_that_breaks_off(hx, oracle, capfd):
    """-A with the hierarchy of A: the first step length is negative.  Only the
    cycle before it prints."""
    A = hx.ParCSRMatrix.laplacian7(9, 9, 9)
    h = A.to_host()
    minus = hx.ParCSRMatrix.from_csr(h.ia, h.ja, -h.a)
    n = h.nrows
    b, x = hx.ParVector(n, 2 * oracle.rand_stream(3, n) - 1), hx.ParVector(n)
    amg = hx.BoomerAMG()
    pcg = hx.PCG(amg, tol=1e-8)
    pcg.setup(A, b, x)
    amg.set(print_level=2)
    assert pcg.solve(minus, b, x) & hx.ERROR_CONV
    ctypes.CDLL(None).fflush(None)
    assert capfd.readouterr().out.count("Average Convergence Factor") == 1
    assert pcg.num_iterations() == 1 and not x.get().any()
