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


def pcg_steps(A, precond, b, skip_break, two_norm=True, eps=1e-16, most=50):
    """pcg.c's iteration: x, iterations, whether an error was flagged, times the
    preconditioner ran."""
    x, runs, error = np.zeros_like(b), [0], False

    def C(r):
        runs[0] += 1
        return precond(r)
    bi = b @ b if two_norm else b @ C(b)
    r = b - A @ x
    p = C(r)
    gamma = r @ p
    tiny, least = 2.0 ** -1074, 2.0 ** -1022
    for i in range(1, most + 1):
        s = A @ p
        sdotp = s @ p
        if sdotp == 0.0:
            return x, i, True, runs[0]
        alpha = gamma / sdotp
        level = 3 if alpha <= 0 else 2 if not alpha >= tiny else 1 if not alpha >= least else 0
        error = error or level > 0
        if level > skip_break:
            return x, i, True, runs[0]
        x = x + alpha * p
        r = r - alpha * s
        s = C(r)
        old, gamma = gamma, r @ s
        if (r @ r if two_norm else gamma) / bi < eps:
            return x, i, error, runs[0]
        level = 3 if gamma <= 0 else 2 if not gamma >= tiny else 1 if not gamma >= least else 0
        error = error or level > 0
        if level > skip_break:
            return x, i, True, runs[0]
        p = s + gamma / old * p
    return x, most, True, runs[0]


# matrices on which the first or a later step length is zero, negative, not a
# number or subnormal, with a right-hand side
BREAKS = {
    "zero": (np.zeros((4, 4)), [1.0, 2.0, -1.0, 0.5]),
    "negative": (-np.diag([1.0, 2.0, 3.0, 4.0]), [1.0, 2.0, -1.0, 0.5]),
    "indefinite_later": (np.diag([5.0, 4.0, 1.0, -0.25]), [1.0, 1.0, 1.0, 1.0]),
    "not_a_number": (np.diag([1e308, -1e308]), [100.0, 100.0]),
    "subnormal": (np.array([[1e308]]), [0.1]),
    "overflow": (np.array([[1e308]]), [100.0]),
    "sound": (np.diag([1.0, 2.0, 3.0, 4.0]), [1.0, 2.0, -1.0, 0.5]),
}


@pytest.mark.parametrize("precond", ["none", "caller"])
@pytest.mark.parametrize("skip_break", [0, 1, 2, 3])
@pytest.mark.parametrize("name", sorted(BREAKS))
def test_breaks_follow_the_serial_iteration(hx, name, skip_break, precond):
    """Error flag, iterations and x of pcg.c's steps; a caller's preconditioner,
    the identity like none, is not called for a step that breaks off."""
    M, b = BREAKS[name]
    b = np.array(b)
    n = len(b)
    full = [np.arange(n)[np.argsort(np.arange(n) != i, kind="stable")] for i in range(n)]
    A = hx.ParCSRMatrix.from_csr(np.arange(n + 1) * n, np.concatenate(full),
                                 np.concatenate([M[i, c] for i, c in enumerate(full)]))
    bv, x = hx.ParVector(n, b), hx.ParVector(n)
    pcg = hx.PCG(None, tol=1e-8, max_iter=50)
    hx.call("HYPRE_PCGSetSkipBreak", pcg.h, skip_break)
    called = [0]

    def apply(_, a, r, z):
        called[0] += 1
        hx.lib().HYPRE_ParVectorCopy(r, z)      # hx.call would clear an error of the iteration
        return 0
    if precond == "caller":
        set_precond(hx, pcg, apply)
    pcg.setup(A, bv, x)
    with np.errstate(all="ignore"):
        want, its, error, runs = pcg_steps(M, np.copy, b, skip_break)
    got = pcg.solve(A, bv, x)
    assert (got == hx.ERROR_CONV) == error and pcg.num_iterations() == its
    np.testing.assert_allclose(x.get(), want, rtol=1e-12, atol=0)
    if precond == "caller":
        assert called[0] == runs


def test_a_hierarchy_s_cycle_before_a_break_leaves_x(hx, oracle):
    """BoomerAMG runs before the host has seen the step: -A breaks off at once,
    and x is what it was."""
    A = hx.ParCSRMatrix.laplacian27(20, 21, 22)
    h = A.to_host()
    minus = hx.ParCSRMatrix.from_csr(h.ia, h.ja, -h.a)
    n = h.nrows
    start = oracle.rand_stream(5, n)
    b, x = hx.ParVector(n, 2 * oracle.rand_stream(3, n) - 1), hx.ParVector(n, start)
    pcg = hx.PCG(hx.BoomerAMG(), tol=1e-8)
    pcg.setup(A, b, x)
    for skip_break in (0, 1, 2):
        hx.call("HYPRE_PCGSetSkipBreak", pcg.h, skip_break)
        assert pcg.solve(minus, b, x) == hx.ERROR_CONV
        assert pcg.num_iterations() == 1 and np.array_equal(x.get(), start)
