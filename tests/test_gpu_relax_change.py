"""Relaxation types chosen after the setup, on levels with a solve-phase copy.

The type is read by the cycle, so a hierarchy set up for l1-Jacobi may be asked
for other sweeps.  The hierarchy of solve_format 0, which has no copies and
keeps every level's values, gives the bits.  What a hierarchy cannot do is an
error and leaves it usable.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def hierarchy(hx, A, fmt, fp32, relax=18):
    amg = hx.BoomerAMG(max_iter=1, tol=0.0, fp32_cycle=fp32, solve_format=fmt, relax_type=relax)
    amg.setup(A)
    return amg


@pytest.mark.parametrize("fp32", [0, 1])
@pytest.mark.parametrize("types", [(0, 0), (7, 7), (13, 13), (3, 3), (18, 13), (0, 18)], ids=str)
def test_type_changed_after_setup(hx, oracle, types, fp32):
    print("[gpu-relax-change]", types, fp32, flush=True)
    A = hx.ParCSRMatrix.laplacian27(50, 51, 49)        # stencil copy, then sliced ELL on level 1
    n, _ = A.dims()
    f = 2 * oracle.rand_stream(9, n) - 1
    got = []
    for fmt in (0, 1):
        amg = hierarchy(hx, A, fmt, fp32)
        assert amg.level_rows(1) >= 4096
        first = amg.cycle_host(f)
        amg.set(relax_down=types[0], relax_up=types[1])
        other = amg.cycle_host(f)
        amg.set(relax_type=18)
        again = amg.cycle_host(f)
        assert np.array_equal(first, again) and not np.array_equal(first, other)
        got.append(other)
        amg.destroy()
    assert np.isfinite(got[0]).all()
    assert np.array_equal(got[0].view(np.int64), got[1].view(np.int64))


@pytest.mark.parametrize("fp32", [0, 1])
def test_sweeps_that_the_hierarchy_has_no_data_for_are_refused(hx, oracle, fp32):
    A = hx.ParCSRMatrix.laplacian27(24, 24, 24)
    n, _ = A.dims()
    f = 2 * oracle.rand_stream(9, n) - 1
    for setup, later in ((18, 14), (18, 6), (0, 18), (0, 13)):   # no reversed rows, no l1 norms
        print("[gpu-relax-change] refused", setup, later, fp32, flush=True)
        amg = hierarchy(hx, A, 1, fp32, setup)
        first = amg.cycle_host(f)
        amg.set(relax_type=later)
        with pytest.raises(hx.HypreError):
            amg.cycle_host(f)
        amg.set(relax_type=setup)
        assert np.array_equal(amg.cycle_host(f), first)
        amg.destroy()


def test_fp32_cycle_of_an_fp64_hierarchy_is_refused(hx, oracle):
    A = hx.ParCSRMatrix.laplacian27(24, 24, 24)
    f = 2 * oracle.rand_stream(9, 24 ** 3) - 1
    amg = hierarchy(hx, A, 1, 0)
    amg.set(fp32_cycle=1)
    with pytest.raises(hx.HypreError):
        amg.cycle_host(f)
