"""The stencil copy of the fine operator gives the bits of the CSR kernels.

solve_format 0 runs the CSR kernels, format 1 (default) the stencil copy where
the fine operator's columns differ from the row by at most 32 offsets: slices
of 128 rows with no values, with a dictionary of at most 256, or with full
values.  A V-cycle in FP64 and FP32 must agree bit for bit between the two on
grids whose slices are cut by lines, planes and the matrix's end, on the
table sizes with an unrolled kernel (5, 7, 9, 19, 27) and others, at 31 and
33 offsets, and on rows that are not sorted (both fall back).  The fine level's
interpolation, which the stencil path forms one lane a row, must be the
general kernels' bits for every threshold, truncation and sign pattern.
"""
import os
import re
import subprocess
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def grid_matrix(nx, ny, nz, offsets, values, seed=1, missing=0.0, shuffle=False, positive=0.0):
    """Rows diagonal first, then ascending, from (dx, dy, dz) offsets in
    symmetric pairs; values 'const', 'few' (64 distinct couplings), 'all'
    (every coupling its own), 'late' (constant up to row 1000, inside a
    slice) or 'mixed' (few, from a third of the rows on constant, from two
    thirds on all); missing: share of the pairs left out; positive: share of small
    couplings of the diagonal's sign."""
    import scipy.sparse as sp
    rng = np.random.default_rng(seed)
    n = nx * ny * nz
    iz, iy, ix = np.unravel_index(np.arange(n), (nz, ny, nx))
    rows, cols, vals = [], [], []
    for dx, dy, dz in offsets:
        if (dz, dy, dx) <= (0, 0, 0):
            continue
        jx, jy, jz = ix + dx, iy + dy, iz + dz
        ok = (jx >= 0) & (jx < nx) & (jy >= 0) & (jy < ny) & (jz >= 0) & (jz < nz)
        ok &= rng.random(n) >= missing
        i = np.nonzero(ok)[0]
        j = i + (dz * ny + dy) * nx + dx
        v = {"const": np.ones(len(i)), "few": 0.5 + rng.integers(0, 64, len(i)) / 64.0,
             "all": 0.5 + rng.random(len(i)),
             "late": np.where(i >= 1000, 1.0 + i % 5 / 8, 1.0),
             "mixed": np.where(i < n // 3, 0.5 + i * 7 % 64 / 64.0,
                               np.where(i < 2 * n // 3, 1.0, 0.5 + i * 0.618034 % 1.0 + dz / 7 + dy / 77 + dx / 777)),
             }[values]
        v = np.where(rng.random(len(i)) < positive, -0.3 * v, v)
        rows += [i, j]
        cols += [j, i]
        vals += [-v, -v]
    off = sp.csr_matrix((np.concatenate(vals), (np.concatenate(rows), np.concatenate(cols))), shape=(n, n))
    off.sort_indices()
    diag = 1e-2 + np.asarray(abs(off).sum(axis=1)).ravel()
    if values in ("const", "late", "mixed"):
        diag[:] = diag.max()
    ia = np.zeros(n + 1, np.int32)
    ia[1:] = np.cumsum(np.diff(off.indptr) + 1)
    ja, a = np.empty(ia[-1], np.int32), np.empty(ia[-1])
    first = ia[:-1]
    ja[first], a[first] = np.arange(n), diag
    rest = np.ones(ia[-1], bool)
    rest[first] = False
    ja[rest], a[rest] = off.indices, off.data
    if shuffle:
        for r in range(0, n, 7):
            s, e = ia[r] + 1, ia[r + 1]
            ja[s:e], a[s:e] = ja[s:e][::-1].copy(), a[s:e][::-1].copy()
    return ia, ja, a


def box(r=1):
    return [(x, y, z) for z in range(-r, r + 1) for y in range(-r, r + 1) for x in range(-r, r + 1)]


P5 = [(0, 0, 0), (1, 0, 0), (-1, 0, 0), (0, 1, 0), (0, -1, 0)]
P7 = P5 + [(0, 0, 1), (0, 0, -1)]
P9 = [o for o in box() if o[2] == 0]
P19 = [o for o in box() if sum(map(abs, o)) <= 2]
P31 = [(k, 0, 0) for k in range(-15, 16)]
# 31 offsets whose sums are more than 128
SCATTERED = [(s * x, s * y, s * z) for s in (-1, 1) for x, y, z in
             ((1, 0, 0), (3, 0, 0), (7, 0, 0), (-9, 1, 0), (0, 1, 0), (4, 1, 0), (0, 3, 0), (2, 5, 0), (-5, 0, 1),
              (0, 0, 1), (6, 1, 1), (0, 5, 1), (0, 0, 2), (1, -3, 3), (0, 1, 4))] + [(0, 0, 0)]
P33 = [(k, 0, 0) for k in range(-16, 17)]

CASES = {
    "27_const_ragged": (17, 19, 23, box(), "const", {}),
    "27_few": (21, 16, 17, box(), "few", {}),
    "27_late": (21, 16, 17, box(), "late", {}),
    "27_all": (19, 17, 16, box(), "all", {}),
    "27_mixed": (16, 16, 48, box(), "mixed", {}),
    "7_mixed": (23, 25, 24, P7, "mixed", {}),
    "31_mixed": (9001, 1, 1, P31, "mixed", {}),
    "27_all_missing": (19, 17, 16, box(), "all", {"missing": 0.2}),
    "27_all_few_entries": (19, 17, 16, box(), "all", {"missing": 0.6}),   # the copy does not pay
    "27_few_few_entries": (19, 17, 16, box(), "few", {"missing": 0.6}),
    "27_thin": (2, 61, 47, box(), "few", {}),        # offsets of lines and planes overlap
    "19_few": (18, 15, 19, P19, "few", {}),
    "19_const": (64, 8, 8, P19, "const", {}),
    "9_all": (131, 67, 1, P9, "all", {}),
    "9_const": (128, 33, 1, P9, "const", {}),
    "7_few_missing": (33, 13, 14, P7, "few", {"missing": 0.1}),
    "7_const": (4, 33, 34, P7, "const", {}),
    "5_all": (67, 71, 1, P5, "all", {}),
    "31_few": (4111, 1, 1, P31, "few", {}),
    "31_all_missing": (5003, 1, 1, P31, "all", {"missing": 0.3}),
    "scattered_all": (17, 19, 16, SCATTERED, "all", {"missing": 0.1}),
    "scattered_few": (18, 17, 19, SCATTERED, "few", {}),
    "33_all": (4999, 1, 1, P33, "all", {}),           # one offset too many
    "27_unsorted": (17, 17, 17, box(), "few", {"shuffle": True}),
}


def cycle(hx, A, fmt, f, fp32):
    amg = hx.BoomerAMG(max_iter=1, tol=0.0, fp32_cycle=1 if fp32 else 0, solve_format=fmt)
    amg.setup(A)
    u = amg.cycle_host(f)
    amg.destroy()
    return u


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("name", sorted(CASES))
def test_vcycle_bits_equal_the_csr_kernels(hx, oracle, name, fp32):
    nx, ny, nz, offsets, values, more = CASES[name]
    print("[gpu-stencil]", name, fp32, flush=True)
    A = hx.ParCSRMatrix.from_csr(*grid_matrix(nx, ny, nz, offsets, values, **more))
    n, _ = A.dims()
    assert n >= 4096
    f = 2 * oracle.rand_stream(7, n) - 1
    u0, u1 = cycle(hx, A, 0, f, fp32), cycle(hx, A, 1, f, fp32)
    assert np.isfinite(u0).all() and np.abs(u0).max() > 0
    bad = np.nonzero(u0.view(np.int64) != u1.view(np.int64))[0]
    assert bad.size == 0, f"{bad.size} entries differ, first at {bad[:5]}"


def test_product_with_dot_matches_the_csr_kernels(hx, oracle):
    """PCG's s = A p on the copy (with <s, p>): same iterations, same solution
    up to the order of the dot product's partial sums."""
    out = []
    for fmt in (0, 1):
        A = hx.ParCSRMatrix.from_csr(*grid_matrix(21, 16, 17, box(), "few"))
        n, _ = A.dims()
        b, x = hx.ParVector(n, 2 * oracle.rand_stream(3, n) - 1), hx.ParVector(n)
        pcg = hx.PCG(hx.BoomerAMG(solve_format=fmt), tol=1e-8)
        pcg.setup(A, b, x)
        pcg.solve(A, b, x)
        out.append((pcg.num_iterations(), np.array(pcg.history()), x.get()))
    assert out[0][0] == out[1][0]
    np.testing.assert_allclose(out[1][1], out[0][1], rtol=1e-9)
    np.testing.assert_allclose(out[1][2], out[0][2], rtol=1e-8, atol=1e-12 * np.abs(out[0][2]).max())


INTERP = {
    "27_const": (17, 19, 23, box(), "const", {}),
    "27_few": (21, 16, 17, box(), "few", {}),
    "27_late": (21, 16, 17, box(), "late", {}),
    "27_mixed": (16, 16, 48, box(), "mixed", {}),
    "27_all_signs": (19, 17, 16, box(), "all", {"positive": 0.2}),
    "27_missing": (19, 17, 16, box(), "few", {"missing": 0.25}),
    "27_thin": (2, 61, 47, box(), "few", {}),
    "19_signs": (18, 15, 19, P19, "few", {"positive": 0.1}),
    "9_all": (131, 67, 1, P9, "all", {}),
    "7_const": (20, 21, 22, P7, "const", {}),
    "7_signs_missing": (33, 13, 14, P7, "few", {"missing": 0.1, "positive": 0.1}),
    "31_all": (5003, 1, 1, P31, "all", {"missing": 0.3}),
    "scattered_few": (18, 17, 19, SCATTERED, "few", {}),                   # too many sums: general kernels
    "scattered_signs": (17, 19, 16, SCATTERED, "all", {"missing": 0.2, "positive": 0.1}),
    "27_half": (19, 17, 16, box(), "all", {"missing": 0.5}),               # a copy for this alone
    "27_half_signs": (19, 17, 16, box(), "all", {"missing": 0.6, "positive": 0.1}),
}


@pytest.mark.parametrize("options", [
    {}, {"strong_threshold": 0.6}, {"strong_threshold": 0.95, "max_row_sum": 1.0},
    {"strong_threshold": 0.01, "P_max_elmts": 32}, {"P_max_elmts": 1, "trunc_factor": 0.3},
    {"coarsen_type": 10, "trunc_factor": 0.1}], ids=lambda o: ",".join(f"{k}={v}" for k, v in o.items()) or "default")
@pytest.mark.parametrize("name", sorted(INTERP))
def test_interpolation_bits_equal_the_general_kernels(hx, name, options):
    nx, ny, nz, offsets, values, more = INTERP[name]
    print("[gpu-stencil] P", name, options, flush=True)
    A = hx.ParCSRMatrix.from_csr(*grid_matrix(nx, ny, nz, offsets, values, **more))
    got = []
    for fmt in (0, 1):
        amg = hx.BoomerAMG(solve_format=fmt, max_levels=2, **options)
        amg.setup(A)
        got.append((amg.level_cf(0), amg.level_matrix(0, "P")))
        amg.destroy()
    (cf0, P0), (cf1, P1) = got
    assert np.array_equal(cf0, cf1)
    assert np.array_equal(P0.ia, P1.ia) and np.array_equal(P0.ja, P1.ja)
    bad = np.nonzero(P0.a.view(np.int64) != P1.a.view(np.int64))[0]
    assert bad.size == 0, f"{bad.size} of {P0.nnz} weights differ, first at {bad[:5]}"


def other_diagonal(rows):
    ia, ja, a = grid_matrix(32, 32, 32, box(), "const")
    a[ia[:-1][rows]] *= 2
    return ia, ja, a


# name: matrix, slices with codes and with full values, whether the copy is kept
FORMS = {
    "27_const": (lambda: grid_matrix(32, 32, 32, box(), "const"), 0, 0, "kept"),
    "27_few": (lambda: grid_matrix(32, 32, 32, box(), "few"), 256, 0, "kept"),
    "27_all": (lambda: grid_matrix(32, 32, 32, box(), "all"), 0, 256, "kept"),
    "27_mixed": (lambda: grid_matrix(32, 32, 30, box(), "mixed"), 88, 80, "kept"),
    "27_all_many": (lambda: grid_matrix(32, 32, 32, box(), "all", missing=0.3), 0, 256, "kept"),
    "27_all_half": (lambda: grid_matrix(32, 32, 32, box(), "all", missing=0.5), 0, 256, "interpolation"),
    "31_all_half": (lambda: grid_matrix(32, 32, 32, P31, "all", missing=0.6), 0, 256, "interpolation"),
    "too_many_sums": (lambda: grid_matrix(32, 32, 32, SCATTERED, "all", missing=0.6), 0, 256, "dropped"),
    "27_few_half": (lambda: grid_matrix(32, 32, 32, box(), "few", missing=0.5), 256, 0, "kept"),
    "27_const_seldom": (lambda: grid_matrix(32, 32, 32, box(), "const", missing=0.9), 0, 0, "kept"),
    "31_const_hardly": (lambda: grid_matrix(32, 32, 32, P31, "const", missing=0.97), 0, 0, "interpolation"),
    # the first and the last plane have another diagonal: values come from inside
    "first_plane": (lambda: other_diagonal(slice(0, 1024)), 8, 0, "kept"),
    "last_plane": (lambda: other_diagonal(slice(31 * 1024, 32 * 1024)), 8, 0, "kept"),
}


def report_forms():
    """Sets every matrix of FORMS up; the library reports to stderr."""
    from hypre_amd import api
    api.initialize()
    for name, (matrix, *_) in FORMS.items():
        A = api.ParCSRMatrix.from_csr(*matrix())
        print("[form]", name, file=sys.stderr, flush=True)
        api.BoomerAMG(max_levels=2).setup(A)


def test_form_of_the_slices():
    """Which slices keep codes and full values, as HYPRE_MI355X_VERBOSE reports."""
    here = os.path.dirname(os.path.abspath(__file__))
    r = subprocess.run([sys.executable, "-c", "import test_gpu_stencil_copy as t; t.report_forms()"],
                       capture_output=True, text=True, timeout=110, cwd=here,
                       env=dict(os.environ, HYPRE_MI355X_VERBOSE="1", PYTHONPATH=os.path.dirname(here)))
    assert r.returncode == 0, r.stderr
    got = re.findall(r"\[form\] (\w+)\n.*?(\d+) with codes, (\d+) in full: (\w+)", r.stderr)
    assert got == [(name, *map(str, want)) for name, (_, *want) in FORMS.items()]
