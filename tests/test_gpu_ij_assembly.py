"""IJ assembly on the device against the serial rule, entry for entry.

Calls of at least 32768 operations (and assemblies of that many staged ones)
are assembled on the device.  The rule: a row's columns stand in the order of
their first operation, a later SetValues overwrites, a later AddToValues adds,
in call order, and the diagonal comes first (moved up, or swapped with the
first entry after SetDiagOffdSizes).  Here it is played out in Python.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def serial(lo, hi, jlo, calls, swap=False):
    rows = [dict() for _ in range(hi - lo + 1)]
    for op, rw, nc, cl, vl in calls:
        k = 0
        for r, m in zip(rw, nc):
            for c, v in zip(cl[k:k + m], vl[k:k + m]):
                if lo <= r <= hi:
                    d = rows[r - lo]
                    d[c] = d[c] + v if op == "add" and c in d else v
            k += m
    ia, ja, a = [0], [], []
    for i, d in enumerate(rows):
        e = [(c - jlo, v) for c, v in d.items()]
        at = next((q for q, (c, _) in enumerate(e) if c == i + lo - jlo), None)
        if at:
            if swap:
                e[0], e[at] = e[at], e[0]
            else:
                e.insert(0, e.pop(at))
        ja += [c for c, _ in e]
        a += [v for _, v in e]
        ia.append(len(ja))
    return np.array(ia), np.array(ja), np.array(a)


def assembled(hx, lo, hi, jlo, jhi, calls, swap=False):
    m = hx.IJMatrix(lo, hi, jlo, jhi)
    if swap:
        m.set_diag_offd_sizes(np.ones(hi - lo + 1))
    m.initialize()
    for op, rw, nc, cl, vl in calls:
        (m.set_values if op == "set" else m.add_to_values)(rw, nc, cl, vl)
    m.assemble()
    return m


def check(hx, lo, hi, jlo, jhi, calls, swap=False):
    m = assembled(hx, lo, hi, jlo, jhi, calls, swap)
    G = m.get_object().to_host()
    ia, ja, a = serial(lo, hi, jlo, calls, swap)
    assert np.array_equal(G.ia, ia) and np.array_equal(G.ja, ja)
    assert np.array_equal(G.a.view(np.int64), a.view(np.int64))
    return m, (ia, ja, a)


def random_call(rng, op, rows, jlo, jhi, most, distinct=True):
    nc = rng.integers(0, most + 1, len(rows))
    if distinct:
        cl = np.concatenate([rng.choice(np.arange(jlo, jhi + 1), m, replace=False) for m in nc])
    else:
        cl = rng.integers(jlo, jhi + 1, nc.sum())
    return op, np.asarray(rows), nc, cl.astype(np.int32), rng.standard_normal(nc.sum())


@pytest.mark.parametrize("swap", [False, True])
@pytest.mark.parametrize("name", ["once", "shuffled_rows", "duplicates", "repeated_rows", "two_large",
                                  "small_between", "long_rows", "outside_rows", "offset_range", "many_large"])
def test_device_assembly_follows_the_serial_rule(hx, name, swap):
    print("[gpu-ij-assembly]", name, swap, flush=True)
    rng = np.random.default_rng(3)
    n, lo, jlo = 3000, 0, 0
    if name == "offset_range":
        lo = jlo = 7
    hi, jhi = lo + n - 1, jlo + n - 1
    rows = np.arange(lo, hi + 1)
    if name == "shuffled_rows":
        rows = rng.permutation(rows)
    calls = [random_call(rng, "set", rows, jlo, jhi if name != "duplicates" else jlo + 30, 27, name != "duplicates")]
    if name == "repeated_rows":
        calls = [random_call(rng, "add", rng.integers(lo, hi + 1, 3 * n), jlo, jlo + 80, 14, False)]
    elif name == "two_large":
        calls.append(random_call(rng, "add", rng.permutation(rows), jlo, jhi, 27))
        calls.append(random_call(rng, "set", rows, jlo, jhi, 24))
    elif name == "small_between":
        calls.insert(0, random_call(rng, "add", rows[:50], jlo, jhi, 9))
        calls.append(random_call(rng, "set", rows[20:90], jlo, jhi, 9))
        calls.append(random_call(rng, "add", rows, jlo, jhi, 27))
        calls.append(random_call(rng, "add", rows[::7], jlo, jhi, 5))
    elif name == "long_rows":
        calls = [random_call(rng, op, rows[:120], jlo, jlo + 700, 600, False) for op in ("add", "set", "add")]
    elif name == "outside_rows":
        calls = [random_call(rng, "set", np.arange(-20, n + 30), jlo, jhi, 27)]
    elif name == "many_large":
        calls = [random_call(rng, "add", rng.integers(lo, hi + 1, 300), jlo, jlo + 2000, 250) for _ in range(40)]
        assert sum(c[2].sum() >= 32768 for c in calls) > 32
    assert sum(int(c[2].sum()) for c in calls) >= 32768
    check(hx, lo, hi, jlo, jhi, calls, swap)


def test_many_small_element_calls(hx):
    """8 x 8 element matrices of a 12^3 grid, one AddToValues call each."""
    rng = np.random.default_rng(5)
    e, n = 12, 13 ** 3
    calls = []
    for k in range(e ** 3):
        z, y, x = np.unravel_index(k, (e, e, e))
        at = [((z + dz) * 13 + y + dy) * 13 + x + dx for dz in (0, 1) for dy in (0, 1) for dx in (0, 1)]
        calls.append(("add", np.array(at), np.full(8, 8), np.tile(at, 8).astype(np.int32), rng.standard_normal(64)))
    check(hx, 0, n - 1, 0, n - 1, calls)


def test_values_after_assembly(hx):
    """GetValues, an update of the assembled pattern and reassembly."""
    rng = np.random.default_rng(7)
    n = 3000
    calls = [random_call(rng, "set", np.arange(n), 0, n - 1, 27)]
    m, (ia, ja, a) = check(hx, 0, n - 1, 0, n - 1, calls)
    r = int(np.argmax(np.diff(ia)))
    cols = ja[ia[r]:ia[r + 1]].astype(np.int32)
    m.add_to_values([r], [len(cols)], cols, np.ones(len(cols)))
    with pytest.raises(hx.HypreError):
        m.add_to_values([r], [1], [int(np.setdiff1d(np.arange(n), cols)[0])], [1.0])
    m.assemble()
    G = m.get_object().to_host()
    want = a.copy()
    want[ia[r]:ia[r + 1]] += 1.0
    assert np.array_equal(G.ja, ja) and np.array_equal(G.a, want)


def test_column_outside_the_range_is_refused(hx):
    rng = np.random.default_rng(9)
    call = random_call(rng, "set", np.arange(3000), 0, 2999, 27)
    call[3][100] = 3000
    with pytest.raises(hx.HypreError) as e:
        assembled(hx, 0, 2999, 0, 2999, [call])
    assert e.value.code & hx.ERROR_GENERIC


class DeviceArray:
    """A device array of the library as torch sees it."""

    def __init__(self, ptr, n, typestr):
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": typestr, "data": (ptr, False), "version": 2}


def test_assembled_arrays_are_complete_on_return(hx):
    """The device arrays, read at once on a stream of the caller's: torch's
    stream and the library's are not ordered.  Memory is recycled between the
    rounds, so each round has values and columns of its own."""
    import ctypes

    import torch
    n, m = 400_000, 27
    for k in range(4):
        print("[gpu-ij-assembly] complete", k, flush=True)
        cols = ((np.arange(n)[:, None] + (k + 1) * np.arange(m)) % n).astype(np.int32)
        vals = np.random.default_rng(k).standard_normal(n * m)
        want = torch.from_numpy(vals).cuda(), torch.from_numpy(cols.reshape(-1)).cuda()
        torch.cuda.synchronize()
        M = hx.IJMatrix(0, n - 1)
        M.initialize()
        M.set_values(np.arange(n), np.full(n, m), cols.reshape(-1), vals)     # the diagonal stands first
        M.assemble()
        rows, nnz, ja, a = ctypes.c_int(), ctypes.c_int(), ctypes.c_void_p(), ctypes.c_void_p()
        hx.call("HYPRE_MI355X_ParCSRMatrixGetDevice", M.get_object().h, ctypes.byref(rows), ctypes.byref(nnz),
                None, ctypes.byref(ja), ctypes.byref(a))
        assert (rows.value, nnz.value) == (n, n * m)
        got = [torch.as_tensor(DeviceArray(p.value, n * m, t), device="cuda").clone()
               for p, t in ((a, "<f8"), (ja, "<i4"))]
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
        M.destroy()


@pytest.mark.parametrize("rows", [3000, 30])
def test_negative_row_lengths_have_no_entries(hx, rows):
    """In large calls, whose prefix sums must not run backwards, and small."""
    rng = np.random.default_rng(11)
    op, rw, nc, cl, vl = random_call(rng, "add", np.arange(rows), 0, 2999, 27)
    none = rng.random(rows) < 0.1
    keep = np.repeat(~none, nc)
    given = ("add", rw, np.where(none, -rng.integers(1, 9, rows), nc), cl[keep], vl[keep])
    same = ("add", rw, np.where(none, 0, nc), cl[keep], vl[keep])
    m = assembled(hx, 0, 2999, 0, 2999, [given, ("set", rw, np.ones(rows, int), rw.astype(np.int32), vl[:rows])])
    ia, ja, a = serial(0, 2999, 0, [same, ("set", rw, np.ones(rows, int), rw.astype(np.int32), vl[:rows])])
    G = m.get_object().to_host()
    assert np.array_equal(G.ia, ia) and np.array_equal(G.ja, ja) and np.array_equal(G.a, a)


def long_row_calls(name, rng):
    """Calls on n rows and columns with one or some long rows."""
    n, at = 6000, 2500
    band = (np.arange(n)[:, None] + np.arange(-4, 5)) % n
    base = ("set", np.arange(n), np.full(n, 9), band.reshape(-1).astype(np.int32), rng.standard_normal(9 * n))

    def row(op, cols, segs=None):
        segs = np.array([len(cols)]) if segs is None else segs
        return op, np.full(len(segs), at), segs, np.asarray(cols, np.int32), rng.standard_normal(len(cols))
    if name == "dense":
        return n, [base, row("add", rng.permutation(n))]
    if name == "duplicates":
        return n, [row("add", rng.integers(0, 1500, 20000)), base, row("set", rng.integers(0, 1500, 900)),
                   row("add", rng.integers(700, 2200, 20000))]
    if name == "one_column":
        return n, [base, row("add", np.full(5000, 7)), row("add", np.full(3000, at), np.ones(3000, int))]
    if name == "no_diagonal":
        return n, [("set", *[np.delete(v, at, 0) for v in base[1:3]], np.delete(base[3].reshape(n, 9), at, 0).ravel(),
                    base[4][9:]), row("set", np.delete(np.arange(n), at)[::-1])]
    if name == "segments":              # of 0 to 5 operations
        segs = rng.integers(0, 6, 5000)
        return n, [base, row("add", rng.integers(0, n, segs.sum()), segs)]
    if name == "edges":                 # rows of n operations, and as many segments
        rw, nc = [], []
        for r, m in enumerate((255, 256, 257, 1023, 1024, 1025, 2049, 4096)):
            rw += [r] + [100 + r] * m + [200 + r] * (m + 1)
            nc += [m] + [1] * m + [1] + [0] * m
        cl = rng.integers(0, 3000, sum(nc))
        return n, [("add", np.array(rw), np.array(nc), cl.astype(np.int32), rng.standard_normal(len(cl))), base]
    assert name == "apart"              # many segments, far apart: several windows, cut at all places
    rw = np.where(rng.random(700_000) < 0.02, at, rng.integers(0, n, 700_000))
    return n, [("add", rw, np.ones(len(rw), int), rng.integers(0, n, len(rw)).astype(np.int32),
                rng.standard_normal(len(rw)))]


@pytest.mark.parametrize("swap", [False, True])
@pytest.mark.parametrize("name", ["dense", "duplicates", "one_column", "no_diagonal", "segments", "edges", "apart"])
def test_long_rows_follow_the_serial_rule(hx, name, swap):
    """Rows over 256 operations or segments are taken by blocks."""
    print("[gpu-ij-assembly] long", name, swap, flush=True)
    n, calls = long_row_calls(name, np.random.default_rng(13))
    if name == "apart":
        at = np.nonzero(calls[0][1] == 2500)[0]
        assert len(at) > 8192 and at[-1] - at[0] > 2 * 262144
    check(hx, 0, n - 1, 0, n - 1, calls, swap)


def test_long_row_by_many_small_calls(hx):
    rng = np.random.default_rng(17)
    n = 4000
    cols = np.concatenate([rng.permutation(n) for _ in range(9)]).astype(np.int32)
    calls = [("add" if k % 7 else "set", [3 if k % 8 else k % n], [1], cols[k:k + 1], rng.standard_normal(1))
             for k in range(len(cols))]
    check(hx, 0, n - 1, 0, n - 1, calls)


def test_column_outside_the_range_in_a_long_row_is_refused(hx):
    n, calls = long_row_calls("dense", np.random.default_rng(19))
    calls[1][3][4000] = n
    with pytest.raises(hx.HypreError) as e:
        assembled(hx, 0, n - 1, 0, n - 1, calls)
    assert e.value.code & hx.ERROR_GENERIC
