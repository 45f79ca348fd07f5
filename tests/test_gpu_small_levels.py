"""Setup kernels at the edges of their small-matrix forms, bits of the oracle.

Matrices of up to 16384 rows are scanned by one block, independent-set rounds
of at most 1024 rows run in one block (where they have few entries), and the rows
a wave or block of the strength kernels takes shrink with the matrix.  Sizes stand
on both sides of each, with rows of 3 and 24 entries, and of 150 up to 1025 rows
and 100 at 4097; `hub` rows all depend on three points, whose rows of S^T are
longer than one wave.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def irregular(n, length, hub, seed=7):
    """Diagonal first, then ascending columns; a symmetric pattern with
    unsymmetric values of mixed size, a tenth of them positive."""
    import scipy.sparse as sp
    rng = np.random.default_rng(seed)
    m = n * length // 2
    i, j = rng.integers(0, n, m), rng.integers(0, n, m)
    near = rng.random(m) < 0.8          # most couplings local, the rest anywhere
    j[near] = np.clip(i[near] + rng.integers(-2 * length, 2 * length + 1, near.sum()), 0, n - 1)
    i, j = np.concatenate([i, j]), np.concatenate([j, i])
    if hub:
        i, j = np.concatenate([i, np.arange(n)]), np.concatenate([j, np.arange(n) % 3])
    keep = i != j
    off = sp.csr_matrix((np.ones(keep.sum()), (i[keep], j[keep])), shape=(n, n))
    off.sort_indices()
    v = -rng.random(off.nnz) * np.where(rng.random(off.nnz) < 0.1, -0.3, 1.0)
    ia = np.zeros(n + 1, np.int32)
    ia[1:] = np.cumsum(np.diff(off.indptr) + 1)
    first = ia[:-1]
    ja, a = np.empty(ia[-1], np.int32), np.empty(ia[-1])
    rest = np.ones(ia[-1], bool)
    rest[first] = False
    ja[rest], a[rest] = off.indices, v
    ja[first] = np.arange(n)
    a[first] = 0.1 + np.bincount(np.repeat(np.arange(n), np.diff(off.indptr)), np.abs(v), minlength=n)
    return ia, ja, a


# rows of 150 on the larger sizes are left out for the oracle's time
SIZES = [(n, length) for n in (1, 5, 63, 65, 1023, 1024, 1025, 4097, 16383, 16384, 16385) for length in (3, 24, 150)
         if n * length <= 1 << 19] + [(4097, 100)]


@pytest.mark.parametrize("hub", [False, True])
@pytest.mark.parametrize("n,length", SIZES)
def test_strength_split_and_interpolation(hx, oracle, n, length, hub):
    ia, ja, a = irregular(n, length, hub)
    A_or, A = oracle.Csr(n, n, ia, ja, a), hx.HostCsr(n, n, ia, ja, a)
    print("[small]", n, length, hub, len(ja), flush=True)
    S_or = oracle.strength(A_or, 0.25, 0.9)
    S = hx.create_s(A, 0.25, 0.9)
    assert np.array_equal(S.ia, S_or.ia) and np.array_equal(S.ja, S_or.ja)
    cf_or, rounds_or = oracle.pmis(S_or)
    cf, rounds = hx.pmis(S)             # the first round is counted on an empty graph too
    assert np.array_equal(cf, cf_or) and rounds == max(rounds_or, 1)
    h_or, rounds_or = oracle.hmis(S_or)
    h, rounds = hx.hmis(S)
    assert np.array_equal(h, h_or) and rounds == max(rounds_or, 1)
    P_or, cf_or = oracle.extpi_interp(A_or, S_or, cf_or, 0.0, 4)
    P, cf = hx.extpi_interp(A, S, cf, 0.0, 4)
    assert np.array_equal(cf, cf_or)
    assert np.array_equal(P.ia, P_or.ia) and np.array_equal(P.ja, P_or.ja)
    assert np.array_equal(P.a, P_or.a)
