"""Precision 1 against an extended-precision solution of each column (64-bit
mantissa): the refinement step must bring the values closer to it than the
FP64 QR alone leaves them, whichever kernel finishes the column.

A refined entry is off by its own rounding, at most u = 2^-53 of the column's
largest entry, and by the rounding of the residual it was refined with (of
the same size on these well-conditioned columns); an unrefined one by the
rounding errors of |J| reflectors.  So the mean over many columns of the
largest error of a column has to be below u, and below half of FP64's.
"""
import numpy as np
import pytest
import scipy.sparse as sp
import torch  # before the library: one HIP runtime per process  # noqa: F401

from mspai_amd import gen

pytestmark = pytest.mark.gpu
U = 2.0 ** -53


def extended_lstsq(A, b):
    """Least-squares solution by Householder QR in long double."""
    assert np.finfo(np.longdouble).nmant >= 63
    A, b = A.astype(np.longdouble), b.astype(np.longdouble)
    n = A.shape[1]
    for i in range(n):
        v = A[i:, i].copy()
        v[0] += np.copysign(np.sqrt((v * v).sum()), v[0])
        v /= np.sqrt((v * v).sum())
        A[i:, i:] -= 2 * np.outer(v, v @ A[i:, i:])
        b[i:] -= 2 * v * (v @ b[i:])
    x = np.zeros(n, np.longdouble)
    for i in range(n - 1, -1, -1):
        x[i] = (b[i] - A[i, i + 1:] @ x[i + 1:]) / A[i, i]
    return x


def column_system(A, J, k):
    sub = A[:, J]
    I = np.unique(sub.indices)
    return sub[I, :].toarray(), (I == k).astype(float), I.size


def column_errors(A, M, cols):
    """Largest error of each column's values, relative to its largest entry."""
    out = []
    for k in cols:
        a, b = M.indptr[k], M.indptr[k + 1]
        Ah, rhs, _ = column_system(A, M.indices[a:b], k)
        x = extended_lstsq(Ah, rhs)
        out.append(float(np.abs(M.data[a:b] - x).max() / np.abs(x).max()))
    return np.array(out)


def assert_refined(e0, e1):
    print(f"   {e0.size} columns, mean error FP64 {e0.mean():.2e}, precision 1 {e1.mean():.2e}", flush=True)
    assert e1.mean() <= U and e1.mean() <= 0.5 * e0.mean()


def test_adaptive_columns_of_the_workgroup_kernel(gpu):
    """Columns of more than 128 rows, which a mixed chain finishes in the
    workgroup kernel."""
    prob = gen.config3(n=32768, bw=2000)
    opts = dict(epsilon=prob.epsilon, maxnew=prob.maxnew, max_impr_steps=prob.max_impr_steps)
    b = gpu.Builder(0)
    try:
        b.upload(prob.A, prob.row_pattern())
        b.set_pattern(prob.P)
        M = []
        for precision in (0, 1):
            print(f"[refined workgroup columns precision={precision}]", flush=True)
            b.set_bin_table(12, precision=precision)
            b.build(binning=2, precision=precision, **opts)
            M.append(b.download())
        fallback = b.column_info()["status"] & 8
    finally:
        b.close()
    assert np.array_equal(M[0].indptr, M[1].indptr) and np.array_equal(M[0].indices, M[1].indices)
    rows = np.array([np.unique(prob.A[:, M[0].indices[M[0].indptr[k]:M[0].indptr[k + 1]]].indices).size
                     for k in range(0, prob.n, 2)])
    wide = [2 * t for t in np.flatnonzero(rows > 128) if not fallback[2 * t]][:80]
    assert len(wide) >= 40
    assert_refined(column_errors(prob.A, M[0], wide), column_errors(prob.A, M[1], wide))


def given_pattern_problem(lens, nnz, band, seed=0, n=400):
    """n columns of `nnz` entries within `band` of a dominant diagonal; column
    k's pattern holds lens[k % len(lens)] indices around k."""
    rng = np.random.Generator(np.random.PCG64(seed))
    rows, cols, vals, ptr, ind = [], [], [], [0], []
    for j in range(n):
        near = np.arange(max(0, j - band), min(n, j + band + 1))
        r = np.union1d(rng.choice(near, size=min(near.size, nnz), replace=False), [j])
        v = rng.standard_normal(r.size)
        v[r == j] = 4.0
        rows.append(r), cols.append(np.full(r.size, j)), vals.append(v)
        want = lens[j % len(lens)]
        near = np.setdiff1d(np.arange(max(0, j - want), min(n, j + want + 1)), [j])
        ind.append(np.union1d(rng.choice(near, size=want - 1, replace=False), [j]).astype(np.int64))
        ptr.append(ptr[-1] + want)
    A = gen._csc(np.concatenate(rows), np.concatenate(cols), np.concatenate(vals), (n, n))
    P = sp.csc_matrix((np.ones(ptr[-1]), np.concatenate(ind), ptr), shape=(n, n))
    return gen.Problem("given", A, P, None, max_impr_steps=0)


STATIC = {  # pattern lengths, entries of a column; the columns' |I|
    "kinds": ((7, 15, 31), 2, (1, 64)),
    "rows_65_to_128": ((20, 24, 30), 5, (65, 128)),
    "columns_32_to_40": ((32, 36, 40), 2, (33, 128)),
    "rows_129_to_384": ((24, 36, 40), 14, (129, 384)),
}


@pytest.mark.parametrize("name", sorted(STATIC))
def test_static_columns(gpu, name):
    lens, nnz, (lo, hi) = STATIC[name]
    prob = given_pattern_problem(lens, nnz, 100)
    b = gpu.Builder(0)
    try:
        b.upload(prob.A, prob.row_pattern())
        b.set_pattern(prob.P)
        M = []
        for precision in (0, 1):
            print(f"[refined static {name} precision={precision}]", flush=True)
            b.build(max_impr_steps=0, precision=precision)
            M.append(b.download())
    finally:
        b.close()
    size = [column_system(prob.A, M[0].indices[M[0].indptr[k]:M[0].indptr[k + 1]], k)[2] for k in range(prob.n)]
    cols = [k for k in range(prob.n) if lo <= size[k] <= hi][::3]
    assert len(cols) >= 60
    assert_refined(column_errors(prob.A, M[0], cols), column_errors(prob.A, M[1], cols))


def extended_adjoint(A, g):
    """A lambda with A^T A lambda = g, by the R of a long double QR."""
    A0, A = A.astype(np.longdouble), A.astype(np.longdouble)
    n = A.shape[1]
    for i in range(n):
        v = A[i:, i].copy()
        v[0] += np.copysign(np.sqrt((v * v).sum()), v[0])
        v /= np.sqrt((v * v).sum())
        A[i:, i:] -= 2 * np.outer(v, v @ A[i:, i:])
    lam = g.astype(np.longdouble)
    for i in range(n):
        lam[i] = (lam[i] - A[:i, i] @ lam[:i]) / A[i, i]
    for i in range(n - 1, -1, -1):
        lam[i] = (lam[i] - A[i, i + 1:n] @ lam[i + 1:]) / A[i, i]
    return A0 @ lam


@pytest.mark.parametrize("name", ["kinds", "rows_65_to_128", "columns_32_to_40"])
def test_adjoint_columns(gpu, name):
    """dL/dB(:, k) = C lambda over I, one column's own values: a target with
    every row of I in it gives all of them.  The step removes what the QR and
    the two triangular solves left; what remains is the rounding of C lambda
    and C^T (C lambda): on average below three quarters of FP64's error."""
    lens, nnz, (lo, hi) = STATIC[name]
    prob = given_pattern_problem(lens, nnz, 100, n=300)
    n, P = prob.n, prob.P
    J = [P.indices[P.indptr[k]:P.indptr[k + 1]] for k in range(n)]
    I = [np.unique(prob.A[:, J[k]].indices) for k in range(n)]
    B = gen._csc(np.concatenate(I), np.repeat(np.arange(n), [i.size for i in I]),
                 np.concatenate([(i == k) + 0.0 for k, i in enumerate(I)]), (n, n))
    assert B.nnz == sum(i.size for i in I)  # the zeros are stored
    g = np.random.Generator(np.random.PCG64(5)).standard_normal(P.nnz)
    b = gpu.Builder(0)
    gbs = []
    try:
        b.upload(prob.A, prob.row_pattern())
        b.set_pattern(P)
        b.set_target(B)
        gm = torch.tensor(g, device="cuda")
        gc = torch.empty(prob.A.nnz, dtype=torch.float64, device="cuda")
        gb = torch.empty(B.nnz, dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        for precision in (0, 1):
            print(f"[refined adjoint {name} precision={precision}]", flush=True)
            b.build(max_impr_steps=0, precision=precision)
            b.backward_device(gm.data_ptr(), gc.data_ptr(), gb.data_ptr(), precision=precision)
            gbs.append(gb.cpu().numpy())
    finally:
        b.close()
    e = [[], []]
    for k in [k for k in range(n) if lo <= I[k].size <= hi][::3]:
        exact = extended_adjoint(prob.A[:, J[k]][I[k], :].toarray(), g[P.indptr[k]:P.indptr[k + 1]])
        for p in (0, 1):
            d = gbs[p][B.indptr[k]:B.indptr[k + 1]] - exact
            e[p].append(float(np.abs(d).max() / np.abs(exact).max()))
    assert len(e[0]) >= 50
    e0, e1 = np.mean(e[0]), np.mean(e[1])
    print(f"   {len(e[0])} columns, mean error FP64 {e0:.2e}, precision 1 {e1:.2e}", flush=True)
    assert e1 <= 0.75 * e0
