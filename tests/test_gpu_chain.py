"""The chain of an untuned build: which bins it begins with, and grid operators
whose first bin holds all but a few columns (M is assembled after that bin and
again once the chain has built the others)."""
import os

import numpy as np
import pytest
import scipy.sparse as sp

from mspai_amd import gen
from tests.util import same_csc_bitwise

pytestmark = pytest.mark.gpu
THREADS = min(16, os.cpu_count() or 1)


def grid_with_heavy_columns(m, heavy, nnz, seed):
    """A 2D transport operator, `heavy` columns of which have nnz more entries."""
    P = gen.config2(m)
    n = P.n
    if not heavy:
        return P
    rng = np.random.Generator(np.random.PCG64(seed))
    cols = np.repeat(rng.choice(n, heavy, replace=False), nnz)
    rows = rng.integers(0, n, cols.size)
    E = sp.coo_matrix((0.3 * rng.standard_normal(cols.size), (rows, cols)), shape=(n, n))
    A = (P.A + E).tocsc()
    A.sum_duplicates()
    A.sort_indices()
    return gen.Problem(P.name, A, P.P, None, epsilon=P.epsilon, maxnew=P.maxnew, max_impr_steps=P.max_impr_steps)


def band(k_off):
    A = gen.random_band(3000, k_off=k_off, bw=300, seed=9)
    return gen.Problem("random_band", A, gen.diag_pattern(3000), None, epsilon=0.3, maxnew=4, max_impr_steps=8)


CASES = {
    "none_moves_on": lambda: grid_with_heavy_columns(40, 0, 0, 0),
    "one_moves_on": lambda: grid_with_heavy_columns(48, 1, 6, 1),
    "some_reach_every_bin": lambda: grid_with_heavy_columns(64, 12, 9, 2),
    "lists_about_the_rule_below": lambda: band(10),  # lists of 121
    "lists_about_the_rule_above": lambda: band(11),  # lists of 144
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_untuned_chain(oracle, gpu, name):
    prob = CASES[name]()
    opts = dict(epsilon=prob.epsilon, maxnew=prob.maxnew, max_impr_steps=prob.max_impr_steps)
    ref = oracle.spai(prob, threads=THREADS)
    Mref = oracle.to_csc(ref, prob.n)
    b = gpu.Builder(0)
    try:
        b.upload(prob.A, prob.row_pattern())
        b.set_pattern(prob.P)
        for precision in (0, 0, 1):
            print(f"[chain {name} precision={precision}]", flush=True)
            st = b.build(precision=precision, **opts)
            M, info = b.download(), b.column_info()
            print(f"   moved on {st['n_overflow']}, declined {st['n_fallback']}", flush=True)
            assert 0.0 < st["first_bin_ms"] <= st["solve_ms"] <= st["build_ms"]
            assert st["nnz"] == Mref.nnz
            assert np.array_equal(Mref.indptr, M.indptr) and np.array_equal(Mref.indices, M.indices)
            assert np.array_equal(ref["nsolve"], info["nsolve"])
            if precision == 0:
                assert same_csc_bitwise(Mref, M)
                assert np.array_equal(ref["res_norm"].view(np.int64), info["res_norm"].view(np.int64))
                assert np.array_equal(ref["status"], info["status"])
            else:
                # every column within 1e-10 of FP64's; the declined ones are FP64's
                err = np.abs(M.data - Mref.data)
                big = np.maximum.reduceat(np.abs(Mref.data), Mref.indptr[:-1])
                assert (np.maximum.reduceat(err, Mref.indptr[:-1]) <= 1e-10 * big).all()
                assert ((info["status"] & 8) != 0).sum() == st["n_fallback"]
    finally:
        b.close()
