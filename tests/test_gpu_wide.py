"""Adaptive builds whose columns reach the workgroup-per-column kernel, at the
edges of the sizes it takes: the oracle's bits, with and without counters."""
import os

import numpy as np
import pytest
import scipy.sparse as sp

from mspai_amd import gen
from tests.util import same_csc_bitwise

pytestmark = pytest.mark.gpu
THREADS = min(16, os.cpu_count() or 1)
WIDE_TABLE = 12  # 64-lane bins to |I| <= 128, then the workgroup bin, then the generic kernel


def band(n, nnz, bw, seed, equal=False, heavy=1):
    """n columns of nnz entries within bw of the diagonal, which dominates all
    but every heavy-th column (those grow)."""
    rng = np.random.Generator(np.random.PCG64(seed))
    cols = np.repeat(np.arange(n), nnz)
    rows = np.clip(cols + rng.integers(-bw, bw + 1, cols.size), 0, n - 1)
    vals = np.ones(rows.size) if equal else rng.standard_normal(rows.size)
    vals[cols % heavy != 0] *= 1e-3
    A = sp.coo_matrix((vals, (rows, cols)), shape=(n, n)).tocsc()
    A.sum_duplicates()
    if equal:
        A.data[:] = 1.0
    A = (A + sp.identity(n) * (6.0 if equal else 3.0)).tocsc()
    A.sort_indices()
    return A


def scattered(n, heavy, nnz, seed):
    """The identity with `heavy` columns of nnz far-apart entries: candidates
    over a range that no bitmap in LDS holds."""
    rng = np.random.Generator(np.random.PCG64(seed))
    cols = np.repeat(rng.choice(n, heavy, replace=False), nnz)
    rows = rng.integers(0, n, cols.size)
    A = sp.coo_matrix((rng.standard_normal(cols.size), (rows, cols)), shape=(n, n)).tocsc()
    A = (A + A.T + sp.identity(n) * 4.0).tocsc()
    A.sum_duplicates()
    A.sort_indices()
    return A


CASES = {
    "rows_to_384": (lambda: band(1200, 30, 500, 1), dict(epsilon=0.05, maxnew=5, max_impr_steps=3)),
    "rows_past_384": (lambda: band(1500, 60, 700, 2), dict(epsilon=0.05, maxnew=4, max_impr_steps=3)),
    "columns_past_40": (lambda: band(900, 6, 60, 3), dict(epsilon=0.01, maxnew=7, max_impr_steps=7)),
    "candidates_past_4096": (lambda: band(12000, 26, 5900, 4, heavy=60), dict(epsilon=0.1, maxnew=3, max_impr_steps=4)),
    "ties_at_the_cut": (lambda: band(600, 40, 90, 5, equal=True), dict(epsilon=0.05, maxnew=3, max_impr_steps=2)),
    "range_past_the_bitmap": (lambda: scattered(700_000, 20, 200, 6),
                              dict(epsilon=0.05, maxnew=3, max_impr_steps=2)),
    "target": (lambda: band(700, 20, 200, 7), dict(max_impr_steps=0)),  # a static build on A's pattern
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_wide_bitwise(oracle, gpu, name):
    make, opts = CASES[name]
    A = make()
    n = A.shape[0]
    B, P = None, gen.pattern_of(sp.identity(n, format="csc"))
    if name == "target":
        rng = np.random.Generator(np.random.PCG64(8))
        d = np.arange(n)
        B = gen._csc(np.concatenate([d, (d * 3 + 1) % n]), np.concatenate([d, d]),
                     np.concatenate([np.ones(n), 0.2 * rng.standard_normal(n)]), (n, n))
        P = gen.pattern_of(A)
    prob = gen.Problem(name, A, P, B, **opts)
    ref = oracle.spai(prob, threads=THREADS)
    Mref = oracle.to_csc(ref, n)
    b = gpu.Builder(0)
    try:
        b.upload(prob.A, prob.row_pattern())
        b.set_pattern(prob.P)
        if B is not None:
            b.set_target(B)
        b.set_bin_table(WIDE_TABLE, precision=0)
        for counters in (1, 0):
            print(f"[wide {name} counters={counters}]", flush=True)
            b.build(binning=2, counters=counters, **opts)
            info = b.column_info()
            if counters:
                ls = {x["name"]: int(x["columns"]) for x in b.launch_stats()}
                print(f"   {ls}", flush=True)
                assert any("G=512" in k for k in ls)
                assert sum(ls.values()) == n
            assert same_csc_bitwise(Mref, b.download())
            assert np.array_equal(ref["res_norm"].view(np.int64), info["res_norm"].view(np.int64))
            assert np.array_equal(ref["nsolve"], info["nsolve"])
            assert np.array_equal(ref["status"], info["status"])
    finally:
        b.close()
