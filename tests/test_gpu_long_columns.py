"""Matrices with a few columns of 10,000 entries: the kernels whose working set
cannot hold such a column pass it on at once (the launches are timed: reading
and inserting every entry takes 13 to 27 ms in the given-pattern kernels and
1.9 ms in the workgroup kernel), and the results are the oracle's bits."""
import os

import numpy as np
import pytest
import scipy.sparse as sp
import torch  # before the library: one HIP runtime per process

from mspai_amd import gen
from tests.util import same_csc_bitwise

pytestmark = pytest.mark.gpu
THREADS = min(16, os.cpu_count() or 1)
N, ENTRIES = 12_000, 10_000


def matrix(seed=1):
    """A tridiagonal matrix, three columns of which have ENTRIES small entries."""
    rng = np.random.Generator(np.random.PCG64(seed))
    A = sp.diags([rng.standard_normal(N - 1), np.full(N, 4.0), rng.standard_normal(N - 1)], [-1, 0, 1])
    heavy = [N // 4, N // 2, 3 * N // 4]
    rows = np.concatenate([rng.choice(N, ENTRIES, replace=False) for _ in heavy])
    E = sp.coo_matrix((1e-3 * rng.standard_normal(rows.size), (rows, np.repeat(heavy, ENTRIES))), shape=(N, N))
    A = sp.csc_matrix(A + E)
    A.sum_duplicates()
    A.sort_indices()
    return A


def pattern(width):
    """`width` neighbouring indices around every column."""
    lo, hi = -((width - 1) // 2), width // 2
    return gen.pattern_of(sp.csc_matrix(sp.diags([np.ones(N - abs(d)) for d in range(lo, hi + 1)],
                                                 range(lo, hi + 1), shape=(N, N))))


@pytest.mark.parametrize("width", [1, 7, 15, 31])
def test_static_long_columns(oracle, gpu, width):
    prob = gen.Problem("long", matrix(), pattern(width), None, max_impr_steps=0)
    print(f"[long columns static |J|<={width}]", flush=True)
    ref = oracle.spai(prob, threads=THREADS)
    Mref = oracle.to_csc(ref, N)
    b = gpu.Builder(0)
    try:
        b.upload(prob.A, prob.row_pattern())
        b.set_pattern(prob.P)
        for _ in range(2):
            b.build(max_impr_steps=0)
        ms = sum(x["ms"] for x in b.launch_stats() if "given pattern" in x["name"])
        assert same_csc_bitwise(Mref, b.download())
        g = np.random.Generator(np.random.PCG64(5)).standard_normal(Mref.nnz)
        gm = torch.tensor(g, device="cuda")
        gc = torch.empty(prob.A.nnz, dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        b.backward_device(gm.data_ptr(), gc.data_ptr())
        ms_back = sum(x["ms"] for x in b.launch_stats() if "given pattern" in x["name"])
    finally:
        b.close()
    print(f"   given-pattern launches {ms:.3f} ms, adjoint {ms_back:.3f} ms", flush=True)
    ref_c, _ = oracle.backward(prob, Mref, g, threads=THREADS)
    assert np.linalg.norm(gc.cpu().numpy() - ref_c) <= 1e-11 * np.linalg.norm(ref_c)
    assert ms <= 2.0 and ms_back <= 2.0


def test_adaptive_long_columns(oracle, gpu):
    opts = dict(epsilon=0.05, maxnew=3, max_impr_steps=2)
    prob = gen.Problem("long", matrix(), gen.diag_pattern(N), None, **opts)
    print("[long columns adaptive]", flush=True)
    ref = oracle.spai(prob, threads=THREADS)
    b = gpu.Builder(0)
    try:
        b.upload(prob.A, prob.row_pattern())
        b.set_pattern(prob.P)
        b.set_bin_table(12, precision=0)
        for _ in range(2):
            b.build(binning=2, **opts)
        ms = sum(x["ms"] for x in b.launch_stats() if "G=512" in x["name"])
        M = b.download()
    finally:
        b.close()
    print(f"   workgroup launch {ms:.3f} ms", flush=True)
    assert same_csc_bitwise(oracle.to_csc(ref, N), M)
    assert ms <= 0.5
