"""Static builds and the adjoint on the given-pattern kernels (builds without
work counters), at the edges of the sizes each kernel takes.

FP64 builds are the oracle's bits; precision 1 keeps the pattern and every
column within 1e-10 of it (a refinement step is taken only when it is no
larger); gradients against the CPU reference with the bars of the adjoint's
tests.
"""
import os

import numpy as np
import pytest
import scipy.sparse as sp
import torch  # before the library: one HIP runtime per process

from mspai_amd import gen
from tests.util import same_csc_bitwise

pytestmark = pytest.mark.gpu
THREADS = min(16, os.cpu_count() or 1)


def system(lens, nnz, band, n=400, seed=0, target=False, degenerate=False):
    """n columns of about `nnz` entries within `band` of a dominant diagonal;
    column k's pattern holds lens[k % len(lens)] indices around k."""
    rng = np.random.Generator(np.random.PCG64(seed))
    rows, cols, vals = [], [], []
    for j in range(n):
        lo, hi = max(0, j - band), min(n, j + band + 1)
        r = rng.choice(np.arange(lo, hi), size=min(hi - lo, int(rng.integers(1, 2 * nnz))), replace=False)
        r = np.union1d(r, [j])
        v = rng.standard_normal(r.size)
        v[r == j] = 8.0
        if degenerate and j % 5 == 0:
            v[:] = 0.0  # a zero pivot
        if degenerate and j % 7 == 0:
            r, v = np.array([j // 2]), np.array([1.0])  # fewer rows than columns, k not among them
        rows.append(r), cols.append(np.full(r.size, j)), vals.append(v)
    A = gen._csc(np.concatenate(rows), np.concatenate(cols), np.concatenate(vals), (n, n))
    ptr, ind = [0], []
    for k in range(n):
        want = lens[k % len(lens)]
        lo, hi = max(0, k - want), min(n, k + want + 1)
        pick = rng.choice(np.setdiff1d(np.arange(lo, hi), [k]), size=max(want - 1, 0), replace=False)
        J = np.union1d(pick, [k] if want else []).astype(np.int64)
        ind.append(J)
        ptr.append(ptr[-1] + J.size)
    P = sp.csc_matrix((np.ones(ptr[-1]), np.concatenate(ind), ptr), shape=(n, n))
    B = None
    if target:
        d = np.arange(n)
        B = gen._csc(np.concatenate([d, (d * 3 + 1) % n]), np.concatenate([d, d]),
                     np.concatenate([np.ones(n), rng.standard_normal(n)]), (n, n))
    return gen.Problem("edges", A, P, B, max_impr_steps=0)


CASES = {
    "one_kind_short": dict(lens=(0, 1, 5, 7), nnz=2, band=4),
    "rows_about_32": dict(lens=(7,), nnz=5, band=40),
    "rows_about_64": dict(lens=(15, 14, 9), nnz=5, band=200),
    "rows_about_64_wide": dict(lens=(31, 30, 16), nnz=2, band=100),
    "columns_past_8_entries": dict(lens=(7, 15), nnz=10, band=12),
    "routed_lengths": dict(lens=(1, 1, 1, 1, 7, 8, 15, 16, 31, 32, 40, 41, 60), nnz=3, band=30),
    "all_past_the_kinds": dict(lens=(33, 40, 48), nnz=4, band=50),
    "target": dict(lens=(5, 7, 6), nnz=3, band=6, target=True),
    "target_routed": dict(lens=(2, 2, 2, 12, 20, 31), nnz=3, band=20, target=True),
    "degenerate": dict(lens=(3, 6, 12, 20), nnz=2, band=9, degenerate=True),
    "tiny": dict(lens=(1, 2), nnz=1, band=1, n=3),
}


def build(gpu, prob, **opts):
    b = gpu.Builder(0)
    b.upload(prob.A, prob.row_pattern())
    b.set_pattern(prob.P)
    if prob.B is not None:
        b.set_target(prob.B)
    st = b.build(max_impr_steps=0, **opts)
    return b, st


@pytest.mark.parametrize("name", sorted(CASES))
def test_static_bitwise(oracle, gpu, name):
    prob = system(**CASES[name])
    print(f"[static {name}]", flush=True)
    ref = oracle.spai(prob, threads=THREADS)
    Mref = oracle.to_csc(ref, prob.n)
    b, st = build(gpu, prob)
    M, info = b.download(), b.column_info()
    b.close()
    print(f"   bins moved on {st['n_overflow']}", flush=True)
    assert same_csc_bitwise(Mref, M)
    assert np.array_equal(ref["res_norm"].view(np.int64), info["res_norm"].view(np.int64))
    assert np.array_equal(ref["nsolve"], info["nsolve"])
    assert np.array_equal(ref["status"], info["status"])
    b, st = build(gpu, prob, precision=1)
    M1, info1 = b.download(), b.column_info()
    b.close()
    assert np.array_equal(Mref.indptr, M1.indptr) and np.array_equal(Mref.indices, M1.indices)
    assert np.array_equal(ref["status"], info1["status"])
    for k in range(prob.n):
        x, y = Mref.data[Mref.indptr[k]:Mref.indptr[k + 1]], M1.data[M1.indptr[k]:M1.indptr[k + 1]]
        assert x.size == 0 or np.abs(x - y).max() <= 1.0000001e-10 * np.abs(x).max()


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("name", sorted(set(CASES) - {"degenerate"}))
def test_adjoint_edges(oracle, gpu, name, precision):
    prob = system(**CASES[name])
    print(f"[adjoint {name} precision={precision}]", flush=True)
    b, _ = build(gpu, prob, precision=precision)
    M = b.download()
    g = np.random.Generator(np.random.PCG64(5)).standard_normal(M.nnz)
    gm = torch.tensor(g, device="cuda")
    gc = torch.empty(prob.A.nnz, dtype=torch.float64, device="cuda")
    gb = torch.empty(prob.B.nnz, dtype=torch.float64, device="cuda") if prob.B is not None else None
    torch.cuda.synchronize()
    b.backward_device(gm.data_ptr(), gc.data_ptr(), gb.data_ptr() if gb is not None else None, precision=precision)
    b.close()
    ref_c, ref_b = oracle.backward(prob, M, g, threads=THREADS)
    bar = 1e-11 if precision == 0 else 1e-9
    assert np.linalg.norm(gc.cpu().numpy() - ref_c) <= bar * np.linalg.norm(ref_c)
    if gb is not None:
        assert np.linalg.norm(gb.cpu().numpy() - ref_b) <= bar * np.linalg.norm(ref_b)
