"""The adjoint of builds with degenerate columns (an exact zero pivot, or fewer
rows than columns): those have no gradient, so dL/dC is the reference's over
the other columns and their part of dL/dB is zero."""
import os

import numpy as np
import pytest
import scipy.sparse as sp
import torch  # before the library: one HIP runtime per process

from mspai_amd import gen
from tests.test_gpu_static import build, system

pytestmark = pytest.mark.gpu
THREADS = min(16, os.cpu_count() or 1)
DEGENERATE = 1 | 2  # zero pivot, underdetermined

CASES = {  # lengths of the patterns, entries of a column, their band; the step from zero column to zero column
    "kinds": (dict(lens=(3, 6, 12, 20), nnz=2, band=9), 30),
    "past_the_kinds": (dict(lens=(33, 36, 20), nnz=4, band=50), 100),
}


def degenerate_problem(kw, step, alike=60):
    """Every step-th column is zero (an exact zero pivot).  The last `alike`
    columns hold one entry each, all in one row, and only patterns among
    themselves reach them: fewer rows than columns.  No pattern holds a part
    of them, which would be singular but for rounding."""
    prob = system(target=True, **kw)
    n, cut = prob.n, prob.n - alike
    a, p = prob.A.tocoo(), prob.P.tocoo()
    zero = np.arange(0, cut, step)
    live = (a.col < cut) & (a.row < cut) & ~np.isin(a.col, zero)
    A = gen._csc(np.concatenate([a.row[live], zero, np.full(alike, cut)]),
                 np.concatenate([a.col[live], zero, np.arange(cut, n)]),
                 np.concatenate([a.data[live], np.zeros(zero.size), np.ones(alike)]), (n, n))
    among = (p.col < cut) == (p.row < cut)
    P = gen._csc(p.row[among], p.col[among], np.ones(among.sum()), (n, n))
    return gen.Problem("degenerate", A, P, prob.B, max_impr_steps=0)


@pytest.mark.parametrize("binning", [1, 0])
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("name", sorted(CASES))
def test_degenerate_columns_have_no_gradient(oracle, gpu, name, precision, binning):
    prob = degenerate_problem(*CASES[name])
    n = prob.n
    print(f"[degenerate adjoint {name} precision={precision} binning={binning}]", flush=True)
    b, _ = build(gpu, prob, precision=precision, binning=binning)
    M, status = b.download(), b.column_info()["status"]
    g = np.random.Generator(np.random.PCG64(5)).standard_normal(M.nnz)
    gm = torch.tensor(g, device="cuda")
    gc = torch.full((prob.A.nnz,), np.nan, dtype=torch.float64, device="cuda")
    gb = torch.full((prob.B.nnz,), np.nan, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    b.backward_device(gm.data_ptr(), gc.data_ptr(), gb.data_ptr(), precision=precision, binning=binning)
    b.close()
    gc, gb = gc.cpu().numpy(), gb.cpu().numpy()
    bad = (status & DEGENERATE) != 0
    assert (status & 1).sum() >= 10 and (status & 2).sum() >= 10 and bad.sum() <= n - 20
    # the reference sees a pattern without the degenerate columns
    keep = np.repeat(~bad, np.diff(M.indptr))
    ptr = np.concatenate([[0], np.cumsum(np.diff(M.indptr) * ~bad)])
    Mk = sp.csc_matrix((M.data[keep], M.indices[keep], ptr), shape=M.shape)
    ref_c, ref_b = oracle.backward(prob, Mk, g[keep], threads=THREADS)
    assert np.isfinite(gc).all() and np.isfinite(gb).all()
    bar = 1e-11 if precision == 0 else 1e-9
    assert np.linalg.norm(gc - ref_c) <= bar * np.linalg.norm(ref_c)
    assert np.linalg.norm(gb - ref_b) <= bar * np.linalg.norm(ref_b)
    assert (gb[np.repeat(bad, np.diff(prob.B.indptr))] == 0.0).all()
