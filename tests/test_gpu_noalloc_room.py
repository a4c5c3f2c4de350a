"""The largest problems that mspai_build_noalloc's scratch array holds: 36 bytes
of queues a column beside its results, so a tridiagonal matrix of 3,190,000
columns with one augmentation step of one index (and of 3,490,000 columns with
none) fits 256 MiB; the build equals mspai_build bit for bit.  (Slot-by-slot:
9 queue entries, |J|, nsolve and status of 4 bytes, the residual of 8 and 12
per output entry are 80 bytes a column, 68 without augmentation, and the rest
is the tie buffers.)"""
import numpy as np
import pytest
import scipy.sparse as sp
import torch  # before the library: one HIP runtime per process

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("n,steps", [(3_190_000, 1), (3_490_000, 0)])
def test_noalloc_room(gpu, n, steps, precision):
    print(f"[noalloc room n={n} steps={steps} precision={precision}]", flush=True)
    v = np.random.Generator(np.random.PCG64(3)).uniform(0.5, 1.5, (2, n - 1))
    A = sp.diags([-v[0], np.full(n, 3.0), -v[1]], [-1, 0, 1], format="csc")
    cap = 1 + steps
    opts = dict(epsilon=0.1, maxnew=1, max_impr_steps=steps, precision=precision)
    b = gpu.Builder(0)
    try:
        b.upload(A)
        b.set_pattern(None)
        colptr = torch.zeros(n + 1, dtype=torch.int32, device="cuda")
        rowind = torch.zeros(n * cap, dtype=torch.int32, device="cuda")
        val = torch.zeros(n * cap, dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        st = b.build_noalloc(colptr.data_ptr(), rowind.data_ptr(), val.data_ptr(), n * cap, **opts)
        nnz = st["nnz"]
        b.build(**opts)
        M = b.download()
    finally:
        b.close()
    assert np.array_equal(M.indptr, colptr.cpu().numpy())
    assert np.array_equal(M.indices, rowind[:nnz].cpu().numpy())
    assert np.array_equal(M.data.view(np.int64), val[:nnz].cpu().numpy().view(np.int64))
