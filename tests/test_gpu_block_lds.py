"""Block columns at the edges of the sizes the LDS kernels take (|I| <= 64 and
|J| <= 24 scalars, then 128 and 36, blocks to 4x4): the block oracle's bits."""
import numpy as np
import pytest
import scipy.sparse as sp
import torch  # noqa: F401  before the library: one HIP runtime per process

from mspai_amd import gen
from tests.test_gpu_block import blk, check_case  # noqa: F401

pytestmark = pytest.mark.gpu


def coupled(nblocks, bs, degree, seed, equal=False):
    """nblocks blocks of bs with `degree` random off-diagonal blocks a block
    column and a diagonal that does not dominate."""
    rng = np.random.Generator(np.random.PCG64(seed))
    c = np.repeat(np.arange(nblocks), degree)
    r = (c + rng.integers(1, 4 * degree, c.size)) % nblocks
    r, c = np.concatenate([r, np.arange(nblocks)]), np.concatenate([c, np.arange(nblocks)])
    i = (r[:, None, None] * bs + np.arange(bs)[None, :, None]).repeat(bs, axis=2)
    j = (c[:, None, None] * bs + np.arange(bs)[None, None, :]).repeat(bs, axis=1)
    v = np.ones(i.shape) if equal else rng.standard_normal(i.shape)
    A = sp.coo_matrix((v.ravel(), (i.ravel(), j.ravel())), shape=(nblocks * bs,) * 2).tocsc()
    A.sum_duplicates()
    A = (A + sp.identity(nblocks * bs) * (2.0 + bs)).tocsc()
    A.sort_indices()
    return A


CASES = {
    "rows_about_64_bs4": (lambda: coupled(150, 4, 3, 1), 4, dict(epsilon=0.05, maxnew=2, max_impr_steps=3)),
    "rows_about_128_bs3": (lambda: coupled(200, 3, 4, 2), 3, dict(epsilon=0.05, maxnew=4, max_impr_steps=3)),
    "columns_about_36_bs2": (lambda: coupled(160, 2, 2, 3), 2, dict(epsilon=0.01, maxnew=5, max_impr_steps=4)),
    "ties_at_the_cut_bs2": (lambda: coupled(120, 2, 3, 4, equal=True), 2,
                            dict(epsilon=0.02, maxnew=2, max_impr_steps=2)),
    "candidates_past_128_bs3": (lambda: coupled(600, 3, 13, 5), 3, dict(epsilon=0.1, maxnew=1, max_impr_steps=1)),
    "blocks_of_5": (lambda: coupled(60, 5, 2, 6), 5, dict(epsilon=0.1, maxnew=2, max_impr_steps=2)),
    "remainder_block_bs4": (lambda: coupled(67, 3, 2, 7), 4, dict(epsilon=0.1, maxnew=3, max_impr_steps=3)),
    "two_blocks": (lambda: coupled(2, 3, 1, 8), 3, dict(epsilon=0.1, maxnew=3, max_impr_steps=3)),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_block_lds_bitwise(blk, gpu, name):  # noqa: F811
    make, bs, opts = CASES[name]
    print(f"[block {name}]", flush=True)
    check_case(blk, gpu, make(), bs, **opts)
