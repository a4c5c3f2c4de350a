"""Work counters of a static build describe the launches that run without them:
the same launches in the same order, every column in one of them, and the
oracle's counts."""
import os

import numpy as np
import pytest

from tests.test_gpu_static import CASES, build, system

pytestmark = pytest.mark.gpu
THREADS = min(16, os.cpu_count() or 1)


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("name", ["one_kind_short", "rows_about_64", "routed_lengths", "target_routed", "degenerate"])
def test_static_counters(oracle, gpu, name, precision):
    prob = system(**CASES[name])
    print(f"[static counters {name} precision={precision}]", flush=True)
    ref = oracle.spai(prob, threads=THREADS)
    b, _ = build(gpu, prob, precision=precision)
    plain, M0 = [x["name"] for x in b.launch_stats()], b.download()
    b.build(max_impr_steps=0, precision=precision, counters=1)
    ls, tot, info, M1 = b.launch_stats(), b.work_totals(), b.column_info(), b.download()
    b.close()
    assert [x["name"] for x in ls] == plain
    assert sum(x["columns"] for x in ls) == prob.n
    assert sum(x["nnz"] for x in ls) == M0.nnz
    assert np.array_equal(M0.data.view(np.int64), M1.data.view(np.int64))
    assert np.array_equal(ref["work"], info["work"])
    per_launch = np.sum([x["work"] for x in ls], axis=0)
    assert np.array_equal(per_launch[1:], tot[1:])  # integers: exact in any order
    assert np.allclose(per_launch[0], tot[0], rtol=1e-12, atol=0)  # QR flop: fractional
    assert np.array_equal(tot[1:], ref["work"].sum(axis=0)[1:])
    if precision == 0:
        assert np.array_equal(np.sum([x["near"] for x in ls], axis=0), ref["near"].sum(axis=0))
