"""The autotuner on static builds, which run on the given-pattern kernels
whatever the bin table: timed once, and the table of adaptive builds stays."""
import pytest

from mspai_amd import gen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1])
def test_static_options_leave_the_table_alone(gpu, precision):
    prob = gen.config3(n=4096, bw=300)
    opts = dict(epsilon=prob.epsilon, maxnew=prob.maxnew, max_impr_steps=prob.max_impr_steps, precision=precision)

    def launches(**kw):
        b.build(**opts, **kw)
        names = [x["name"] for x in b.launch_stats()]
        # a mixed build's FP64 remainder takes its route by the length the last one had
        return [x for x in names if precision == 0 or x.startswith("mixed")]

    b = gpu.Builder(0)
    try:
        print(f"[autotune static precision={precision}]", flush=True)
        b.upload(prob.A, prob.row_pattern())
        untuned = launches(binning=1)
        rep = b.autotune(repeats=1, max_impr_steps=0, precision=precision)
        assert sum(t >= 0 for t in rep["candidate_ms"]) == 1 and rep["candidate_ms"][rep["chosen"]] >= 0
        assert launches(binning=2) == untuned
        name = b.set_bin_table(9, precision=precision)
        pinned = launches(binning=2)
        assert pinned != untuned
        rep = b.autotune(repeats=1, max_impr_steps=0, precision=precision)
        assert rep["chosen"] == 9 and rep["name"] == name
        assert launches(binning=2) == pinned
        # adaptive options tune as before
        rep = b.autotune(repeats=1, **opts)
        assert sum(t >= 0 for t in rep["candidate_ms"]) > 10
    finally:
        b.close()
