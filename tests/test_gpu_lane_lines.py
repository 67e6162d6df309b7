"""Lanes per node change at a count of active nodes (3-D: the mixed SPH pass after 49152, the grad-h
pass at 2^18); a small run equals itself beside another that takes the count over the line."""
import numpy as np
import pytest

from spheral_amd import abi, problems

pytestmark = pytest.mark.gpu

FIELDS = ("position", "velocity", "mass density", "specific thermal energy", "H", "grad h corrections",
          "velocity gradient", "max viscous pressure")


@pytest.mark.parametrize("n1d,precision", [(37, abi.SPX_PREC_MIXED), (64, abi.SPX_PREC_MIXED), (64, abi.SPX_PREC_FP64)])
def test_small_run_beside_one_over_the_line(gpu, n1d, precision):
    cfg, small = problems.taylor_green_3d(12, precision=precision)
    large = problems.taylor_green_3d(n1d, precision=precision)[1]
    print(f"[case] 12^3 + {n1d}^3 nodes, precision {precision}", flush=True)
    t_end = 0.002
    b = gpu.Batch(cfg, capacity=len(small["m"]) + len(large["m"]), max_runs=2)
    rid = b.add_run(small, t_end)
    b.add_run(large, 1.0)
    while b.status(rid)["state"] != gpu.RUN_DONE:
        b.step()
    r = gpu.make_run(cfg, small)
    r.initialize()
    r.advance(t_end, 10000)
    for f in FIELDS:
        assert np.array_equal(b.field(rid, f), r.field(f)), f
