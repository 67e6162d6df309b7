"""Kernel tables of other sizes than the default 1000 points: staged in LDS up to 1023 points (FP64
passes that read both halves of the table) or 2047 (mixed precision; the FP64 step's SPH pass), read
from memory beyond, beside the SPH pass's own LDS.  Derivatives, sum density and three steps against
the oracle, whose table has as many points."""
import numpy as np
import pytest

from spheral_amd import abi, problems

pytestmark = pytest.mark.gpu

STEP_FIELDS = ("position", "velocity", "mass density", "specific thermal energy", "H", "grad h corrections")


def state(dim):
    return (problems.sod_1d(120), problems.kelvin_helmholtz_2d(900), problems.taylor_green_3d(9))[dim - 1]


@pytest.mark.parametrize("points", [101, 1023, 1024, 2047, 2048])
@pytest.mark.parametrize("dim", [1, 2, 3])
def test_table_sizes(gpu, oracle_mod, dim, points):
    for precision, bar in ((abi.SPX_PREC_FP64, 1.0e-10), (abi.SPX_PREC_MIXED, 1.0e-5)):
        print(f"[case] {dim}-D, {points} points, precision {precision}", flush=True)
        cfg, st = state(dim)
        cfg.precision, cfg.kernel_points = precision, points
        g = gpu.make_run(cfg, st)
        o = oracle_mod.OracleRun(cfg, len(st["m"]))
        o.set_state(**st)
        for r in (g, o):
            r.initialize()
            r.evaluate_derivatives()
        S = o.field("abs delta velocity hydro")
        assert np.all(np.abs(g.field("delta velocity hydro") - o.field("delta velocity hydro")) <= bar*S + 1.0e-300)
        g.set_group_sizes((8, 8, 8))
        for _ in range(3):
            dg, do = g.step(), o.step()
            assert abs(dg - do) <= bar*do
        for f in STEP_FIELDS:
            a, b = g.field(f), o.field(f)
            assert np.all(np.abs(a - b) <= 10.0*bar*np.abs(b).max()), f
