"""In mixed precision, whose sums run in list order, the package-level sum density and the one that
rides on a step's neighbour pass are the same bits, whatever place a neighbour has in the list."""
import numpy as np
import pytest

from spheral_amd import abi, problems

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim", [1, 2, 3])
def test_package_sum_density_is_the_steps(gpu, dim):
    print(f"[case] {dim}-D", flush=True)
    cfg, st = (problems.sod_1d(200), problems.kelvin_helmholtz_2d(2000), problems.taylor_green_3d(11))[dim - 1]
    cfg.precision = abi.SPX_PREC_MIXED
    cfg.dt_max = 1.0e-300                        # a step that moves nothing: its density is the sum density
    a, b = gpu.make_run(cfg, st), gpu.make_run(cfg, st)
    for r in (a, b):
        r.initialize()
    a.sum_density()
    b.step()
    assert np.array_equal(a.field("mass density"), b.field("mass density"))
