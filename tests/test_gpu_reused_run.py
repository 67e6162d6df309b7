"""A run that has stepped and is given a new state steps from it as a fresh run does, bit for bit,
also where nodes of the new state lie behind a wall (what the last steps left pending is dropped)."""
import numpy as np
import pytest

from spheral_amd import abi, problems

pytestmark = pytest.mark.gpu

FIELDS = ("position", "velocity", "mass density", "specific thermal energy", "H")


def walled(dim):
    cfg, st = problems.uniform_lattice(dim, {1: 60, 2: 16, 3: 9}[dim])
    for a in range(dim):
        cfg.bc_lo[a] = cfg.bc_hi[a] = abi.SPX_BC_REFLECTING
        cfg.xmin[a], cfg.xmax[a] = 0.0, 1.0
    g = np.random.default_rng(dim)
    st["x"] = st["x"] + g.uniform(-0.1, 0.1, st["x"].shape)*(st["m"][0]**(1.0/dim))
    st["v"] = g.normal(size=st["x"].shape)
    return cfg, st


@pytest.mark.parametrize("dim", [1, 2, 3])
def test_new_state_on_a_stepped_run(gpu, dim):
    print(f"[case] {dim}-D", flush=True)
    cfg, st = walled(dim)
    other = dict(st, x=st["x"].copy())
    k = int(np.argmin(other["x"][:, 0]))
    other["x"][k, 0] = -0.2*st["m"][0]**(1.0/dim)      # behind the lower wall, moving on
    other["v"] = st["v"][::-1].copy()
    other["v"][k, 0] = -1.0
    used, fresh = gpu.make_run(cfg, st), gpu.make_run(cfg, other)
    for r in (used, fresh):
        r.set_group_sizes((8, 8, 8))                   # no measuring steps: steady ones from the first
    used.initialize()
    for _ in range(3):
        used.step()
    used.set_state(**other)
    for r in (used, fresh):
        r.initialize()
    for step in range(3):
        assert used.step() == fresh.step(), step
        for f in FIELDS:
            assert np.array_equal(used.field(f), fresh.field(f)), (step, f)
