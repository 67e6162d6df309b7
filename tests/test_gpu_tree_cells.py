"""A batch slot with TreeGravity that holds a small run, then one of so many cells that the tree's
arrays grow, then the small run again: the small run steps as before, bit for bit, and the outgrown
arrays were given back."""
import numpy as np
import pytest

from spheral_amd import abi

pytestmark = pytest.mark.gpu

FIELDS = ("position", "velocity", "mass density", "specific thermal energy", "H")
CELLS = 20*2**18 + 2            # allocated at first: 20 per point of up to 2^18 points
CELL_BYTES = 56


def points(x, nperh=1.0):
    n = len(x)
    h = nperh*2.0/n**(1.0/3.0)
    return dict(x=x, v=np.zeros((n, 3)), m=np.full(n, 1.0/n), rho=np.full(n, 0.125), eps=np.ones(n),
                H=np.broadcast_to(np.eye(3)/h, (n, 3, 3)).copy())


def test_cells_grow_and_the_small_run_returns(gpu):
    print("[case] 4000 points, 860000 in close pairs, 4000 again", flush=True)
    g = np.random.default_rng(3)
    small = points(g.uniform(-1.0, 1.0, (4000, 3)))
    pairs = g.uniform(-1.0, 1.0, (430000, 3))
    large = points(np.concatenate([pairs, pairs + 1.0e-9]))      # a chain of cells down to each pair: 6.2 million
    held, out = {}, []
    for gravity in (0, 1):
        cfg = abi.default_config(3, nperh=1.0)
        cfg.gravity, cfg.G, cfg.softening, cfg.opening, cfg.ftimestep = gravity, 1.0e-30, 0.01, 1.0, 0.1
        b = gpu.Batch(cfg, capacity=len(large["m"]), max_runs=1)
        b.set_group_sizes((8, 8, 8))

        def run(state, steps):
            rid = b.add_run(state, 1.0)
            for _ in range(steps):
                b.step()
            fields = [b.field(rid, f) for f in FIELDS]
            b.remove_run(rid)
            return fields

        first = run(small, 8)
        held[gravity] = [b.device_bytes()]
        run(large, 1)
        held[gravity].append(b.device_bytes())
        again = run(small, 8)
        if gravity:
            assert b.step_stats()["graph_replays"] > 0
        for x, y in zip(first, again):
            assert np.array_equal(x, y)
        b.close()
    tree = [w - wo for w, wo in zip(held[1], held[0])]           # the tree's own memory, before and after it grew
    assert 0 < tree[1] - tree[0] < CELL_BYTES*CELLS
