"""Steps replayed from graphs equal the same steps launched one by one, bit for bit, also with the
Limited Q (its gradient's copy) and with TreeGravity (its tree on a second stream), across
boundaries and candidate-list rebuilds; and the tree a replay leaves behind is the current one."""
import numpy as np
import pytest

from spheral_amd import abi, problems

pytestmark = pytest.mark.gpu

FIELDS = ("position", "velocity", "mass density", "specific thermal energy", "H")


def setup(name):
    if name == "limited Q":
        cfg, st = problems.noh_planar_1d(100)
        cfg.viscosity = abi.SPX_Q_LIMITED_MONAGHAN_GINGOLD
        return cfg, st
    if name == "periodic":
        cfg, st = problems.kelvin_helmholtz_2d(4096)
        st["v"] = st["v"] + 3.0               # everything crosses the box
        return cfg, st
    return problems.gravity_disk_2d(3000) if name == "disk" else problems.evrard_3d(4000)


@pytest.mark.parametrize("name", ["limited Q", "periodic", "disk", "collapse"])
def test_replayed_steps_equal_launched_steps(gpu, name):
    print(f"[case] {name}", flush=True)
    cfg, st = setup(name)
    a, b = gpu.make_run(cfg, st), gpu.make_run(cfg, st)
    b.set_step_graphs(False)
    a.initialize()
    b.initialize()
    for block in range(5):
        for _ in range(8):
            assert a.step() == b.step(), block
        for f in FIELDS:
            assert np.array_equal(a.field(f), b.field(f)), (block, f)
        if cfg.gravity:
            assert tuple(a.gravity_interactions()) == tuple(b.gravity_interactions())
            assert np.array_equal(a.field("gravitational potential"), b.field("gravitational potential"))
    sa, sb = a.step_stats(), b.step_stats()
    assert sa["graph_replays"] > 0 and sb["graph_replays"] == 0


def test_a_batch_of_many_slots_waits_on_the_stream(gpu):
    """The host polls for a step's end when one block writes the runs' scalars; with more than 256
    slots several do, and it waits on the stream.  The same steps either way."""
    print("[case] 1 and 300 slots", flush=True)
    cfg, st = problems.kelvin_helmholtz_2d(4096)
    out = []
    for slots in (1, 300):
        b = gpu.Batch(cfg, capacity=len(st["m"]), max_runs=slots)
        rid = b.add_run(st, 1.0)
        for _ in range(70):                      # past a step that waits on the stream by its number
            b.step()
        assert b.step_stats()["graph_replays"] > 0
        out.append([b.field(rid, f) for f in FIELDS] + [b.status(rid)["t"]])
        b.close()
    for x, y in zip(*out):
        assert np.array_equal(x, y)
