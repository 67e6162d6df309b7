"""The pair passes' lanes per node never show in the results.

The grad-h pass takes four lanes per node for small active particle counts and one beyond; a run
stepped alone (four lanes) equals the same run inside a batch whose other run pushes the active
count over the line (one lane), bit for bit, in FP64 and mixed precision.  Lists shorter than a
quad, and lists that end anywhere within one, are compared with the oracle."""
import numpy as np
import pytest

from spheral_amd import abi, problems

pytestmark = pytest.mark.gpu

FIELDS = ("position", "velocity", "mass density", "specific thermal energy", "H", "grad h corrections")


@pytest.mark.parametrize("precision", [abi.SPX_PREC_FP64, abi.SPX_PREC_MIXED], ids=["fp64", "mixed"])
def test_small_run_beside_a_large_one_equals_it_alone(gpu, precision):
    t_end = 0.004
    cfg, small = problems.kelvin_helmholtz_2d(1500, precision=precision)
    _, large = problems.kelvin_helmholtz_2d(260000, precision=precision)
    print(f"[case] 1500 + {len(large['m'])} nodes, precision {precision}", flush=True)
    b = gpu.Batch(cfg, capacity=len(small["m"]) + len(large["m"]), max_runs=2)
    rid = b.add_run(small, t_end)
    b.add_run(large, 10.0*t_end)
    while b.status(rid)["state"] != gpu.RUN_DONE:
        b.step()
    r = gpu.make_run(cfg, small)
    r.initialize()
    r.advance(t_end, 10000)
    for f in FIELDS:
        assert np.array_equal(b.field(rid, f), r.field(f)), f


@pytest.mark.parametrize("reach", [0.55, 1.05, 1.55, 2.05, 2.55, 4.05])
def test_short_lists_match_oracle(gpu, oracle_mod, reach):
    """Open 1-D chains whose nodes reach `reach` spacings: 0 to 8 neighbours, fewer at the ends."""
    print(f"[case] chain reach {reach}", flush=True)
    n, dx = 37, 0.1
    x = np.arange(n)*dx + 0.01*dx*np.sin(1.7*np.arange(n))
    cfg = abi.default_config(1, nperh=2.01)
    H = np.full((n, 1, 1), 2.0/(reach*dx))
    st = dict(x=x.reshape(n, 1), v=0.1*np.cos(0.3*np.arange(n)).reshape(n, 1), m=np.full(n, dx), rho=np.ones(n),
              eps=np.full(n, 0.5), H=H)
    g = gpu.make_run(cfg, st)
    g.initialize()
    o = oracle_mod.OracleRun(cfg, n)
    o.set_state(**st)
    o.initialize()
    assert np.array_equal(g.neighbors()[1], o.neighbors()[1])
    for _ in range(3):
        dg, do = g.step(), o.step()
        assert abs(dg - do) <= 1e-10*do
    for f in FIELDS:
        a, c = g.field(f), o.field(f)
        assert np.all(np.abs(a - c) <= 1e-9*max(np.abs(c).max(), 1e-300)), f


@pytest.mark.parametrize("wide", [1, 15, 16, 17, 40, 70])
@pytest.mark.parametrize("dim", [2, 3])
def test_handed_over_entries_match_oracle(gpu, oracle_mod, dim, wide):
    """`wide` nodes whose support covers a cluster of nodes with an eighth of it: every cluster node
    receives `wide` entries its own support does not find, below, at and beyond the 16 that one
    row of lanes ranks at a time."""
    print(f"[case] {wide} wide nodes, {dim}-D", flush=True)
    rng = np.random.default_rng(100*dim + wide)
    n = 60
    x = np.concatenate([0.05*rng.uniform(-1, 1, (n, dim)), 0.5 + 0.1*rng.uniform(-1, 1, (wide, dim))])
    h = np.concatenate([np.full(n, 0.1), np.full(wide, 0.8)])
    H = np.zeros((n + wide, dim, dim))
    for a in range(dim):
        H[:, a, a] = 1.0/h
    st = dict(x=x, v=np.zeros_like(x), m=np.full(n + wide, 1.0/(n + wide)), rho=np.ones(n + wide), eps=np.ones(n + wide),
              H=H)
    cfg = abi.default_config(dim, nperh=2.01)
    g = gpu.make_run(cfg, st)
    g.initialize()
    o = oracle_mod.OracleRun(cfg, n + wide)
    o.set_state(**st)
    o.initialize()
    for a, c in zip(g.neighbors(), o.neighbors()):
        assert np.array_equal(a, c)
    assert g.neighbor_counts()[:n].min() >= wide
