"""The tree walk visits cells by one point or by four neighbouring points together (by particle
count); what a point gets does not depend on which, bit for bit.  With an opening angle that
accepts no monopole, both equal the direct sum over the points, coincident ones included."""
import numpy as np
import pytest
import torch

from spheral_amd import abi

pytestmark = pytest.mark.gpu

ALONE = 98304          # largest count whose points walk by themselves
SOFT = 0.01


def tree_run(gpu, x, m, opening, hinv=None):
    n, dim = x.shape
    hinv = hinv or n**(1.0/dim)
    cfg = abi.default_config(dim, nperh=2.01)
    cfg.integrator = abi.SPX_INTEGRATOR_SYNCHRONOUS_RK2
    cfg.gravity = cfg.gravity_only = 1
    cfg.G, cfg.softening, cfg.opening, cfg.ftimestep = 1.0, SOFT, opening, 0.1
    H = np.broadcast_to(np.eye(dim)*hinv, (n, dim, dim)).copy()
    r = gpu.make_run(cfg, dict(x=x, v=np.zeros((n, dim)), m=m, rho=np.ones(n), eps=np.zeros(n), H=H))
    r.initialize()
    r.evaluate_derivatives()
    return r


def evaluate(gpu, x, m, opening, hinv=None):
    r = tree_run(gpu, x, m, opening, hinv)
    return r.field("delta velocity"), r.field("gravitational potential")


def ball(n, dim, seed=5):
    g = np.random.default_rng(seed)
    d = g.normal(size=(n, dim))
    return d/np.sqrt((d*d).sum(1))[:, None]*np.sqrt(g.uniform(0.0, 1.0, n))[:, None]


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("opening", [0.5, 1.0])
def test_alone_and_together_give_the_same_bits(gpu, dim, opening):
    print(f"[case] {dim}-D {ALONE} + 1 points, opening {opening}", flush=True)
    x, m = ball(ALONE, dim), np.full(ALONE, 1.0/ALONE)
    # corners of the box, so that it does not change; then a weightless point in an empty cell
    x[0], x[1] = -1.0, 1.0
    more = np.concatenate([x, np.full((1, dim), 0.9)*np.where(np.arange(dim) == 0, -1.0, 1.0)])
    a, p = evaluate(gpu, x, m, opening)
    a1, p1 = evaluate(gpu, more, np.append(m, 1.0e-200), opening)
    assert np.array_equal(a, a1[:-1]) and np.array_equal(p, p1[:-1])


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("n", [2, 3, 5, 63, 64, 65, 257, 2051, ALONE + 3])
def test_opened_walk_is_the_direct_sum(gpu, dim, n):
    print(f"[case] {dim}-D {n} points, direct", flush=True)
    x, m = ball(n, dim, seed=n), np.linspace(1.0, 2.0, n)/n
    if n > 4:
        x[n//2] = x[0]                       # a coincident pair, and a close one
        x[n//2 + 1] = x[1] + 1e-9
    a, p = evaluate(gpu, x, m, 1.0e-9)
    X, M = torch.tensor(x, device="cuda"), torch.tensor(m, device="cuda")
    # a term is a dozen roundings, and a sum of n terms errs by at most n more of its terms' sizes
    eps = 2.3e-16*(n + 30)
    for i0 in range(0, n, 1024):
        d = X[None, :, :] - X[i0:i0 + 1024, None, :]
        r2 = (d*d).sum(2)
        on = r2/SOFT**2 > 1.0e-10
        s = r2 + SOFT**2
        f = M[None, :]/(s if dim == 3 else s.sqrt())*on
        u = d/torch.where(on, r2, 1.0).sqrt()[:, :, None]
        acc = (f[:, :, None]*u).sum(1).cpu().numpy()
        pot = -(M[None, :]/s.sqrt() if dim == 3 else M[None, :]*0.5*s.log())*on
        size, psize = f.sum(1).cpu().numpy(), pot.abs().sum(1).cpu().numpy()
        assert np.all(np.abs(a[i0:i0 + 1024] - acc) <= eps*size[:, None])
        assert np.all(np.abs(p[i0:i0 + 1024] - pot.sum(1).cpu().numpy()) <= eps*psize)


def sampled(n):
    """The points that the build's sort samples."""
    ns = min(n, 512 if n <= 65536 else 1024)
    j = np.arange(ns, dtype=np.uint64)
    i0, i1 = j*np.uint64(n)//np.uint64(ns), (j + np.uint64(1))*np.uint64(n)//np.uint64(ns)
    return (i0 + (((j*np.uint64(2654435769)) & np.uint64(0xffffffff))*(i1 - i0) >> np.uint64(32))).astype(np.int64)


@pytest.mark.parametrize("case", ["chunk - 1", "chunk", "chunk + 1", "two chunks", "lattice", "clump", "chains", "one place"])
def test_tree_build_edges(gpu, oracle_mod, case):
    """Builds at the edges of the sort and of the cells' chunks (512 points) against the oracle's tree."""
    print(f"[case] {case}", flush=True)
    if case == "lattice":                      # 64 points a row: the sampling stride is a row's
        n = 65536
        k = np.arange(n)
        x = np.stack([k % 64, k//64 % 32, k//2048], 1)/32.0 + 0.01
    elif case == "clump":                      # one bucket with all but the sampled points: sorted in memory
        n = 20000
        x = 0.25 + 0.05*ball(n, 3)
        around = ball(8192, 3)
        x[sampled(n)] = around[((around - 0.25)**2).sum(1) > 0.01][:512]
    elif case == "chains":                     # pairs at 1e-5: up to 16 single-daughter cells above each
        n = 3000
        x = ball(n, 3)
        x[1::2] = x[::2] + 1.0e-5
    elif case == "one place":                  # lists of coincident points over several chunks, in two places
        n = 2600
        x = np.where(np.arange(n)[:, None] % 2 == 0, 0.25, -0.5)*np.ones((n, 3))
    else:
        n = {"chunk - 1": 511, "chunk": 512, "chunk + 1": 513, "two chunks": 1024}[case]
        x = ball(n, 3)
    m = np.linspace(1.0, 2.0, n)/n
    hinv = 200.0 if case == "clump" else n**(1.0/3.0)
    a, p = evaluate(gpu, x, m, 0.7, hinv)
    cfg = abi.default_config(3, nperh=2.01)
    cfg.integrator = abi.SPX_INTEGRATOR_SYNCHRONOUS_RK2
    cfg.gravity = cfg.gravity_only = 1
    cfg.G, cfg.softening, cfg.opening, cfg.ftimestep = 1.0, SOFT, 0.7, 0.1
    H = np.broadcast_to(np.eye(3)*hinv, (n, 3, 3)).copy()
    o = oracle_mod.OracleRun(cfg, n)
    o.set_state(x=x, v=np.zeros((n, 3)), m=m, rho=np.ones(n), eps=np.zeros(n), H=H)
    o.initialize()
    o.evaluate_derivatives()
    ao, po = o.field("delta velocity"), o.field("gravitational potential")
    assert np.all(np.abs(a - ao) <= 1e-10*np.abs(ao).max())
    assert np.all(np.abs(p - po) <= 1e-10*np.abs(po).max())


def test_the_two_sorts_give_the_same_bits(gpu):
    """2^18 points are sorted by the sample sort, more by the library's radix sort."""
    n = 1 << 18
    print(f"[case] {n} + 1 points", flush=True)
    x, m = ball(n, 3), np.full(n, 1.0/n)
    x[0], x[1] = -1.0, 1.0
    a, p = evaluate(gpu, x, m, 1.0)
    a1, p1 = evaluate(gpu, np.concatenate([x, [[-0.9, 0.9, 0.9]]]), np.append(m, 1.0e-200), 1.0)
    assert np.array_equal(a, a1[:-1]) and np.array_equal(p, p1[:-1])


@pytest.mark.parametrize("n", [3, 65, 2051])
def test_interaction_counts(gpu, n):
    """Opened all the way, a walk's interactions are the pairs of points farther apart than the screen."""
    print(f"[case] counts of {n} points", flush=True)
    x = ball(n, 3, seed=n)
    x[n//2] = x[0]
    r = tree_run(gpu, x, np.full(n, 1.0/n), 1.0e-9)
    r2 = ((x[:, None, :] - x[None, :, :])**2).sum(2)
    before = r.field("delta velocity")
    assert tuple(r.gravity_interactions()) == (0, int((r2/SOFT**2 > 1.0e-10).sum()))
    r.evaluate_derivatives()
    assert np.array_equal(r.field("delta velocity"), before)
