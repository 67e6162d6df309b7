"""State moves between the caller's Field records and the engine's arrays unchanged, in one piece
and in several (a field of more than 2^21 doubles goes through the staging buffer in pieces), before
and after the engine has re-ordered its particles."""
import numpy as np
import pytest

from spheral_amd import abi

pytestmark = pytest.mark.gpu


def lattice(dim, n1d, seed):
    rng = np.random.default_rng(seed)
    g = (np.arange(n1d) + 0.5)/n1d
    x = np.stack([a.ravel() for a in np.meshgrid(*([g]*dim), indexing="ij")], 1)
    x = x + rng.uniform(-0.1, 0.1, x.shape)/n1d
    n = len(x)
    order = rng.permutation(n)
    H = np.zeros((n, dim, dim))
    for a in range(dim):
        H[:, a, a] = n1d/2.0*rng.uniform(0.99, 1.01, n) if a == 0 else H[:, 0, 0]
    return dict(x=x[order], v=rng.normal(size=(n, dim)), m=rng.uniform(1, 2, n)/n, rho=rng.uniform(1, 2, n),
                eps=rng.uniform(1, 2, n), H=H)


def check(r, st):
    for name, key in (("position", "x"), ("velocity", "v"), ("mass", "m"), ("mass density", "rho"),
                      ("specific thermal energy", "eps"), ("H", "H")):
        assert np.array_equal(r.field(name), st[key]), name


@pytest.mark.parametrize("dim,n1d", [(1, 1), (1, 257), (2, 33), (2, 800), (3, 7), (3, 65)])
def test_state_round_trip(gpu, dim, n1d):
    print(f"[case] {n1d}^{dim}", flush=True)
    st = lattice(dim, n1d, 5)
    cfg = abi.default_config(dim, kernel=abi.SPX_KERNEL_WENDLANDC4, nperh=2.0)
    cfg.kernel = abi.SPX_KERNEL_WENDLANDC4
    cfg.neighbor_extent = 1.0
    r = gpu.make_run(cfg, st)
    check(r, st)
    r.initialize()
    check(r, st)
    if len(st["m"]) > 1:
        r.evaluate_derivatives()
        M = r.field("M SPH correction")
        assert M.shape == (len(st["m"]), dim, dim) and np.isfinite(M).all()
    other = lattice(dim, n1d, 6)
    r.update_state(**other)
    check(r, other)
