"""A state with one bad node, the first or the last, is refused before anything is transferred: by its
H (not a positive multiple of the identity), its mass or its density; the run keeps the state it has."""
import numpy as np
import pytest

from spheral_amd import abi, problems
from spheral_amd.engine import SpxError

pytestmark = pytest.mark.gpu


def bad_values(dim):
    cases = [("H", (a, b), 1.0e-300, abi.SPX_ERR_UNSUPPORTED) for a in range(dim) for b in range(dim) if a != b]
    cases += [("H", (a, a), v, abi.SPX_ERR_UNSUPPORTED) for a in range(1, dim) for v in (0.0, np.nan)]
    cases += [("H", "all", 0.0, abi.SPX_ERR_ARG), ("H", "all", -1.0, abi.SPX_ERR_ARG), ("H", "all", np.inf, abi.SPX_ERR_ARG),
              ("H", "all", np.nan, abi.SPX_ERR_UNSUPPORTED)]
    return cases + [(k, (), v, abi.SPX_ERR_ARG) for k in ("m", "rho") for v in (0.0, -1.0, np.nan)]


@pytest.mark.parametrize("dim", [1, 2, 3])
def test_one_bad_node(gpu, dim):
    cfg, st = problems.uniform_lattice(dim, 7)
    r = gpu.make_run(cfg, st)
    r.initialize()
    before = r.field("position")
    for key, at, value, code in bad_values(dim):
        for node in (0, -1):
            print(f"[case] {dim}-D {key}{at} = {value} of node {node}", flush=True)
            other = dict(st, x=st["x"][::-1].copy())
            other[key] = st[key].copy()
            if at == "all":
                other[key][node] = np.eye(dim)*value if np.isfinite(value) else np.where(np.eye(dim) > 0, value, 0.0)
            else:
                other[key][(node,) + at] = value
            with pytest.raises(SpxError) as err:
                r.update_state(**other)
            assert err.value.code == code
            assert np.array_equal(r.field("position"), before)
            with pytest.raises(SpxError) as err:
                gpu.make_run(cfg, other)
            assert err.value.code == code
