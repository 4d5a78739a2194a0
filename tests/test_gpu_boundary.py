"""Value and copy boundaries of bounded grids (pamhd_apply_boundaries) against
the FP64 oracle, bit for bit, with values set on boundary cells only (one
launch for all stages) and on normal cells that copy cells read (the copies
wait for each variable's values)."""
import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu

CASES = [((9, 1, 1), (0, 1, 1)), ((33, 9, 1), (0, 1, 1)), ((70, 6, 5), (0, 1, 1)), ((6, 70, 3), (1, 0, 1))]


def _grid(cells, periodic):
    """closed in one dimension with value cells at its lower and copy cells
    at its upper end"""
    n = cells[0] * cells[1] * cells[2]
    k, j, i = np.meshgrid(*[np.arange(c) for c in cells[::-1]], indexing="ij")
    d = [i, j, k][periodic.index(0)].reshape(-1)
    lo = np.tile(d == 0, (4, 1))
    hi = np.tile(d == cells[periodic.index(0)] - 1, (4, 1))
    G = O.BoundedGrid(cells, (0.1, 0.2, 0.3), 5 / 3, 1.0, 1.5, periodic, lo, hi)
    assert G.status == 0 and (G.vtype == 4).any()
    return G, lo, n


@pytest.mark.parametrize("cells,periodic", CASES)
@pytest.mark.parametrize("on_normal", [(), (0,), (1,), (2,), (0, 1, 2, 3)])
def test_boundary_values_bit_exact_vs_oracle(gpu, cells, periodic, on_normal):
    from pamhd_amd import solver as S
    G, lo, n = _grid(cells, periodic)
    rng = np.random.default_rng(11)
    with S.Grid(cells, (0.1, 0.2, 0.3), 5 / 3, 1.0, 1.5, periodic=periodic,
                types=(G.vtype, G.ctype, G.finfo)) as g:
        for extra in (on_normal, ()):
            mask = lo.copy()
            for v in extra:
                mask[v] |= rng.random(n) < 0.7
            assert (mask & (G.ctype == 1)).any() == bool(extra)
            u = lambda k, a, b: rng.uniform(a, b, (k, n) if k > 1 else n)
            values = (mask, u(1, 0.5, 2), u(3, -1, 1), u(1, 0.1, 1), u(6, -1, 1))
            state = np.concatenate([u(1, 0.5, 2)[None], u(3, -1, 1), u(1, 9, 12)[None], u(9, -1, 1)])
            ref = state.copy()
            assert G.apply(ref, *values) == 0
            G.sync(ref)
            print("cells", cells, "values on normal cells of", extra, flush=True)
            g.upload(state)
            g.set_boundary_values(*values)
            g.apply_boundaries()
            np.testing.assert_array_equal(g.download(), ref)
