"""The default boundary step of Butcher-table integrators -- ghosts written by
the stage launch, both walls of an axis in one fill -- against the same steps
with a callback that exchanges and fills one face after the other: the same
array, ghost cells included, on blocks of the staged pushes' cross-section,
narrower than two ghost layers' width, single along an axis, and with walls on
one side, on both, and on several axes (corner ghosts)."""
import numpy as np
import pytest

from cases import GAMMA, R
from gpu_helpers import RawFlux

pytestmark = pytest.mark.gpu

FLUX = [dict(kind=1, order=2), dict(kind=7, law=1, mu=2e-3, T_ref=1.1, power=0.76, prandtl=0.72)]
T_WALL = 1.13
WALLS = {"periodic": (), "y": (2, 3), "y_low": (2,), "y_high": (3,), "xyz": (0, 1, 2, 3, 4, 5), "x_z": (0, 1, 4, 5)}


def _advance(sa, cells, blocks, walls, table, callback):
    periodic = tuple(not (2 * a in walls or 2 * a + 1 in walls) for a in range(3))
    g = sa.CartesianGrid(cells, blocks, ((0.0, 2.0), (-1.0, 1.0), (0.0, 1.5)), num_exch=2, periodic=periodic)
    q = np.random.default_rng(sum(cells)).standard_normal(g.host_shape)
    q[..., 0] = (1.0 + 0.02 * q[..., 0]) / GAMMA
    q[..., 1] = 1.1 * (1.0 + 0.005 * q[..., 1])
    q[..., 2:] *= 0.1
    arr = sa.GridArray(g).upload(q)

    def bc(sol, t):
        sa.create_exchange(sol).exchange(sol)
        for face in walls:
            sa.boundary_fill_wall(sol, face, T_WALL)
    kw = dict(bc=bc) if callback else dict(walls=walls, t_wall=T_WALL)
    it = sa.RKIntegrator(arr, getattr(sa, table), 1e-4, gas=sa.IdealGas(GAMMA, R), flux=RawFlux(FLUX, GAMMA, R), **kw)
    it.advance(2)
    out = arr.download()
    it.close()
    assert not np.array_equal(out, q)
    return out


@pytest.mark.parametrize("walls", sorted(WALLS))
@pytest.mark.parametrize("cells, blocks", [((16, 16, 8), (2, 2, 1)), ((16, 16, 16), (1, 1, 2)), ((3, 5, 4), (2, 1, 3)),
                                           ((2, 2, 2), (1, 2, 2)), ((11, 9, 6), (2, 2, 2)), ((16, 3, 3), (1, 2, 2))],
                         ids=["16x16x8", "16x16x16", "3x5x4", "2x2x2", "11x9x6", "16x3x3"])
def test_default_boundary_equals_callback(cells, blocks, walls):
    import spade_amd as sa
    for table in ("rk4", "ssprk3_table"):
        a = _advance(sa, cells, blocks, WALLS[walls], table, False)
        b = _advance(sa, cells, blocks, WALLS[walls], table, True)
        print(cells, blocks, walls, table, flush=True)
        assert np.all(np.isfinite(a))
        assert np.array_equal(a, b)
