"""The 16 x 16 kernel with a block's planes shared out unevenly between
workgroups (shares of one plane, odd ones, more than the planes divide into):
flux_div in both modes and fused SSP-RK3 steps have the bits of whole blocks."""
import os

import numpy as np
import pytest

from cases import GAMMA, R
from gpu_helpers import RawFlux

pytestmark = pytest.mark.gpu

FLUX = [dict(kind=1, order=2), dict(kind=7, law=1, mu=2e-3, T_ref=1.1, power=0.76, prandtl=0.72)]


def _run(sa, host, nz, shares, stretch):
    os.environ["SPD_FAST_ZSPLIT"] = str(shares)
    try:
        g = sa.CartesianGrid((16, 16, nz), (2, 1, 2), ((0.0, 2.0), (-1.0, 1.0), (0.0, 1.5)),
                             periodic=(True, not stretch, True),
                             maps=(None, sa.tanh_map(-1.0, 1.0, 1.5) if stretch else None, None))
        q = sa.GridArray(g).upload(host)
        sa.create_exchange(q).exchange(q)
        walls = dict(walls=(2, 3), t_wall=1.1) if stretch else {}
        for face in walls.get("walls", ()):
            sa.boundary_fill_wall(q, face, 1.1)
        flux = RawFlux(FLUX, GAMMA, R)
        assert sa.flux_div_kernel(q, flux) == "fast"
        out = []
        for increment in (False, True):
            rhs = sa.GridArray(g, fill=0.25)
            sa.flux_div(q, rhs, flux, increment=increment)
            out.append(rhs.download())
        it = sa.Integrator(q, flux, 1e-4, **walls)
        assert it.fused
        it.advance(1)
        it.advance(2)
        out.append(q.download())
        it.close()
        return out
    finally:
        os.environ.pop("SPD_FAST_ZSPLIT", None)


@pytest.mark.parametrize("stretch", [False, True], ids=["periodic", "channel"])
@pytest.mark.parametrize("nz", [5, 16])
def test_uneven_shares_equal_whole_blocks(nz, stretch):
    import spade_amd as sa
    sa.load()
    rng = np.random.default_rng(nz)
    host = rng.standard_normal((4, nz + 4, 20, 20, 5))
    host[..., 0] = 70.0 + 0.5 * host[..., 0]
    host[..., 1] = 1.1 * (1.0 + 0.005 * host[..., 1])
    host[..., 2:] *= 0.1
    host[0, 4, 5, 5, 1] = 2.0                 # outside the power law's series
    whole = _run(sa, host, nz, 1, stretch)
    for shares in (2, 3, nz, 200):
        print(nz, stretch, shares, flush=True)
        for a, b in zip(whole, _run(sa, host, nz, shares, stretch)):
            assert np.all(np.isfinite(a))
            assert np.array_equal(a, b)
