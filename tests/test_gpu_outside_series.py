"""Faces whose temperatures leave the power law's series take the library pow
inside the 16x16 kernel: with hot and cold cells at every place a face is
evaluated from (a block's first and last plane, its closing rows and columns,
its ghost layers, a whole block), the residual has the bits of the generic
per-cell kernel, in whole blocks and in shares of planes."""
import os

import numpy as np
import pytest

from cases import GAMMA, R
from gpu_helpers import RawFlux

pytestmark = pytest.mark.gpu

VISC = dict(kind=7, law=1, mu=2e-3, T_ref=1.1, power=0.76, prandtl=0.72)
PDISS = dict(kind=3, sensor=1, sensor_param=1e-6, eps_p=0.1, eps_T=0.05)
# (block, k, j, i) with the ghost layers counted, and a factor on T
PLACES = {
    "inside": [((0, 9, 8, 7), 1.9)],
    "planes": [((0, 2, 5, 6), 1.9), ((1, -3, 9, 12), 0.4)],
    "closing": [((0, 8, 6, 17), 0.4), ((1, 7, 17, 4), 1.9), ((1, 10, 17, 17), 2.5)],
    "ghosts": [((0, 1, 7, 7), 1.9), ((0, 9, 7, 18), 0.4), ((1, 9, 18, 9), 1.9), ((1, -2, 4, 11), 1.9)],
    "block": [((1, slice(None), slice(None), slice(None)), 1.5)],
}


@pytest.mark.parametrize("stretch", [False, True], ids=["identity", "stretched"])
@pytest.mark.parametrize("T_ref", [1.1, 1.0])
@pytest.mark.parametrize("place", sorted(PLACES))
def test_staged_kernel_equals_per_cell(place, T_ref, stretch):
    import spade_amd as sa
    g = sa.CartesianGrid((16, 16, 13), (2, 1, 1), ((0.0, 2.0), (-1.0, 1.0), (0.0, 1.5)), num_exch=2,
                         maps=(None, sa.tanh_map(-1.0, 1.0, 1.5) if stretch else None, None))
    rng = np.random.default_rng(12)
    q = rng.standard_normal(g.host_shape)
    q[..., 0] = (1.0 + 0.02 * q[..., 0]) / GAMMA
    q[..., 1] = T_ref * (1.0 + 0.005 * q[..., 1])
    q[..., 2:] *= 0.1
    for at, factor in PLACES[place]:
        q[at + (1,)] *= factor
    arr = sa.GridArray(g).upload(q)
    init = rng.standard_normal(g.host_shape)
    for terms in ([dict(kind=1, order=2), dict(VISC, T_ref=T_ref)],
                  [dict(kind=1, order=2), PDISS, dict(VISC, T_ref=T_ref)]):
        flux = RawFlux(terms, GAMMA, R)
        for increment in (False, True):
            out = []
            for env in (dict(SPD_DISABLE_FAST="1", SPD_DISABLE_SPEC="1"), dict(SPD_FAST_ZSPLIT="1"),
                        dict(SPD_FAST_ZSPLIT="5")):
                os.environ.update(env)
                try:
                    kind = sa.flux_div_kernel(arr, flux)
                    rhs = sa.GridArray(g).upload(init)
                    sa.flux_div(arr, rhs, flux, increment=increment)
                finally:
                    for name in env:
                        os.environ.pop(name, None)
                assert kind == ("fast" if out else "generic")
                out.append(rhs.download())
            print(place, T_ref, stretch, len(terms), increment, flush=True)
            assert np.all(np.isfinite(out[0]))
            assert np.array_equal(out[1], out[0])
            assert np.array_equal(out[2], out[0])
