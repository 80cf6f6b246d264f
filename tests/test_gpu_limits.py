"""Viscous laws at the ends of their parameters' ranges: the face-once kernels
(16x16 and tiled) have the bits of the generic per-cell kernel."""
import os

import numpy as np
import pytest

from cases import GAMMA, R
from gpu_helpers import RawFlux

pytestmark = pytest.mark.gpu

POWER = dict(kind=7, law=1, mu=2e-3, T_ref=1.1, power=0.76, prandtl=0.72)
WALE = dict(sgs=1, sgs_cw=0.5, sgs_delta=0.3, sgs_prt=0.9)


def _both(cells, terms, ng=2, maps=(None, None, None), touch=None):
    """The residual from the kernel the library chooses and from the generic one."""
    import spade_amd as sa
    g = sa.CartesianGrid(cells, (2, 1, 1), ((0.0, 2.0), (-1.0, 1.0), (0.0, 1.5)), num_exch=ng,
                         maps=tuple(None if m is None else sa.tanh_map(*m) for m in maps))
    q = np.random.default_rng(sum(cells)).standard_normal(g.host_shape)
    q[..., 0] = (1.0 + 0.02 * q[..., 0]) / GAMMA
    q[..., 1] = 1.1 * (1.0 + 0.005 * q[..., 1])
    q[..., 2:] *= 0.1
    if touch is not None:
        touch(q)
    arr = sa.GridArray(g).upload(q)
    flux = RawFlux(terms, GAMMA, R)
    out = []
    for generic in (False, True):
        if generic:
            os.environ["SPD_DISABLE_SPEC"] = os.environ["SPD_DISABLE_FAST"] = "1"
        try:
            kind = sa.flux_div_kernel(arr, flux)
            rhs = sa.GridArray(g)
            sa.flux_div(arr, rhs, flux)
            out.append((kind, rhs.download()))
        finally:
            os.environ.pop("SPD_DISABLE_SPEC", None)
            os.environ.pop("SPD_DISABLE_FAST", None)
    (kind, got), (ref_kind, ref) = out
    print(cells, kind, np.max(np.abs(got - ref)), flush=True)
    assert ref_kind == "generic" and kind != "generic"
    return got, ref


@pytest.mark.parametrize("cells", [(16, 16, 16), (11, 9, 6)], ids=["staged", "tiled"])
@pytest.mark.parametrize("changes", [dict(prandtl=np.inf), dict(T_ref=np.inf), dict(prandtl=np.inf, **WALE)],
                         ids=["prandtl", "T_ref", "prandtl_wale"])
def test_infinite_parameters(changes, cells):
    """An infinite Prandtl number switches heat conduction off, an infinite
    reference temperature the viscosity."""
    got, ref = _both(cells, [dict(kind=1, order=2), dict(POWER, **changes)])
    assert np.all(np.isfinite(ref))
    assert np.array_equal(got, ref)


@pytest.mark.parametrize("cells", [(16, 16, 16), (11, 9, 6)], ids=["staged", "tiled"])
@pytest.mark.parametrize("var", [2, 3, 4])
def test_infinite_velocity_on_a_stretched_axis(var, cells):
    """An infinite velocity gradient divided by dy/deta stays infinite, so the
    Ducros sensor's denominator gives the finite values that the division gives:
    wherever the generic kernel's residual is a number, so is this one, and the
    same one."""
    def touch(q):
        q[1, 5, 6, 7, var] = np.inf
    pdiss = dict(kind=3, sensor=1, sensor_param=1e-6, eps_p=0.1, eps_T=0.05)
    got, ref = _both(cells, [dict(kind=1, order=2), pdiss], maps=(None, (-1.0, 1.0, 1.5), None), touch=touch)
    assert np.isnan(ref).any()
    number = ~np.isnan(ref)
    assert np.array_equal(got[number], ref[number])
