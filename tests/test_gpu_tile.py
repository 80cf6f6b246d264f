"""The tiled face-once kernel on block shapes at its edges: blocks narrower
than a wavefront's row, wider than a tile, with remainders in every axis, one
or several workgroups along k, one and two ghost layers, three mapped axes.

It evaluates the per-cell kernel's expressions once per face, so the bar is
the generic per-cell kernel (SPD_DISABLE_SPEC=1) bit for bit, in overwrite and
increment mode, with hot and cold cells too, whose face temperatures leave the
power law's series and send their planes through the library pow.
"""
import os

import numpy as np
import pytest

from cases import GAMMA, R
from gpu_helpers import RawFlux

pytestmark = pytest.mark.gpu

VC = dict(kind=7, law=0, mu=2e-3, prandtl=0.72)
VP = dict(kind=7, law=1, mu=2e-3, T_ref=1.1, power=0.76, prandtl=0.72)
WALE = dict(sgs=1, sgs_cw=0.5, sgs_delta=0.3, sgs_prt=0.9)
PDD = dict(kind=3, sensor=1, sensor_param=1e-6, eps_p=0.1, eps_T=0.05)
FLUXES = {
    "keep2_visc": [dict(kind=1, order=2), VP],
    "keep2_ducros_wale": [dict(kind=1, order=2), PDD, dict(VP, **WALE)],
    "keep4_wale": [dict(kind=1, order=4), dict(VC, **WALE)],
    "weno_visc": [dict(kind=4, split=0, smooth=1), VP],
    "fweno_visc": [dict(kind=5, smooth=1), VC],
    "totani_visc": [dict(kind=2), VP],
    "first_wale": [dict(kind=6), dict(VC, **WALE)],
    "fds_visc": [dict(kind=9, smooth=0), VC],
}
SHAPES = [((2, 2, 2), (2, 1, 1)), ((3, 5, 7), (2, 2, 1)), ((17, 15, 3), (1, 2, 2)), ((24, 20, 12), (1, 1, 2)),
          ((40, 6, 5), (1, 2, 1)), ((5, 67, 4), (1, 1, 1)), ((16, 16, 16), (2, 1, 1)), ((4, 4, 70), (1, 1, 1))]


def _compare(cells, blocks, terms, maps=(None, None, None), ng=2, hot=False):
    import spade_amd as sa
    g = sa.CartesianGrid(cells, blocks, ((0.0, 2.0), (-1.0, 1.0), (0.0, 1.5)), num_exch=ng,
                         maps=tuple(None if m is None else sa.tanh_map(*m) for m in maps))
    rng = np.random.default_rng(sum(cells))
    q = rng.standard_normal(g.host_shape)
    q[..., 0] = (1.0 + 0.02 * q[..., 0]) / GAMMA
    q[..., 1] = 1.1 * (1.0 + 0.005 * q[..., 1])
    q[..., 2:] *= 0.1
    if hot:
        q[0, ng, ng, ng, 1] = 2.3
        q[-1, -1 - ng, -1 - ng, -1, 1] = 0.4
    arr = sa.GridArray(g).upload(q)
    init = rng.standard_normal(g.host_shape)
    flux = RawFlux(terms, GAMMA, R)
    for increment in (False, True):
        out = []
        for generic in (False, True):
            rhs = sa.GridArray(g).upload(init)
            if generic:
                os.environ["SPD_DISABLE_SPEC"] = "1"
            os.environ["SPD_DISABLE_FAST"] = "1"
            try:
                sa.flux_div(arr, rhs, flux, increment=increment)
            finally:
                os.environ.pop("SPD_DISABLE_SPEC", None)
                os.environ.pop("SPD_DISABLE_FAST", None)
            out.append(rhs.download())
        print(cells, blocks, increment, np.max(np.abs(out[0] - out[1])), flush=True)
        assert np.all(np.isfinite(out[0]))
        assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("name", sorted(FLUXES))
@pytest.mark.parametrize("cells, blocks", SHAPES, ids=["x".join(map(str, s[0])) for s in SHAPES])
def test_shapes_equal_per_cell(cells, blocks, name):
    _compare(cells, blocks, FLUXES[name])


@pytest.mark.parametrize("name", sorted(FLUXES))
@pytest.mark.parametrize("maps", [(None, (-1.0, 1.0, 1.5), None), ((0.0, 2.0, 0.8), (-1.0, 1.0, 1.5), (0.0, 1.5, 1.1))],
                         ids=["y", "xyz"])
def test_mapped_equal_per_cell(maps, name):
    _compare((11, 9, 6), (2, 1, 2), FLUXES[name], maps=maps)


@pytest.mark.parametrize("name", ["keep2_visc", "keep2_ducros_wale", "weno_visc", "totani_visc"])
def test_planes_outside_the_series_equal_per_cell(name):
    _compare((11, 9, 6), (2, 1, 2), FLUXES[name], hot=True)


def test_one_ghost_layer_equal_per_cell():
    _compare((7, 10, 5), (1, 2, 1), FLUXES["keep2_visc"], ng=1)


@pytest.mark.parametrize("name", ["weno_visc", "fweno_visc"])
@pytest.mark.parametrize("p, jump", [(1e-12, 1.0), (1.0, 0.0), (1.0, 1e6), (1e55, 1.0), (1.0, np.inf)],
                         ids=["faint", "uniform", "shock", "huge", "infinite"])
def test_weno_quotients_equal_per_cell(p, jump, name):
    """The smooth weights' own quotients over the range of their squares (1e-32
    for equal fluxes, about 1e220 for "huge") and through an infinite cell."""
    import spade_amd as sa
    g = sa.CartesianGrid((19, 18, 5), (1, 2, 1), ((0.0, 2.0), (-1.0, 1.0), (0.0, 1.5)), num_exch=2)
    q = np.random.default_rng(4).standard_normal(g.host_shape)
    q *= 0.0 if jump == 0.0 else 1.0
    q[..., 0] = p * (1.0 + 0.3 * np.tanh(q[..., 0]))
    q[..., 1] = 1.1 * (1.0 + 0.005 * q[..., 1])
    q[..., 2:] = 0.3 + 0.2 * q[..., 2:]
    if jump:
        q[0, 6, 9:, :, 0] *= jump
    arr = sa.GridArray(g).upload(q)
    flux = RawFlux(FLUXES[name], GAMMA, R)
    out = []
    for generic in (False, True):
        if generic:
            os.environ["SPD_DISABLE_SPEC"] = "1"
        try:
            rhs = sa.GridArray(g)
            sa.flux_div(arr, rhs, flux)
            out.append(rhs.download())
        finally:
            os.environ.pop("SPD_DISABLE_SPEC", None)
    print(name, p, jump, np.isnan(out[0]).sum(), flush=True)
    assert np.array_equal(out[0], out[1], equal_nan=True)
    assert np.isfinite(out[0]).all() == np.isfinite(jump)


@pytest.mark.parametrize("nz", [16, 17, 40])
def test_tall_mapped_blocks_equal_per_cell(nz):
    """16x16 cross-sections with x and z mapped: more than 16 planes exceed the
    staged kernel's metric tables, so those take the tiled kernel."""
    import spade_amd as sa
    g = sa.CartesianGrid((16, 16, nz), (1, 2, 1), ((0.0, 2.0), (-1.0, 1.0), (0.0, 1.5)), num_exch=2,
                         maps=(sa.tanh_map(0.0, 2.0, 0.8), None, sa.tanh_map(0.0, 1.5, 1.1)))
    q = np.random.default_rng(nz).standard_normal(g.host_shape)
    q[..., 0] = (1.0 + 0.02 * q[..., 0]) / GAMMA
    q[..., 1] = 1.1 * (1.0 + 0.005 * q[..., 1])
    arr = sa.GridArray(g).upload(q)
    flux = RawFlux([dict(kind=1, order=2), VC], GAMMA, R)
    out = []
    for generic in (False, True):
        if generic:
            os.environ["SPD_DISABLE_SPEC"] = os.environ["SPD_DISABLE_FAST"] = "1"
        try:
            rhs = sa.GridArray(g)
            sa.flux_div(arr, rhs, flux)
            out.append(rhs.download())
        finally:
            os.environ.pop("SPD_DISABLE_SPEC", None)
            os.environ.pop("SPD_DISABLE_FAST", None)
    print("tall mapped block", nz, flush=True)
    assert np.array_equal(*out)


@pytest.mark.parametrize("name", ["keep2", "weno_visc"])
@pytest.mark.parametrize("cells", [(16, 16, 16), (11, 9, 6)], ids=["staged", "tiled"])
def test_cell_quotients_equal_per_cell(cells, name):
    """Densities and energies of cells at the ends: zero, NaN and negative
    temperatures and pressures (densities zero, infinite, NaN), and far from
    one.  (Infinite pressures and temperatures themselves the per-cell kernel
    multiplies by the zero components of a face normal, which the face-once
    kernels leave out.)"""
    import spade_amd as sa
    g = sa.CartesianGrid(cells, (1, 2, 1), ((0.0, 2.0), (-1.0, 1.0), (0.0, 1.5)), num_exch=2)
    rng = np.random.default_rng(9)
    q = rng.standard_normal(g.host_shape)
    q[..., 0] = 1.0 + 0.02 * q[..., 0]
    q[..., 1] = 1.1 * (1.0 + 0.005 * q[..., 1])
    pts = [(0.0, 1.0), (1.0, 0.0), (0.0, 0.0), (np.nan, 1.0), (1.0, -2.0), (-1.0, 1.0),
           (1e200, 1.0), (1e-200, 1.0), (1.0, 1e100), (1.0, 1e-100), (-0.0, 1.0)]
    for p, t in pts:
        at = (rng.integers(q.shape[0]),) + tuple(rng.integers(2, n - 2) for n in q.shape[1:4])
        q[at][:2] = p, t
    arr = sa.GridArray(g).upload(q)
    flux = RawFlux([dict(kind=1, order=2), VC] if name == "keep2" else FLUXES[name], GAMMA, R)
    out = []
    for generic in (False, True):
        if generic:
            os.environ["SPD_DISABLE_SPEC"] = os.environ["SPD_DISABLE_FAST"] = "1"
        try:
            rhs = sa.GridArray(g)
            sa.flux_div(arr, rhs, flux)
            out.append(rhs.download())
        finally:
            os.environ.pop("SPD_DISABLE_SPEC", None)
            os.environ.pop("SPD_DISABLE_FAST", None)
    print("cell quotients", name, cells, np.isnan(out[0]).sum(), flush=True)
    assert np.isnan(out[0]).any() and np.isfinite(out[0]).any()
    assert np.array_equal(*out, equal_nan=True)
