"""GPU tests of the batched FP32-flux / FP64-state engine.

* against the FP64 path (which equals the reference bit for bit): state and
  kinetic-energy history of a TGV case; tolerance 1e-6 relative max-norm per
  variable on the state after 20 steps, 1e-7 relative on kinetic energy (the
  stated bar for this form is 1e-5 on kinetic energy);
* periodic conservation of mass and total energy to round-off;
* a case's result is bit-for-bit the same alone and in a mix, with or without
  the hipGraph, after the autotuner ran, with every stage kernel shape
  (prefetch depth, register budget) the autotuner chooses between, and with
  the work items taken in XCD runs or every eighth per XCD;
* admission fails cleanly when a case does not fit the HBM budget.
"""
import numpy as np
import pytest

import spade_amd as sa
from spade_amd.serve import Request, Server

pytestmark = pytest.mark.gpu

MB = 1 << 20


def cons_to_prim(cons, gamma, R):
    rho, E, mu, mv, mw = (cons[:, v] for v in range(5))
    u, v, w = mu / rho, mv / rho, mw / rho
    p = (gamma - 1.0) * (E - 0.5 * rho * (u * u + v * v + w * w))
    T = p / (R * rho)
    return np.stack([p, T, u, v, w], axis=-1)        # (blocks, 16, 16, 16, 5)


def prim_to_cons(prim, gamma, R):
    p, T, u, v, w = (prim[..., v] for v in range(5))
    rho = p / (R * T)
    E = 0.5 * rho * (u * u + v * v + w * w) + p / (gamma - 1.0)
    return np.stack([rho, E, rho * u, rho * v, rho * w], axis=1)


def _tgv(cells=32, steps=20, mach=0.1, re=1600.0):
    return sa.CaseSpec("tgv", (cells,) * 3, mach=mach, reynolds=re, steps=steps)


def test_batch_tracks_fp64_path():
    spec = _tgv(32, 20)
    b = sa.Batch(256 * MB)
    cid = b.add(spec)
    cons0 = b.download(cid)
    dt = b.info(cid)["dt"]
    gamma = 1.4
    c0 = 1.0 / spec.mach
    R = c0 * c0 / gamma            # p0 / (rho0 T0)
    # FP64 path on the same initial state
    g = sa.CartesianGrid((16, 16, 16), (2, 2, 2), ((0.0, 2 * np.pi),) * 3, num_exch=2)
    host = np.zeros(g.host_shape)
    host[:, 2:-2, 2:-2, 2:-2] = cons_to_prim(cons0, gamma, R)
    q = sa.GridArray(g).upload(host)
    sa.create_exchange(q).exchange(q)
    gas = sa.IdealGas(gamma, R)
    flux = sa.compose(sa.cent_keep(2, gas), sa.visc_lr(sa.power_law(1.0 / spec.reynolds, 1.0, 0.76, 0.72), gas))
    it = sa.Integrator(q, flux, dt)
    ke64 = []
    for _ in range(spec.steps):
        ke64.append(sa.diagnostics(q, gas)[0])
        it.advance(1)
    b.step(spec.steps)
    ke32, _ = b.diag(cid)
    got = cons_to_prim(b.download(cid), gamma, R)
    ref = q.download()[:, 2:-2, 2:-2, 2:-2]
    scale = np.max(np.abs(ref.reshape(-1, 5)), axis=0)
    err = np.max(np.abs((got - ref).reshape(-1, 5)), axis=0) / scale
    kerr = np.max(np.abs(ke32 - np.array(ke64)) / np.array(ke64))
    print("state rel err per var", err, "KE rel err", kerr)
    assert np.all(err <= 1e-6), err
    assert kerr <= 1e-7, kerr


def test_batch_conserves_mass_and_energy():
    b = sa.Batch(256 * MB)
    cid = b.add(sa.CaseSpec("vortex", (48, 32, 16), mach=0.3, reynolds=500.0, steps=10))
    c0 = b.download(cid)
    b.step(10)
    c1 = b.download(cid)
    for v in (0, 1):
        s0, s1 = c0[:, v].sum(), c1[:, v].sum()
        assert abs(s1 - s0) <= 1e-13 * abs(s0), (v, s0, s1)


def _run_alone(spec, steps, graph=True):
    b = sa.Batch(256 * MB)
    b.use_graph(graph)
    cid = b.add(spec)
    b.step(steps)
    return b.download(cid), b.diag(cid)


def test_alone_equals_mix_bitwise():
    a = _tgv(32, 12, mach=0.2, re=800.0)
    ref_state, (ref_ke, ref_en) = _run_alone(a, 12)
    b = sa.Batch(512 * MB)
    b.add(sa.CaseSpec("vortex", (48, 48, 16), mach=0.4, reynolds=300.0))
    cid = b.add(a)
    b.add(_tgv(16, 4))
    b.step(5)
    other = b.add(sa.CaseSpec("vortex", (32, 16, 32), mach=0.15, reynolds=2000.0))
    g, inter = b.tune()
    print("tuned shape", g, inter)
    b.step(4)
    b.remove(other)
    b.use_graph(False)
    b.step(3)
    st = b.download(cid)
    ke, en = b.diag(cid)
    assert np.array_equal(st, ref_state)
    assert np.array_equal(ke, ref_ke) and np.array_equal(en, ref_en)


SHAPES = [(r, p, o) for r in (16, 8) for p in (1, 2) for o in (3, 2)]


@pytest.mark.parametrize("grid,interleaved", [(300, False), (1024, False), (77, True)])
def test_xcd_runs_agree_bitwise(grid, interleaved):
    """Work items in contiguous runs per XCD (the default) or every eighth
    per XCD: the same states and diagnostics, bit for bit, for persistent
    grids that are and are not multiples of eight."""
    import os
    specs = [sa.CaseSpec("vortex", (48, 32, 16), mach=0.3, reynolds=500.0), _tgv(32, 5),
             sa.CaseSpec("vortex", (16, 48, 32), mach=0.2, reynolds=900.0), _tgv(16, 5)]

    def run(x):
        os.environ["SPD_BATCH_XCD"] = str(x)
        try:
            b = sa.Batch(512 * MB)
            b.set_shape(grid, interleaved=interleaved)
            ids = [b.add(sp) for sp in specs]
            b.step(5)
            return [(b.download(c), b.diag(c)) for c in ids]
        finally:
            os.environ.pop("SPD_BATCH_XCD", None)
    print("batch xcd runs, grid", grid, "interleaved", interleaved, flush=True)
    a, c = run(0), run(1)
    for (sa_, (ka, ea)), (sc, (kc, ec)) in zip(a, c):
        assert np.isfinite(sa_).all()
        assert np.array_equal(sa_, sc)
        assert np.array_equal(ka, kc) and np.array_equal(ea, ec)


@pytest.mark.parametrize("rows,prefetch,occupancy", SHAPES)
def test_kernel_shapes_agree_bitwise(rows, prefetch, occupancy):
    spec = sa.CaseSpec("vortex", (32, 16, 32), mach=0.3, reynolds=700.0)
    ref_state, (ref_ke, ref_en) = _run_alone(spec, 6)
    b = sa.Batch(256 * MB)
    b.set_kernel_shape(rows, prefetch, occupancy)
    b.set_shape(3 * 256 * (16 // rows), interleaved=True)
    cid = b.add(spec)
    b.add(_tgv(16, 4))
    b.step(6)
    sh = b.shape()
    assert (sh["rows"], sh["prefetch"], sh["occupancy"]) == (rows, prefetch, occupancy), sh
    assert np.array_equal(b.download(cid), ref_state)
    ke, en = b.diag(cid)
    assert np.array_equal(ke, ref_ke) and np.array_equal(en, ref_en)


def test_tuner_reports_a_candidate_shape():
    b = sa.Batch(256 * MB)
    b.add(_tgv(32, 2))
    b.add(sa.CaseSpec("vortex", (32, 16, 16), mach=0.2, reynolds=900.0))
    g, inter = b.tune()
    sh = b.shape()
    assert sh["grid"] == g and sh["interleaved"] == inter
    log = b.tune_log()
    assert len(log) == 2 * 8 * 4                       # orders x kernel shapes x grids
    best = min(log, key=lambda e: e["ms_per_step"])
    assert {k: best[k] for k in sh} == sh
    assert sh["rows"] in (16, 8) and sh["prefetch"] in (1, 2) and sh["occupancy"] in (2, 3)
    for bad in ((16, 3, 3), (12, 1, 3), (8, 1, 4)):
        with pytest.raises(sa.SpadeError):
            b.set_kernel_shape(*bad)


def test_graph_and_direct_launch_agree_bitwise():
    spec = sa.CaseSpec("vortex", (32, 32, 16), mach=0.25, reynolds=1000.0)
    s1, d1 = _run_alone(spec, 7, graph=True)
    s2, d2 = _run_alone(spec, 7, graph=False)
    assert np.array_equal(s1, s2) and np.array_equal(d1[0], d2[0])


def test_admission_respects_budget():
    b = sa.Batch(30 * MB)                     # 30 MiB / ~0.5 MiB per block
    big = _tgv(64)                            # 64 blocks: does not fit
    assert not b.fits(big)
    with pytest.raises(sa.SpadeError):
        b.add(big)
    small = _tgv(32)                          # 8 blocks
    ids = [b.add(small) for _ in range(7)]
    assert not b.fits(small)
    b.remove(ids[0])
    assert b.fits(small)


def test_served_results_equal_alone_runs():
    specs = [_tgv(32, 6, mach=0.1), sa.CaseSpec("vortex", (32, 32, 16), mach=0.3, reynolds=400.0, steps=9),
             _tgv(16, 4, mach=0.4, re=200.0), sa.CaseSpec("vortex", (16, 16, 16), mach=0.2, reynolds=3000.0, steps=5)]
    reqs = [Request(i, s, arrival=0.002 * i) for i, s in enumerate(specs)]
    srv = Server(sa.Batch(64 * MB), max_chunk=2)
    res = srv.run(reqs)
    assert len(res) == 4
    for r in res:
        st, (ke, en) = _run_alone(r.request.spec, r.request.spec.steps)
        assert np.array_equal(r.state, st), r.request.rid
        assert np.array_equal(r.ke, ke)


def test_full_ensemble_conserves_and_equals_alone_runs():
    """The 300-case ensemble bench.py times (65.9 M cells, all resident):
    10 steps conserve every case's mass and energy to the round-off of its
    FP64 sums, and three of its cases run alone give the same bits as in the
    mix."""
    from spade_amd import studies
    specs = studies.ensemble_specs(300, 10)
    blocks = sum(s.blocks for s in specs)
    b = sa.Batch(int(blocks * studies.BYTES_PER_BLOCK * 1.02) + (64 << 20))
    ids = [b.add(s) for s in specs]
    print("ensemble:", len(ids), "cases,", blocks, "blocks", flush=True)

    def sums(cid):
        c = b.download(cid)
        return c[:, 0].sum(), c[:, 1].sum()

    s0 = [sums(cid) for cid in ids]
    b.step(10)
    s1 = [sums(cid) for cid in ids]
    drift = np.array([[abs(z[v] - a[v]) / abs(a[v]) for v in (0, 1)] for a, z in zip(s0, s1)])
    print("ensemble: largest relative mass / energy drift", drift.max(axis=0), flush=True)
    # round-off of the FP64 sums: the energy residual carries p_ref D(U) and
    # e_ref d(rho) terms that cancel over a periodic case only up to rounding
    assert np.all(drift <= 1e-10), drift.max(axis=0)
    for n in (0, 150, 299):
        alone, _ = _run_alone(specs[n], 10)
        assert np.array_equal(alone, b.download(ids[n])), n


def test_served_stream_at_its_sizes_equals_alone_runs():
    """The served form at the sizes its request stream draws (cells per axis
    from {32, 64, 96, 128}, 100-2000 steps, Mach 0.1-0.5, Re 100-5000): eight
    requests from the stream's own sampler, the first forced to 128^3, arriving
    as a Poisson stream fast enough that they overlap on the device (continuous
    batching: admitted while others run, retired as they finish).  Every served
    result -- final conserved fields and the per-step kinetic-energy and
    enstrophy history -- equals the same case run alone, bit for bit."""
    from spade_amd import studies
    from spade_amd.serve import poisson_requests
    reqs = poisson_requests(8, 40.0, studies.serving_spec, seed=31)
    s0 = reqs[0].spec
    reqs[0].spec = sa.CaseSpec(s0.kind, (128, 128, 128), mach=s0.mach, reynolds=s0.reynolds, steps=s0.steps)
    for r in reqs:
        print("request", r.rid, r.spec.kind, r.spec.cells, "steps", r.spec.steps, f"arrival {r.arrival:.3f}s",
              flush=True)
        assert r.spec.steps >= 100
    srv = Server(sa.Batch(8 << 30), max_chunk=8)
    res = srv.run(reqs)
    assert len(res) == len(reqs)
    overlap = sum(1 for r in res for o in res if o is not r and o.admitted < r.completed and r.admitted < o.completed)
    print("served: rounds", srv.rounds, "overlapping pairs", overlap // 2, flush=True)
    assert overlap > 0
    for r in res:
        b = sa.Batch(1 << 30)
        cid = b.add(r.request.spec)
        b.step(r.request.spec.steps)
        st = b.download(cid)
        ke, en = b.diag(cid)
        b.close()
        assert np.array_equal(r.state, st), r.request.rid
        assert np.array_equal(r.ke, ke) and np.array_equal(r.enstrophy, en), r.request.rid
        print("request", r.request.rid, "served == alone", flush=True)


class _PoisonBatch(sa.Batch):
    """The device engine, with one NaN density planted in the cases whose
    request is marked, right after admission (a case that has diverged)."""

    def __init__(self, budget, poisoned):
        super().__init__(budget)
        self.poisoned = poisoned

    def add(self, spec):
        cid = super().add(spec)
        if id(spec) in self.poisoned:
            st = self.download(cid)
            st[0, 0, 3, 4, 5] = np.nan
            self.upload(cid, st)
        return cid


def test_served_case_that_diverges_is_retired_others_unaffected():
    """A served case whose state is no longer finite is retired with an error
    after the round in which its kinetic energy turned non-finite; the other
    cases, sharing the device with it, still equal their alone runs bit for
    bit, and its slots return to the pool."""
    specs = [_tgv(32, 12, mach=0.1), _tgv(32, 12, mach=0.2), sa.CaseSpec("vortex", (32, 32, 16), mach=0.3,
                                                                          reynolds=400.0, steps=12)]
    reqs = [Request(i, s, arrival=0.002 * i) for i, s in enumerate(specs)]
    eng = _PoisonBatch(64 * MB, {id(specs[1])})
    srv = Server(eng, max_chunk=3)
    res = srv.run(reqs)
    by = {r.request.rid: r for r in res}
    assert len(res) == 3
    assert by[1].error is not None and "diverged" in by[1].error, by[1].error
    assert len(by[1].ke) < 12 and not np.isfinite(by[1].ke[-1])
    for rid in (0, 2):
        assert by[rid].error is None
        st, (ke, en) = _run_alone(specs[rid], specs[rid].steps)
        assert np.array_equal(by[rid].state, st), rid
        assert np.array_equal(by[rid].ke, ke), rid
    assert eng.fits(specs[0]) and eng.fits(specs[1])


@pytest.mark.parametrize("grid", [None, 5, 70, 4096])
def test_plane_shares_agree_bitwise(grid):
    """The default shape and its 1, 2 or 4 workgroups along a block's planes
    follow the number of blocks (16 here, then 412); a case's bits do not, nor
    do its diagnostics, under the graph or launched directly."""
    spec = sa.CaseSpec("vortex", (32, 64, 32), mach=0.3, reynolds=700.0)
    b = sa.Batch(512 * MB)
    b.set_kernel_shape(16, 1, 3)
    b.set_shape(768)
    ref = b.add(spec)
    filler = [b.add(_tgv(48, 3)) for _ in range(28)]
    b.step(4)
    assert len(filler) == 28
    c = sa.Batch(512 * MB)
    if grid:
        c.set_shape(grid)
    cid = c.add(spec)
    c.step(2)
    more = [c.add(_tgv(48, 3)) for _ in range(15)]
    c.step(1)
    for m in more:
        c.remove(m)
    c.use_graph(False)
    c.step(1)
    print("plane shares, grid", grid, c.shape(), flush=True)
    assert np.array_equal(b.download(ref), c.download(cid))
    for x, y in zip(b.diag(ref), c.diag(cid)):
        assert len(x) == 4 and np.array_equal(x, y)
