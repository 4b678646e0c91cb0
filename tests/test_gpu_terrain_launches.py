"""Launch shapes of the terrain kernels that the autotuner or an ensemble may
pick: level chunks and tile heights of every form, the recorded (batched)
march with its column reference, and the FP32 column reference itself."""
import re

import numpy as np
import pytest

import gwm_amd as G
import pyoracle as O

pytestmark = pytest.mark.gpu
FIELDS = (O.RHO, O.RHO_THETA, O.MOM_U, O.MOM_V, O.MOM_W)


def _state(ctx, nx, ny, nz, height, ntr=0, pert=False, seed=0, **kw):
    zi = np.linspace(0.0, 350.0 * nz, nz + 1)
    grid = G.Grid(ctx, nx, ny, nz, dx=1500.0, dy=900.0, z_interfaces=zi,
                  terrain=G.cosine_mountain(nx, ny, height), **kw)
    st = G.State(grid, ntr, perturbation=pert)
    st.init_constant_n(u=7.0)
    rng = np.random.default_rng(seed)
    for f in FIELDS[2:]:
        a = st.get(f)
        st.set(f, (a + 0.3 * rng.standard_normal(a.shape)).astype(ctx.dtype))
    rho = st.get(O.RHO).astype(np.float64)
    for t in range(ntr):
        st.set(O.TRACER0 + t, (rho * (2e-2, 2e-3, 1e-3)[t] * rng.random(rho.shape)).astype(ctx.dtype))
    return st


@pytest.mark.parametrize("form,prec", [("full", G.F64), ("full", G.F32), ("pert", G.F32),
                                       ("tiny", G.F64), ("tiny", G.F32)])
@pytest.mark.parametrize("nx,ny,nz,open_x,open_y", [
    (70, 13, 33, True, False), (130, 9, 12, False, True), (33, 20, 9, True, True)])
def test_terrain_launch_codes_agree(form, prec, nx, ny, nz, open_x, open_y):
    """Whole columns in 8-row tiles against 2, 3 and 8 chunks and 4-row tiles
    (16 more): two steps and the slow tendencies after them, bit for bit.  The
    column reference (full), the per-cell bases (pert) and the level means of
    heights below 1e-6 m (tiny) are forms of the march; the slow stage takes
    the chunks."""
    first = None
    for code in (1, 2, 3, 8, 17, 18, 24):
        ctx = G.Context(0, prec)
        ctx.set_chunks(code)
        st = _state(ctx, nx, ny, nz, 1e-7 if form == "tiny" else 20.0 * nz, pert=form == "pert",
                    periodic_x=not open_x, periodic_y=not open_y)
        assert st.grid.terrain_active == (form != "tiny")
        st.capture_boundary()
        bc = G.BoundaryConfig(G.BOUNDARY_RELAX, 3.0, G.BOUNDARY_FN(), None)
        for _ in range(2):
            st.ssprk3_step(G.step_config(0.3, 3), bc)
        st.slow_tendencies(G.step_config(0.3, 3))
        got = {f: st.get(f) for f in FIELDS + (6, 7, 8, 9, 10)}
        first = first or got
        assert np.isfinite(got[O.MOM_W]).all() and np.abs(got[O.MOM_W]).max() > 0
        for f, v in got.items():
            np.testing.assert_array_equal(v, first[f], err_msg=f"code {code}, field {f}")


@pytest.mark.parametrize("prec", [G.F32, G.F64])
@pytest.mark.parametrize("height", [200.0, 1e-7])
def test_ensemble_of_terrain_members(prec, height):
    """Uneven terrain members advanced in batched launches (the candidates of
    the ensemble's tuner among them: chunks 2, 4 and 8) against their own
    steps, bit for bit."""
    ctx = G.Context(0, prec)
    sizes = ((70, 33, 36), (40, 20, 32), (130, 9, 33), (33, 5, 40), (64, 16, 35))
    members, alone = ([_state(ctx, *s, height, ntr=3, seed=e, periodic_x=e != 1)
                       for e, s in enumerate(sizes)] for _ in range(2))
    cfg, wr = G.step_config(0.3, 3), G.warm_rain_config(dt=0.3, rain_terminal_velocity=8.0)
    steps = 1 + 2 * 4 + 2  # a warm one, a pair for each candidate, one with the fastest
    G.ensemble_steps(members, cfg, wr, steps)
    lines = [s for s in G.ensemble_tuning_report().splitlines() if s.startswith("5 members:")]
    assert any(re.search(r"own codes [0-9.]+ ms chunks 2 rows 8 [0-9.]+ ms", s) for s in lines), lines
    for m, a in zip(members, alone):
        for _ in range(steps):
            a.moist_step(cfg, wr)
        for f in FIELDS + (16, 17, 18, G.PRECIP):
            np.testing.assert_array_equal(m.get(f), a.get(f), err_msg=f"{a.grid.nx}: field {f}")
        assert np.isfinite(a.get(O.MOM_W)).all()


@pytest.mark.parametrize("nz,z_top", [(1, 800.0), (7, 9000.0), (8, 12000.0), (40, 16000.0),
                                      (6, 24000.0), (4, 26000.0)])
def test_fp32_column_reference(nz, z_top):
    """w after one FP32 substep against the FP64 oracle from the same state:
    levels around a segment of the reference, and layers so deep (4000 m and
    more) that the series gives way to the power.  A face's w holds the
    roundings of two pressures (about three each), two of the reference and a
    few of the product: below 10 of 1.2e5 Pa, over dz."""
    nx, ny, dt = 67, 9, 0.2
    kw = dict(z_top=z_top, terrain=G.cosine_mountain(nx, ny, 0.02 * z_top))
    w = O.World(nx, ny, nz, precision=8, **kw)
    w.init_mountain_wave(1.18, 300.0, 0.0)
    rng = np.random.default_rng(nz)
    rho = (w.get(O.RHO) * (1.0 + 0.01 * rng.random((nz, ny, nx)))).astype(np.float32)
    theta = 300.0 + 5.0 * rng.random(rho.shape)
    rt = (rho * theta).astype(np.float32)
    ctx = G.Context(0, G.F32)
    grid = G.Grid(ctx, nx, ny, nz, **kw)
    st = G.State(grid, 0)
    for f, v in zip(FIELDS, (rho, rt, 0.0, 0.0, 0.0)):
        v = np.broadcast_to(np.float32(v), w.get(f).shape)
        w.set(f, v.astype(np.float64))
        st.set(f, v)
    w.fast_modes(O.step_cfg(dt=dt, fast_substeps=1))
    st.fast_modes(G.step_config(dt=dt, fast_substeps=1))
    idz = grid.metric(3).astype(np.float64)
    got, want = st.get(O.MOM_W).astype(np.float64), w.get(O.MOM_W)
    err = np.abs(got - want)[1:nz]
    bound = dt * idz[1:nz] * 10 * 2.0 ** -23 * 1.2e5 + 4 * 2.0 ** -23 * np.abs(want[1:nz])
    assert (err <= bound).all(), float((err / bound).max())
