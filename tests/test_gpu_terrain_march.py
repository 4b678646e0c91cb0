"""The terrain march and its column reference against the FP64 oracle at the
edges of their tiles: columns not a multiple of the 64 of a work-group, levels
around the seven that one segment prepares, a single level, layers so deep
that the density series gives way to the power, a cell on the EOS's floors,
partial tiles, and level chunks (whose results are the whole march's)."""
import numpy as np
import pytest

import gwm_amd as G
import pyoracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nz,z_top,open_x,thin", [
    (5, 3, 1, 800.0, False, False), (67, 9, 2, 1500.0, True, False),
    (70, 13, 7, 9000.0, False, False), (65, 5, 8, 12000.0, True, True),
    (64, 8, 15, 16000.0, False, False), (130, 4, 6, 24000.0, False, False)])
def test_terrain_substeps_against_oracle(nx, ny, nz, z_top, open_x, thin):
    terrain = G.cosine_mountain(nx, ny, 0.02 * z_top)
    kw = dict(periodic_x=not open_x, z_top=z_top, terrain=terrain)
    w = O.World(nx, ny, nz, precision=8, **kw)
    w.init_mountain_wave(1.18, 300.0, 10.0)
    rng = np.random.default_rng(nz)
    rho = w.get(O.RHO) * (1.0 + 0.002 * rng.random((nz, ny, nx)))
    if thin:
        rho[nz // 2, ny // 2, nx // 2] = 2e-7
    w.set(O.RHO, rho)
    start = {f: w.get(f) for f in (O.RHO, O.RHO_THETA, O.MOM_U, O.MOM_V, O.MOM_W)}
    w.fast_modes(O.step_cfg(dt=0.2, fast_substeps=3))
    first = None
    for code in (1, 2, 3, 16 + 1, 16 + 2):  # chunks, with 16: tiles of 4 rows
        if (code & 15) > nz:
            continue
        ctx = G.Context(0, G.F64)
        ctx.set_chunks(code)
        st = G.State(G.Grid(ctx, nx, ny, nz, **kw), 0)
        for f, v in start.items():
            st.set(f, v)
        st.fast_modes(G.step_config(dt=0.2, fast_substeps=3))
        got = {f: st.get(f) for f in start}
        first = first or got
        for f, v in got.items():
            np.testing.assert_array_equal(v, first[f], err_msg=f"chunks {code}")
            want = w.get(f)
            # rounding of p (some 1e5 Pa at 2^-52 times a few ulp) through
            # dt / d over three substeps, relative to the field's own size
            scale = np.abs(want).max() + 1.0
            assert np.abs(v - want).max() <= 2e-11 * scale, (f, code)


@pytest.mark.parametrize("prec", [G.F64, G.F32])
@pytest.mark.parametrize("case", ["overflow", "thin"])
def test_column_reference_outside_the_series(prec, case):
    """Levels where the density series does not hold.  A cell whose pressure
    overflows (its theta is finite, so the power gives the reference a finite
    density there): w is not finite on the cell's two faces only.  Pressures
    between one and two Pascal (too near the floor of one Pascal), with layers
    whose weight the series' variable would take for a small departure: the
    reference ends on the floor.  Against the oracle of the same precision;
    each p carries a few roundings on both sides, so p - p_ref of a face is off
    by at most 16 of them (the floored case is exact in p_ref)."""
    nx, ny, nz = 70, 6, 9
    if case == "thin":
        theta, p = 300.0, 1.5
        rho0 = p / (287.05 * theta * (p / 1e5) ** 0.2854)
        z_top = nz * (p + 1.0) / (9.81 * rho0)
    else:
        theta, rho0, z_top = 300.0, 1.0, 9000.0
    kw = dict(z_top=z_top, terrain=G.cosine_mountain(nx, ny, 0.001 * z_top))
    cfg = dict(dt=0.2, fast_substeps=1)
    w = O.World(nx, ny, nz, precision=8 if prec == G.F64 else 4, **kw)
    ctx = G.Context(0, prec)
    rho = np.full((nz, ny, nx), rho0)
    rt = rho * theta
    if case == "overflow":
        rt[4, 3, 65] = 1e30 if prec == G.F32 else 1e250
    st = G.State(G.Grid(ctx, nx, ny, nz, **kw), 0)
    for f, v in ((O.RHO, rho), (O.RHO_THETA, rt), (O.MOM_U, 0.0), (O.MOM_V, 0.0), (O.MOM_W, 0.0)):
        v = np.broadcast_to(v, w.get(f).shape).astype(ctx.dtype)
        w.set(f, v.astype(w.get(f).dtype))
        st.set(f, v)
    w.fast_modes(O.step_cfg(**cfg))
    st.fast_modes(G.step_config(**cfg))
    got, want = st.get(O.MOM_W), w.get(O.MOM_W)
    faces = np.isfinite(got)
    if case == "overflow":
        assert not faces[4:6, 3, 65].any() and faces.sum() == faces.size - 2
    else:
        assert faces.all()
    p_max = 1.3e5 if case == "overflow" else 1.5
    bound = 0.2 * nz / z_top * 1.01 * 16 * np.finfo(ctx.dtype).eps * p_max
    err = np.abs(got[faces] - want[faces]).max()
    assert err <= bound + 4 * np.finfo(ctx.dtype).eps * np.abs(want[faces]).max()


@pytest.mark.parametrize("prec", [G.F64, G.F32])
def test_reference_differences_hold_one_rounding(prec):
    """K14 takes differences of the column reference between neighbouring
    levels; each holds one rounding, that of the upper level's pressure.  All
    cells share one state, so p cancels from w but for the start of the
    reference, and the layers are thin: the rounding (half an ulp of 1e5, over
    dz) outweighs the others, which are relative to the layer's 60 Pa."""
    nx, ny, nz = 70, 9, 40
    z_top, dt = 200.0, 0.5
    ctx = G.Context(0, prec)
    R, ld = ctx.dtype, np.longdouble
    kw = dict(z_top=z_top, terrain=G.cosine_mountain(nx, ny, 10.0))
    grid = G.Grid(ctx, nx, ny, nz, **kw)
    st = G.State(grid, 0)
    for f, v in ((O.RHO, 1.16), (O.RHO_THETA, 1.16 * 300.0), (O.MOM_U, 0.0), (O.MOM_V, 0.0),
                 (O.MOM_W, 0.0)):
        st.fill(f, v)
    st.fast_modes(G.step_config(dt=dt, fast_substeps=1))
    rho, th = ld(R(1.16)), ld(R(R(1.16 * 300.0) / R(1.16)))
    rd, kappa, grav = ld(R(287.05)), ld(R(0.2854)), ld(R(9.81))
    zc, idz = grid.metric(1).astype(ld), grid.metric(3).astype(ld)

    def density(p):
        return p / (rd * th * (p / 1e5) ** kappa)

    p = np.empty((nz, ny, nx), ld)
    r = np.empty_like(p)
    p[0] = 1e5 * (rho * rd * th / 1e5) ** (1 / (1 - kappa))
    r[0] = density(p[0])
    for k in range(1, nz):
        dz = zc[k] - zc[k - 1]
        p[k] = p[k - 1] - grav * r[k - 1] * dz
        for _ in range(4):
            p[k] = p[k - 1] - grav * (r[k - 1] + density(p[k])) * dz / 2
        r[k] = density(p[k])
    want = ld(R(dt)) * ((p[1:] - p[:-1]) * idz[1:nz] - grav * (2 * rho - r[1:] - r[:-1]) / 2)
    bound = dt * idz[1:nz] * np.spacing(R(0.99e5)) * ld(0.55)
    err = np.abs(st.get(O.MOM_W)[1:nz] - want)
    assert (err <= bound).all(), float((err / bound).max())
