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
