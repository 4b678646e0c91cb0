"""Warm rain in level chunks: the number of chunks follows from the number of
64-column waves, and the columns do not depend on each other, so the same
columns repeated to more rows (eight, four and two chunks, and one where the
levels are few) give the same bits; the few-row run is checked against the
FP64 oracle.  70 columns leave a ragged second wave."""
import numpy as np
import pytest

import gwm_amd as G
import pyoracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nz,prec,metric", [(1, G.F64, True), (7, G.F32, True), (9, G.F64, False),
                                            (17, G.F32, False), (33, G.F64, True),
                                            (33, G.F32, False)])
def test_chunk_counts_agree(nz, prec, metric):
    nx, ny = 70, 4
    ctx = G.Context(0, prec)
    rng = np.random.default_rng(nz)
    zi = np.linspace(0.0, 400.0 * nz, nz + 1)
    rho = np.repeat(1.2 * np.exp(-zi[:nz] / 8000.0)[:, None, None], ny, 1).repeat(nx, 2)
    f = {O.RHO: rho * (1.0 + 0.01 * rng.random(rho.shape))}
    f[O.RHO_THETA] = f[O.RHO] * (295.0 + 0.004 * zi[:nz, None, None])
    for t, q in enumerate((2e-2, 2e-3, 2e-3)):
        f[O.TRACER0 + t] = f[O.RHO] * q * rng.random(rho.shape)
    f = {k: v.astype(ctx.dtype) for k, v in f.items()}
    cfg = dict(dt=5.0, rain_terminal_velocity=12.0, sedimentation_layer_depth_m=400.0)
    first = None
    for rows in (ny, 256, 2048) + ((65600,) if nz == 1 else ()):
        st = G.State(G.Grid(ctx, nx, rows, nz, z_interfaces=zi), 3)
        for k, v in f.items():
            st.set(k, np.tile(v, (1, rows // ny, 1)))
        st.warm_rain(G.warm_rain_config(**cfg), metric_fallout=metric)
        got = {k: st.get(k) for k in list(f) + [G.PRECIP]}
        first = first or got
        for k, v in got.items():
            np.testing.assert_array_equal(v.reshape(-1, rows, nx)[:, -ny:], first[k].reshape(-1, ny, nx),
                                          err_msg=f"rows {rows}")
    w = O.World(nx, ny, nz, z_interfaces=zi, n_tracers=3, precision=8)
    for k, v in f.items():
        w.set(k, v.astype(np.float64))
    w.warm_rain(O.warm_rain_cfg(**cfg), metric_fallout=metric)
    # the bounds of the whole-column parity test, on the largest values
    tol = 1e-12 if prec == G.F64 else 1e-5
    for k in first:
        want = w.get(k)
        assert np.abs(first[k] - want).max() <= 4 * tol * max(np.abs(want).max(), 1e-6), k


def test_ensemble_member_of_a_million_rows():
    """A batched launch numbers a member's work-groups in 20 bits: a member
    whose warm rain has 2^20 + 1 rows of waves batches beside a small one
    (rows in fours, the last one short), and both equal steps by themselves."""
    ctx = G.Context(0, G.F32)
    cfg, wr = G.step_config(0.5, 2), G.warm_rain_config(dt=0.5, rain_terminal_velocity=5.0)
    members, alone = [], []
    for e, (nx, ny, nz) in enumerate(((2, 2 ** 20 + 1, 1), (40, 24, 9))):
        grid = G.Grid(ctx, nx, ny, nz, z_interfaces=np.linspace(0.0, 500.0 * nz, nz + 1))
        for group in (members, alone):
            rng = np.random.default_rng(e)
            st = G.State(grid, 3)
            st.init_constant_n(u=3.0)
            rho = st.get(O.RHO)
            for t, q in enumerate((2e-2, 2e-3, 2e-3)):
                st.set(O.TRACER0 + t, rho * (q * rng.random(rho.shape)).astype(ctx.dtype))
            group.append(st)
    G.ensemble_steps(members, cfg, wr, 3)
    for m, a in zip(members, alone):
        for _ in range(3):
            a.moist_step(cfg, wr)
        for k in (0, 1, 2, 3, 4, 16, 17, 18, G.PRECIP):
            np.testing.assert_array_equal(m.get(k), a.get(k), err_msg=str(k))
        assert a.get(G.PRECIP).max() > 0
