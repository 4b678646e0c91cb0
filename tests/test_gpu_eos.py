"""The step kernels' equation of state against extended precision, through
the slow tendency of u at rest: -(p_i - p_{i-1}) / dx on a flat grid.

rho theta spans the model's range and beyond it (thin densities below the
1e-6 floor, ratios below theirs, rho theta = 0).  Roundings of a pressure:
the ratio's two products (times gamma), the power (2 ulp: log2, its sum with
the exponent's part, 2^f), the last product; together below 6 ulp, and the
quotient's own."""
import numpy as np
import pytest

import gwm_amd as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,thin", [(G.F64, False), (G.F64, True), (G.F32, False), (G.F32, True)])
def test_pressure_of_the_step_kernels(prec, thin):
    nx, ny, nz = 130, 6, 40
    ctx = G.Context(0, prec)
    grid = G.Grid(ctx, nx, ny, nz, z_interfaces=np.linspace(0.0, 12000.0, nz + 1))
    st = G.State(grid, 0)
    rng = np.random.default_rng(5)
    shape = (nz, ny, nx)
    rho = 1.3 * np.exp(-5.0 * rng.random(shape))
    rt = rho * (250.0 + 300.0 * rng.random(shape))
    if thin:
        pick = rng.random(shape)
        rho = np.where(pick < 0.2, 3e-7, rho)
        rt = np.where(pick > 0.8, rng.choice([0.0, 1e-5, 1e-3, 2e4], shape), rt)
    rho, rt = rho.astype(ctx.dtype), rt.astype(ctx.dtype)
    st.set(0, rho)
    st.set(1, rt)
    st.slow_tendencies(G.step_config(1.0, 1))
    got = st.get(8)[:, :, :nx].astype(np.longdouble)
    ld = np.longdouble
    one = ctx.dtype(1)  # R_d and gamma as the working precision has them
    rd, gamma = ld(ctx.dtype(287.05)), ld(one / (one - ctx.dtype(0.2854)))
    r, t = rho.astype(ld), rt.astype(ld)
    ratio = np.maximum(r * rd * (t / np.maximum(r, ld(ctx.dtype(1e-6)))) / ld(1e5), ld(1e-6))
    p = ld(1e5) * ratio ** gamma
    left = np.roll(p, 1, axis=2)
    eps = ld(np.finfo(ctx.dtype).eps)
    want = (left - p) / 1000
    bound = 6 * eps * (np.abs(p) + np.abs(left)) / 1000 + 2 * eps * np.abs(want)
    assert (np.abs(got - want) <= bound).all(), float((np.abs(got - want) / bound).max())


def test_fp64_pressure_of_a_state_that_is_not_finite():
    """A density that is infinite or NaN makes the ratio NaN, which takes the
    floor (p0 1e-6^gamma), whatever rho theta is; so do a NaN and a negative
    infinity of rho theta.  Through the slow tendency of u at rest, on the
    faces beside the cell: its other terms are zero."""
    nx, ny, nz = 66, 12, 3
    ctx = G.Context(0, G.F64)
    grid = G.Grid(ctx, nx, ny, nz, z_interfaces=np.linspace(0.0, 900.0, nz + 1))
    st = G.State(grid, 0)
    rho, rt = np.full((nz, ny, nx), 1.1), np.full((nz, ny, nx), 330.0)
    inf, nan = np.inf, np.nan
    cells = [(inf, 330.0), (-inf, 330.0), (nan, 330.0), (inf, inf), (nan, inf), (inf, 0.0),
             (inf, nan), (1.1, nan), (1.1, -inf)]
    for j, (r, t) in enumerate(cells):
        rho[1, j, 64], rt[1, j, 64] = r, t
    st.set(0, rho.astype(ctx.dtype))
    st.set(1, rt.astype(ctx.dtype))
    st.slow_tendencies(G.step_config(1.0, 1))
    du = st.get(8)[1].astype(np.float64)
    p = 1e5 * (330.0 * 287.05 / 1e5) ** (1.0 / (1.0 - 0.2854))
    p_floor = 1e5 * 1e-6 ** (1.0 / (1.0 - 0.2854))
    bound = 12 * 2.0 ** -52 * p / 1000  # six roundings of p, the kernel's and numpy's
    for j, cell in enumerate(cells):
        assert abs(du[j, 64] - (p - p_floor) / 1000) <= bound, cell
        assert abs(du[j, 65] - (p_floor - p) / 1000) <= bound, cell
