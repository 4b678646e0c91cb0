"""The one-launch budget sums against numpy on ragged sizes: rows shorter and
longer than a wave, a last batch of loads that ends inside it, fewer rows than
waves, every tracer count, terrain and the perturbation form.  Extremes and
counts are exact (single operations on the same values; the device's FP64
division misses numpy's only beside a tie, closer than 2^-52 ulp); sums are
compensated on both sides, so they agree to the rounding of the result and of
each term (2^-53 of the sum of magnitudes bounds both)."""
import math

import numpy as np
import pytest

import gwm_amd as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nz,ntr,prec,form", [
    (3, 2, 2, 0, G.F32, "full"), (63, 5, 3, 1, G.F32, "full"), (65, 9, 7, 2, G.F64, "full"),
    (257, 31, 5, 3, G.F32, "full"), (600, 7, 4, 4, G.F64, "full"), (130, 40, 6, 3, G.F32, "pert"),
    (70, 33, 5, 3, G.F64, "terrain"), (70, 33, 5, 0, G.F32, "terrain pert")])
def test_budget_sums_on_ragged_sizes(nx, ny, nz, ntr, prec, form):
    rng = np.random.default_rng(nx)
    ctx = G.Context(0, prec)
    terrain = G.cosine_mountain(nx, ny, 300.0) if "terrain" in form else None
    grid = G.Grid(ctx, nx, ny, nz, terrain=terrain, z_interfaces=np.linspace(0, 9000.0, nz + 1) ** 1.02)
    st = G.State(grid, ntr, perturbation="pert" in form)
    f = {0: 0.4 + rng.random((nz, ny, nx)), 1: 300.0 * (0.4 + rng.random((nz, ny, nx))),
         2: rng.standard_normal((nz, ny, nx + 1)), 3: rng.standard_normal((nz, ny + 1, nx)),
         4: rng.standard_normal((nz + 1, ny, nx))}
    f.update({16 + t: rng.random((nz, ny, nx)) * 0.01 for t in range(ntr)})
    for k, a in f.items():
        st.set(k, a.astype(ctx.dtype))
    rain = (rng.random((ny, nx)) * (rng.random((ny, nx)) < 0.5)).astype(ctx.dtype)
    st.set(G.PRECIP, rain)
    s = st.summary()
    f = {k: (st.get_f64(k) if k < 2 else st.get(k).astype(np.float64)) for k in f}

    def close(got, terms):
        terms = np.asarray(terms, np.float64).ravel()
        bound = 2.0 ** -52 * np.abs(terms).sum()
        if "pert" in form:  # FP64 base sums added term by term on the host
            bound *= 64.0
        assert abs(got - math.fsum(terms)) <= bound

    for name, k in (("total_dry_mass", 0), ("total_rho_theta_m", 1),
                    ("total_horizontal_momentum_x", 2), ("total_horizontal_momentum_y", 3),
                    ("total_vertical_momentum", 4)):
        close(s[name], f[k])
    ends = [("rho", f[0]), ("theta", f[1] / np.maximum(f[0], 1e-12)), ("u", f[2]), ("v", f[3]),
            ("w", f[4])]
    idz = grid.metric(2).astype(np.float64)
    for t, (path, q) in enumerate((("vapor_path", "qv"), ("cloud_path", "qc"), ("rain_path", "qr"))):
        if t < ntr:
            close(s[path], f[16 + t] * (1.0 / idz))
            ends.append((q, f[16 + t] / np.maximum(f[0], 1e-12)))
        else:
            assert s[path] == s[q + "_min"] == s[q + "_max"] == 0.0
    for name, a in ends:
        # the perturbation form's device base is the FP32 one, get_f64's the FP64 one
        rel = 3e-7 if "pert" in form else 0.0
        assert abs(s[name + "_min"] - a.min()) <= rel * abs(a.min()), name
        assert abs(s[name + "_max"] - a.max()) <= rel * abs(a.max()), name
    close(s["precip_sum"], rain)
    assert s["precip_max"] == rain.max() and s["precipitating_cells"] == (rain > 0).sum()
    assert s["precip_cells"] == nx * ny and s["nonfinite_values"] == 0
    bad = st.get(4)
    bad[nz, ny - 1, nx - 1] = np.inf
    bad[0, 0, 0] = np.nan
    st.set(4, bad)
    s = st.summary()
    assert s["nonfinite_values"] == 2 and np.isnan(s["w_min"]) and np.isfinite(s["u_max"])


def test_overflowing_theta_is_reported():
    """rho theta and rho finite, their quotient not: the field's extremes are
    NaN, the count of non-finite prognostic values is zero."""
    ctx = G.Context(0, G.F64)
    st = G.State(G.Grid(ctx, 66, 5, 3), 1)
    for f, v in ((0, 1.0), (1, 300.0), (16, 0.01)):
        st.fill(f, v)
    rt, rho = st.get(1), st.get(0)
    rt[2, 4, 65], rho[2, 4, 65] = 1e300, 1e-10
    st.set(1, rt)
    st.set(0, rho)
    s = st.summary()
    assert np.isnan(s["theta_min"]) and np.isnan(s["theta_max"]) and s["nonfinite_values"] == 0
    assert s["rho_min"] == 1e-10 and s["qv_max"] == 0.01 / 1e-10
