"""GPU parity: the HIP path (through the C-ABI) against the CPU oracle.

Bars (written per test):
  - halo maps, interface averaging, metrics, initial states: bit-exact;
  - FP64 operators and steps: relative L2 <= 1e-11 against the FP64 oracle;
  - FP32 operators: relative L2 <= 1e-5 against the FP32 oracle and
    <= 1e-4 against the FP64 oracle.
Momentum fields that start at rest are compared with an absolute floor
scaled to the field's own magnitude.
"""
import numpy as np
import pytest

import gwm_amd as G
import pyoracle as O

pytestmark = pytest.mark.gpu

FIELDS = (O.RHO, O.RHO_THETA, O.MOM_U, O.MOM_V, O.MOM_W)
NAMES = {O.RHO: "rho", O.RHO_THETA: "rho_theta", O.MOM_U: "u", O.MOM_V: "v", O.MOM_W: "w"}


@pytest.fixture(scope="module")
def ctx32():
    c = G.Context(0, G.F32)
    yield c
    c.close()


@pytest.fixture(scope="module")
def ctx64():
    c = G.Context(0, G.F64)
    yield c
    c.close()


def ctx_for(prec, ctx32, ctx64):
    return ctx64 if prec == 8 else ctx32


def rel_l2(a, b, floor=0.0):
    a = np.asarray(a, np.float64)
    b = np.asarray(b, np.float64)
    den = max(np.linalg.norm(b), floor * np.sqrt(b.size), 1e-300)
    return np.linalg.norm(a - b) / den


def pair(prec, ctx32, ctx64, nx, ny, nz, n_tracers=0, **kw):
    ctx = ctx_for(prec, ctx32, ctx64)
    gkw = {k: v for k, v in kw.items() if k in ("halo", "periodic_x", "periodic_y", "dx", "dy",
                                                  "z_top", "z_interfaces", "terrain")}
    grid = G.Grid(ctx, nx, ny, nz, **gkw)
    gs = G.State(grid, n_tracers)
    w = O.World(nx, ny, nz, n_tracers=n_tracers, precision=prec, **gkw)
    return w, gs


def copy_state(w, gs, tracers=0):
    for f in FIELDS:
        gs.set(f, w.get(f))
    for t in range(tracers):
        gs.set(O.TRACER0 + t, w.get(O.TRACER0 + t))


FLOORS = {O.RHO: 1.0, O.RHO_THETA: 300.0, O.MOM_U: 1.0, O.MOM_V: 1.0, O.MOM_W: 1.0}


def compare(w, gs, tol, fields=FIELDS, tracers=0, label=""):
    """Relative L2 with a physical floor per field (rho 1 kg m-3, rho*theta
    300 K kg m-3, momenta 1 kg m-2 s-1, tracers 1e-3 kg m-3), so fields that
    are pure round-off (a state at rest) are judged against a meaningful
    scale rather than against their own noise."""
    worst = {}
    for f in list(fields) + [O.TRACER0 + t for t in range(tracers)]:
        a, b = gs.get(f), w.get(f)
        e = rel_l2(a, b, FLOORS.get(f, 1e-3))
        worst[NAMES.get(f, f"tracer{f - O.TRACER0}")] = e
    bad = {k: v for k, v in worst.items() if not v <= tol}
    assert not bad, f"{label} rel-L2 above {tol}: {bad} (all: {worst})"
    return worst


# ------------------------------------------------------------- bit-exact ---

@pytest.mark.parametrize("px,py,halo", [(True, True, 1), (False, True, 1), (True, False, 2),
                                        (False, False, 1)])
@pytest.mark.parametrize("field", [O.RHO, O.MOM_U, O.MOM_V, O.MOM_W])
def test_halo_fill_bit_exact(ctx64, px, py, halo, field):
    nx, ny, nz = 9, 7, 3
    w, gs = pair(8, None, ctx64, nx, ny, nz, halo=halo, periodic_x=px, periodic_y=py)
    rng = np.random.default_rng(field * 10 + halo)
    st = rng.standard_normal(w.rank_storage(0, field).shape)
    w.set_rank_storage(0, field, st)
    gs.set_storage(field, st)
    w.exchange(field)
    gs.halo_fill(field)
    np.testing.assert_array_equal(gs.storage(field), w.rank_storage(0, field))


@pytest.mark.parametrize("field", [O.MOM_U, O.MOM_V])
def test_interface_sync_bit_exact(ctx32, field):
    w, gs = pair(4, ctx32, None, 8, 6, 2)
    v = np.random.default_rng(5).standard_normal(w.global_shape(field)).astype(np.float32)
    w.set(field, v)
    gs.set(field, v)
    w.sync_interfaces(field)
    gs.sync_interfaces(field)
    np.testing.assert_array_equal(gs.get(field), w.get(field))


@pytest.mark.parametrize("orient,field", [(0, O.RHO), (1, O.MOM_U), (2, O.MOM_V), (3, O.MOM_W)])
@pytest.mark.parametrize("rx,ry,px,py", [(2, 2, True, True), (3, 2, False, True)])
def test_multirank_exchange_bit_exact(ctx32, orient, field, rx, ry, px, py):
    """gwm_halo_exchange_layout on per-rank device arrays reproduces the
    virtual-rank exchange, including absent neighbours and corners."""
    import ctypes
    nx, ny, nz, h = 8, 8, 2, 1
    w = O.World(nx, ny, nz, halo=h, ranks_x=rx, ranks_y=ry, periodic_x=px, periodic_y=py,
                precision=4)
    rng = np.random.default_rng(orient + 7 * rx)
    L = G.lib()
    descs, ptrs, host = [], [], []
    for r in range(w.num_ranks):
        d = w.rank_desc(r)
        descs += [d[k] for k in ("rank", "coord_x", "coord_y", "ranks_x", "ranks_y", "global_nx",
                                 "global_ny", "nz", "halo", "i_begin", "i_end", "j_begin", "j_end")]
        st = rng.standard_normal(w.rank_storage(r, field).shape).astype(np.float32)
        w.set_rank_storage(r, field, st)
        p = ctypes.c_void_p()
        G.check(L.gwm_device_alloc(ctx32.h, st.nbytes, ctypes.byref(p)))
        G.check(L.gwm_memcpy_h2d(ctx32.h, p, st.ctypes.data_as(ctypes.c_void_p), st.nbytes))
        ptrs.append(p.value)
        host.append(st)
    w.exchange(field)
    d13 = np.array(descs, np.int32)
    parr = (ctypes.c_void_p * len(ptrs))(*ptrs)
    G.check(L.gwm_halo_exchange_layout(ctx32.h, len(ptrs), d13.ctypes.data_as(ctypes.c_void_p),
                                       int(px), int(py), orient, parr))
    for r, p in enumerate(ptrs):
        out = np.empty_like(host[r])
        G.check(L.gwm_memcpy_d2h(ctx32.h, out.ctypes.data_as(ctypes.c_void_p), p, out.nbytes))
        G.check(L.gwm_device_free(ctx32.h, p))
        np.testing.assert_array_equal(out, w.rank_storage(r, field))


def test_multirank_known_answers_on_gpu(ctx32):
    # tests/unit/test_halo_exchange.cpp:16-19 on the device
    import ctypes
    w = O.World(8, 8, 1, ranks_x=2, ranks_y=2, precision=4)
    j, i = np.mgrid[0:8, 0:8]
    w.set(O.RHO, (100 * j + i)[None].astype(np.float32))
    L = G.lib()
    descs, ptrs = [], []
    for r in range(4):
        d = w.rank_desc(r)
        descs += [d[k] for k in ("rank", "coord_x", "coord_y", "ranks_x", "ranks_y", "global_nx",
                                 "global_ny", "nz", "halo", "i_begin", "i_end", "j_begin", "j_end")]
        st = w.rank_storage(r, O.RHO)
        p = ctypes.c_void_p()
        G.check(L.gwm_device_alloc(ctx32.h, st.nbytes, ctypes.byref(p)))
        G.check(L.gwm_memcpy_h2d(ctx32.h, p, st.ctypes.data_as(ctypes.c_void_p), st.nbytes))
        ptrs.append(p.value)
    d13 = np.array(descs, np.int32)
    G.check(L.gwm_halo_exchange_layout(ctx32.h, 4, d13.ctypes.data_as(ctypes.c_void_p), 1, 1, 0,
                                       (ctypes.c_void_p * 4)(*ptrs)))
    out = np.empty(w.rank_storage(0, O.RHO).shape, np.float32)
    G.check(L.gwm_memcpy_d2h(ctx32.h, out.ctypes.data_as(ctypes.c_void_p), ptrs[0], out.nbytes))
    for p in ptrs:
        G.check(L.gwm_device_free(ctx32.h, p))
    assert out[0, 1, 0] == 7.0 and out[0, 1, 5] == 4.0
    assert out[0, 0, 1] == 700.0 and out[0, 5, 1] == 400.0


@pytest.mark.parametrize("prec", [4, 8])
@pytest.mark.parametrize("case", ["flat", "mountain", "stretched", "open"])
def test_metrics_bit_exact(ctx32, ctx64, prec, case):
    nx, ny, nz = 21, 13, 12
    kw = dict(z_top=18000.0)
    if case in ("mountain", "open"):
        kw["terrain"] = O_cosine(nx, ny, 1200.0)
    if case == "stretched":
        kw["z_interfaces"] = G.stretched_levels(nz, 100.0, 900.0, 18000.0)
        kw["terrain"] = O_cosine(nx, ny, 800.0)
    if case == "open":
        kw["periodic_x"] = False
        kw["periodic_y"] = False
    w, gs = pair(prec, ctx32, ctx64, nx, ny, nz, **kw)
    for m in range(11):
        np.testing.assert_array_equal(gs.grid.metric(m), w.metric(m), err_msg=f"metric {m}")


def O_cosine(nx, ny, h):
    return G.cosine_mountain(nx, ny, h, hx=0.25, hy=0.3)


@pytest.mark.parametrize("prec", [4, 8])
def test_initial_states_bit_exact(ctx32, ctx64, prec):
    nx, ny, nz = 16, 12, 10
    t = O_cosine(nx, ny, 900.0)
    for init in ("constant", "hydro", "bubble", "cold_bubble", "hydro_bubble", "mountain"):
        w, gs = pair(prec, ctx32, ctx64, nx, ny, nz, terrain=t, z_top=12000.0)
        if init == "constant":
            w.init_constant(1.1, 301.0, 5.0, -2.0, 0.5)
            gs.init_constant(1.1, 301.0, 5.0, -2.0, 0.5)
        elif init == "hydro":
            w.init_hydrostatic_rest(1.22, 300.0)
            gs.init_hydrostatic_rest(1.22, 300.0)
        elif init in ("bubble", "cold_bubble", "hydro_bubble"):
            kw = dict(rho_background=-1.16 if init == "hydro_bubble" else 1.0, theta_background=300.0,
                      center=(0.5, 0.4, 0.3), radius=(0.2, 0.25, 0.2), theta_perturbation=2.5,
                      sign=-1 if init == "cold_bubble" else 1)
            w.init_bubble(**kw)
            gs.init_bubble(**kw)
        else:
            w.init_mountain_wave(1.18, 300.0, 15.0, 2.0)
            gs.init_mountain_wave(1.18, 300.0, 15.0, 2.0)
        for f in FIELDS:
            np.testing.assert_array_equal(gs.get(f), w.get(f), err_msg=f"{init} {NAMES[f]}")


# ------------------------------------------------------------- operators ---

@pytest.mark.parametrize("prec,tol", [(8, 1e-14), (4, 2e-7)])
def test_pressure(ctx32, ctx64, prec, tol):
    w, gs = pair(prec, ctx32, ctx64, 12, 10, 6, periodic_y=False)
    w.init_bubble(1.0, 300.0, center=(0.4, 0.5, 0.5), radius=(0.3, 0.3, 0.3), theta_perturbation=3.0)
    copy_state(w, gs)
    for f in (O.RHO, O.RHO_THETA):
        w.exchange(f)
    w.pressure()
    gs.pressure()
    a, b = gs.storage(O.PRESSURE), w.rank_storage(0, O.PRESSURE)
    assert np.max(np.abs(a - b) / np.abs(b)) <= tol


def bubble_world(w, sign=+1, u=0.0, v=0.0):
    w.init_bubble(1.0, 300.0, u=u, v=v, center=(0.45, 0.55, 0.35), radius=(0.2, 0.25, 0.25),
                  theta_perturbation=3.0, sign=sign)


@pytest.mark.parametrize("prec,tol", [(8, 1e-12), (4, 2e-5)])
@pytest.mark.parametrize("case", ["periodic", "open", "terrain"])
def test_slow_tendencies(ctx32, ctx64, prec, tol, case):
    if prec == 4 and case == "terrain":
        # The terrain pressure gradient is a difference of two large
        # hydrostatic terms; in FP32 one ulp of p (8 mPa) in either library's
        # powf moves it by ~1e-4 relative.
        tol = 3e-4
    nx, ny, nz = 20, 16, 10
    kw = {}
    if case == "open":
        kw = dict(periodic_x=False, periodic_y=False)
    if case == "terrain":
        kw = dict(terrain=O_cosine(nx, ny, 900.0), z_top=12000.0)
    w, gs = pair(prec, ctx32, ctx64, nx, ny, nz, **kw)
    if case == "terrain":
        w.init_mountain_wave(1.18, 300.0, 12.0, -3.0)
    else:
        bubble_world(w, u=7.0, v=-3.0)
    # add vertical motion so every flux branch is exercised
    wf = w.get(O.MOM_W)
    k = np.arange(nz + 1)[:, None, None]
    wf = wf + (0.05 * np.sin(np.pi * k / nz) * np.cos(np.arange(nx)[None, None, :])).astype(wf.dtype)
    w.set(O.MOM_W, wf)
    copy_state(w, gs)
    cfg = O.step_cfg(dt=2.0, fast_substeps=3)
    w.slow_tendencies(cfg)
    gs.slow_tendencies(G.step_config(dt=2.0, fast_substeps=3))
    for f in (O.TEND_RHO, O.TEND_RHO_THETA, O.TEND_U, O.TEND_V, O.TEND_W):
        a, b = gs.get(f), w.get(f)
        e = rel_l2(a, b, 1e-3 * np.abs(b).max() + 1e-30)
        assert e <= tol, (f, e)


@pytest.mark.parametrize("prec,tol", [(8, 1e-12), (4, 2e-5)])
@pytest.mark.parametrize("case", ["pulse", "terrain", "open"])
def test_fast_modes(ctx32, ctx64, prec, tol, case):
    nx, ny, nz = 20, 18, 10
    kw = {}
    if case == "terrain":
        kw = dict(terrain=O_cosine(nx, ny, 900.0), z_top=12000.0)
    if case == "open":
        kw = dict(periodic_x=False)
    w, gs = pair(prec, ctx32, ctx64, nx, ny, nz, **kw)
    if case == "terrain":
        w.init_mountain_wave(1.18, 300.0, 10.0)
    else:
        w.init_constant(1.0, 300.0, 3.0, -2.0)
    rho = w.get(O.RHO)
    rho[nz // 2, ny // 2, nx // 2] += 0.02
    rho[2, 3, 4] -= 0.01
    w.set(O.RHO, rho)
    w.set(O.RHO_THETA, rho * np.asarray(300.0, rho.dtype))
    copy_state(w, gs)
    for _ in range(2):
        w.fast_modes(O.step_cfg(dt=2.0, fast_substeps=4))
        gs.fast_modes(G.step_config(dt=2.0, fast_substeps=4))
    compare(w, gs, tol, label=case)


CASES = {
    "hydrostatic_rest": dict(nx=18, ny=18, nz=12, dx=3000.0, dy=3000.0, z_top=18000.0),
    "warm_bubble": dict(nx=24, ny=20, nz=12),
    "density_current": dict(nx=24, ny=20, nz=12),
    "mountain_wave": dict(nx=32, ny=12, nz=14, dx=1000.0, dy=1000.0, z_top=18000.0, terrain=1200.0),
    "terrain_rest": dict(nx=24, ny=16, nz=12, dx=2000.0, dy=2000.0, z_top=18000.0, terrain=900.0),
    "open_bubble": dict(nx=20, ny=16, nz=10, periodic_x=False, periodic_y=False),
    # Several 64 x 4 column tiles, a ragged last tile in x and a tile count
    # divisible by 8 (the XCD-banded tile order of the column kernel).
    "wide_bubble": dict(nx=130, ny=32, nz=8),
    "wide_mountain": dict(nx=128, ny=16, nz=10, dx=1000.0, dy=1000.0, z_top=15000.0,
                          terrain=800.0),
}


def build_case(name, prec, ctx32, ctx64, n_tracers=0):
    c = dict(CASES[name])
    nx, ny, nz = c.pop("nx"), c.pop("ny"), c.pop("nz")
    if "terrain" in c:
        c["terrain"] = G.cosine_mountain(nx, ny, c["terrain"], hx=0.15, hy=0.35)
    w, gs = pair(prec, ctx32, ctx64, nx, ny, nz, n_tracers=n_tracers, **c)
    if name == "hydrostatic_rest":
        w.init_hydrostatic_rest(1.22, 300.0)
    elif name == "warm_bubble":
        bubble_world(w, +1, u=4.0)
    elif name in ("density_current", "open_bubble"):
        bubble_world(w, -1)
    elif name == "wide_bubble":
        bubble_world(w, +1, u=3.0)
    elif name in ("mountain_wave", "wide_mountain"):
        w.init_mountain_wave(1.18, 300.0, 15.0)
    elif name == "terrain_rest":
        w.init_hydrostatic_rest(1.18, 300.0)
    copy_state(w, gs)
    return w, gs


# FP32: the device and host powf/expf differ by an ulp now and then; three
# steps of the reference scheme (whose perturbations grow) amplify that to a
# few 1e-5 in the momenta.
@pytest.mark.parametrize("prec,tol", [(8, 1e-11), (4, 2e-4)])
@pytest.mark.parametrize("name", list(CASES))
def test_ssprk3_steps(ctx32, ctx64, prec, tol, name):
    w, gs = build_case(name, prec, ctx32, ctx64)
    cfg = dict(dt=2.0, fast_substeps=3)
    for _ in range(3):
        w.ssprk3_step(O.step_cfg(**cfg))
        gs.ssprk3_step(G.step_config(**cfg))
    compare(w, gs, tol, label=name)


def test_fp32_step_against_fp64_oracle(ctx32):
    """The reference's FP32 formulation (full rho*theta and p in FP32) vs the
    FP64 oracle.  One ulp of rho*theta (3e-5 K kg m-3) moves p by ~10 mPa,
    against ~1 Pa horizontal pressure differences, so the momenta carry a
    ~1e-3 relative error after five steps; that is the bound this path meets
    (the north-star 1e-4 needs the perturbation-form storage)."""
    w64, _ = build_case("warm_bubble", 8, ctx32, ctx32)
    w32, gs = build_case("warm_bubble", 4, ctx32, ctx32)
    cfg = dict(dt=2.0, fast_substeps=3)
    for _ in range(5):
        w64.ssprk3_step(O.step_cfg(**cfg))
        gs.ssprk3_step(G.step_config(**cfg))
    compare(w64, gs, 3e-3, label="fp32 vs fp64 oracle")


def test_ssprk3_boundary_strips(ctx32, ctx64):
    w, gs = build_case("open_bubble", 8, ctx32, ctx64)
    w.set_boundary_from_current()
    gs.capture_boundary()
    for _ in range(2):
        w.ssprk3_step(O.step_cfg(dt=2.0, fast_substeps=2), boundary=O.BOUNDARY_STRIPS)
        gs.ssprk3_step(G.step_config(dt=2.0, fast_substeps=2),
                       G.BoundaryConfig(G.BOUNDARY_STRIPS, 0.0, G.BOUNDARY_FN(), None))
    compare(w, gs, 1e-11, label="strips")


def test_ssprk3_boundary_relaxation(ctx32, ctx64):
    w, gs = build_case("open_bubble", 8, ctx32, ctx64)
    w.set_boundary_from_current()
    gs.capture_boundary()
    for _ in range(2):
        w.ssprk3_step(O.step_cfg(dt=2.0, fast_substeps=2), boundary=O.BOUNDARY_RELAX,
                      relax_width=4.0)
        gs.ssprk3_step(G.step_config(dt=2.0, fast_substeps=2),
                       G.BoundaryConfig(G.BOUNDARY_RELAX, 4.0, G.BOUNDARY_FN(), None))
    compare(w, gs, 1e-11, label="relax")


def moist_world(prec, ctx32, ctx64, nx=16, ny=14, nz=12, seed=3, z_interfaces=None):
    """Convection sounding with perturbed moisture.  Uniform 1 km levels by
    default: the reference's explicit acoustic scheme diverges on fine
    (100 m) levels at dt 5 s, so dynamics tests use coarse levels."""
    zi = z_interfaces if z_interfaces is not None else np.linspace(0.0, 12000.0, nz + 1)
    ctx = ctx_for(prec, ctx32, ctx64)
    grid = G.Grid(ctx, nx, ny, nz, dx=1000.0, dy=1000.0, z_interfaces=zi)
    gs = G.State(grid, 3)
    gs.init_convection(1.0e5, seed, 0.5, 1000.0)
    w = O.World(nx, ny, nz, dx=1000.0, dy=1000.0, z_interfaces=zi, n_tracers=3, precision=prec)
    for f in FIELDS:
        w.set(f, gs.get(f))
    qv = gs.get(O.TRACER0)
    rng = np.random.default_rng(seed)
    qv = qv * (1.0 + 0.25 * rng.random(qv.shape)).astype(qv.dtype)  # supersaturate some cells
    qc = (np.abs(rng.standard_normal(qv.shape)) * 2e-4).astype(qv.dtype) * gs.get(O.RHO)
    qr = (np.abs(rng.standard_normal(qv.shape)) * 1e-4).astype(qv.dtype) * gs.get(O.RHO)
    for t, q in enumerate((qv, qc, qr)):
        w.set(O.TRACER0 + t, q)
        gs.set(O.TRACER0 + t, q)
    return w, gs


@pytest.mark.parametrize("prec,tol", [(8, 1e-11), (4, 3e-5)])
def test_tracers_ssprk3(ctx32, ctx64, prec, tol):
    w, gs = moist_world(prec, ctx32, ctx64, z_interfaces=G.stretched_levels(12, 150.0, 900.0, 6000.0))
    u = w.get(O.MOM_U) + np.asarray(8.0, w.dtype)
    w.set(O.MOM_U, u)
    gs.set(O.MOM_U, u)
    for _ in range(2):
        w.tracers_ssprk3(O.step_cfg(dt=5.0))
        gs.tracers_ssprk3(G.step_config(dt=5.0))
    compare(w, gs, tol, fields=(), tracers=3, label="tracers")


@pytest.mark.parametrize("prec,tol", [(8, 1e-12), (4, 1e-5)])
@pytest.mark.parametrize("metric", [True, False])
def test_warm_rain(ctx32, ctx64, prec, tol, metric):
    w, gs = moist_world(prec, ctx32, ctx64, z_interfaces=G.stretched_levels(12, 150.0, 900.0, 6000.0))
    cfg = dict(dt=5.0, rain_terminal_velocity=12.0, sedimentation_layer_depth_m=400.0,
               cloud_autoconversion_rate=1e-3, rain_evaporation_rate=5e-3)
    for _ in range(3):
        w.warm_rain(O.warm_rain_cfg(**cfg), metric_fallout=metric)
        gs.warm_rain(G.warm_rain_config(**cfg), metric_fallout=metric)
    compare(w, gs, tol, fields=(O.RHO_THETA,), tracers=3, label="warm rain")
    a, b = gs.get(O.PRECIP), w.get(O.PRECIP)
    assert rel_l2(a, b, 1e-30) <= tol


@pytest.mark.parametrize("prec,tol", [(8, 1e-11), (4, 2e-4)])
def test_moist_step(ctx32, ctx64, prec, tol):
    """gwm_moist_step == the prepared driver's loop body: dry SSPRK3, tracer
    SSPRK3, warm rain with metric fallout (gwm_prepared_case_driver.cpp:427-463)."""
    w, gs = moist_world(prec, ctx32, ctx64)
    cfg = dict(dt=2.0, fast_substeps=3)
    wr = dict(dt=2.0, rain_terminal_velocity=12.0)
    for _ in range(2):
        w.ssprk3_step(O.step_cfg(**cfg))
        w.tracers_ssprk3(O.step_cfg(**cfg))
        w.warm_rain(O.warm_rain_cfg(**wr), metric_fallout=True)
        gs.moist_step(G.step_config(**cfg), G.warm_rain_config(**wr))
    compare(w, gs, tol, tracers=3, label="moist step")


@pytest.mark.parametrize("prec", [8, 4])
def test_nominal_fallout_leaves_columns_alone_when_nothing_falls(ctx32, ctx64, prec):
    """dt 0 with a terminal velocity and a layer depth: the fallout fraction
    is 0 and the reference's nominal sweep returns before touching the column
    (warm_rain.cu:134-136), so the result equals the call without fallout,
    bit for bit (a sweep that ran would rewrite rho*qr as (rho*qr*dz)/dz)."""
    _, a = moist_world(prec, ctx32, ctx64, seed=4)
    _, b = moist_world(prec, ctx32, ctx64, seed=4)
    base = dict(dt=0.0, cloud_autoconversion_rate=1e-3, rain_evaporation_rate=5e-3)
    a.warm_rain(G.warm_rain_config(rain_terminal_velocity=12.0, sedimentation_layer_depth_m=400.0,
                                   **base), metric_fallout=False)
    b.warm_rain(G.warm_rain_config(rain_terminal_velocity=0.0, **base), metric_fallout=False)
    for f in (O.RHO_THETA, O.TRACER0, O.TRACER0 + 1, O.TRACER0 + 2, O.PRECIP):
        assert np.array_equal(a.get(f), b.get(f)), f


def test_summary_counts_nonfinite_values(ctx32):
    """Sums and extremes cover the finite values; NaN and infinities are
    counted over every prognostic field, and the extremes of a field holding
    one are NaN."""
    _, gs = moist_world(4, ctx32, None)
    s0 = gs.summary()
    assert s0["nonfinite_values"] == 0
    assert all(np.isfinite(v) for v in s0.values())
    w = gs.get(O.MOM_W)
    w[3, 2, 1] = np.nan
    w[5, 1, 1] = np.inf
    gs.set(O.MOM_W, w)
    q = gs.get(O.TRACER0 + 2)
    q[0, 0, 0] = np.nan
    gs.set(O.TRACER0 + 2, q)
    p = gs.get(O.PRECIP)
    p[0, 0, 0] = -np.inf
    gs.set(O.PRECIP, p)
    s = gs.summary()
    assert s["nonfinite_values"] == 4
    assert np.isnan(s["w_min"]) and np.isnan(s["w_max"])
    assert np.isnan(s["qr_min"]) and np.isnan(s["qr_max"])
    for k in ("u_min", "u_max", "rho_min", "theta_max", "qv_max", "total_dry_mass"):
        assert s[k] == s0[k], k
    assert np.isfinite(s["total_vertical_momentum"]) and np.isfinite(s["precip_sum"])


@pytest.mark.parametrize("prec", [4, 8])
def test_budget_sums(ctx32, ctx64, prec):
    w, gs = moist_world(prec, ctx32, ctx64)
    wr = G.warm_rain_config(dt=5.0, rain_terminal_velocity=12.0)
    w.warm_rain(O.warm_rain_cfg(dt=5.0, rain_terminal_velocity=12.0), metric_fallout=True)
    gs.warm_rain(wr, metric_fallout=True)
    for f in FIELDS:
        gs.set(f, w.get(f))
    for t in range(3):
        gs.set(O.TRACER0 + t, w.get(O.TRACER0 + t))
    gs.set(O.PRECIP, w.get(O.PRECIP))
    a, b = gs.summary(), w.summary()
    for k in O.SUMMARY_KEYS:
        assert abs(a[k] - b[k]) <= 1e-12 * max(1.0, abs(b[k])), (k, a[k], b[k])


@pytest.mark.parametrize("prec", [8, 4])
@pytest.mark.parametrize("ny", [16, 20])
def test_level_chunks_do_not_change_results(ctx32, ctx64, prec, ny):
    """The column kernels split columns into level chunks, and the flat fast
    kernel runs tiles of 8 or 4 rows (both autotuned); every chunk count and
    tile height must give bit-identical states, tracers included (ny 20:
    the 8-row tiles end in a partial one, the 4-row tiles do not)."""
    ctx = ctx_for(prec, ctx32, ctx64)
    nx, nz = 130, 12
    zi = np.linspace(0.0, 12000.0, nz + 1)
    grid = G.Grid(ctx, nx, ny, nz, dx=1000.0, dy=1000.0, z_interfaces=zi)
    ref = None
    try:
        for chunks in (1, 2, 3, 4, 6, 8, 16 | 1, 16 | 2, 16 | 3, 16 | 8, 64 | 1, 64 | 16 | 1, 0):
            ctx.set_chunks(chunks)
            gs = G.State(grid, 3)
            gs.init_convection(1.0e5, 5, 0.5, 1000.0)
            qv = gs.get(O.TRACER0)
            gs.set(O.TRACER0 + 1, (0.02 * qv).astype(qv.dtype))
            gs.set(O.TRACER0 + 2, (0.01 * qv).astype(qv.dtype))
            for _ in range(2):
                gs.moist_step(G.step_config(dt=2.0, fast_substeps=3),
                              G.warm_rain_config(dt=2.0, rain_terminal_velocity=12.0))
            out = [gs.get(f) for f in FIELDS + (O.TRACER0, O.TRACER0 + 1, O.TRACER0 + 2)]
            if ref is None:
                ref = out
            else:
                for a, b in zip(out, ref):
                    assert np.array_equal(a, b), f"chunks={chunks}"
    finally:
        ctx.set_chunks(0)
    report = ctx.tuning_report()
    assert any(k.startswith(f"fast_column:130x{ny}x12") for k in report), report
    assert all(v & 15 in (1, 2, 3, 4, 6, 8, 12) and v >> 4 in (0, 1) for v in report.values())


@pytest.mark.parametrize("perturbation", [False, True])
@pytest.mark.parametrize("ty4", [0, 16])
def test_downward_march_does_not_change_results(ctx32, perturbation, ty4):
    """Every other fast substep of a flat whole-column launch marches its
    columns from the top down (launch code bit 6 keeps them all upward);
    each cell's arithmetic is the same either way, so the moist steps give
    bit-identical states, in the full and the perturbation form, on a grid
    whose tiles end in partial ones."""
    nx, ny, nz = 130, 20, 12
    zi = np.linspace(0.0, 12000.0, nz + 1)
    grid = G.Grid(ctx32, nx, ny, nz, dx=1000.0, dy=1000.0, z_interfaces=zi)
    outs = []
    try:
        for code in (1 | ty4, 64 | 1 | ty4):
            ctx32.set_chunks(code)
            gs = G.State(grid, 3, perturbation=perturbation)
            gs.init_convection(1.0e5, 5, 0.5, 1000.0)
            qv = gs.get(O.TRACER0)
            gs.set(O.TRACER0 + 1, (0.02 * qv).astype(qv.dtype))
            for _ in range(2):
                gs.moist_step(G.step_config(dt=2.0, fast_substeps=4),
                              G.warm_rain_config(dt=2.0, rain_terminal_velocity=12.0))
            assert gs.summary()["nonfinite_values"] == 0
            outs.append([gs.get_f64(f) for f in FIELDS + (O.TRACER0, O.TRACER0 + 1,
                                                          O.TRACER0 + 2, O.PRECIP)])
    finally:
        ctx32.set_chunks(0)
    for a, b in zip(*outs):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("prec", [8, 4])
def test_column_reference_tile_heights_do_not_change_results(ctx32, ctx64, prec):
    """On terrain the fast kernel's tile height (8 or 4 rows) is autotuned
    like its level chunks (the column reference, a recurrence from the ground,
    has a kernel of its own); both heights give bit-identical states on an
    open-x ridge grid whose 8-row tiles end in a partial one, here in whole
    columns."""
    ctx = ctx_for(prec, ctx32, ctx64)
    nx, ny, nz, dx = 96, 20, 16, 2000.0
    zi = G.stretched_levels(nz, 50.0, 600.0, 8000.0)
    ter = G.agnesi_ridge(nx, ny, dx, 0.5 * nx * dx, 10000.0, 400.0)
    grid = G.Grid(ctx, nx, ny, nz, dx=dx, dy=dx, z_interfaces=zi, terrain=ter,
                  periodic_x=False)
    cfg = G.step_config(dt=0.25, fast_substeps=4)
    bc = G.BoundaryConfig(G.BOUNDARY_RELAX, 4.0, G.BOUNDARY_FN(), None)
    out = []
    try:
        for code in (1, 16 | 1):
            ctx.set_chunks(code)
            st = G.State(grid, 0)
            st.init_constant_n(theta_surface=288.0, brunt_vaisala=0.01, p_surface=1.0e5, u=10.0)
            st.capture_boundary()
            for _ in range(3):
                st.ssprk3_step(cfg, bc)
            assert st.summary()["nonfinite_values"] == 0
            out.append([st.get(f) for f in FIELDS])
    finally:
        ctx.set_chunks(0)
    assert np.abs(out[0][O.MOM_W]).max() > 0.0
    for a, b, f in zip(out[0], out[1], FIELDS):
        assert np.array_equal(a, b), f


def _moist_pair(prec, ctx, seed=21, shape=(40, 24, 12)):
    nx, ny, nz = shape
    zi = np.linspace(0.0, 12000.0, nz + 1)
    grid = G.Grid(ctx, nx, ny, nz, dx=1000.0, dy=1000.0, z_interfaces=zi)
    out = []
    for _ in range(2):
        gs = G.State(grid, 3)
        gs.init_convection(1.0e5, seed, 0.5, 1000.0)
        qv = gs.get(O.TRACER0)
        gs.set(O.TRACER0 + 1, (0.03 * qv).astype(qv.dtype))
        gs.set(O.TRACER0 + 2, (0.02 * qv).astype(qv.dtype))
        out.append(gs)
    return grid, out


def assert_all_finite(*states):
    for st in states:
        s = st.summary()
        assert s["nonfinite_values"] == 0, s
        for f in FIELDS + (O.TRACER0, O.TRACER0 + 1, O.TRACER0 + 2, O.PRECIP):
            assert np.all(np.isfinite(st.get(f))), f


# dt 1 s: this moist case stays bounded (|w| < 0.3 m/s over ten steps in the
# FP32 oracle); at dt 2 s the reference scheme overflows by the seventh step,
# and equality of overflowed states would show nothing.
@pytest.mark.parametrize("prec", [8, 4])
def test_graph_replayed_steps_equal_eager_steps(ctx32, ctx64, prec):
    ctx = ctx_for(prec, ctx32, ctx64)
    grid, (a, b) = _moist_pair(prec, ctx)
    cfg = G.step_config(dt=1.0, fast_substeps=3)
    wr = G.warm_rain_config(dt=1.0, rain_terminal_velocity=12.0)
    for _ in range(7):
        a.moist_step(cfg, wr)
    b.moist_steps_graph(cfg, wr, 3)   # eager + one graph replay
    b.moist_steps_graph(cfg, wr, 4)   # replays
    assert_all_finite(a, b)
    assert a.summary()["w_max"] > 1e-3  # the state moved
    for f in FIELDS + (O.TRACER0, O.TRACER0 + 1, O.TRACER0 + 2, O.PRECIP):
        x, y = a.get(f), b.get(f)
        assert np.array_equal(x, y), (f, int((x != y).sum()))


@pytest.mark.parametrize("streams", [False, True])
def test_ensemble_steps_equal_member_steps(streams):
    """Members of different sizes advanced together -- one launch per kernel
    of the step over all members (batched), or one context (stream) each
    from their graphs -- equal the same members stepped one by one."""
    shapes = [(40, 24, 12), (64, 32, 10), (24, 40, 14)]
    cfg = G.step_config(dt=1.0, fast_substeps=4)
    wr = G.warm_rain_config(dt=1.0, rain_terminal_velocity=12.0)
    ctxs = [G.Context(0, G.F32) for _ in shapes]
    members, refs, keep = [], [], []
    for i, (ctx, shape) in enumerate(zip(ctxs, shapes)):
        grid, (a, b) = _moist_pair(4, ctx, seed=30 + i, shape=shape)
        keep.append(grid)
        members.append(a)
        refs.append(b)
    G.ensemble_steps(members, cfg, wr, 5, streams=streams)
    # a second call reuses the members' warm-up and records again
    G.ensemble_steps(members, cfg, wr, 4, streams=streams)
    for r in refs:
        for _ in range(9):
            r.moist_step(cfg, wr)
    assert_all_finite(*members, *refs)
    for m, r in zip(members, refs):
        for f in FIELDS + (O.TRACER0, O.TRACER0 + 1, O.TRACER0 + 2, O.PRECIP):
            assert np.array_equal(m.get(f), r.get(f)), f
    del members, refs, keep
    for c in ctxs:
        c.close()


@pytest.mark.parametrize("prec", [8, 4])
def test_batched_ensemble_on_one_context_and_mixed_members(ctx32, ctx64, prec):
    """Batched members may share one context; FP32 members in the
    perturbation form and with the surrogate (the same network per member)
    batch as well.  A mixed-precision ensemble cannot batch and runs its
    members on their own streams.  Every member equals its own steps."""
    ctx = ctx_for(prec, ctx32, ctx64)
    cfg = G.step_config(dt=1.0, fast_substeps=3)
    wr = G.warm_rain_config(dt=1.0, rain_terminal_velocity=12.0)
    shapes = [(40, 24, 12), (24, 16, 12), (72, 40, 12)]
    keep, members, refs = [], [], []
    for i, shape in enumerate(shapes):
        grid, (a, b) = _moist_pair(prec, ctx, seed=40 + i, shape=shape)
        keep.append(grid)
        members.append(a)
        refs.append(b)
    G.ensemble_steps(members, cfg, wr, 6)
    for r in refs:
        for _ in range(6):
            r.moist_step(cfg, wr)
    assert_all_finite(*members, *refs)
    for m, r in zip(members, refs):
        for f in FIELDS + (O.TRACER0, O.TRACER0 + 2, O.PRECIP):
            assert np.array_equal(m.get(f), r.get(f)), f
    if prec == 4:
        import gwm_amd.surrogate as SG
        import surrogate_oracle as SO
        sur = G.Surrogate(ctx, seed=3)
        big = 1e30
        sur.set_norm(x_mean=np.zeros(7), x_std=np.ones(7) * 1e3, y_mean=np.zeros(4),
                     y_std=np.array([1e-6, 1e-6, 1e-6, 1e-2]), box_lo=-big * np.ones(7),
                     box_hi=big * np.ones(7))
        sur.set_params((SO.init_xavier(2) * 0.5).astype(np.float32))
        pm, pr = [], []
        for i, shape in enumerate(shapes[:2]):
            zi = np.linspace(0.0, 12000.0, shape[2] + 1)
            grid = G.Grid(ctx, *shape, dx=1000.0, dy=1000.0, z_interfaces=zi)
            keep.append(grid)
            for lst in (pm, pr):
                st = G.State(grid, 3, perturbation=True)
                st.init_convection(1.0e5, 50 + i, 0.5, 1000.0)
                qv = st.get(O.TRACER0)
                st.set(O.TRACER0 + 1, (0.03 * qv).astype(qv.dtype))
                lst.append(st)
        G.ensemble_steps(pm, cfg, wr, 4, surrogates=[sur, sur])
        for r in pr:
            for _ in range(4):
                r.moist_step_surrogate(cfg, wr, sur)
        assert_all_finite(*pm, *pr)
        for m, r in zip(pm, pr):
            for f in FIELDS + (O.TRACER0, O.TRACER0 + 1, O.TRACER0 + 2, O.PRECIP):
                assert np.array_equal(m.get(f), r.get(f)), f
        del SG
    # mixed precision: streams, one context each
    other = ctx64 if prec == 4 else ctx32
    grid2, (c2, d2) = _moist_pair(8 if prec == 4 else 4, other, seed=60, shape=(32, 24, 12))
    keep.append(grid2)
    a0 = G.State(keep[0], 3)
    a0.copy_from(refs[0])
    G.ensemble_steps([a0, c2], cfg, wr, 2)
    for _ in range(2):
        refs[0].moist_step(cfg, wr)
        d2.moist_step(cfg, wr)
    assert_all_finite(a0, c2)
    for x, y in ((a0, refs[0]), (c2, d2)):
        for f in FIELDS + (O.TRACER0, O.PRECIP):
            assert np.array_equal(x.get(f), y.get(f)), f


@pytest.mark.parametrize("prec", [4, 8])
def test_theta_ref_from_last_substep_matches_separate_pass(ctx32, ctx64, prec):
    """Without boundaries the last fast substep of SSPRK3 stages 1-2 emits the
    next stage's theta_ref level sums; with a boundary callback (one that
    changes nothing) a separate pass over the state computes them.  Same
    per-cell theta summed in another order, so the states agree to the
    working precision's rounding; a wrong fused sum (another quantity, level or state) would move
    theta_ref by O(1) K and the buoyancy with it."""
    nx, ny, nz = 96, 64, 24
    zi = np.linspace(0.0, 12000.0, nz + 1)
    grid = G.Grid(ctx_for(prec, ctx32, ctx64), nx, ny, nz, dx=1000.0, dy=1000.0,
                  z_interfaces=zi)
    a, b = G.State(grid, 3), G.State(grid, 3)
    for s in (a, b):
        s.init_convection(1.0e5, 7, 0.5, 1000.0)
    times = []

    def noop(_state, t, _user):
        times.append(t)
        return 0

    cb = G.BOUNDARY_FN(noop)
    bc = G.BoundaryConfig(G.BOUNDARY_NONE, 0.0, cb, None)
    cfg = G.step_config(dt=2.0, fast_substeps=3)
    for _ in range(3):
        a.ssprk3_step(cfg)
        b.ssprk3_step(cfg, bc)
    assert times == [0.0, 2.0, 1.0] * 3  # entry state, after stages 1 and 2
    for f in FIELDS:
        x, y = a.get(f).astype(np.float64), b.get(f).astype(np.float64)
        scale = np.max(np.abs(y))
        assert np.all(np.isfinite(x)), f
        tol = 1e-5 if prec == 4 else 1e-11
        assert np.max(np.abs(x - y)) <= tol * scale, (f, np.max(np.abs(x - y)) / scale)
