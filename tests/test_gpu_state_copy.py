"""State copies in one launch: whole storage (halos too) of every field, for
sizes below, at and across the 4096-word chunks and words past a chunk, with
no, some and the most tracers, full and perturbation form; the source stays."""
import numpy as np
import pytest

import gwm_amd as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nz,ntr,prec,pert", [
    (1, 1, 1, 0, G.F32, False), (62, 62, 1, 3, G.F32, False), (61, 63, 3, 8, G.F64, False),
    (30, 14, 8, 3, G.F32, True), (127, 33, 40, 1, G.F32, False), (254, 254, 33, 3, G.F32, False)])
def test_copy_is_whole(nx, ny, nz, ntr, prec, pert):
    ctx = G.Context(0, prec)
    grid = G.Grid(ctx, nx, ny, nz)
    a, b = (G.State(grid, ntr, perturbation=pert) for _ in range(2))
    rng = np.random.default_rng(nx)
    fields = list(range(5)) + [16 + t for t in range(ntr)]
    for f in fields:
        a.set_storage(f, rng.random(a.storage_shape(f)).astype(ctx.dtype) + 1)
    a.set(G.PRECIP, rng.random((ny, nx)).astype(ctx.dtype))
    before = {f: a.storage(f) for f in fields}
    b.copy_from(a)
    for f in fields:
        np.testing.assert_array_equal(a.storage(f), before[f], err_msg=f"source {f}")
        np.testing.assert_array_equal(b.storage(f), before[f], err_msg=f"copy {f}")
    np.testing.assert_array_equal(b.get(G.PRECIP), a.get(G.PRECIP))
