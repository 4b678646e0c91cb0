"""Level means summed by the substep and the slow stage themselves on small
grids against the launch that larger and batched ones use: an ensemble step
(always the launch) gives the bits of single steps.  One, two and ragged lanes
of partials (rows x 64-column segments: 3, 64, 65, 127, 128; 129 takes the
launch), in both precisions and the perturbation form, with an odd and an even
number of substeps (the partials' two halves)."""
import numpy as np
import pytest

import gwm_amd as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,prec,pert,ns", [
    (20, 3, G.F32, False, 1), (64, 64, G.F32, True, 2), (63, 65, G.F64, False, 3),
    (30, 127, G.F32, False, 4), (65, 64, G.F64, False, 2), (17, 129, G.F32, True, 3)])
def test_single_and_batched_steps_agree(nx, ny, prec, pert, ns):
    ctx = G.Context(0, prec)
    grid = G.Grid(ctx, nx, ny, 10, z_interfaces=np.linspace(0.0, 9000.0, 11))
    a, b = (G.State(grid, 3, perturbation=pert) for _ in range(2))
    a.init_convection(1.0e5, 7, 0.5, 1000.0)
    b.copy_from(a)
    cfg, wr = G.step_config(0.5, ns), G.warm_rain_config(0.5, rain_terminal_velocity=12.0)
    for _ in range(3):
        a.moist_step(cfg, wr)
    G.ensemble_steps([b], cfg, wr, 3)
    for f in (0, 1, 2, 3, 4, 16, 17, 18, G.PRECIP):
        np.testing.assert_array_equal(a.get(f), b.get(f), err_msg=f"field {f}")
