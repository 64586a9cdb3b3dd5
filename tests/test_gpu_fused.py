"""The fused line operators of the constant-property sub-step against the
oracle, at the line lengths where their chunks go wrong first: lines of one
chunk, of 17-row chunks, of a short last chunk, of few lines per wave, odd
lengths (no 16-byte accesses) and lengths below the fused form's smallest
(single operators), with and without walls, in every accuracy."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LX, LZ = 4 * np.pi, 4 * np.pi / 3
TOL = 1e-12  # relative to each field's largest value, as the step parity tests


def rel(a, b):
    return float(np.abs(a - b).max() / np.abs(b).max())


# (nx, ny, nz): chunks of ceil(n / P) rows: 16, 17, 18 (2 x 9), 20 (2 x 10), 32, 33 (17 + 16), 34 (2 x 17),
# 45 (3 x 15), 48, 50 (3 x 17 - 1), 64, 65, 80, 90, 100 (6 x 17 - 2), 8 and 9 (too short)
GRIDS = [(16, 16, 16), (18, 17, 18), (20, 15, 10), (32, 32, 27), (36, 33, 20), (54, 34, 45), (50, 49, 25), (64, 64, 12),
         (90, 19, 30), (100, 50, 50), (24, 64, 75), (16, 12, 9), (10, 65, 8), (270, 16, 16), (16, 20, 288)]


@pytest.mark.parametrize("nc", GRIDS)
def test_fused_substeps_vs_oracle(po, nc):
    from chapsim2_amd.domain import Domain
    from chapsim2_amd.initial import channel_fields

    cfg = dict(istret=2, rstret=0.075, dt=5e-4, ren=2800.0, idriven=1)
    f = channel_fields(nc, LX, -1.0, 1.0, LZ, 2, 0.075, noise=0.1, seed=3)
    dm = Domain(nc, LX, -1.0, 1.0, LZ, **cfg)
    of = po.Flow(list(nc), LX, -1.0, 1.0, LZ, wall_y=True, iacc=4, poisson=2, **cfg)
    try:
        for o in (dm, of):
            o.set_state(*f)
            o.update_re(0)
        # right-hand sides (not yet applied), then two sub-steps that use rhs0
        for g, r in zip(dm.momentum_rhs(1), of.momentum_rhs(1)):
            assert rel(g, r) < TOL
        for isub in (1, 2):
            dm.substep(isub)
            of.substep(isub)
        for name, g, r in zip(("qx", "qy", "qz"), dm.get_state(), of.get_state()):
            assert rel(g, r) < TOL, name
    finally:
        dm.close()


@pytest.mark.parametrize("iacc", [1, 2, 3, 4])
def test_fused_accuracies_and_moving_walls_vs_oracle(po, iacc):
    from chapsim2_amd.domain import Domain
    from chapsim2_amd.initial import channel_fields

    nc = (36, 25, 20)
    cfg = dict(istret=2, rstret=0.075, dt=5e-4, ren=2800.0, idriven=1, uwall=((0.1, 0.0, -0.05), (-0.2, 0.0, 0.1)))
    f = channel_fields(nc, LX, -1.0, 1.0, LZ, 2, 0.075, noise=0.1, seed=5)
    dm = Domain(nc, LX, -1.0, 1.0, LZ, iacc=iacc, **cfg)
    of = po.Flow(list(nc), LX, -1.0, 1.0, LZ, wall_y=True, iacc=iacc, poisson=2, **cfg)
    try:
        for o in (dm, of):
            o.set_state(*f)
            o.update_re(0)
        for g, r in zip(dm.momentum_rhs(0), of.momentum_rhs(0)):
            assert rel(g, r) < TOL
        dm.substep(1)
        of.substep(1)
        for name, g, r in zip(("qx", "qy", "qz"), dm.get_state(), of.get_state()):
            assert rel(g, r) < TOL, name
    finally:
        dm.close()


@pytest.mark.parametrize("nc", [(16, 16, 16), (20, 18, 30), (32, 27, 12), (64, 48, 10)])
def test_fused_periodic_box_vs_oracle(po, nc):
    from chapsim2_amd.domain import FFT_2DECOMP_3DFFT, Domain
    from chapsim2_amd.initial import tgv_fields

    p2 = 2 * np.pi
    cfg = dict(dt=1e-3, ren=1600.0)
    f = tgv_fields(nc, p2, 0.0, p2, p2)
    rng = np.random.default_rng(1)
    f = [np.asfortranarray(a + 0.05 * rng.uniform(-1, 1, a.shape)) for a in f]
    dm = Domain(nc, p2, 0.0, p2, p2, periodic_y=True, poisson=FFT_2DECOMP_3DFFT, **cfg)
    of = po.Flow(list(nc), p2, 0.0, p2, p2, wall_y=False, iacc=4, poisson=3, **cfg)
    try:
        for o in (dm, of):
            o.set_state(*f)
            o.update_re(0)
        for isub in (1, 2, 3):
            dm.substep(isub)
            of.substep(isub)
        for name, g, r in zip(("qx", "qy", "qz"), dm.get_state(), of.get_state()):
            assert rel(g, r) < TOL, name
    finally:
        dm.close()


def test_fused_mixed_form_ragged_grid(po):
    """The FP32 right-hand side on a grid of short last chunks: velocities within the mixed form's 1e-6."""
    from chapsim2_amd.domain import PREC_MIXED, PROJ_EXACT, Domain
    from chapsim2_amd.initial import channel_fields

    nc = (90, 49, 45)
    cfg = dict(istret=2, rstret=0.075, dt=5e-4, ren=2800.0, idriven=1)
    f = channel_fields(nc, LX, -1.0, 1.0, LZ, 2, 0.075, noise=0.1, seed=9)
    dm = Domain(nc, LX, -1.0, 1.0, LZ, projection=PROJ_EXACT, precision=PREC_MIXED, **cfg)
    of = po.Flow(list(nc), LX, -1.0, 1.0, LZ, wall_y=True, iacc=4, poisson=2, projection=1, **cfg)
    try:
        for o in (dm, of):
            o.set_state(*f)
            o.update_re(0)
        dm.run(0, 2)
        of.step(1)
        of.step(2)
        for name, g, r in zip(("qx", "qy", "qz"), dm.get_state(), of.get_state()):
            assert rel(g, r) < 1e-6, name
        assert float(dm.mass_check().max()) < 1e-11
    finally:
        dm.close()
