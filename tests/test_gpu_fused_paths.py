"""Which operators a sub-step runs: the fused ones wherever the lines have them, in the chunk form that every direction
has, and one operator per launch only where listed; and the sub-steps of long thin grids against the oracle."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_fused_pressure import CFG, LX, LZ, TOL, _domain_kw, check

pytestmark = pytest.mark.gpu


def path(dm):
    from chapsim2_amd import _lib

    out = (C.c_int * 5)()
    _lib.check(dm.lib.chs_inspect_substep(dm.h, out))
    return tuple(out)


# grid: short chunks; chunks along x, y (nodes) and z.  x lines take chunks of 8 (16) rows, the last one shorter; the
# others too when they are a multiple, else the fewest of at most 9 (17).  A line's chunks must be decoupled beyond the
# ends that its coupling reads, rows of the type's precision apart: a last chunk of a few rows brings them too close
FUSED = {
    (16, 16, 16): (1, 2, 2, 2), (18, 17, 18): (1, 3, 2, 2), (20, 15, 10): (1, 3, 2, 2), (32, 32, 27): (1, 4, 4, 3),
    (36, 33, 20): (1, 5, 4, 3), (54, 34, 45): (1, 7, 4, 5), (50, 49, 25): (1, 7, 6, 3), (64, 64, 12): (1, 8, 8, 2),
    (90, 19, 30): (0, 6, 2, 2), (24, 64, 75): (1, 3, 8, 9), (32, 24, 16): (1, 4, 3, 2),
    (60, 49, 200): (0, 4, 3, 12), (96, 128, 64): (0, 6, 8, 4),
    # the most chunks of the short form; beyond it along x, y or z, on grids of few cells: the long form for all
    (256, 16, 16): (1, 32, 2, 2), (16, 20, 288): (1, 2, 3, 32), (16, 287, 20): (1, 2, 32, 3),
    (270, 16, 16): (0, 17, 1, 1), (288, 32, 32): (0, 18, 2, 2), (512, 24, 32): (0, 32, 2, 2), (24, 300, 18): (0, 2, 18, 2),
    (16, 20, 300): (0, 1, 2, 18), (16, 16, 540): (0, 1, 1, 32),
    # a line of more than 256 points on a grid of more than 2^19 cells
    (288, 48, 48): (0, 18, 3, 3), (64, 48, 288): (0, 4, 3, 18),
}
# fewer ends in FP32: there these have the long chunks only
MIXED = {(54, 34, 45): (0, 4, 3, 3), (50, 49, 25): (0, 4, 3, 2), (24, 64, 75): (0, 2, 4, 5)}
# z lines below ten points; x and z lines beyond 32 chunks of 16 and 17; last chunks of 4 and 3 rows on lines of many
SINGLE = [(16, 12, 9), (10, 65, 8), (540, 16, 16), (16, 16, 576), (100, 50, 50), (180, 16, 16), (16, 16, 360)]


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("nc", list(FUSED) + SINGLE)
def test_path(nc, mixed):
    from chapsim2_amd.domain import Domain

    dm = Domain(nc, LX, -1.0, 1.0, LZ, **CFG, **_domain_kw(mixed))
    try:
        want = (1,) + (mixed and MIXED.get(nc) or FUSED[nc]) if nc in FUSED else (0,) * 5
        assert path(dm) == want
    finally:
        dm.close()


@pytest.mark.parametrize("iacc", [1, 2, 3, 4])
def test_path_accuracies_and_periodic_box(iacc):
    from chapsim2_amd.domain import FFT_2DECOMP_3DFFT, Domain

    dm = Domain((36, 25, 20), LX, -1.0, 1.0, LZ, iacc=iacc, **CFG)
    try:
        assert path(dm)[:2] == (1, 1)
    finally:
        dm.close()
    dm = Domain((32, 27, 12), LX, 0.0, LX, LX, periodic_y=True, poisson=FFT_2DECOMP_3DFFT, iacc=iacc, dt=1e-3, ren=1600.0)
    try:
        assert path(dm)[:2] == (1, 1)
    finally:
        dm.close()


@pytest.mark.parametrize("nc", [(288, 32, 32), (512, 24, 32), (16, 20, 288), (16, 16, 540), (288, 48, 48), (64, 48, 288)])
@pytest.mark.parametrize("mixed", [False, True])
def test_long_lines_vs_oracle(po, nc, mixed):
    from chapsim2_amd.domain import Domain
    from chapsim2_amd.initial import channel_fields

    print(f"long lines {nc} mixed {mixed}", flush=True)

    def make():
        of = po.Flow(list(nc), LX, -1.0, 1.0, LZ, wall_y=True, iacc=4, poisson=2, **CFG)
        of.update_re(0)
        return of

    fields = channel_fields(nc, LX, -1.0, 1.0, LZ, 2, 0.075, noise=0.1, seed=17)
    dm, of = Domain(nc, LX, -1.0, 1.0, LZ, **CFG, **_domain_kw(mixed)), make()
    try:
        for o in (dm, of):
            o.set_state(*fields)
            o.update_re(0)
            for isub in (1, 2):
                o.substep(isub)
        check(f"long lines {nc} mixed {mixed}:", dm.get_state(), of.get_state(), fields, make, (1, 2), mixed)
    finally:
        dm.close()


@pytest.mark.parametrize("nc", [(16, 287, 20), (24, 300, 18), (16, 512, 16)])
def test_long_y_lines_vs_oracle(po, nc):
    """Lines between the walls of the most short chunks and of the long form: the right-hand side (walls this finely
    resolved leave the projection's pressure ill-conditioned) and, by the divergence, the y derivative of the sum."""
    from chapsim2_amd.domain import Domain
    from chapsim2_amd.initial import channel_fields

    print(f"long y lines {nc}", flush=True)
    fields = channel_fields(nc, LX, -1.0, 1.0, LZ, 2, 0.075, noise=0.1, seed=18)
    dm = Domain(nc, LX, -1.0, 1.0, LZ, **CFG)
    of = po.Flow(list(nc), LX, -1.0, 1.0, LZ, wall_y=True, iacc=4, poisson=2, **CFG)
    try:
        assert path(dm)[0] == 1
        for o in (dm, of):
            o.set_state(*fields)
            o.update_re(0)
        for g, r in list(zip(dm.momentum_rhs(1), of.momentum_rhs(1))) + [(dm.divergence(), of.divergence())]:
            assert float(np.abs(g - r).max() / np.abs(r).max()) < TOL
    finally:
        dm.close()
