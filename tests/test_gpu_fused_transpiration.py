"""Walls with a wall-normal velocity on the fused operators: the -v_w^2 term of the y-normal flux at the walls, the
interpolated v next to them and the wall rows that the last y operator and the correction write, against the oracle in
every accuracy.  The walls also slide, each its own way."""
import numpy as np
import pytest

from test_gpu_fused_pressure import TOL, _domain_kw, check

pytestmark = pytest.mark.gpu

LX, LZ = 4 * np.pi, 4 * np.pi / 3
NC = (36, 25, 20)


def _setup(po, iacc, v, mixed=False):
    from chapsim2_amd.domain import Domain
    from chapsim2_amd.initial import channel_fields

    cfg = dict(istret=2, rstret=0.075, dt=5e-4, ren=2800.0, idriven=1, iacc=iacc,
               uwall=((0.1, v[0], -0.05), (-0.2, v[1], 0.1)))
    fields = channel_fields(NC, LX, -1.0, 1.0, LZ, 2, 0.075, noise=0.1, seed=8)
    # the wall-normal velocity runs from one wall's value to the other's
    y = np.linspace(0.0, 1.0, NC[1] + 1)[None, :, None]
    fields[1] = np.asfortranarray(fields[1] + v[0] + (v[1] - v[0]) * y)

    def make():
        of = po.Flow(list(NC), LX, -1.0, 1.0, LZ, wall_y=True, poisson=2, **cfg)
        of.update_re(0)
        return of

    dm, of = Domain(NC, LX, -1.0, 1.0, LZ, **cfg, **_domain_kw(mixed)), make()
    for o in (dm, of):
        o.set_state(*fields)
        o.update_re(0)
    return dm, of, fields, make


# (walls of different wall-normal velocity change the channel's volume: the right-hand side alone)
@pytest.mark.parametrize("v", [(0.07, 0.07), (0.07, -0.04)])
@pytest.mark.parametrize("iacc", [1, 2, 3, 4])
def test_momentum_rhs(po, iacc, v):
    dm, of, _, _ = _setup(po, iacc, v)
    try:
        for isub in (0, 1):
            for name, g, r in zip(("mx", "my", "mz"), dm.momentum_rhs(isub), of.momentum_rhs(isub)):
                err = float(np.abs(g - r).max() / np.abs(r).max())
                assert err < TOL, (isub, name, err)
    finally:
        dm.close()


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("iacc", [1, 2, 3, 4])
def test_substeps(po, iacc, mixed):
    dm, of, fields, make = _setup(po, iacc, (0.07, 0.07), mixed)
    try:
        for o in (dm, of):
            for isub in (1, 2):
                o.substep(isub)
        got = dm.get_state()
        assert np.all(got[1][:, [0, -1], :] == 0.07)
        check(f"transpiration iacc {iacc} mixed {mixed}:", got, of.get_state(), fields, make, (1, 2), mixed)
    finally:
        dm.close()
