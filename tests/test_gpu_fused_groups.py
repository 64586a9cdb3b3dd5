"""y and z lines of different chunk counts in one launch (short and long chunks, more of them in y and in z), with the
right-hand side in FP64 and in FP32, against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LX, LZ = 4 * np.pi, 4 * np.pi / 3


# y 3 chunks (of 9) to z 2, 2 to 6, 16 to 1, 6 to 8; 16- and 17-row chunks of 2^19 to 2^20 cells: 8 to 4, 3 to 13
@pytest.mark.parametrize("nc", [(32, 24, 16), (24, 16, 48), (16, 128, 12), (30, 49, 60), (96, 128, 64), (60, 49, 200)])
@pytest.mark.parametrize("mixed", [False, True])
def test_groups_vs_oracle(po, nc, mixed):
    from chapsim2_amd.domain import PREC_MIXED, Domain
    from chapsim2_amd.initial import channel_fields

    print(f"group {nc} mixed {mixed}", flush=True)
    cfg = dict(istret=2, rstret=0.075, dt=5e-4, ren=2800.0, idriven=1)
    f = channel_fields(nc, LX, -1.0, 1.0, LZ, 2, 0.075, noise=0.1, seed=6)
    dm = Domain(nc, LX, -1.0, 1.0, LZ, **cfg, **(dict(precision=PREC_MIXED) if mixed else {}))
    of = po.Flow(list(nc), LX, -1.0, 1.0, LZ, wall_y=True, iacc=4, poisson=2, **cfg)
    try:
        for o in (dm, of):
            o.set_state(*f)
            o.update_re(0)
        for isub in (1, 2):
            dm.substep(isub)
            of.substep(isub)
        for name, g, r, q0 in zip(("qx", "qy", "qz"), dm.get_state(), of.get_state(), f):
            # FP64: as the step parity tests; FP32: the change of the step is a sum of some ten terms of a few
            # roundings each, cancelling by up to ten
            step = float(np.abs(r - q0).max())
            tol = 100 * 2.0 ** -24 * step if mixed else 1e-12 * float(np.abs(r).max())
            assert float(np.abs(g - r).max()) < tol, (name, step)
    finally:
        dm.close()
