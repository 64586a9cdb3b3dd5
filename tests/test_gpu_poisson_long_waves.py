"""TRID0's rule for a singular last pivot (at most 1e-10: last unknown 0) holds for every mode of the FISHPACK solve, not
only the mean one: on a domain so long in x and z that all modes meet it, and on one where none but the mean does."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# last pivots grow with the mode's eigenvalue, at least (2 pi / length)^2: 4e-14 to 5e-12 at 1e8, from 2e-4 on at 2e3
@pytest.mark.parametrize("length", [1e8, 2e3])
@pytest.mark.parametrize("ny", [16, 33])
def test_long_domain_vs_oracle(po, length, ny):
    from chapsim2_amd.domain import Domain
    from chapsim2_amd.poisson import solve_fft_poisson

    nc = (16, ny, 12)
    cfg = dict(istret=2, rstret=0.075)
    dm = Domain(nc, length, -1.0, 1.0, length, **cfg)
    of = po.Flow(list(nc), length, -1.0, 1.0, length, wall_y=True, iacc=4, poisson=2, **cfg)
    try:
        # per mode a right-hand side the singular rows admit, as the divergence's are up to rounding
        dom = po.Dom(list(nc), [1, 0, 1], length, -1.0, 1.0, length, 2, 0.075)
        w = 1.0 / np.array(dom.ymc)
        rhs = np.random.default_rng(ny).uniform(-1, 1, nc)
        rhs = np.asfortranarray(rhs - ((rhs * w[None, :, None]).sum(axis=1) / w.sum())[:, None, :])
        ref = np.asarray(of.poisson(rhs.copy(order="F")))
        got = solve_fft_poisson(rhs.copy(order="F"), dm)
        err = float(np.abs(got - ref).max() / np.abs(ref).max())
        print(f"long domain {length:g} ny {ny}: rel {err:.2e}, max|phi| {np.abs(ref).max():.2e}", flush=True)
        # a mode's sum over its line is rounding, ny eps, which the smallest pivot divides: 33 * 2.2e-16 / 2e-4 = 4e-11
        assert err < 1e-9
    finally:
        dm.close()
