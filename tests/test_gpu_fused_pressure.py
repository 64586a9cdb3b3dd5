"""The pressure after sub-steps on the fused operators (p += phi and its FP32 rounding are done in the x correction), and
with it the velocity, against the oracle: ragged and odd grids, whose last waves and chunks are partial, channel, periodic
box and heated channel, FP64 and mixed."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LX, LZ = 4 * np.pi, 4 * np.pi / 3
CFG = dict(istret=2, rstret=0.075, dt=5e-4, ren=2800.0, idriven=1)
TOL = 1e-12  # of the field's largest value, as the step parity tests
ALPHA = (1.0, 8.0 / 15.0, 2.0 / 15.0, 1.0 / 3.0)


def pressure_tol(make, fields, delta, subs):
    """Absolute bound of the pressure (mean removed) after the sub-steps `subs`, for a difference of up to delta in the
    velocity before each projection.

    An increment solves div(u*) / (alpha dt), so the difference reaches the pressure through the solve and over dt.
    That is measured on the oracle: one sub-step from velocities that differ by uniform noise of that size (none at the
    walls), and by how much its pressure then moves; the other sub-steps count with their own 1 / alpha."""
    make_one = make()
    make_one.set_state(*fields)
    make_one.substep(1)
    p0 = make_one.get_state()[3]
    move = 0.0
    for seed in (1, 2):
        rng = np.random.default_rng(seed)
        pert = [f + delta * rng.uniform(-1, 1, f.shape) for f in fields[:3]]
        if fields[1].shape[1] != fields[0].shape[1]:
            pert[1][:, [0, -1], :] = fields[1][:, [0, -1], :]
        of = make()
        of.set_state(*[np.asfortranarray(f) for f in pert], fields[3])
        of.substep(1)
        d = of.get_state()[3] - p0
        move = max(move, float(np.abs(d - d.mean()).max()))
    return move * sum(ALPHA[1] / ALPHA[i] for i in subs)


def delta_fp64(fields):
    """sixteen roundings of the largest velocity: q + rhs, and a right-hand side of some ten terms times dt"""
    return 16 * 2.0 ** -52 * max(float(np.abs(f).max()) for f in fields[:3])


def delta_mixed(fields, ref):
    """the FP32 right-hand side: the change of the steps is a sum of some ten terms of a few roundings each, cancelling
    by up to ten"""
    return 100 * 2.0 ** -24 * max(float(np.abs(r - f).max()) for r, f in zip(ref[:3], fields[:3]))


def check(tag, got, ref, fields, make, subs, mixed):
    delta = delta_mixed(fields, ref) if mixed else delta_fp64(fields)
    ptol = max(pressure_tol(make, fields, delta, subs), TOL * float(np.abs(ref[3]).max()))
    d = (got[3] - got[3].mean()) - (ref[3] - ref[3].mean())
    errs = [float(np.abs(g - r).max()) for g, r in zip(got[:3], ref[:3])] + [float(np.abs(d).max())]
    tols = [max(TOL * float(np.abs(r).max()), delta if mixed else 0.0) for r in ref[:3]] + [ptol]
    print(tag, " ".join(f"{n} {e:.2e} (of {t:.1e})" for n, e, t in zip(("qx", "qy", "qz", "pr"), errs, tols)), flush=True)
    bad = [n for n, e, t in zip(("qx", "qy", "qz", "pr"), errs, tols) if not e < t]
    assert not bad, bad


def _domain_kw(mixed):
    from chapsim2_amd.domain import PREC_MIXED

    return dict(precision=PREC_MIXED) if mixed else {}


# one chunk; short last chunks; odd lengths; few lines in the last wave; long chunks; a line over 256 points
CHANNELS = [(16, 16, 16), (18, 17, 18), (20, 15, 10), (54, 34, 45), (50, 49, 25), (90, 19, 30), (24, 64, 75),
            (60, 49, 200), (270, 16, 16), (16, 20, 288)]


@pytest.mark.parametrize("nc", CHANNELS)
@pytest.mark.parametrize("mixed", [False, True])
def test_channel(po, nc, mixed):
    from chapsim2_amd.domain import Domain
    from chapsim2_amd.initial import channel_fields

    print(f"pressure, channel {nc} mixed {mixed}", flush=True)

    def make():
        of = po.Flow(list(nc), LX, -1.0, 1.0, LZ, wall_y=True, iacc=4, poisson=2, **CFG)
        of.update_re(0)
        return of

    fields = channel_fields(nc, LX, -1.0, 1.0, LZ, 2, 0.075, noise=0.1, seed=31)
    dm, of = Domain(nc, LX, -1.0, 1.0, LZ, **CFG, **_domain_kw(mixed)), make()
    try:
        for o in (dm, of):
            o.set_state(*fields)
            o.update_re(0)
            for isub in (1, 2):
                o.substep(isub)
        check(f"channel {nc} mixed {mixed}:", dm.get_state(), of.get_state(), fields, make, (1, 2), mixed)
    finally:
        dm.close()


@pytest.mark.parametrize("nc", [(20, 18, 30), (32, 27, 12)])
@pytest.mark.parametrize("mixed", [False, True])
def test_periodic_box(po, nc, mixed):
    from chapsim2_amd.domain import FFT_2DECOMP_3DFFT, Domain
    from chapsim2_amd.initial import tgv_fields

    print(f"pressure, box {nc} mixed {mixed}", flush=True)
    p2 = 2 * np.pi
    cfg = dict(dt=1e-3, ren=1600.0)

    def make():
        of = po.Flow(list(nc), p2, 0.0, p2, p2, wall_y=False, iacc=4, poisson=3, **cfg)
        of.update_re(0)
        return of

    rng = np.random.default_rng(1)
    fields = [np.asfortranarray(a + 0.05 * rng.uniform(-1, 1, a.shape)) for a in tgv_fields(nc, p2, 0.0, p2, p2)]
    dm, of = Domain(nc, p2, 0.0, p2, p2, periodic_y=True, poisson=FFT_2DECOMP_3DFFT, **cfg, **_domain_kw(mixed)), make()
    try:
        for o in (dm, of):
            o.set_state(*fields)
            o.update_re(0)
            for isub in (1, 2, 3):
                o.substep(isub)
        check(f"box {nc} mixed {mixed}:", dm.get_state(), of.get_state(), fields, make, (1, 2, 3), mixed)
    finally:
        dm.close()


@pytest.mark.parametrize("nc", [(18, 21, 15), (30, 50, 25), (270, 16, 18)])
@pytest.mark.parametrize("mixed", [False, True])
def test_heated_channel(po, nc, mixed):
    from test_gpu_thermo import CFG as HCFG, _initial, _pair

    print(f"pressure, heated {nc} mixed {mixed}", flush=True)
    tab, fields, rhoh, tw, t0 = _initial(po, nc, 21)

    class Heated:
        """the oracle's heated channel from a velocity, with the enthalpy of _pair"""

        def __init__(self):
            self.of = po.Flow(list(nc), LX, -1.0, 1.0, LZ, wall_y=True, iacc=4, poisson=2, projection=1, **HCFG)
            self.get_state = self.of.get_state

        def set_state(self, *f):
            self.of.set_state(*f)
            self.of.thermo_enable(po.Props(tab, -1.0), tw, 1.0, t0)
            assert self.of.thermo_set_rhoh(rhoh) == 0
            self.of.update_re(0)

        def substep(self, isub):
            self.of.energy_substep(isub)
            self.of.substep(isub)

    dm, unused, keep = _pair(po, nc, 21, precision=1 if mixed else 0)
    of = Heated()
    of.set_state(*fields)
    try:
        dm.update_re(0)
        for isub in (1, 2, 3):
            dm.substep(isub)
            of.substep(isub)
        check(f"heated {nc} mixed {mixed}:", dm.get_state(), of.get_state(), fields, Heated, (1, 2, 3), mixed)
    finally:
        dm.close()
