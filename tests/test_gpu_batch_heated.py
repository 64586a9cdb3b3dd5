"""Heated channels in a batch: captured steps, eager ones and new states in between give what the same channel gives by
itself, in FP64 and in the mixed form, whose FP32 copies of rho u and of the properties outlive a step."""
import numpy as np
import pytest

from test_gpu_thermo import CFG, LX, LZ, _initial

pytestmark = pytest.mark.gpu

NC = (32, 24, 16)


@pytest.mark.parametrize("mixed", [False, True])
def test_heated_batch_matches_single(po, mixed):
    from chapsim2_amd.domain import PREC_FP64, PREC_MIXED, PROJ_EXACT, Batch, Domain
    from chapsim2_amd.props import PropertyTable

    print(f"heated batch mixed {mixed}", flush=True)
    spec = dict(nc=NC, lxx=LX, lyb=-1.0, lyt=1.0, lzz=LZ, projection=PROJ_EXACT,
                precision=PREC_MIXED if mixed else PREC_FP64, **CFG)
    tab, fields, rhoh, tw, t0 = _initial(po, NC, 5)
    _, fields2, rhoh2, _, _ = _initial(po, NC, 6)
    tables = [PropertyTable(tab, -1.0), PropertyTable(tab, -1.0)]
    b = Batch([spec])
    one = Domain(NC, LX, -1.0, 1.0, LZ, **{k: v for k, v in spec.items() if k not in ("nc", "lxx", "lyb", "lyt", "lzz")})
    try:
        for d, t in zip((b.domains[0], one), tables):
            d.set_state(*fields)
            d.thermo_enable(t, tw, 1.0, t0, 0)
            d.thermo_set_rhoh(rhoh)
            d.update_re(0)
            d.substep(0)

        def both(it, n, graph):
            b.run(it, n, graph=graph)
            one.run(it, n)
            x, y = b.domains[0], one
            tx, ty = x.thermo_get(), y.thermo_get()
            for name, p, q in list(zip(("qx", "qy", "qz", "pr"), x.get_state(), y.get_state())) + [
                    (k, tx[k], ty[k]) for k in tx]:
                assert np.array_equal(p, q), (it, n, graph, name, np.abs(p - q).max())

        both(0, 3, True)
        for d in (b.domains[0], one):
            d.set_state(*fields2)
        both(3, 1, True)
        both(4, 1, False)
        for d in (b.domains[0], one):
            d.thermo_set_rhoh(rhoh2)
        both(5, 1, False)
        for d in (b.domains[0], one):
            d.set_state(*fields)
        both(6, 2, True)
    finally:
        one.close()
        b.close()
