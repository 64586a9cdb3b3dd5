"""The from-rho*h searches by bins and neighbours against the oracle's bisections, bit for bit: rows on, beside and
between nodes (kMinP's gap included), rising, falling and folded rho*h, two rows to 12000."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _table(kind, rows):
    h = np.linspace(0.5, 2.0, rows) ** 1.5
    if kind == "rising":
        d = 1.0 + 0.2 * np.sin(3.0 * h)
    elif kind == "falling":
        d = h ** -2.5
    else:  # rho*h rises, folds over and rises again
        d = (h + 0.4 * np.sin(6.0 * h)) / h
    t = np.zeros((rows, 8))
    t[:, 1], t[:, 2], t[:, 3] = h, 1.0 + np.arange(rows) / rows, d
    t[:, 4], t[:, 5], t[:, 6], t[:, 7] = np.sqrt(h), 1.0 / h, 2.0 + np.cos(h), h * h
    return t


@pytest.mark.parametrize("kind", ["rising", "falling", "folded"])
@pytest.mark.parametrize("rows", [2, 3, 17, 1000, 4096, 9000, 12000])
def test_search_is_the_bisection(po, kind, rows):
    from chapsim2_amd.props import NAMES, PropertyTable

    op = po.Props(_table(kind, rows), -1.0)
    pt = PropertyTable(_table(kind, rows), -1.0)
    try:
        lo, hi, _ = pt.info()
        rng = np.random.default_rng(rows)
        node = op.column("rhoh")[rng.integers(0, rows, 4000)]
        gaps = np.array([0.0, 1e-10, -1e-10, 9.99e-11, 1.002e-10, -1.002e-10, 1e-9, -1e-9, 1e-15])
        x = np.concatenate([rng.uniform(lo, hi, 40000), node + gaps[rng.integers(0, gaps.size, node.size)], [lo, hi]])
        x = np.clip(x, lo, hi)
        got = pt.from_rhoh(x)
        res, flags = op.from_dh(x)
        assert not flags.any()
        for j, n in enumerate(NAMES):
            assert np.array_equal(got[n], res[:, j]), (n, np.abs(got[n] - res[:, j]).max())
    finally:
        pt.close()
