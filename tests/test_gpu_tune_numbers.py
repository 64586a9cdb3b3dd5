"""The numbers of the transforms' launch shapes (chs_tune_report, chs_tune_set, chs_tune_force): 1 and 2 are the two-pass
kernels with 8 and 16 lines per workgroup, 3 the general kernel, so that a saved report keeps its meaning; 0 (4 lines) is
no longer built and takes the next that applies."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_fft_lengths import LENGTHS, LX, LZ, NY, _reference

pytestmark = pytest.mark.gpu


def _report(lib):
    buf = C.create_string_buffer(1 << 20)
    lib.chs_tune_report(buf, len(buf))
    out = {}
    for line in buf.value.decode().splitlines():
        key, _, rest = line.partition("=")
        out[key] = (int(rest.split()[0]), rest[rest.index("(") + 1:rest.index(" us")].split("/"))
    return out


def test_reported_choices():
    from chapsim2_amd.domain import Domain

    nc = (2 * 72, 11, 60)
    dm = Domain(nc, LX, -1.0, 1.0, LZ, istret=2, rstret=0.075)
    try:
        rep = _report(dm.lib)
        nxh = nc[0] // 2 + 1
        keys = [f"fft_x{s}/f64/72/{nc[1] * nc[2]}x1" for s in "+-"] + [f"fft_s{s}/f64/60/{nxh}x{nc[1]}" for s in "+-"]
        for key in keys:
            choice, us = rep[key]
            assert choice in (1, 2), (key, choice, us)
            assert len(us) == 3 and float(us[0]) < 0 and min(float(us[1]), float(us[2])) > 0, (key, us)
            assert float(us[choice]) == min(float(us[1]), float(us[2])), (key, choice, us)
    finally:
        dm.close()


@pytest.mark.parametrize("n", LENGTHS)
def test_sixteen_lines(po, n):
    """Shape 2 on every two-pass length, as nx/2 and as nz, on ragged line counts."""
    from chapsim2_amd import _lib
    from chapsim2_amd.domain import Domain
    from chapsim2_amd.poisson import solve_fft_poisson

    lib = _lib.load()
    for nc in ((2 * n, NY, 9), (10, NY, n)):
        print(f"transform length {n} with 16 lines nc={nc}", flush=True)
        _lib.check(lib.chs_tune_force(b"fft_", 2))
        dm = Domain(nc, LX, -1.0, 1.0, LZ, istret=2, rstret=0.075)
        try:
            rhs = np.random.default_rng(n).standard_normal(nc)
            rhs -= rhs.mean(axis=(0, 2), keepdims=True)
            ref = _reference(rhs, po.Dom(list(nc), [1, 0, 1], LX, -1.0, 1.0, LZ, 2, 0.075))
            out = solve_fft_poisson(np.array(rhs, order="F"), dm)
            # numpy's elimination of rows whose diagonal is up to ~2000 times the smallest eigenvalue
            assert np.abs(out - ref).max() / np.abs(ref).max() < 1e-12, nc
        finally:
            dm.close()
            _lib.check(lib.chs_tune_force(b"fft_", -1))
