"""The y solves of the FISHPACK pressure path on lines of one chunk, of whole
and ragged chunks, of the most chunks the partitioned solve takes, and beyond
(factor tables), FP64 and FP32, against an extended-precision elimination of
the same rows.  The mean mode, which carries the singular-pivot rule, is
compared apart with the oracle's."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LX, LZ = 4 * np.pi, 4 * np.pi / 3


def _reference(rhs, dom, nc):
    """phi with every mode's tridiagonal rows (the rounded double coefficients) solved in extended precision; the
    (0, 0) mode left out."""
    nx, ny, nz = nc
    h2 = 1.0 / np.array(dom.h) ** 2
    ymp, ymc = np.array(dom.ymp), np.array(dom.ymc)
    a = h2[1] * ymc * ymp[:ny]
    c = h2[1] * ymc * ymp[1:]
    b = -(a + c)
    b[0] = b[0] + a[0]
    b[-1] = b[-1] + c[-1]
    a[0] = c[-1] = 0.0
    spec = np.fft.fft(np.fft.rfft(rhs, axis=0), axis=2)
    kx, kz = np.arange(nx // 2 + 1), np.arange(nz)
    xr = -4.0 * h2[0] * np.sin(np.pi * kx / nx) ** 2
    zr = -4.0 * h2[2] * np.sin(np.pi * np.minimum(kz, nz - kz) / nz) ** 2
    re, im = spec.real.astype(np.longdouble), spec.imag.astype(np.longdouble)
    bb = ((b[None, :, None] + xr[:, None, None]) + zr[None, None, :]).astype(np.longdouble)
    bb[0, -1, 0] += 1.0
    al, cl = a.astype(np.longdouble), c.astype(np.longdouble)
    d = np.zeros_like(re)
    for j in range(ny):
        piv = bb[:, j] - (al[j] * d[:, j - 1] if j else 0)
        d[:, j] = cl[j] / piv
        for v in (re, im):
            v[:, j] = (v[:, j] - (al[j] * v[:, j - 1] if j else 0)) / piv
    for j in range(ny - 2, -1, -1):
        for v in (re, im):
            v[:, j] -= d[:, j] * v[:, j + 1]
    out = re.astype(float) + 1j * im.astype(float)
    out[0, :, 0] = 0.0
    return np.fft.irfft(np.fft.ifft(out, axis=2), n=nx, axis=0)


# one chunk; whole, short and long chunks; 32 chunks; tables
@pytest.mark.parametrize("ny", [8, 15, 16, 17, 33, 96, 129, 511, 512, 520])
@pytest.mark.parametrize("f32", [False, True])
def test_y_lines_vs_extended_precision(po, ny, f32):
    import torch

    from chapsim2_amd import _lib
    from chapsim2_amd.domain import Domain

    nc = (18, ny, 10)
    dm = Domain(nc, LX, -1.0, 1.0, LZ, istret=2, rstret=0.075)
    dom = po.Dom(list(nc), [1, 0, 1], LX, -1.0, 1.0, LZ, 2, 0.075)
    try:
        rhs = np.random.default_rng(ny).uniform(-1, 1, nc)
        # (no mean mode, and errors against the whole result: beyond 500 rows the mean mode's last pivot is rounding
        # above the rule's 1e-10, and its constant then rounds off in the inverse transforms)
        rhs = rhs - rhs.mean(axis=(0, 2), keepdims=True)
        rhs = np.asfortranarray(rhs.astype(np.float32).astype(np.float64) if f32 else rhs)
        dt = torch.float32 if f32 else torch.float64
        t = torch.from_numpy(np.ascontiguousarray(rhs.transpose(2, 1, 0))).to(dt).cuda()
        p = C.c_void_p(t.data_ptr())
        torch.cuda.synchronize()
        _lib.check(dm.lib.chs_poisson_f32(dm.h, p) if f32 else dm.lib.chs_poisson(dm.h, p, _lib.MEM_DEVICE))
        got = t.double().cpu().numpy().transpose(2, 1, 0)
        fluct = got - got.mean(axis=(0, 2), keepdims=True)
        ref = _reference(rhs, dom, nc)
        # transforms in the type: log2(n) roundings of each coefficient, twice
        tol = 16 * (2.0 ** -23 if f32 else 2.0 ** -52) * np.log2(nc[0] * nc[2]) * 2
        if ny > 512 and not f32:
            tol = 1e-11  # TRID0's own elimination: eps times max|b| / min row sum over the line
        if ny > 512 and f32:
            tol = 1e-3
        err = float(np.abs(fluct - ref).max() / max(np.abs(ref).max(), np.abs(got).max()))
        assert err < tol
    finally:
        dm.close()


@pytest.mark.parametrize("ny", [16, 33, 130])
def test_mean_mode_vs_oracle(po, ny):
    """The (0, 0) mode keeps TRID0's order and pivot rule: the oracle's values."""
    from chapsim2_amd.domain import Domain
    from chapsim2_amd.poisson import solve_fft_poisson

    nc = (16, ny, 12)
    cfg = dict(istret=2, rstret=0.075)
    dm = Domain(nc, LX, -1.0, 1.0, LZ, **cfg)
    of = po.Flow(list(nc), LX, -1.0, 1.0, LZ, wall_y=True, iacc=4, poisson=2, **cfg)
    try:
        dom = po.Dom(list(nc), [1, 0, 1], LX, -1.0, 1.0, LZ, 2, 0.075)
        rhs = np.random.default_rng(7).uniform(-1, 1, nc)
        w = 1.0 / np.array(dom.ymc)
        rhs = np.asfortranarray(rhs - (rhs.mean(axis=(0, 2)) * w).sum() / w.sum())
        ref = np.asarray(of.poisson(rhs.copy(order="F")))
        got = solve_fft_poisson(rhs.copy(order="F"), dm)
        err = float(np.abs(got - ref).max() / np.abs(ref).max())
        assert err < 1e-11
    finally:
        dm.close()
