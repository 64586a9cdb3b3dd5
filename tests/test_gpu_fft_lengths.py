"""Every length of the two-pass transforms (CHS_FFT2_LENGTHS), as nx/2 and as nz, with 8 and with 16 lines per
workgroup on ragged line counts, FP64 and FP32, through the FISHPACK pressure solve against numpy's transforms and
an FP64 elimination per mode."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LENGTHS = (16, 20, 24, 25, 27, 30, 32, 36, 40, 45, 48, 50, 54, 60, 64, 72, 75, 80, 81, 90, 96, 100, 108, 120, 128, 135,
           144, 150, 160, 162, 180, 192, 200, 216, 225, 240, 256, 270, 288, 300, 320, 360, 384, 400, 432, 480, 512)
NY = 8
LX, LZ = 4 * np.pi, 4 * np.pi / 3


def _reference(rhs, dom):
    nx, ny, nz = rhs.shape
    h2 = 1.0 / np.array(dom.h) ** 2
    ymp, ymc = np.array(dom.ymp), np.array(dom.ymc)
    a = h2[1] * ymc * ymp[:ny]
    c = h2[1] * ymc * ymp[1:]
    b = -(a + c)
    b[0] += a[0]
    b[-1] += c[-1]
    spec = np.fft.fft(np.fft.rfft(rhs, axis=0), axis=2)
    kx, kz = np.arange(nx // 2 + 1), np.arange(nz)
    lam = (-4.0 * h2[0] * np.sin(np.pi * kx / nx) ** 2)[:, None] - 4.0 * h2[2] * np.sin(np.pi * kz / nz)[None] ** 2
    m = np.zeros(lam.shape + (ny, ny))
    j = np.arange(ny)
    m[..., j, j] = b + lam[..., None]
    m[..., j[1:], j[:-1]] = a[1:]
    m[..., j[:-1], j[1:]] = c[:-1]
    m[0, 0] = np.eye(ny)
    out = np.moveaxis(np.linalg.solve(m, np.moveaxis(spec, 1, 2)[..., None])[..., 0], 2, 1).copy()
    out[0, :, 0] = 0.0
    return np.fft.irfft(np.fft.ifft(out, axis=2), n=nx, axis=0)


@pytest.mark.parametrize("variant", [0, 1])
@pytest.mark.parametrize("n", LENGTHS)
def test_transform_length(po, n, variant):
    import torch

    from chapsim2_amd import _lib
    from chapsim2_amd.domain import Domain

    lib = _lib.load()
    for nc in ((2 * n, NY, 9), (10, NY, n)):
        print(f"transform length {n} variant {variant} nc={nc}", flush=True)
        _lib.check(lib.chs_tune_force(b"fft_", variant))
        dm = Domain(nc, LX, -1.0, 1.0, LZ, istret=2, rstret=0.075)
        try:
            rhs = np.random.default_rng(n).standard_normal(nc)
            rhs -= rhs.mean(axis=(0, 2), keepdims=True)
            ref = _reference(rhs, po.Dom(list(nc), [1, 0, 1], LX, -1.0, 1.0, LZ, 2, 0.075))
            # four transforms of at most 9 levels of a few roundings each; FP64: numpy's elimination of rows whose
            # diagonal is up to ~2000 times the smallest eigenvalue
            for dt, tol in ((torch.float64, 1e-12), (torch.float32, 1e-5)):
                t = torch.from_numpy(np.ascontiguousarray(rhs.transpose(2, 1, 0))).to("cuda", dt)
                p = C.c_void_p(t.data_ptr())
                torch.cuda.synchronize()
                _lib.check(lib.chs_poisson(dm.h, p, _lib.MEM_DEVICE) if tol < 1e-9 else lib.chs_poisson_f32(dm.h, p))
                out = t.double().cpu().numpy().transpose(2, 1, 0)
                err = np.abs(out - ref).max() / np.abs(ref).max()
                assert err < tol, (nc, dt, err)
        finally:
            dm.close()
            _lib.check(lib.chs_tune_force(b"fft_", -1))
