"""The pressure solves on device arrays that start at an odd element (views into a larger array): values as on an array
of its own, nothing written beside it."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LX, LZ = 4 * np.pi, 4 * np.pi / 3


# two-pass x transforms of lines of one wave and of several, general x transforms (nx/2 = 18), and the solves
@pytest.mark.parametrize("nc,kind", [((64, 16, 12), "fishpack"), ((240, 9, 10), "fishpack"), ((36, 12, 9), "fishpack"),
                                     ((32, 16, 12), "periodic"), ((64, 16, 10), "channel")])
@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("offset", [1, 3])
def test_offset_view(nc, kind, f32, offset):
    import torch

    from chapsim2_amd import _lib
    from chapsim2_amd.domain import FFT_2DECOMP_3DFFT, Domain

    print(f"view {nc} {kind} f32 {f32} offset {offset}", flush=True)
    kw = {"fishpack": dict(istret=2, rstret=0.075), "periodic": dict(periodic_y=True, poisson=FFT_2DECOMP_3DFFT),
          "channel": dict(poisson=FFT_2DECOMP_3DFFT)}[kind]
    dm = Domain(nc, LX, -1.0, 1.0, LZ, **kw)
    try:
        dt = torch.float32 if f32 else torch.float64
        n = int(np.prod(nc))
        rhs = np.random.default_rng(n).uniform(-1, 1, n)
        rhs -= rhs.mean()
        own = torch.from_numpy(rhs).to(dt).cuda()
        guard = 7.25
        big = torch.full((n + 16,), guard, dtype=dt, device="cuda")
        view = big[offset:offset + n]
        view.copy_(own)
        assert view.data_ptr() % (2 * own.element_size()) != 0
        torch.cuda.synchronize()
        for t in (own, view):
            p = C.c_void_p(t.data_ptr())
            _lib.check(dm.lib.chs_poisson_f32(dm.h, p) if f32 else dm.lib.chs_poisson(dm.h, p, _lib.MEM_DEVICE))
        assert torch.equal(view, own)
        assert bool((big[:offset] == guard).all()) and bool((big[offset + n:] == guard).all())
    finally:
        dm.close()
