"""The launch profile's algorithmic bytes: every field an operator reads or writes, counted once, by direction."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LX, LZ = 4 * np.pi, 4 * np.pi / 3
NC = (36, 25, 20)


def _bytes(dm, cls, what):
    from chapsim2_amd import _lib

    ms, nl, byt = C.c_double(), C.c_longlong(), C.c_double()
    _lib.check(dm.lib.chs_profile_begin(dm.h, cls))
    what()
    _lib.check(dm.lib.chs_profile_end(dm.h, C.byref(ms), C.byref(nl), C.byref(byt)))
    return nl.value, byt.value


def _fields():
    """points at the cells, and at the cells with y at its nodes"""
    nx, ny, nz = NC
    return nx * ny * nz, nx * (ny + 1) * nz


def _domain(mixed=False):
    from chapsim2_amd.domain import PREC_MIXED, Domain
    from chapsim2_amd.initial import channel_fields

    dm = Domain(NC, LX, -1.0, 1.0, LZ, istret=2, rstret=0.075, dt=5e-4, ren=2800.0, idriven=1,
                **(dict(precision=PREC_MIXED) if mixed else {}))
    dm.set_state(*channel_fields(NC, LX, -1.0, 1.0, LZ, 2, 0.075, noise=0.1, seed=3))
    dm.update_re(0)
    return dm


def test_divergence_bytes():
    """d = D_x u, then d += D_y v and d += D_z w: the component read, the sum written or read and written."""
    dm = _domain()
    c, n = _fields()
    try:
        for cls, words in ((0, 2 * c), (1, n + 2 * c), (2, 3 * c)):
            assert _bytes(dm, cls, dm.divergence) == (1, 8.0 * words), cls
    finally:
        dm.close()


@pytest.mark.parametrize("mixed", [False, True])
def test_substep_bytes(mixed):
    """A sub-step's operators along each direction (constant properties, the second sub-step: its rhs0 is read).

    Right-hand side, words of its type, with c points at the cells and n with y at its nodes: a pair reads one field
    and writes two; a shear flux reads one and two operands and writes one; the normal fluxes read one and four operands
    and write three; a single reads and writes one; the last operator of a component reads two and three operands and
    writes rhs0, and reads and writes the FP64 state.  Projection, FP64: the divergence as above; a correction reads the
    increment, reads and writes the velocity, and x also the pressure."""
    dm = _domain(mixed)
    c, n = _fields()
    t = 4.0 if mixed else 8.0
    rhs = {0: (c + 2 * c) + 2 * n + n + (c + 2 * c)  # pairs of u, v, w
           + (n + n) + (c + c)                       # x derivatives of f_xy, f_xz
           + (2 * c + 3 * c + c),                    # last x operator
           1: (c + 2 * n) + (n + 2 * c)              # pairs of w, v
           + (c + 2 * n + n)                         # f_xy
           + (n + c) + (n + c)                       # y derivatives of f_xy, f_yz
           + (2 * c + 3 * n + n),
           2: (c + 2 * c + c) + (n + 2 * n + n)      # f_xz, f_yz
           + (c + 4 * c + 3 * c)                     # normal fluxes
           + (c + c) + (n + n)                       # z derivatives of f_xz, f_yz
           + (2 * c + 3 * c + c)}
    state = {0: 2 * c, 1: 2 * n, 2: 2 * c}
    div = {0: 2 * c, 1: n + 2 * c, 2: 3 * c}
    corr = {0: c + 2 * c + 2 * c, 1: c + 2 * n, 2: c + 2 * c}
    rounded = {0: 2 * c, 1: n, 2: c}                 # FP32 copies of the velocity and, in x, of the pressure
    try:
        dm.substep(1)
        for cls in (0, 1, 2):
            want = t * rhs[cls] + 8.0 * (state[cls] + div[cls] + corr[cls]) + (4.0 * rounded[cls] if mixed else 0.0)
            assert _bytes(dm, cls, lambda: dm.substep(2))[1] == want, cls
    finally:
        dm.close()
