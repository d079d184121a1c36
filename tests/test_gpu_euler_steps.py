"""Two forward Euler steps per launch: odd and even step counts, sizes at
the edges of a brick (16x16x8 points, halo of two), grid spacings that are and are not a power of
two, padded fields, in place -- bit for bit the oracle's steps."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

import oracle as O  # noqa: E402


def check(shape, steps, dx, upwind, nufreq=0.0, kind="compact", in_place=False):
    import stencilparareal_amd as sp
    ni, nj, nk = shape
    c = (1.0, -0.5, 0.25)
    q0 = np.random.default_rng(ni + nj + nk + steps).standard_normal((nk, nj, ni))
    conv = sp.Convection(ni, nj, nk, dx, 0.01, nufreq, *c, upwind=upwind)
    a = conv.field(kind=kind)
    b = a if in_place else conv.field()
    a.set(q0)
    conv.DoEuler(a, b, 0.2, 1e-4, steps)
    oc = O.OConvection(ni, nj, nk, dx, 0.01, nufreq, *c, upwind=upwind)
    assert np.array_equal(b.get(), oc.euler(q0, 0.2, 1e-4, steps))


@pytest.mark.parametrize("steps", [1, 2, 3, 4, 5, 6, 9])
@pytest.mark.parametrize("upwind", [True, False])
def test_euler_steps_bitwise(steps, upwind):
    check((32, 32, 32), steps, 1. / 32, upwind, nufreq=50.0)


@pytest.mark.parametrize("shape", [(2, 2, 8), (3, 5, 9), (16, 16, 8), (17, 15, 10), (48, 33, 15), (31, 64, 7)],
                         ids=lambda s: "%dx%dx%d" % s)
@pytest.mark.parametrize("steps", [2, 3, 4])
def test_euler_steps_brick_edges(shape, steps):
    check(shape, steps, 1. / 24, True)


@pytest.mark.parametrize("steps", [2, 4, 8])
@pytest.mark.parametrize("kind,in_place", [("stella", False), ("compact", True)])
def test_euler_steps_padded_and_in_place(steps, kind, in_place):
    check((40, 20, 17), steps, 1. / 32, True, kind=kind, in_place=in_place)


@pytest.mark.parametrize("steps", [2, 4, 6, 10])
@pytest.mark.parametrize("shift", [2, 33, 32 * 32 * 9])
def test_euler_steps_overlapping_storage(steps, shift):
    """An output that overlaps the input `shift` points on: an even number of steps reads the input
    only while it writes to the scratch."""
    import ctypes as C
    import stencilparareal_amd as sp
    from stencilparareal_amd import _lib as L
    n, c = 32, (1.0, -0.5, 0.25)
    conv = sp.Convection(n, n, n, 1. / n, 0.01, 30.0, *c)
    lay = L.Layout()
    L.call("sp_layout_compact", n, n, n, L.SP_F64, C.byref(lay))
    q0 = np.random.default_rng(shift + steps).standard_normal((n, n, n))
    buf = torch.zeros(n**3 + shift, dtype=torch.float64, device="cuda")
    buf[:n**3] = torch.from_numpy(q0.ravel())
    conv.ctx.sync_stream()
    L.call("sp_do_euler", conv.h, C.byref(lay), C.c_void_p(buf.data_ptr()), C.byref(lay),
           C.c_void_p(buf.data_ptr() + 8 * shift), 0.2, 1e-4, steps)
    torch.cuda.synchronize()
    want = O.OConvection(n, n, n, 1. / n, 0.01, 30.0, *c).euler(q0, 0.2, 1e-4, steps)
    assert np.array_equal(buf[shift:].cpu().numpy().reshape(n, n, n), want)
