"""Who may share a propagator's scratch and work fields.  An out-of-place single step holds nothing
but its input and output: single steps of one propagator run on several streams at once, and a
captured one stays valid whatever the propagator runs later.  The scalar kernel's result, one
launch per step, is the reference, bit for bit."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

SIZES = [(64, 64, 64), (45, 38, 29)]  # the built-in choice of longer runs: bricks


@pytest.fixture(scope="module")
def sp():
    import stencilparareal_amd as spm
    from stencilparareal_amd import field
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    field.Context.default(0)
    return spm


def convection(sp, shape, tile=None):
    conv = sp.Convection(*shape, 1. / 64, 0.02, 0.0, 1.0, -0.5, 0.25)
    if tile:
        conv.set_tile(*tile, variant="scalar")
    return conv


def scalar_steps(sp, shape, u, steps):
    conv = convection(sp, shape, (32, 16, 512, 0))
    a, b = conv.field(), conv.field()
    a.set(u)
    conv.DoRK4(a, b, 0.0, 1e-4, steps)
    return b.get()


def batched(conv, slices, steps):
    """A batched call of `steps` steps on fields of its own: (input, output)."""
    from stencilparareal_amd import _lib as L
    ni, nj, nk = conv.sizes
    lay = L.Layout()
    L.call("sp_layout_compact", ni, nj, nk, L.SP_F64, C.byref(lay))
    a = torch.rand(slices, nk, nj, ni, dtype=torch.float64, device="cuda")
    b = torch.empty_like(a)
    conv.ctx.sync_stream()
    L.call("sp_do_rk4_batched", conv.h, slices, C.byref(lay), C.c_void_p(a.data_ptr()), C.byref(lay),
           C.c_void_p(b.data_ptr()), ni * nj * nk, 0.0, 1e-4, steps)
    torch.cuda.synchronize()
    return a, b


def seeded(shape, seed):
    return np.random.default_rng(seed).standard_normal(shape[::-1])


@pytest.mark.parametrize("tuned", [False, True])
@pytest.mark.parametrize("shape", SIZES, ids=lambda s: "%dx%dx%d" % s)
def test_single_steps_on_two_streams(sp, shape, tuned):
    conv = convection(sp, shape)
    if tuned:
        conv.autotune(1)
    fields = [[conv.field(), conv.field()] for _ in range(2)]
    conv.DoRK4Timestep(*fields[0], 0.0, 1e-4)  # allocations happen here
    for s, (a, _) in enumerate(fields):
        a.set(seeded(shape, s))
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in fields]
    for _ in range(8):  # one stream's step starts before the other's has ended
        for stream, (a, b) in zip(streams, fields):
            with torch.cuda.stream(stream):
                conv.DoRK4Timestep(a, b, 0.0, 1e-4)
    torch.cuda.synchronize()
    for s, (_, b) in enumerate(fields):
        assert np.array_equal(b.get(), scalar_steps(sp, shape, seeded(shape, s), 1))


@pytest.mark.parametrize("shape", SIZES, ids=lambda s: "%dx%dx%d" % s)
def test_captured_single_step_after_larger_calls(sp, shape):
    conv = convection(sp, shape)
    a, b = conv.field(), conv.field()
    a.set(seeded(shape, 0))
    conv.DoRK4Timestep(a, b, 0.0, 1e-4)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        conv.DoRK4Timestep(a, b, 0.0, 1e-4)
    for i, later in enumerate((lambda: batched(conv, 5, 3), lambda: conv.autotune(7), lambda: batched(conv, 9, 2))):
        later()
        a.set(seeded(shape, i))
        b.set(np.zeros(shape[::-1]))
        g.replay()
        torch.cuda.synchronize()
        assert np.array_equal(b.get(), scalar_steps(sp, shape, seeded(shape, i), 1))


@pytest.mark.parametrize("shape", [(64, 64, 64), (63, 64, 64)], ids=lambda s: "%dx%dx%d" % s)
@pytest.mark.parametrize("warm", [False, True])
def test_captured_steps_after_larger_calls(sp, shape, warm):
    """Several steps captured once the scratch is there: without a work field (never used before)
    and with one, which later calls, all within the scratch, and the autotuner outgrow."""
    conv = convection(sp, shape)
    batched(conv, 64, 2)  # too many bricks for the built-in choice: a scratch of 64 slices, no work field
    a, b = conv.field(), conv.field()
    a.set(seeded(shape, 0))
    if warm:
        conv.DoRK4(a, b, 0.0, 1e-4, 3)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        conv.DoRK4(a, b, 0.0, 1e-4, 3)
    for i, later in enumerate((lambda: batched(conv, 5, 3), lambda: conv.autotune(7), lambda: batched(conv, 9, 2))):
        later()
        a.set(seeded(shape, i))
        b.set(np.zeros(shape[::-1]))
        g.replay()
        torch.cuda.synchronize()
        assert np.array_equal(b.get(), scalar_steps(sp, shape, seeded(shape, i), 3))
