"""Fused RK4 kernels at the edges of their tiles and k chunks: widths below, at and past a
tile, the thinnest k extent, chunks of a plane count that is no multiple of the planes a loop
turn takes, strided batches.  Every FP64 variant evaluates each point with the same operation
sequence, so the scalar kernel's result is the reference, bit for bit; the oracle bounds both
(1e-12 of the largest value, the bound stated for the fused kernels)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

import oracle as O  # noqa: E402

C3 = (1.0, -0.5, 0.25)


@pytest.fixture(scope="module")
def sp():
    import stencilparareal_amd as spm
    from stencilparareal_amd import field
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    field.Context.default(0)
    return spm


def run(sp, shape, variant, tile, kchunk, steps=3, nufreq=0.0):
    ni, nj, nk = shape
    q0 = np.random.default_rng(ni * 100 + nj + nk).standard_normal((nk, nj, ni))
    conv = sp.Convection(ni, nj, nk, 1. / 32, 0.02, nufreq, *C3)
    conv.set_tile(*tile, kchunk, variant=variant)
    a, b = conv.field(), conv.field()
    a.set(q0)
    conv.DoRK4(a, b, 0.0, 1e-4, steps)
    return q0, b.get()


@pytest.mark.parametrize("shape", [(2, 2, 8), (8, 8, 8), (30, 31, 9), (32, 32, 10), (34, 33, 11), (66, 2, 17), (96, 64, 16)],
                         ids=lambda s: "%dx%dx%d" % s)
@pytest.mark.parametrize("kchunk", [0, 1, 3, 6])
def test_quad_kernel_edges(sp, shape, kchunk):
    q0, ref = run(sp, shape, "scalar", (32, 16, 512), 0)
    _, got = run(sp, shape, "quad", (32, 32, 512), kchunk)
    assert np.array_equal(got, ref)
    exact = O.OConvection(*shape, 1. / 32, 0.02, 0.0, *C3).rk4(q0, 0.0, 1e-4, 3)
    assert np.abs(got - exact).max() <= 1e-12 * np.abs(exact).max()


@pytest.mark.parametrize("shape", [(2, 2, 8), (3, 5, 8), (8, 8, 8), (16, 16, 16), (17, 16, 9), (18, 33, 15), (31, 7, 24), (48, 34, 33)],
                         ids=lambda s: "%dx%dx%d" % s)
def test_brick_kernel_edges(sp, shape):
    q0, ref = run(sp, shape, "scalar", (32, 16, 512), 0, steps=4, nufreq=30.0)
    _, got = run(sp, shape, "split", (16, 16, 384), 8, steps=4, nufreq=30.0)
    assert np.array_equal(got, ref)
    exact = O.OConvection(*shape, 1. / 32, 0.02, 30.0, *C3).rk4(q0, 0.0, 1e-4, 4)
    assert np.abs(got - exact).max() <= 1e-12 * np.abs(exact).max()


@pytest.mark.parametrize("shape", [(96, 98, 72), (145, 131, 40), (272, 258, 17)], ids=lambda s: "%dx%dx%d" % s)
@pytest.mark.parametrize("kind", ["compact", "stella"])
def test_bricks_in_turn(sp, shape, kind):
    """More bricks than blocks: 378 to 867, the last ones partial in every direction."""
    ni, nj, nk = shape
    q0 = np.random.default_rng(ni).standard_normal((nk, nj, ni))
    out = []
    for variant, tile, kchunk in (("scalar", (32, 16, 512), 0), ("split", (16, 16, 384), 8)):
        conv = sp.Convection(ni, nj, nk, 1. / 64, 0.02, 0.0, *C3)
        conv.set_tile(*tile, kchunk, variant=variant)
        a, b = conv.field(kind=kind), conv.field(kind=kind)
        a.set(q0)
        conv.DoRK4(a, b, 0.0, 1e-4, 3)
        out.append(b.get())
    assert np.isfinite(out[0]).all() and np.array_equal(*out)


@pytest.mark.parametrize("shape,slices,pad", [((50, 34, 41), 7, 0), ((50, 34, 41), 7, 3), ((45, 38, 29), 8, 1), ((16, 16, 8), 601, 0)],
                         ids=lambda v: "%dx%dx%d" % v if isinstance(v, tuple) else str(v))
def test_bricks_of_several_slices_in_turn(sp, shape, slices, pad):
    """More bricks than blocks over a batch: a block's bricks lie in several slices, which are `pad`
    elements more than a field apart (an odd stride: no 16-byte accesses)."""
    import ctypes as C
    from stencilparareal_amd import _lib as L
    ni, nj, nk = shape
    lay = L.Layout()
    L.call("sp_layout_compact", ni, nj, nk, L.SP_F64, C.byref(lay))
    stride = ni * nj * nk + pad
    assert -(-ni // 16) * -(-nj // 16) * -(-nk // 8) * slices > 256
    a = torch.from_numpy(np.random.default_rng(slices).standard_normal(stride * slices)).cuda()
    out = []
    for variant, tile, kchunk in (("scalar", (32, 16, 512), 0), ("split", (16, 16, 384), 8)):
        conv = sp.Convection(ni, nj, nk, 1. / 64, 0.02, 20.0, *C3)
        conv.set_tile(*tile, kchunk, variant=variant)
        b = torch.zeros_like(a)
        conv.ctx.sync_stream()
        L.call("sp_do_rk4_batched", conv.h, slices, C.byref(lay), C.c_void_p(a.data_ptr()), C.byref(lay),
               C.c_void_p(b.data_ptr()), stride, 0.0, 1e-4, 2)
        torch.cuda.synchronize()
        out.append(b)
    assert torch.isfinite(out[0]).all() and torch.equal(*out)


def test_bricks_with_a_viscosity_per_slice(sp):
    """Time-dependent viscosity in a Parareal: every slice has its own coefficients, and a block's
    bricks lie in several slices."""
    from stencilparareal_amd.config import RuntimeConfiguration
    n, slices = 48, 8
    u0 = O.fill_gaussians(n, [0.3, 0.7], [0.4, 0.6], [0.5, 0.2], [0.1, 0.15], [1.0, 0.5])
    out = []
    for variant, tile, kchunk in (("scalar", (32, 16, 512), 0), ("split", (16, 16, 384), 8)):
        conf = RuntimeConfiguration(gridSize=n, endTime=0.004, timeStepsFine=4 * slices, timeStepsCoarse=2 * slices,
                                    nu0=0.02, nufreq=900.0, cx=C3[0], cy=C3[1], cz=C3[2], kmax=2, async_=False,
                                    timeSlices=slices)
        conv = sp.Convection(n, n, n, conf.dx(), conf.nu0, conf.nufreq, *C3)
        conv.set_tile(*tile, kchunk, variant=variant)
        init, sol = conv.field(), conv.field()
        init.set(u0)
        sp.Parareal(conv, init, sol, conf, coarse="rk4").DoParallel()
        out.append(sol.get())
    assert np.isfinite(out[0]).all() and np.array_equal(*out)
