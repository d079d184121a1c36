"""The fused step's built-in tile choice over sizes on either side of its lines: fields of one
tile and less, more blocks than compute units, odd extents, the padded storage, every storage
type.  Each kernel evaluates a point with the same operation sequence in the same precision, so
the scalar kernel's result is the reference, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

SIZES = [(8, 8, 8), (34, 18, 9), (35, 18, 9), (64, 64, 64), (96, 80, 40), (129, 40, 33), (160, 96, 72), (288, 288, 10)]


@pytest.fixture(scope="module")
def sp():
    import stencilparareal_amd as spm
    from stencilparareal_amd import field
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    field.Context.default(0)
    return spm


@pytest.mark.parametrize("shape", SIZES, ids=lambda s: "%dx%dx%d" % s)
@pytest.mark.parametrize("storage", ["f64", "f64 padded", "f32", "bf16"])
def test_default_tile(sp, shape, storage):
    ni, nj, nk = shape
    dtype, kind = storage.split()[0], "stella" if "padded" in storage else "compact"
    q0 = np.random.default_rng(ni + nk).standard_normal((nk, nj, ni))
    out = []
    for tile in (None, (32, 16, 512, 0)):
        conv = sp.Convection(ni, nj, nk, 1. / 64, 0.02, 0.0, 1.0, -0.5, 0.25)
        if tile:
            conv.set_tile(*tile, variant="scalar")
        a, b = conv.field(kind=kind, dtype=dtype), conv.field(kind=kind, dtype=dtype)
        a.set(q0)
        conv.DoRK4(a, b, 0.0, 1e-4, 3)
        out.append(b.get())
    assert np.isfinite(out[1]).all() and np.array_equal(*out)


def test_single_batched_step_keeps_no_scratch(sp):
    """A batched call of one step holds nothing between its input and output: captured before any
    other call, each replay gives the bits of the scalar kernel, on inputs changed in between."""
    import ctypes as C
    from stencilparareal_amd import _lib as L

    n, S = 32, 3
    lay = L.Layout()
    L.call("sp_layout_compact", n, n, n, 0, C.byref(lay))

    def step(conv, a, b):
        conv.ctx.sync_stream()
        L.call("sp_do_rk4_batched", conv.h, S, C.byref(lay), C.c_void_p(a.data_ptr()), C.byref(lay),
               C.c_void_p(b.data_ptr()), n**3, 0.0, 1e-4, 1)

    conv, ref = (sp.Convection(n, n, n, 1. / n, 0.02, 0.0, 1.0, -0.5, 0.25) for _ in range(2))
    ref.set_tile(32, 16, 512, 0, variant="scalar")
    a = torch.empty(S, n, n, n, dtype=torch.float64, device="cuda")
    b, want = torch.empty_like(a), torch.empty_like(a)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        step(conv, a, b)
    for seed in range(3):
        a.copy_(torch.from_numpy(np.random.default_rng(seed).standard_normal((S, n, n, n))))
        g.replay()
        step(ref, a, want)
        torch.cuda.synchronize()
        assert torch.equal(b, want)


@pytest.mark.parametrize("n", [32, 90, 130])
@pytest.mark.parametrize("steps", [1, 2])
def test_default_tile_odd_rows(sp, n, steps):
    """Rows of n + 1 doubles, n even: no aligned x pairs in the output."""
    import ctypes as C
    from stencilparareal_amd import _lib as L

    lay = L.Layout()
    L.call("sp_layout_compact", n, n, n, 0, C.byref(lay))
    lay.sj, lay.sk = n + 1, (n + 1) * n
    a = torch.from_numpy(np.random.default_rng(n).standard_normal((n, n, n + 1))).cuda()
    out = []
    for tile in (None, (32, 16, 512, 0)):
        conv = sp.Convection(n, n, n, 1. / 64, 0.02, 0.0, 1.0, -0.5, 0.25)
        if tile:
            conv.set_tile(*tile, variant="scalar")
        b = torch.zeros_like(a)
        conv.ctx.sync_stream()
        L.call("sp_do_rk4", conv.h, C.byref(lay), C.c_void_p(a.data_ptr()), C.byref(lay), C.c_void_p(b.data_ptr()),
               0.0, 1e-4, steps)
        torch.cuda.synchronize()
        out.append(b)
    assert torch.isfinite(out[1]).all() and torch.equal(*out)


@pytest.mark.parametrize("shape", [(48, 48, 40), (47, 48, 40), (192, 192, 192)], ids=lambda s: "%dx%dx%d" % s)
def test_k_chunk_set_alone(sp, shape):
    """A k chunk without a tile is the chunk of the kernel that runs, whatever the size's own choice."""
    ni, nj, nk = shape
    q0 = np.random.default_rng(ni).standard_normal((nk, nj, ni))
    out = []
    for kwargs in (dict(kchunk=12), dict(tx=32, ty=16, nthreads=512, variant="scalar")):
        conv = sp.Convection(ni, nj, nk, 1. / 64, 0.02, 0.0, 1.0, -0.5, 0.25)
        conv.set_tile(**kwargs)
        tile = conv.get_tile(1)
        assert tile["variant"] != "split" and tile["kchunk"] == kwargs.get("kchunk", 0)
        a, b = conv.field(), conv.field()
        a.set(q0)
        conv.DoRK4(a, b, 0.0, 1e-4, 3)
        out.append(b.get())
    assert np.isfinite(out[1]).all() and np.array_equal(*out)
