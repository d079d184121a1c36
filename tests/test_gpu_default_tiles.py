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
