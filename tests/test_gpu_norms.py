"""Norms of fields with remainders in the four-points-per-turn sweep, compact and padded, against
numpy (sums in another order: 1e-13 relative; the maxima are exact)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("shape", [(2, 2, 2), (7, 5, 3), (64, 33, 62), (101, 75, 87)], ids=lambda s: "%dx%dx%d" % s)
@pytest.mark.parametrize("kind", ["compact", "stella"])
def test_norms_remainders_and_layouts(shape, kind):
    import stencilparareal_amd as sp
    from stencilparareal_amd.field import ConvectionField, norms
    ni, nj, nk = shape
    rng = np.random.default_rng(ni + nj)
    x, y = rng.standard_normal((nk, nj, ni)), rng.standard_normal((nk, nj, ni))
    a, b = ConvectionField("a", ni, nj, nk, kind=kind), ConvectionField("b", ni, nj, nk)
    a.set(x)
    b.set(y)
    e, m, d2, r2 = norms(a, b, sp.Context.default(0))
    assert e == np.abs(x - y).max() and m == np.abs(x).max()
    assert abs(d2 - ((x - y) ** 2).sum()) <= 1e-13 * d2 and abs(r2 - (y ** 2).sum()) <= 1e-13 * r2
