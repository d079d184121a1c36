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
