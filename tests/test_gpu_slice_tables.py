"""Slice loops whose layers share, repeat or differ in thickness: the propagator
factors are kept per distinct thickness, whichever layer takes them.

A layer's propagation does not depend on the other layers of the stack, so a
stack run in one call equals its slices run one call each, to the rounding of
the extra transforms (FP64: 1e-12).
"""
import numpy as np
import pytest

import multislice_amd as msx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cz", [[2.0, 2.0, 2.0], [2.0, 1.5, 2.0], [1.0, 2.0, 3.0], [2.0, 1.0, 1.0]])
def test_mixed_thicknesses(ctx, cz):
    rng = np.random.default_rng(2)
    nx, ny, a, b, kev = 64, 128, 8.0, 14.0, 200.0
    t = ctx.transmission(rng.uniform(0, 300, (3, nx, ny)), a, b, kev)
    layer = np.array([0, 2, 1, 1, 0, 2, 2])
    psi = np.ones((2, nx, ny), np.complex128)
    ctx.multislice(t, cz, layer, psi, a, b, kev, tilt=(0.002, -0.001))
    ref = np.ones((2, nx, ny), np.complex128)
    for l in layer:
        ctx.multislice(t[l:l + 1], [cz[l]], [0], ref, a, b, kev, tilt=(0.002, -0.001))
    assert np.linalg.norm(psi - ref) < 1e-12 * np.linalg.norm(ref)
