"""exp(i sigma V / 1000) of the transmission build over the range of its phases:
the FP32 sine and cosine below their limit (60000 rad), the general ones above
it, one large value in a row of small ones, infinities and NaN; and more layers
than one work-group takes, whose potentials are loaded a layer ahead.

The FP32 phase fl(fl(sigma / 1000) V) is the kernel's own, so the reference is
the FP64 exponential of that phase.  Tolerance: the reduction and polynomials
are within 1.1 units of 2^-24 of the exact value (0.7e-7 absolute), the general
functions within 2 units (1.2e-7): 1.5e-7 absolute per component.
"""
import numpy as np
import pytest

import multislice_amd as msx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [16, 256, 1024])
@pytest.mark.parametrize("top", [1.0, 40.0, 59999.0, 61000.0, 3e6])
def test_phase_range(ctx, n, top):
    kev = 300.0
    vs = np.float32(msx.sigma(kev) / 1000.0)
    rng = np.random.default_rng(n)
    V = (rng.uniform(-top, top, (3, n, n)) / vs).astype(np.float32)
    t = ctx.transmission(V, 10.0, 10.0, kev, bw=0.0)
    ph = (vs * V).astype(np.float64)
    assert np.abs(t.real - np.cos(ph)).max() < 1.5e-7
    assert np.abs(t.imag - np.sin(ph)).max() < 1.5e-7


def test_mixed_and_special(ctx):
    kev, n = 200.0, 64
    vs = np.float32(msx.sigma(kev) / 1000.0)
    V = np.random.default_rng(1).uniform(-3, 3, (2, n, n)).astype(np.float32) / vs
    V[0, 5, 7], V[0, 6, 1], V[1, 0, 0], V[1, 63, 63] = 1e6 / vs, np.inf, np.nan, 0.0
    t = ctx.transmission(V, 10.0, 10.0, kev, bw=0.0)
    bad = ~np.isfinite(V)
    assert np.isnan(t[bad]).all() and np.isfinite(t[~bad]).all()
    ph = (vs * V).astype(np.float64)[~bad]
    assert np.abs(t[~bad] - np.exp(1j * ph)).max() < 2.2e-7
    assert t[1, 63, 63] == 1


@pytest.mark.parametrize("prec", ["f32", "f64"])
def test_layers_and_absorption(ctx, prec):
    dt = np.float32 if prec == "f32" else np.float64
    rng = np.random.default_rng(3)
    V = rng.uniform(0, 2e3, (70, 32, 64)).astype(dt)
    Va = rng.uniform(0, 1e2, V.shape).astype(dt)
    many = ctx.transmission(V, 6.0, 9.0, 200.0, Vabs=Va)
    for l in (0, 1, 35, 69):
        one = ctx.transmission(V[l:l + 1], 6.0, 9.0, 200.0, Vabs=Va[l:l + 1])
        np.testing.assert_array_equal(many[l], one[0])
