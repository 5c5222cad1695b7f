"""STEM probes whose aperture reaches past the band limit: the first transmission
takes the whole probe, in the persistent slice loop as in the sweeps.

200 kV, 40 mrad: |k| to 1.59 1/A; the band ends at 0.83 1/A with 0.4 A pixels
and at 0.83 1/A with 0.1 A pixels and a band limit of 1/6.  Grids in both axis
orders (the loop prunes y), a checkpoint late enough for a loop before it.
Tolerances: the loop and the sweeps make the same transforms in the same
order (equal bits); against the FP64 oracle 1e-11 in FP64 and in FP32 2e-5 of
the largest sum, 24 slices of rounding."""
import numpy as np
import pytest

import multislice_amd as msx
from oracle import Oracle as O

pytestmark = pytest.mark.gpu

KEV, ALPHA = 200.0, 0.040


@pytest.mark.parametrize("f64", [False, True])
@pytest.mark.parametrize("nx,ny,pixel,bw", [(128, 128, 0.4, 2 / 3), (128, 256, 0.4, 2 / 3), (256, 128, 0.4, 2 / 3),
                                            (128, 128, 0.1, 1 / 6), (384, 128, 0.1, 1 / 6)])
def test_aperture_past_the_band(ctx, nx, ny, pixel, bw, f64):
    a, b, ns = nx * pixel, ny * pixel, 24
    lam = msx.wavelength(KEV)
    kband = float(np.sqrt(O.k2max(nx, ny, a, b, bw)))
    assert ALPHA / lam > 1.5 * kband
    rng = np.random.default_rng(nx + ny)
    t = O.transmission(rng.random((4, nx, ny)) * 200, a, b, KEV, bw=bw)
    cz, layer = np.array([2.0, 1.5, 2.0, 1.0]), np.arange(ns) % 4
    pos = rng.random((18, 2)) * [a, b]
    det, ck = [(0.0, 0.3 * kband), (0.5 * kband, 1.1 * kband)], [20, ns]
    ref = O.stem(t, cz, layer, a, b, KEV, ALPHA, pos, det, ck, cs=1e4, df=50.0, bw=bw, nthreads=4)
    tt = t if f64 else t.astype(np.complex64)
    got = []
    for graphs in (True, False):  # graphs run the sweeps
        ctx.set_graphs(graphs)
        before = ctx.loop_stats()[0]
        got.append(ctx.stem(tt, cz, layer, a, b, KEV, dict(alpha_max=ALPHA, cs=1e4, df=50.0), pos, det, ck, bw=bw))
        assert (ctx.loop_stats()[0] > before) == (not graphs)
    ctx.set_graphs(False)
    np.testing.assert_array_equal(got[0], got[1])
    assert np.abs(got[1] - ref).max() <= (1e-11 if f64 else 2e-5) * np.abs(ref).max()
