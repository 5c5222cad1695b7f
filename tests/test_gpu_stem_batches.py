"""A scan that chooses no batch: one batch, several equal ones, a rounded one
with a shorter last one, in both precisions and on a grid with the fixed bound;
the images do not depend on the batches (equal bit for bit)."""
import numpy as np
import pytest

import multislice_amd as msx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nprobe,f64", [
    (16, 32, 1537, False), (64, 64, 1600, True), (256, 512, 325, False), (512, 512, 161, False), (512, 512, 90, True),
    (256, 256, 1, False), (384, 128, 270, False),
])
def test_default_batches_match_chosen_ones(ctx, nx, ny, nprobe, f64):
    import torch
    g = torch.Generator(device="cuda").manual_seed(nprobe)
    V = torch.rand((2, nx, ny), generator=g, device="cuda", dtype=torch.float64 if f64 else torch.float32) * 100
    a, b = 0.2 * nx, 0.2 * ny
    t = ctx.transmission(V, a, b, 200.0)
    pos = np.random.default_rng(nprobe).uniform(0, min(a, b), (nprobe, 2))
    args = (t, np.full(2, 2.0), np.arange(2), a, b, 200.0, dict(alpha_max=0.02), pos, [(0.0, 0.4), (0.5, 2.0)], [1, 2])
    got = ctx.stem(*args)
    want = ctx.stem(*args, batch=100)
    assert np.isfinite(got).all() and got.max() > 0
    np.testing.assert_array_equal(got, want)
