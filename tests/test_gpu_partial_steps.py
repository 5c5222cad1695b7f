"""Partial coherence with several defocus steps per launch: the image does not
depend on how the angles fall into batches, and with them the steps into
launches (one step, all, some with a shorter last launch).  A wave's sum over
its steps is formed in the same order and precision; the FP64 sum over waves is
grouped differently, hence 1e-12."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,cone,batches,spread,f64,astig", [
    (64, 6e-3, (0, 1, 7), 30.0, False, 0.0),    # every step in one launch
    (128, 4e-3, (0, 1), 30.0, True, 30.0),
    (512, 3.2e-3, (41, 23), 20.0, False, 0.0),  # 3 and 6 of 11 steps per launch
    (2048, 3e-4, (3, 1), 8.0, False, 0.0),      # 3 and all 5 steps per launch
    (128, 4e-3, (0, 3), 0.0, False, 20.0),      # one step
])
def test_image_is_independent_of_batches(ctx, n, cone, batches, spread, f64, astig):
    import torch
    g = torch.Generator(device="cuda").manual_seed(n)
    V = torch.rand((2, n, n), generator=g, device="cuda", dtype=torch.float64 if f64 else torch.float32) * 200
    a = 0.2 * n
    t = ctx.transmission(V, a, a, 200.0)
    lens = dict(cs=1.2e7, df=600.0, aobj=0.015, dfa2=astig, dfa2phi=0.3)
    out = []
    for b in batches:
        img, nang, nstep = ctx.partial_coherence(t, np.full(2, 2.0), np.arange(2), a, a, 200.0, lens, 0.0, cone, spread,
                                                 10.0, batch=b)
        out.append(img.cpu().numpy() if hasattr(img, "cpu") else np.asarray(img))
    assert nstep == (1 if spread == 0 else 2 * int(2.5 * spread / 10.0) + 1)
    assert nang > max(batches) - 1
    np.testing.assert_allclose(out[0], out[1], rtol=1e-12, atol=0)
    for o in out[2:]:
        np.testing.assert_allclose(out[0], o, rtol=1e-12, atol=0)
