"""Calls whose larger workspaces find no room do with the smaller ones, and
give the same bits: the defocus steps of a partial-coherence image one by one,
an exit wave in place by the sweeps, a STEM scan in batches of 256, the surrogate without packed weights and with
the weight gradients of one layer after the other.  Allocations above a limit
are refused on the host."""
import ctypes as C

import numpy as np
import pytest

import multislice_amd as msx

pytestmark = pytest.mark.gpu

KEV = 200.0


@pytest.fixture
def limit():
    fn = msx.load().msx_test_alloc_limit
    fn.argtypes, fn.restype = [C.c_size_t], None
    yield fn
    fn(0)


def trans(nl, n):
    import torch
    ph = torch.rand((nl, n, n), generator=torch.Generator(device="cuda").manual_seed(n), device="cuda")
    return torch.polar(torch.ones_like(ph), ph)


def test_partial_coherence(ctx, limit):
    n, a, ns = 128, 12.8, 4
    args = (trans(ns, n), np.full(ns, 2.0), np.arange(ns), a, a, KEV, dict(cs=1e7, df=500.0, aobj=0.02), 0.0, 4e-3,
            30.0, 15.0)
    want, nang, nd = ctx.partial_coherence(*args)
    c = msx.Context(0)
    limit(2 * nang * n * n * 8)  # room for one or two of the steps
    got, _, _ = c.partial_coherence(*args)
    c.close()
    assert nd > 2 and bool((got == want).all())


def test_exit_wave_in_place(ctx, limit):
    """The copy that a persistent loop keeps of its incident waves: without room the sweeps run."""
    import torch
    n, a, ns = 128, 12.8, 20
    t = trans(ns, n)
    want, got = (torch.ones((4, n, n), dtype=torch.complex64, device="cuda") for _ in range(2))
    ctx.multislice(t, np.full(ns, 2.0), np.arange(ns), want, a, a, KEV)
    c = msx.Context(0)
    limit(300000)  # the tables, less than four waves
    c.multislice(t, np.full(ns, 2.0), np.arange(ns), got, a, a, KEV)
    assert c.loop_stats() == (0, 0)
    c.close()
    assert bool((got == want).all())


def test_stem(ctx, limit):
    n, a, ns = 64, 12.8, 3
    pos = np.random.default_rng(1).uniform(0, a, (700, 2))
    args = (trans(ns, n), np.full(ns, 2.0), np.arange(ns), a, a, KEV, dict(alpha_max=0.02), pos, [(0, 0.5), (1.0, 2.0)],
            [ns])
    want = ctx.stem(*args)
    c = msx.Context(0)
    limit(300 * n * n * 8)
    got = c.stem(*args)
    with pytest.raises(msx.MsxError):
        c.stem(*args, batch=400)  # asked for: not changed
    np.testing.assert_array_equal(got, want)
    np.testing.assert_array_equal(c.stem(*args), want)  # and no error left behind
    c.close()


def unet_run(net, x, t):
    y = net.forward(x)
    loss = [net.train_step(x, t, 1e-3) for _ in range(2)]
    return y, loss, net.params()


def same(a, b):
    np.testing.assert_array_equal(a[0], b[0])
    assert a[1] == b[1]
    np.testing.assert_array_equal(a[2], b[2])


def test_surrogate(ctx, limit):
    rng = np.random.default_rng(2)
    x, t = rng.random((3, 32, 32), np.float32), rng.random((3, 32, 32), np.float32)
    want = unet_run(msx.UNet(ctx, 3, 16, 5), x, t)
    limit(1000)
    plain = msx.UNet(ctx, 3, 16, 5)  # no packed weights
    limit(0)
    same(unet_run(plain, x, t), want)
    net = msx.UNet(ctx, 3, 16, 5)
    p = net.params()
    for k in range(12, 31):  # the first power of two that holds the largest layer's slices
        limit(1 << k)
        try:
            net.train_step(x, t, 1e-3)
            break
        except msx.MsxError:
            np.testing.assert_array_equal(net.params(), p)
    assert k > 12
    net.set_params(p)
    same(unet_run(net, x, t), want)


def test_one_convolution(ctx, limit):
    import torch
    L = msx.load()
    n, cin, cout, h, w = 2, 20, 40, 12, 16
    g = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randn((n, cin, h, w), generator=g, device="cuda")
    wt = torch.randn((cout, cin, 3, 3), generator=g, device="cuda")
    out = [torch.empty((n, cout, h, w), device="cuda") for _ in range(2)]
    torch.cuda.synchronize()
    for k, o in enumerate(out):
        c = msx.Context(0)
        limit(0 if k == 0 else 1000)
        assert L.msx_unet_conv(c.h, 0, 3, C.c_void_p(x.data_ptr()), C.c_void_p(wt.data_ptr()), None, None, None,
                               C.c_void_p(o.data_ptr()), n, cin, cout, h, w, 0) == 0
        c.close()
    assert bool((out[0] == out[1]).all())
