"""The persistent slice loop against the sweeps: the same transforms in the same
order, so every result is equal bit for bit.  With graphs on, a context runs
the sweeps (captured); with graphs off, the loop where its rule takes it.

Shapes cover the loop's lengths in both orders, one and several waves per team
of work-groups, both precisions, repeated layers and unequal thicknesses, the
STEM segments between checkpoints, the partial-coherence loop (which stops
before the last inverse transform), job sets, and two contexts at once.
"""
import threading

import numpy as np
import pytest

import multislice_amd as msx

pytestmark = pytest.mark.gpu

KEV = 200.0


def stack(nl, nx, ny, f64, seed=0):
    import torch
    g = torch.Generator(device="cuda").manual_seed(seed)
    V = torch.rand((nl, nx, ny), generator=g, device="cuda", dtype=torch.float64 if f64 else torch.float32) * 200
    return V


def both(ctx, fn):
    out = []
    for graphs in (True, False):
        ctx.set_graphs(graphs)
        out.append(fn())
    ctx.set_graphs(False)
    return out


def equal(a, b):
    return bool((a == b).all())


@pytest.mark.parametrize("nx,ny,nwave,nslice,f64", [
    (128, 128, 1, 6, False), (128, 512, 3, 9, False), (512, 128, 2, 7, True), (256, 256, 1, 20, False),
    (256, 384, 5, 8, False), (384, 256, 2, 8, True), (384, 384, 24, 6, False), (512, 512, 16, 6, False),
    (512, 512, 2, 7, True), (128, 128, 256, 6, False), (256, 256, 60, 7, True), (512, 256, 9, 6, False),
])
def test_exit_waves_equal_sweeps(ctx, nx, ny, nwave, nslice, f64):
    import torch
    a, b = 0.1 * nx, 0.1 * ny
    t = ctx.transmission(stack(4, nx, ny, f64), a, b, KEV)
    cz = [2.0, 1.0, 2.0, 1.5]
    layer = np.arange(nslice) % 4
    psi0 = torch.randn((nwave, nx, ny), dtype=t.dtype, device="cuda")

    def own():
        psi = psi0.clone()
        ctx.multislice(t, cz, layer, psi, a, b, KEV, tilt=(0.003, -0.002))
        return psi

    def shared():
        psi = torch.empty_like(psi0)
        ctx.multislice(t, cz, layer, psi, a, b, KEV, psi0=psi0[0].contiguous())
        return psi
    for fn in (own, shared):
        x, y = both(ctx, fn)
        assert equal(x, y) and float(x.abs().max()) > 0


@pytest.mark.parametrize("nprobe,ck", [(3, [20]), (40, [7, 8, 20]), (9, [1, 12])])
def test_stem_equals_sweeps(ctx, nprobe, ck):
    n, a = 256, 25.6
    t = ctx.transmission(stack(20, n, n, False), a, a, KEV)
    pos = np.random.default_rng(nprobe).uniform(5, 20, (nprobe, 2))
    x, y = both(ctx, lambda: ctx.stem(t, np.full(20, 2.0), np.arange(20), a, a, KEV, dict(alpha_max=0.02), pos,
                                      [(0, 0.4), (1.0, 3.0)], ck))
    np.testing.assert_array_equal(x, y)


def test_partial_coherence_equals_sweeps(ctx):
    n, a = 128, 25.6
    t = ctx.transmission(stack(12, n, n, False), a, a, KEV)
    lens = dict(cs=1e7, df=500.0, aobj=0.02)
    x, y = both(ctx, lambda: ctx.partial_coherence(t, np.full(12, 2.0), np.arange(12), a, a, KEV, lens, 0.0, 3e-3,
                                                   30.0, 15.0, batch=5)[0])
    assert equal(x, y)


@pytest.mark.parametrize("f64", [False, True])
def test_job_set_equals_jobs_alone(ctx, f64):
    import torch
    rng = np.random.default_rng(4)
    jobs = []
    for k, (n, ns) in enumerate([(128, 9), (256, 6), (128, 17), (256, 30), (512, 8), (128, 1)]):
        a = 0.1 * n
        t = ctx.transmission(stack(ns, n, n, f64, k), a, a, 200.0 + 100 * (k % 2))
        psi0 = torch.ones((n, n), dtype=t.dtype, device="cuda")
        jobs.append(dict(trans=t, psi=torch.empty_like(psi0), psi0=psi0, ax=a, by=a, kev=200.0 + 100 * (k % 2),
                         cz=rng.uniform(1, 2, ns), layer=np.arange(ns)))
    ctx.multislice_batch(jobs)
    ctx.set_graphs(True)
    for j in jobs:
        psi = torch.empty_like(j["psi"])[None]
        ctx.multislice(j["trans"], j["cz"], j["layer"], psi, j["ax"], j["by"], j["kev"], psi0=j["psi0"])
        assert equal(psi[0], j["psi"])
    ctx.set_graphs(False)


def test_job_set_with_shared_buffers(ctx):
    """Jobs that read or write each other's buffers: every incident wave is read before any result is written."""
    import torch
    n, ns = 128, 9
    t = ctx.transmission(stack(ns, n, n, False), 12.8, 12.8, KEV)
    w0 = torch.randn((2, n, n), dtype=torch.complex64, device="cuda")

    def jobs(w):
        base = dict(trans=t, ax=12.8, by=12.8, kev=KEV, cz=np.full(ns, 2.0), layer=np.arange(ns))
        return [dict(base, psi=w[0], psi0=w[1]), dict(base, psi=w[1], psi0=w[0])]
    want = w0.flip(0).contiguous()
    ctx.set_graphs(True)
    ctx.multislice(t, np.full(ns, 2.0), np.arange(ns), want, 12.8, 12.8, KEV)
    ctx.set_graphs(False)
    w = w0.clone()
    ctx.multislice_batch(jobs(w))
    assert equal(w, want)


def test_two_contexts_at_once():
    import torch
    n, ns = 256, 40
    ref = msx.Context(0)
    t = ref.transmission(stack(ns, n, n, False), 25.6, 25.6, KEV)
    cz, layer = np.full(ns, 2.0), np.arange(ns)
    psi0 = torch.ones((n, n), dtype=torch.complex64, device="cuda")
    want = torch.empty((20, n, n), dtype=torch.complex64, device="cuda")
    ref.multislice(t, cz, layer, want, 25.6, 25.6, KEV, psi0=psi0)
    bad = []

    def work():
        c = msx.Context(0)
        for _ in range(5):
            psi = torch.empty_like(want)
            c.multislice(t, cz, layer, psi, 25.6, 25.6, KEV, psi0=psi0)
            if not equal(psi, want):
                bad.append(1)
        c.close()
    th = [threading.Thread(target=work) for _ in range(3)]
    for x in th:
        x.start()
    for x in th:
        x.join()
    ref.close()
    assert not bad
