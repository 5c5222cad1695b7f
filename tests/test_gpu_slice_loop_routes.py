"""Which calls the persistent slice loop takes: its launches are counted, so
that the tests that compare it with the sweeps cannot compare the sweeps with
themselves."""
import numpy as np
import pytest

import multislice_amd as msx

pytestmark = pytest.mark.gpu

KEV = 200.0


def trans(n, ns, f64=False):
    import torch
    g = torch.Generator(device="cuda").manual_seed(n)
    ph = torch.rand((ns, n, n), generator=g, device="cuda", dtype=torch.float64 if f64 else torch.float32)
    return torch.polar(torch.ones_like(ph), ph)


def launched(ctx, fn):
    n0, bad0 = ctx.loop_stats()
    fn()
    n1, bad1 = ctx.loop_stats()
    assert bad1 == bad0
    return n1 - n0


@pytest.mark.parametrize("f64", [False, True])
@pytest.mark.parametrize("n,nwave", [(128, 1), (128, 256), (256, 5), (384, 2), (512, 2)])
def test_exit_waves(ctx, n, nwave, f64):
    import torch
    ns, a = 20, 0.1 * n
    t = trans(n, ns, f64)
    psi = torch.ones((nwave, n, n), dtype=t.dtype, device="cuda")

    def go(m=ns):
        ctx.multislice(t, np.full(ns, 2.0), np.arange(m), psi, a, a, KEV)
    assert launched(ctx, go) == 1
    assert launched(ctx, lambda: go(2)) == 0  # few slices
    ctx.set_graphs(True)
    assert launched(ctx, go) == 0
    ctx.set_graphs(False)
    ctx.profile(True)
    assert launched(ctx, go) == 0
    ctx.profile(False)


@pytest.mark.parametrize("f64", [False, True])
@pytest.mark.parametrize("nx", [128, 256, 384, 512])
@pytest.mark.parametrize("ny", [128, 256, 384, 512])
def test_every_shape_equals_sweeps(ctx, nx, ny, f64):
    """One kernel per shape and precision, with as many waves as the rule asks
    for and one more: bits of the sweeps (graphs), repeated layers of unequal
    thickness, and with 16 slices and no loop with 15, or 6 and 5 from 8 MiB on."""
    import torch
    size = nx * ny * (16 if f64 else 8)
    few = 1
    if (nx == 512 and not f64) or (nx, ny) in ((128, 256), (512, 128)):
        few = (8 if (nx, ny, f64) == (512, 128, False) else 4) * 2**20 // size
        few += few * size < 4 * 2**20  # (not a whole number of waves)
    many = -(-8 * 2**20 // size)
    a, b = 0.1 * nx, 0.1 * ny
    g = torch.Generator(device="cuda").manual_seed(nx + 7 * ny)
    ph = torch.rand((3, nx, ny), generator=g, device="cuda", dtype=torch.float64 if f64 else torch.float32)
    t = torch.polar(torch.ones_like(ph), ph)
    first = torch.randn((max(few, many) + 1, nx, ny), dtype=t.dtype, device="cuda", generator=g)

    def run(n, ns):
        w = first[:n].clone()
        ctx.multislice(t, [2.0, 1.5, 2.0], np.arange(ns) % 3, w, a, b, KEV)
        return w
    for n, ns in ((few, 16), (few + 1, 17), (many, 6), (many + 1, 7)):
        if n < many and n * size >= 8 * 2**20:
            continue
        ctx.set_graphs(True)
        want = run(n, ns)
        ctx.set_graphs(False)
        got = []
        assert launched(ctx, lambda: got.append(run(n, ns))) == 1
        assert bool((got[0] == want).all())
    assert launched(ctx, lambda: run(many, 5)) == 0
    if few < many:
        assert launched(ctx, lambda: run(few, 15)) == 0
    if few > 1:
        assert launched(ctx, lambda: run(few - 1, 40)) == 0


def test_lengths_without_a_loop(ctx):
    import torch
    for n in (64, 768):
        t = trans(n, 20)
        psi = torch.ones((1, n, n), dtype=t.dtype, device="cuda")
        assert launched(ctx, lambda: ctx.multislice(t, np.full(20, 2.0), np.arange(20), psi, 10.0, 10.0, KEV)) == 0


def taken(ctx, fn, loops):
    """fn() by loops, so many of them, and by the sweeps (profiled): the same bits."""
    got = []
    assert launched(ctx, lambda: got.append(fn())) == loops
    ctx.profile(True)
    assert launched(ctx, lambda: got.append(fn())) == 0
    ctx.profile(False)
    assert all(bool((x == y).all()) for x, y in zip(*got))


def test_stem_partial_coherence_and_job_sets(ctx):
    import torch
    n, ns, a = 128, 40, 12.8
    t, cz, layer = trans(n, ns), np.full(ns, 2.0), np.arange(ns)
    pos = np.random.default_rng(0).uniform(0, a, (8, 2))
    # a loop up to each checkpoint's slice, for each of three batches
    taken(ctx, lambda: ctx.stem(t, cz, layer, a, a, KEV, dict(alpha_max=0.02), pos, [(0, 1.0), (1.0, 3.0)], [20, 40],
                                batch=3), 6)
    lens = dict(cs=1e7, df=500.0, aobj=0.02)
    taken(ctx, lambda: ctx.partial_coherence(t, cz, layer, a, a, KEV, lens, 0.0, 5e-3, 30.0, 15.0)[:1], 1)

    def job_set():  # one class with uneven ends, more waves than one team; another cell
        g = torch.Generator(device="cuda").manual_seed(1)
        jobs = [dict(trans=t, psi=torch.randn((n, n), dtype=t.dtype, device="cuda", generator=g), ax=a,
                     by=a + (k == 5), kev=KEV + k % 2, cz=cz, layer=layer[:ns - k]) for k in range(24)]
        jobs[3]["psi0"] = torch.ones_like(jobs[3]["psi"])
        ctx.multislice_batch(jobs)
        return [j["psi"] for j in jobs]
    taken(ctx, job_set, 2)


def test_waves_in_pinned_memory(ctx):
    """The work-groups exchange waves in this device's memory only: others go through the sweeps."""
    import ctypes as C
    import torch
    n, ns, a = 128, 20, 12.8
    t, cz, layer = trans(n, ns), np.full(ns, 2.0), np.arange(ns)
    want = torch.ones((1, n, n), dtype=t.dtype, device="cuda")
    psi = torch.empty(want.shape, dtype=want.dtype, pin_memory=True)
    psi.copy_(want)
    ctx.multislice(t, cz, layer, want, a, a, KEV)
    st, keep = ctx._stack(n, n, a, a, KEV, cz, layer, (0.0, 0.0), 2.0 / 3.0)
    assert launched(ctx, lambda: msx.load().msx_multislice(ctx.h, C.byref(st), C.c_void_p(t.data_ptr()), None,
                                                           C.c_void_p(psi.data_ptr()), 1, msx.F32, 1)) == 0
    assert bool((psi == want.cpu()).all())
